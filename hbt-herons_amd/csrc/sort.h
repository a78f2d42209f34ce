// Segmented sort of (uint64 key, int32 value) pairs.
//  * segments of <= SORT_WAVE4_MAX elements: one wave each, bitonic sort in lanes;
//  * segments of <= SORT_SMALL_MAX elements: one workgroup each, the same bitonic
//    network in registers, lane moves and three steps through LDS;
//  * where no segment is longer than SORT_BLOCK_MAX, those above: one workgroup each, a
//    stable LSD radix sort whose passes stay in registers and LDS (the order of the next);
//  * else the segments above SORT_SMALL_MAX: tiled LSD radix sort (8- or 9-bit digits,
//    whichever needs fewer passes) where every tile of SORT_TILE elements ranks its keys
//    stably with wave ballots (match of the digit bits) and LDS per-digit counters, so
//    all large segments advance together in one launch per pass.
#pragma once
#include "common.h"
#include "scan.h"

namespace hbtx
{
#ifndef SORT_THREADS
#define SORT_THREADS 256
#endif
#define SORT_SMALL_MAX 2048
#define SORT_WAVE_MAX HBTX_WAVE // segments of at most one wave: k_sort_wave
#define SORT_WAVE4_MAX (4 * HBTX_WAVE) // segments of at most four per lane: k_sort_wave4
#ifndef SORT_TILE
#define SORT_TILE 2048
#endif
#define RADIX_MAX_BINS 512 // (9-bit digits)
#define SORT_BLOCK_THREADS 1024
#define SORT_BLOCK_ITEMS 16
#define SORT_BLOCK_MAX (SORT_BLOCK_THREADS * SORT_BLOCK_ITEMS)

// v of the lane whose number differs in the bit X, by moves of the vector unit.
template <int X>
HBTX_DEV uint32_t lane_xor(uint32_t v)
{
  if constexpr (X == 1)
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xf, 0xf, true); // quad_perm [1,0,3,2]
  else if constexpr (X == 2)
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xf, 0xf, true); // quad_perm [2,3,0,1]
  else if constexpr (X == 4)
  {
    const int m = __builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xf, 0xf, true); // row_half_mirror: lane ^ 7
    return (uint32_t)__builtin_amdgcn_update_dpp(0, m, 0x1B, 0xf, 0xf, true);    // quad_perm [3,2,1,0]: lane ^ 3
  }
  else if constexpr (X == 8)
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xf, 0xf, true); // row_ror:8
  else if constexpr (X == 16)
  {
    const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false); // the even rows twice, the odd ones
    return (lane_id() & 16) ? r[0] : r[1];
  }
  else
  {
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false); // the lower half twice, the upper
    return (lane_id() & 32) ? r[0] : r[1];
  }
}

// One step of the network between lanes X apart: up, the pair's direction.
template <int R, int X>
HBTX_DEV void net_lanes(uint64_t (&key)[R], int32_t (&val)[R], bool up)
{
  const bool low = (lane_id() & X) == 0; // this lane holds the pairs' first elements
#pragma unroll
  for (int r = 0; r < R; r++)
  {
    const uint64_t ok =
      ((uint64_t)lane_xor<X>((uint32_t)(key[r] >> 32)) << 32) | lane_xor<X>((uint32_t)key[r]);
    const int32_t ov = (int32_t)lane_xor<X>((uint32_t)val[r]);
    if ((low ? key[r] > ok : ok > key[r]) == up)
    {
      key[r] = ok;
      val[r] = ov;
    }
  }
}

// The bitonic network over 256 R elements, element R t + r in register r of thread t:
// pairs less than R apart meet in a thread's registers, less than 64 R apart through lane
// moves, and only the three steps beyond that in LDS, between barriers.
template <int R>
HBTX_DEV void sort_net(uint64_t *__restrict__ keys, int32_t *__restrict__ vals, int len, uint64_t *sk, int32_t *sv)
{
  const int t = threadIdx.x;
  uint64_t key[R];
  int32_t val[R];
#pragma unroll
  for (int r = 0; r < R; r++)
  {
    const int e = R * t + r;
    key[r] = (e < len) ? keys[e] : ~0ull;
    val[r] = (e < len) ? vals[e] : 0;
  }
  for (int k = 2; k <= SORT_THREADS * R; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1)
    {
      const bool up_t = (t & (k / R)) == 0; // (k >= R: the direction of all the thread's elements)
      if (j >= HBTX_WAVE * R)
      {
#pragma unroll
        for (int r = 0; r < R; r++)
        {
          sk[r * SORT_THREADS + t] = key[r];
          sv[r * SORT_THREADS + t] = val[r];
        }
        __syncthreads();
        const int o = t ^ (j / R);
#pragma unroll
        for (int r = 0; r < R; r++)
        {
          const uint64_t ok = sk[r * SORT_THREADS + o];
          const int32_t ov = sv[r * SORT_THREADS + o];
          if ((t < o ? key[r] > ok : ok > key[r]) == up_t)
          {
            key[r] = ok;
            val[r] = ov;
          }
        }
        __syncthreads();
      }
      else if (j >= R)
      {
        switch (j / R)
        {
        case 1:
          net_lanes<R, 1>(key, val, up_t);
          break;
        case 2:
          net_lanes<R, 2>(key, val, up_t);
          break;
        case 4:
          net_lanes<R, 4>(key, val, up_t);
          break;
        case 8:
          net_lanes<R, 8>(key, val, up_t);
          break;
        case 16:
          net_lanes<R, 16>(key, val, up_t);
          break;
        default:
          net_lanes<R, 32>(key, val, up_t);
        }
      }
      else
      {
#pragma unroll
        for (int jr = 1; jr < R; jr <<= 1)
          if (jr == j)
          {
#pragma unroll
            for (int r = 0; r < R; r++)
            {
              const int r2 = r ^ jr;
              if (r2 < r)
                continue;
              const bool up = (k < R) ? (r & k) == 0 : up_t;
              if ((key[r] > key[r2]) == up)
              {
                const uint64_t tk = key[r];
                key[r] = key[r2];
                key[r2] = tk;
                const int32_t tv = val[r];
                val[r] = val[r2];
                val[r2] = tv;
              }
            }
          }
      }
    }
#pragma unroll
  for (int r = 0; r < R; r++)
  {
    const int e = R * t + r;
    if (e < len)
    {
      keys[e] = key[r];
      vals[e] = val[r];
    }
  }
}

// Segments of SORT_WAVE4_MAX + 1 .. SORT_SMALL_MAX elements, a workgroup each, padded to
// 512, 1024 or 2048.  Through LDS and a barrier a step (45 to 66 steps): one segment of
// 300, 18 us, the segments of a set of 1e6 particles 65 us a launch; by sort_net 13 and
// 30 us.
__global__ __launch_bounds__(SORT_THREADS) void k_sort_small(uint64_t *__restrict__ keys, int32_t *__restrict__ vals,
                                                            const int32_t *__restrict__ seg_begin,
                                                            const int32_t *__restrict__ seg_len, int32_t nseg)
{
  __shared__ uint64_t sk[SORT_SMALL_MAX];
  __shared__ int32_t sv[SORT_SMALL_MAX];
  for (int s = blockIdx.x; s < nseg; s += gridDim.x)
  {
    const int len = seg_len[s];
    if (len <= SORT_WAVE4_MAX || len > SORT_SMALL_MAX)
      continue; // (segments of up to four per lane: k_sort_wave, k_sort_wave4)
    const int b = seg_begin[s];
    if (len <= 2 * SORT_THREADS)
      sort_net<2>(keys + b, vals + b, len, sk, sv);
    else if (len <= 4 * SORT_THREADS)
      sort_net<4>(keys + b, vals + b, len, sk, sv);
    else
      sort_net<8>(keys + b, vals + b, len, sk, sv);
  }
}
static_assert(SORT_SMALL_MAX == 8 * SORT_THREADS, "sort_net's forms cover k_sort_small's segments");

// Segments of at most one wave (the common case for small subhaloes): one wave per
// segment, element i in lane i, the same bitonic network as k_sort_small (so the
// same permutation, ties included) through lane shuffles, with no barrier.
__global__ __launch_bounds__(SORT_THREADS) void k_sort_wave(uint64_t *__restrict__ keys, int32_t *__restrict__ vals,
                                                           const int32_t *__restrict__ seg_begin,
                                                           const int32_t *__restrict__ seg_len, int32_t nseg)
{
  const int lane = lane_id();
  const int wpb = SORT_THREADS / HBTX_WAVE;
  for (int s = uniform(blockIdx.x * wpb + (int)(threadIdx.x / HBTX_WAVE)); s < nseg; s += gridDim.x * wpb)
  {
    const int len = seg_len[s];
    if (len <= 1 || len > SORT_WAVE_MAX)
      continue;
    const int b = seg_begin[s];
    int P = 1;
    while (P < len)
      P <<= 1;
    uint64_t key = (lane < len) ? keys[b + lane] : ~0ull;
    int32_t val = (lane < len) ? vals[b + lane] : 0;
    for (int k = 2; k <= P; k <<= 1)
      for (int j = k >> 1; j > 0; j >>= 1)
      {
        const uint64_t ok = __shfl_xor(key, j, HBTX_WAVE);
        const int32_t ov = __shfl_xor(val, j, HBTX_WAVE);
        const bool low = (lane & j) == 0;     // this lane holds the pair's first element
        const bool up = (lane & k) == 0;      // the pair's direction (the same for both lanes)
        const uint64_t a = low ? key : ok, c = low ? ok : key;
        const bool swap = (a > c) == up;
        if (swap)
        {
          key = ok;
          val = ov;
        }
      }
    if (lane < len)
    {
      keys[b + lane] = key;
      vals[b + lane] = val;
    }
  }
}

// Segments of SORT_WAVE_MAX + 1 .. SORT_WAVE4_MAX elements: one wave each, element
// lane + 64 r in register r, padded to 128 or 256 like k_sort_small, and the same
// bitonic network (so the same permutation, ties included): pairs less than 64
// apart meet through lane shuffles, pairs 64 or more apart in a lane's registers.
// No LDS and no barrier.
__global__ __launch_bounds__(SORT_THREADS) void k_sort_wave4(uint64_t *__restrict__ keys, int32_t *__restrict__ vals,
                                                            const int32_t *__restrict__ seg_begin,
                                                            const int32_t *__restrict__ seg_len, int32_t nseg)
{
  const int lane = lane_id();
  const int wpb = SORT_THREADS / HBTX_WAVE;
  for (int s = uniform(blockIdx.x * wpb + (int)(threadIdx.x / HBTX_WAVE)); s < nseg; s += gridDim.x * wpb)
  {
    const int len = seg_len[s];
    if (len <= SORT_WAVE_MAX || len > SORT_WAVE4_MAX)
      continue;
    const int b = seg_begin[s];
    const int P = (len > 2 * HBTX_WAVE) ? 4 * HBTX_WAVE : 2 * HBTX_WAVE;
    const int R = P / HBTX_WAVE; // registers in use: 2 or 4
    uint64_t key[4];
    int32_t val[4];
#pragma unroll
    for (int r = 0; r < 4; r++)
    {
      const int e = lane + HBTX_WAVE * r;
      key[r] = (r < R && e < len) ? keys[b + e] : ~0ull;
      val[r] = (r < R && e < len) ? vals[b + e] : 0;
    }
    for (int k = 2; k <= P; k <<= 1)
      for (int j = k >> 1; j > 0; j >>= 1)
      {
        if (j < HBTX_WAVE)
        {
#pragma unroll
          for (int r = 0; r < 4; r++)
          {
            if (r >= R)
              continue;
            const int e = lane + HBTX_WAVE * r;
            const uint64_t ok = __shfl_xor(key[r], j, HBTX_WAVE);
            const int32_t ov = __shfl_xor(val[r], j, HBTX_WAVE);
            const bool low = (lane & j) == 0; // this lane holds the pair's first element
            const bool up = (e & k) == 0;     // the pair's direction (the same for both lanes)
            const uint64_t a = low ? key[r] : ok, c = low ? ok : key[r];
            if ((a > c) == up)
            {
              key[r] = ok;
              val[r] = ov;
            }
          }
        }
        else
        {
          const int jr = j / HBTX_WAVE; // the pair's registers differ by jr (1 or 2)
#pragma unroll
          for (int r = 0; r < 4; r++)
          {
            const int r2 = r ^ jr;
            if (r >= R || r2 < r)
              continue; // (r2 < R: pairs stay inside the padded length)
            const int e = lane + HBTX_WAVE * r;
            const bool up = (e & k) == 0;
            if ((key[r] > key[r2]) == up)
            {
              const uint64_t tk = key[r];
              key[r] = key[r2];
              key[r2] = tk;
              const int32_t tv = val[r];
              val[r] = val[r2];
              val[r2] = tv;
            }
          }
        }
      }
#pragma unroll
    for (int r = 0; r < 4; r++)
    {
      const int e = lane + HBTX_WAVE * r;
      if (r < R && e < len)
      {
        keys[b + e] = key[r];
        vals[b + e] = val[r];
      }
    }
  }
}

// Segments of SORT_SMALL_MAX + 1 .. SORT_BLOCK_MAX elements (tiles: one a segment), one
// workgroup each, by stable 8-bit LSD passes over (32 key bits, place in the segment)
// in registers: wave w owns elements [64 R w, 64 R (w + 1)), R = ceil(n / 1024), ranks
// them by ballot match against its own digit counters, and they change places through
// LDS.  A pass in which every key has the same digit moves nothing.  The keys' top 32
// bits come first; an element among equals of those (a few in 12,000 with spatial
// keys) then counts the members of its run that go before it by the bits below.  A run
// of more than SORT_RUN_MAX sends the segment through the passes of the lower bits
// first, then the upper ones.
// Bound: the match (8 ballots an element) and the LDS on the one CU of the segment,
// some 12 us a pass.  A segment of 12,000, 63 bits: 67 us; through the tiled passes (four
// launches of 2 to 12 us a pass) 115 us; eight passes with key and value in registers
// and LDS 93 us.
#define SORT_RUN_MAX 32
struct SortBlockLds
{
  uint64_t x[SORT_BLOCK_MAX];                        // the elements in passage
  uint16_t cnt[SORT_BLOCK_THREADS / HBTX_WAVE][256]; // per wave and digit (at most 1024), then its base
  int32_t base[256];
  int32_t scan[4];
  int32_t same, long_run;
};

// The lanes whose digit (bits [shift, shift + 8) of v) is this lane's.
HBTX_DEV uint64_t match_digit(uint32_t v, int shift)
{
  uint32_t lo = ~0u, hi = ~0u;
#pragma unroll
  for (int bit = 0; bit < 8; bit++)
  {
    const int32_t on = __builtin_amdgcn_sbfe((int32_t)v, shift + bit, 1); // 0 or -1
    const uint64_t bb = __builtin_amdgcn_sicmp(on, 0, 33 /* ne */);
    lo &= ~((uint32_t)bb ^ (uint32_t)on);
    hi &= ~((uint32_t)(bb >> 32) ^ (uint32_t)on);
  }
  return ((uint64_t)hi << 32) | lo;
}

__global__ __launch_bounds__(SORT_BLOCK_THREADS) void k_sort_block(uint64_t *__restrict__ keys,
                                                                  int32_t *__restrict__ vals,
                                                                  const int4 *__restrict__ tiles,
                                                                  const int32_t *__restrict__ ntiles_p, int key_bits)
{
  extern __shared__ __align__(16) unsigned char sort_lds[];
  SortBlockLds &L = *reinterpret_cast<SortBlockLds *>(sort_lds);
  constexpr int NW = SORT_BLOCK_THREADS / HBTX_WAVE;
  const int tid = threadIdx.x, w = uniform(tid / HBTX_WAVE), lane = lane_id();
  const int low_bits = max(0, key_bits - 32), top_bits = key_bits - low_bits;
  const uint64_t low_mask = (1ull << low_bits) - 1ull;
  const int nt = *ntiles_p;
  for (int t = blockIdx.x; t < nt; t += gridDim.x)
  {
    const int4 tl = tiles[t];
    const int b = tl.y, n = tl.z - tl.y;
    // R rows of a wave's lanes; the places past n hold the largest key, which no pass
    // moves off the end
    const int R = (n + SORT_BLOCK_THREADS - 1) / SORT_BLOCK_THREADS;
    const int i0 = w * R * HBTX_WAVE + lane; // this thread's places: i0 + 64 r, r < R
    uint64_t el[SORT_BLOCK_ITEMS];           // key bits above, the element's place at the start below
    int32_t pos[SORT_BLOCK_ITEMS];
    auto passes = [&](int bits) {
      for (int shift = 0; shift < bits; shift += 8)
      {
        for (int i = tid; i < NW * 256 / 2; i += SORT_BLOCK_THREADS)
          reinterpret_cast<uint32_t *>(&L.cnt[0][0])[i] = 0u;
        if (tid == 0)
          L.same = 0;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < SORT_BLOCK_ITEMS; r++)
        {
          if (r >= R)
            break;
          const uint32_t v = (uint32_t)(el[r] >> 32);
          const int d = (int)((v >> shift) & 255u);
          const uint64_t m = match_digit(v, shift);
          const int before = (int)L.cnt[w][d];
          pos[r] = before + mask_rank(m, 0);
          // (the wave's LDS accesses are in order: the read above comes before this write)
          if ((m >> lane) == 1ull)
            L.cnt[w][d] = (uint16_t)(pos[r] + 1);
        }
        __syncthreads();
        if (tid < 256)
        {
          // digit tid: the waves' bases among its elements, then the digits' own
          int run = 0;
#pragma unroll
          for (int k = 0; k < NW; k++)
          {
            const int c = L.cnt[k][tid];
            L.cnt[k][tid] = (uint16_t)run;
            run += c;
          }
          if (run - (tid == 255 ? R * SORT_BLOCK_THREADS - n : 0) == n)
            L.same = 1;
          const int incl = wave_incl_scan(run);
          if (lane == HBTX_WAVE - 1)
            L.scan[w] = incl;
          L.base[tid] = incl - run;
        }
        __syncthreads();
        if (L.same)
        {
          __syncthreads(); // every thread has read it before the next pass clears it
          continue;
        }
        if (tid < 256)
        {
          int off = L.base[tid];
#pragma unroll
          for (int k = 0; k < 3; k++)
            off += (tid >= 64 * (k + 1)) ? L.scan[k] : 0;
          L.base[tid] = off;
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < SORT_BLOCK_ITEMS; r++)
        {
          if (r >= R)
            break;
          const int d = (int)((uint32_t)(el[r] >> 32) >> shift & 255u);
          L.x[L.base[d] + (int)L.cnt[w][d] + pos[r]] = el[r];
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < SORT_BLOCK_ITEMS; r++)
        {
          if (r >= R)
            break;
          el[r] = L.x[i0 + HBTX_WAVE * r];
        }
        // (the next pass writes x only after its own barriers)
      }
    };
    bool low_first = false;
    for (;;)
    {
#pragma unroll
      for (int r = 0; r < SORT_BLOCK_ITEMS; r++)
      {
        if (r >= R)
          break;
        const int i = i0 + HBTX_WAVE * r;
        const uint64_t k = keys[b + min(i, n - 1)];
        const uint32_t part = (uint32_t)(low_first ? k & low_mask : k >> low_bits);
        el[r] = ((uint64_t)(i < n ? part : 0xffffffffu) << 32) | (uint32_t)i;
      }
      if (low_first)
      {
        passes(low_bits);
#pragma unroll
        for (int r = 0; r < SORT_BLOCK_ITEMS; r++)
        {
          if (r >= R)
            break;
          const int i = (int)(uint32_t)el[r];
          const uint32_t part = (uint32_t)(keys[b + min(i, n - 1)] >> low_bits);
          el[r] = ((uint64_t)(i < n ? part : 0xffffffffu) << 32) | (uint32_t)i;
        }
      }
      passes(top_bits);
      // the elements' places among equals of the top bits
#pragma unroll
      for (int r = 0; r < SORT_BLOCK_ITEMS; r++)
        pos[r] = i0 + HBTX_WAVE * r;
      if (low_bits == 0 || low_first)
        break;
      if (tid == 0)
        L.long_run = 0;
#pragma unroll
      for (int r = 0; r < SORT_BLOCK_ITEMS; r++)
      {
        if (r >= R)
          break;
        L.x[pos[r]] = el[r]; // (again: passes that moved nothing left it as it was)
      }
      __syncthreads();
#pragma unroll
      for (int r = 0; r < SORT_BLOCK_ITEMS; r++)
      {
        if (r >= R)
          break;
        const int i = i0 + HBTX_WAVE * r;
        const uint32_t top = (uint32_t)(el[r] >> 32);
        int a = i, e = i + 1; // the run
        while (a > 0 && i - a < SORT_RUN_MAX && (uint32_t)(L.x[a - 1] >> 32) == top)
          a--;
        while (e < n && e - i < SORT_RUN_MAX && (uint32_t)(L.x[e] >> 32) == top)
          e++;
        if (e - a == 1 || i >= n)
          continue;
        if (e - a > SORT_RUN_MAX)
        {
          L.long_run = 1;
          continue;
        }
        const uint64_t low = keys[b + (int)(uint32_t)el[r]] & low_mask;
        int to = a;
        for (int j = a; j < e; j++)
        {
          const uint64_t lj = keys[b + (int)(uint32_t)L.x[j]] & low_mask;
          to += (lj < low || (lj == low && j < i)) ? 1 : 0;
        }
        pos[r] = to;
      }
      __syncthreads();
      if (!L.long_run)
        break;
      low_first = true;
      __syncthreads(); // every thread has read it before anything below is written
    }
    int32_t val[SORT_BLOCK_ITEMS];
#pragma unroll
    for (int r = 0; r < SORT_BLOCK_ITEMS; r++)
    {
      if (r >= R)
        break;
      const int i = b + min((int)(uint32_t)el[r], n - 1);
      el[r] = keys[i];
      val[r] = vals[i];
    }
    __syncthreads(); // every key and value has been read
#pragma unroll
    for (int r = 0; r < SORT_BLOCK_ITEMS; r++)
    {
      if (r >= R || i0 + HBTX_WAVE * r >= n)
        break;
      keys[b + pos[r]] = el[r];
      vals[b + pos[r]] = val[r];
    }
    __syncthreads();
  }
}

template <int RB>
__global__ __launch_bounds__(SORT_THREADS) void k_radix_hist(const uint64_t *__restrict__ kin,
                                                            const int4 *__restrict__ tiles,
                                                            const int32_t *__restrict__ ntiles_p, int shift,
                                                            int32_t *__restrict__ ghist)
{
  constexpr int BINS = 1 << RB;
  __shared__ int32_t hist[BINS];
  const int nt = *ntiles_p;
  const int tid = threadIdx.x;
  for (int t = blockIdx.x; t < nt; t += gridDim.x)
  {
    for (int b = tid; b < BINS; b += SORT_THREADS)
      hist[b] = 0;
    __syncthreads();
    const int4 tl = tiles[t];
    for (int i = tl.y + tid; i < tl.z; i += SORT_THREADS)
      atomicAdd(&hist[(int)((kin[i] >> shift) & (BINS - 1))], 1);
    __syncthreads();
    for (int b = tid; b < BINS; b += SORT_THREADS)
      ghist[(int64_t)t * BINS + b] = hist[b];
    __syncthreads();
  }
}

// Tile histograms -> global scatter bases, in two steps so that no block walks a
// large segment's whole column of tile counts:
//  * k_radix_chunk_scan: every chunk of SORT_CHUNK consecutive tiles of a segment
//    turns its counts into exclusive prefixes within the chunk (in place) and
//    stores the chunk's totals at its head tile in gchunk;
//  * k_radix_seg_scan: per large segment, the chunk totals become exclusive
//    prefixes over the segment's chunks plus the digit's base in the segment
//    (segment start + the counts of the smaller digits).
// A tile's base for digit d is then ghist[t][d] + gchunk[head(t)][d].  Both are
// driven by the radix tiles, so launches with no large segment cost nothing;
// thread i owns digits [PER i, PER i + PER).
#define SORT_CHUNK 16
template <int RB>
__global__ __launch_bounds__(SORT_THREADS) void k_radix_chunk_scan(const int4 *__restrict__ tiles,
                                                                  const int32_t *__restrict__ ntiles_p,
                                                                  const int32_t *__restrict__ tile_off,
                                                                  const int32_t *__restrict__ ntile,
                                                                  int32_t *__restrict__ ghist,
                                                                  int32_t *__restrict__ gchunk)
{
  constexpr int BINS = 1 << RB, PER = BINS / SORT_THREADS;
  const int d0 = threadIdx.x * PER;
  const int nt_all = *ntiles_p;
  for (int t = blockIdx.x; t < nt_all; t += gridDim.x)
  {
    const int s = tiles[t].x;
    const int t0 = tile_off[s], te = t0 + ntile[s];
    if ((t - t0) % SORT_CHUNK != 0)
      continue; // not a chunk's head tile
    const int ce = min(te, t + SORT_CHUNK);
#pragma unroll
    for (int j = 0; j < PER; j++)
    {
      const int d = d0 + j;
      int c[SORT_CHUNK];
#pragma unroll
      for (int k = 0; k < SORT_CHUNK; k++)
        c[k] = (t + k < ce) ? ghist[(int64_t)(t + k) * BINS + d] : 0;
      int run = 0;
#pragma unroll
      for (int k = 0; k < SORT_CHUNK; k++)
      {
        if (t + k < ce)
          ghist[(int64_t)(t + k) * BINS + d] = run;
        run += c[k];
      }
      gchunk[(int64_t)t * BINS + d] = run;
    }
  }
}

template <int RB>
__global__ __launch_bounds__(SORT_THREADS) void k_radix_seg_scan(const int32_t *__restrict__ seg_begin,
                                                                const int4 *__restrict__ tiles,
                                                                const int32_t *__restrict__ ntiles_p,
                                                                const int32_t *__restrict__ tile_off,
                                                                const int32_t *__restrict__ ntile,
                                                                int32_t *__restrict__ gchunk)
{
  constexpr int BINS = 1 << RB, PER = BINS / SORT_THREADS;
  __shared__ int32_t lds[SORT_THREADS / HBTX_WAVE];
  const int d0 = threadIdx.x * PER;
  const int nt_all = *ntiles_p;
  for (int t = blockIdx.x; t < nt_all; t += gridDim.x)
  {
    const int4 tl = tiles[t];
    const int s = tl.x;
    if (tl.y != seg_begin[s])
      continue; // not the segment's first tile
    const int t0 = tile_off[s], te = t0 + ntile[s];
    int run[PER];
#pragma unroll
    for (int j = 0; j < PER; j++)
    {
      const int d = d0 + j;
      run[j] = 0;
      // eight chunks' totals are loaded together: the chain is the additions, not the
      // loads (one load a chunk: 26 us for the 61 chunks of a 2 million key segment)
      for (int u = t0; u < te; u += 8 * SORT_CHUNK)
      {
        int c[8];
#pragma unroll
        for (int k = 0; k < 8; k++)
          c[k] = (u + k * SORT_CHUNK < te) ? gchunk[(int64_t)(u + k * SORT_CHUNK) * BINS + d] : 0;
#pragma unroll
        for (int k = 0; k < 8; k++)
        {
          if (u + k * SORT_CHUNK < te)
            gchunk[(int64_t)(u + k * SORT_CHUNK) * BINS + d] = run[j];
          run[j] += c[k];
        }
      }
    }
    int mine = 0;
#pragma unroll
    for (int j = 0; j < PER; j++)
      mine += run[j];
    int tot;
    int base = block_excl_scan(mine, lds, &tot) + seg_begin[s];
#pragma unroll
    for (int j = 0; j < PER; j++)
    {
      const int d = d0 + j;
      for (int u = t0; u < te; u += 8 * SORT_CHUNK)
      {
        int c[8];
#pragma unroll
        for (int k = 0; k < 8; k++)
          c[k] = (u + k * SORT_CHUNK < te) ? gchunk[(int64_t)(u + k * SORT_CHUNK) * BINS + d] : 0;
#pragma unroll
        for (int k = 0; k < 8; k++)
          if (u + k * SORT_CHUNK < te)
            gchunk[(int64_t)(u + k * SORT_CHUNK) * BINS + d] = c[k] + base;
      }
      base += run[j];
    }
    __syncthreads();
  }
}

// One pass of the tiled LSD radix sort.  Wave w ranks elements [1024 w, 1024 w +
// 1024) of the tile in order (ballot match of the digit bits, wave-private digit
// counters in LDS), the tile is then reordered by digit in LDS, and threads write
// it out in that order, so consecutive threads store to consecutive addresses of
// each digit's run.
#define SCAT_ITEMS (SORT_TILE / SORT_THREADS)
template <int RB>
__global__ __launch_bounds__(SORT_THREADS) void k_radix_scatter(const uint64_t *__restrict__ kin,
                                                               const int32_t *__restrict__ vin,
                                                               uint64_t *__restrict__ kout,
                                                               int32_t *__restrict__ vout,
                                                               const int4 *__restrict__ tiles,
                                                               const int32_t *__restrict__ ntiles_p, int shift,
                                                               const int32_t *__restrict__ ghist,
                                                               const int32_t *__restrict__ tile_off,
                                                               const int32_t *__restrict__ gchunk)
{
  constexpr int BINS = 1 << RB, PER = BINS / SORT_THREADS;
  __shared__ uint64_t sk[SORT_TILE];
  __shared__ int32_t sv[SORT_TILE];
  __shared__ int32_t wcnt[SORT_THREADS / HBTX_WAVE][BINS];
  __shared__ int32_t dbase[BINS];
  __shared__ int32_t scan_lds[SORT_THREADS / HBTX_WAVE];
  const int nt = *ntiles_p;
  const int tid = threadIdx.x;
  const int w = tid / HBTX_WAVE;
  const int lane = lane_id();
  const int per_wave = SCAT_ITEMS * HBTX_WAVE;
  // Workgroups are dispatched round-robin over the 8 XCDs.  With a grid that is a
  // multiple of 8, XCD x takes the x-th eighth of the tiles, so the short digit
  // runs that neighbouring tiles write next to each other meet in one L2 instead
  // of leaving partial lines in eight of them.
  const bool by_xcd = (gridDim.x & 7) == 0;
  const int xcd = by_xcd ? (int)(blockIdx.x & 7) : 0;
  const int step = by_xcd ? (int)(gridDim.x >> 3) : (int)gridDim.x;
  const int per_xcd = by_xcd ? (nt + 7) / 8 : nt;
  const int t_lo = xcd * per_xcd, t_hi = min(nt, t_lo + per_xcd);
  for (int t = t_lo + (by_xcd ? (int)(blockIdx.x >> 3) : (int)blockIdx.x); t < t_hi; t += step)
  {
    const int4 tl = tiles[t];
    const int n = tl.z - tl.y;
#pragma unroll
    for (int k = 0; k < SORT_THREADS / HBTX_WAVE; k++)
#pragma unroll
      for (int j = 0; j < PER; j++)
        wcnt[k][tid * PER + j] = 0;
    __syncthreads();
    uint64_t key[SCAT_ITEMS];
    int32_t val[SCAT_ITEMS];
    int32_t rank[SCAT_ITEMS];
#pragma unroll
    for (int r = 0; r < SCAT_ITEMS; r++)
    {
      const int li = w * per_wave + r * HBTX_WAVE + lane;
      const bool valid = li < n;
      key[r] = valid ? kin[tl.y + li] : 0ull;
      val[r] = valid ? vin[tl.y + li] : 0;
      const int d = (int)((key[r] >> shift) & (BINS - 1));
      uint64_t m = ballot(valid);
#pragma unroll
      for (int bit = 0; bit < RB; bit++)
      {
        const bool on = (d >> bit) & 1;
        const uint64_t bb = ballot(valid && on);
        m &= on ? bb : ~bb;
      }
      const int base = valid ? wcnt[w][d] : 0;
      rank[r] = base + __popcll(m & lanemask_lt());
      // the highest lane of each digit group advances the wave's counter
      if (valid && (m >> lane) == 1ull)
        wcnt[w][d] = base + __popcll(m);
    }
    __syncthreads();
    {
      // digits PER tid ..: offsets of the waves' runs and the first slot of the digit in the tile
      int tot[PER];
      int mine = 0;
#pragma unroll
      for (int j = 0; j < PER; j++)
      {
        const int d = tid * PER + j;
        tot[j] = 0;
#pragma unroll
        for (int k = 0; k < SORT_THREADS / HBTX_WAVE; k++)
        {
          const int c = wcnt[k][d];
          wcnt[k][d] = tot[j];
          tot[j] += c;
        }
        mine += tot[j];
      }
      int all;
      int b = block_excl_scan(mine, scan_lds, &all);
#pragma unroll
      for (int j = 0; j < PER; j++)
      {
        dbase[tid * PER + j] = b;
        b += tot[j];
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < SCAT_ITEMS; r++)
    {
      const int li = w * per_wave + r * HBTX_WAVE + lane;
      if (li < n)
      {
        const int d = (int)((key[r] >> shift) & (BINS - 1));
        const int pos = dbase[d] + wcnt[w][d] + rank[r];
        sk[pos] = key[r];
        sv[pos] = val[r];
      }
    }
    __syncthreads();
    const int32_t *off = ghist + (int64_t)t * BINS;
    const int t0 = tile_off[tl.x];
    const int32_t *coff = gchunk + (int64_t)(t0 + ((t - t0) / SORT_CHUNK) * SORT_CHUNK) * BINS;
    for (int i = tid; i < n; i += SORT_THREADS)
    {
      const uint64_t k = sk[i];
      const int d = (int)((k >> shift) & (BINS - 1));
      const int dst = off[d] + coff[d] + (i - dbase[d]);
      kout[dst] = k;
      vout[dst] = sv[i];
    }
    __syncthreads();
  }
}

} // namespace hbtx
