// Tile lists over ranges of slots (one range per subhalo or segment), and prefix
// sums of short arrays, in one or two launches.
//
// A round builds several such lists, and each used to take five launches (counts,
// three scan passes, tiles).  One block of LIST_THREADS threads now counts and scans
// up to LIST_ONE_MAX ranges (steps of LIST_STEP, read and written in rows so that
// the accesses are contiguous), and up to LIST_THREADS ranges it writes the tiles
// too; beyond that a second launch does, since one CU's stores would take longer
// (65 us for 20,000 ranges).  300 ranges: 4 us in one launch (five launches: 9 us and
// their gaps); 20,000: 19 us in two (18 us and the gaps).  A step takes 4 us, so
// arrays of more than four steps take the passes over many blocks.
#pragma once
#include "common.h"
#include "scan.h"
#include "unbind.h"

namespace hbtx
{
#define LIST_THREADS 1024
#define LIST_WAVES (LIST_THREADS / HBTX_WAVE)
#define LIST_ROWS 8
#define LIST_STEP (LIST_THREADS * LIST_ROWS)
#define LIST_ONE_MAX (4 * LIST_STEP)

// v of lane l, l the same for the whole wave
HBTX_DEV int32_t lane_value(int32_t v, int l)
{
  return __builtin_amdgcn_readlane(v, l);
}
HBTX_DEV int64_t lane_value(int64_t v, int l)
{
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(uint64_t)v, l);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)((uint64_t)v >> 32), l);
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

// Exclusive prefixes of LIST_ROWS rows of LIST_THREADS values (row k, thread t is
// element k LIST_THREADS + t), and their total.
template <typename T>
HBTX_DEV T list_excl_scan(T v[LIST_ROWS], T *lds /* [LIST_ROWS * LIST_WAVES] */)
{
  static_assert(LIST_ROWS * LIST_WAVES == 2 * HBTX_WAVE, "two wave sums a lane");
  const int w = uniform(threadIdx.x / HBTX_WAVE);
  const int lane = lane_id();
#pragma unroll
  for (int k = 0; k < LIST_ROWS; k++)
  {
    const T incl = wave_incl_scan(v[k]);
    if (lane == HBTX_WAVE - 1)
      lds[k * LIST_WAVES + w] = incl;
    v[k] = incl - v[k];
  }
  __syncthreads();
  // every wave scans the 128 wave sums, two a lane
  const T a = lds[2 * lane], b = lds[2 * lane + 1];
  const T incl = wave_incl_scan(a + b);
  const T total = lane_value(incl, HBTX_WAVE - 1);
#pragma unroll
  for (int k = 0; k < LIST_ROWS; k++)
  {
    const int i = k * LIST_WAVES + w;
    const T first = lane_value(incl - a - b, i >> 1), even = lane_value(a, i >> 1);
    v[k] += first + ((i & 1) ? even : (T)0);
  }
  __syncthreads(); // lds may be written again
  return total;
}

// out[i] = sum(in[0..i)), out[n] = total, n = min(n, *n_dev); one block (in may be out)
template <typename T>
__global__ __launch_bounds__(LIST_THREADS) void k_scan_one(const T *in, T *out, int64_t n, const int32_t *n_dev)
{
  __shared__ T lds[LIST_ROWS * LIST_WAVES];
  if (n_dev)
    n = min(n, (int64_t)*n_dev);
  T carry = 0;
  for (int64_t b = 0; b < n; b += LIST_STEP)
  {
    const int64_t i0 = b + threadIdx.x;
    T v[LIST_ROWS];
#pragma unroll
    for (int k = 0; k < LIST_ROWS; k++)
      v[k] = in[min(i0 + k * LIST_THREADS, n - 1)];
#pragma unroll
    for (int k = 0; k < LIST_ROWS; k++)
      v[k] = (i0 + k * LIST_THREADS < n) ? v[k] : (T)0;
    const T tot = list_excl_scan(v, lds);
#pragma unroll
    for (int k = 0; k < LIST_ROWS; k++)
      if (i0 + k * LIST_THREADS < n)
        out[i0 + k * LIST_THREADS] = carry + v[k];
    carry += tot;
  }
  if (threadIdx.x == 0)
    out[n] = carry;
}

// --- ranges: r(s, begin, len) ---------------------------------------------------
// (every value is loaded before any is tested, so that the loads of a thread's rows
// are in flight together)
struct RangeArray // given arrays
{
  const int32_t *begin, *len;
  HBTX_DEV void operator()(int s, int &b, int &n) const
  {
    b = begin[s];
    n = len[s];
  }
};
struct RangeActive // the slots of the subhaloes of this round
{
  SubArrays S;
  HBTX_DEV void operator()(int s, int &b, int &n) const
  {
    const int a = S.off[s], e = S.off[s + 1], md = S.mode[s];
    b = a;
    n = (md != MODE_IDLE) ? e - a : 0;
  }
};
struct RangeAll // every slot
{
  SubArrays S;
  HBTX_DEV void operator()(int s, int &b, int &n) const
  {
    b = S.off[s];
    n = S.off[s + 1] - b;
  }
};
struct RangeTreeSrc // dense sources of the tree-mode subhaloes
{
  SubArrays S;
  HBTX_DEV void operator()(int s, int &b, int &n) const
  {
    const int a = S.src_off[s], ns = S.nsrc[s], md = S.mode[s], tm = S.treemode[s];
    b = a;
    n = (md != MODE_IDLE && tm) ? ns : 0;
  }
};
struct RangeCom // subhaloes still active after the round's decision
{
  SubArrays S;
  HBTX_DEV void operator()(int s, int &b, int &n) const
  {
    const int a = S.off[s], e = S.off[s + 1], md = S.mode[s], st = S.status[s];
    b = a;
    n = (md != MODE_IDLE && st == ST_ACTIVE) ? e - a : 0;
  }
};
struct RangeConverged
{
  SubArrays S;
  HBTX_DEV void operator()(int s, int &b, int &n) const
  {
    const int a = S.off[s], e = S.off[s + 1], st = S.status[s];
    b = a;
    n = (st == ST_CONVERGED) ? e - a : 0;
  }
};
struct RangeUpscale // full-mode subhaloes that subsample this round
{
  SubArrays S;
  HBTX_DEV void operator()(int s, int &b, int &n) const
  {
    const int a = S.off[s], e = S.off[s + 1], md = S.mode[s], ns = S.nsrc[s], nt = S.ntgt[s];
    b = a;
    n = (md == MODE_FULL && ns < nt) ? e - a : 0;
  }
};
struct RangeRefine // the most bound particles whose order is refined
{
  SubArrays S;
  HBTX_DEV void operator()(int s, int &b, int &n) const
  {
    const int a = S.off[s], ns = S.nsrc[s], md = S.mode[s];
    b = a;
    n = (md == MODE_REFINE) ? ns : 0;
  }
};
struct RangeWarm // the targets of the warm rounds in tree mode
{
  SubArrays S;
  HBTX_DEV void operator()(int s, int &b, int &n) const
  {
    const int a = S.off[s], e = S.off[s + 1], md = S.mode[s], tm = S.treemode[s], ns = S.nsrc[s], nt = S.ntgt[s],
              w = S.warm[s];
    b = a;
    n = (w == WARM_PENDING && md == MODE_FULL && tm && ns < nt) ? e - a : 0;
  }
};

// tiles of a range of n slots: none at or below `over`
HBTX_DEV int list_count(int n, int tile, int over)
{
  return (n > over) ? (n + tile - 1) / tile : 0;
}

// the tiles [k0, nt) step `step` of a range: (subhalo, first, end, first tile or 0)
HBTX_DEV void list_write(int4 *tiles, int s, int b, int n, int t0, int nt, int tile, bool first, int k0, int step)
{
  for (int k = k0; k < nt; k += step)
    tiles[t0 + k] = make_int4(s, b + k * tile, min(b + n, b + (k + 1) * tile), first ? t0 : 0);
}

// The tiles of one wave's ranges (count c, first tile t0): a lane writes its own
// range's few, the wave together those of a range of many.
HBTX_DEV void list_write_wave(int4 *tiles, int s, int b, int n, int t0, int c, int tile, bool first)
{
  if (c > 0 && c <= 8)
    list_write(tiles, s, b, n, t0, c, tile, first, 0, 1);
  for (uint64_t m = ballot(c > 8); m; m &= m - 1)
  {
    const int l = __ffsll((long long)m) - 1;
    list_write(tiles, __shfl(s, l, HBTX_WAVE), __shfl(b, l, HBTX_WAVE), __shfl(n, l, HBTX_WAVE),
               __shfl(t0, l, HBTX_WAVE), __shfl(c, l, HBTX_WAVE), tile, first, lane_id(), HBTX_WAVE);
  }
}

// One block: ranges (begin_out, len_out), counts ntile, offsets toff (toff[ns] =
// total) and, if tiles is given (ns <= LIST_THREADS then), the tiles.
template <class R>
__global__ __launch_bounds__(LIST_THREADS) void k_list_one(R r, int32_t ns, int tile, int over, bool first,
                                                           int32_t *ntile, int32_t *toff, int4 *tiles,
                                                           int32_t *begin_out, int32_t *len_out)
{
  __shared__ int32_t lds[LIST_ROWS * LIST_WAVES];
  int32_t carry = 0;
  for (int base = 0; base < ns; base += LIST_STEP)
  {
    const int s0 = base + (int)threadIdx.x;
    int b[LIST_ROWS], n[LIST_ROWS];
    int32_t c[LIST_ROWS], ex[LIST_ROWS];
#pragma unroll
    for (int k = 0; k < LIST_ROWS; k++)
      r(min(s0 + k * LIST_THREADS, ns - 1), b[k], n[k]);
#pragma unroll
    for (int k = 0; k < LIST_ROWS; k++)
    {
      c[k] = (s0 + k * LIST_THREADS < ns) ? list_count(n[k], tile, over) : 0;
      ex[k] = c[k];
    }
    const int32_t tot = list_excl_scan(ex, lds);
#pragma unroll
    for (int k = 0; k < LIST_ROWS; k++)
    {
      const int s = s0 + k * LIST_THREADS;
      if (s < ns)
      {
        ntile[s] = c[k];
        toff[s] = carry + ex[k];
        if (begin_out)
        {
          begin_out[s] = b[k];
          len_out[s] = n[k];
        }
      }
    }
    if (tiles)
      list_write_wave(tiles, s0, b[0], n[0], ex[0], c[0], tile, first);
    carry += tot;
  }
  if (threadIdx.x == 0)
    toff[ns] = carry;
}

// The same in passes over many blocks: ranges and counts, (a scan), tiles.
template <class R>
__global__ void k_list_counts(R r, int32_t ns, int tile, int over, int32_t *ntile, int32_t *begin_out,
                              int32_t *len_out)
{
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= ns)
    return;
  int b, n;
  r(s, b, n);
  if (begin_out)
  {
    begin_out[s] = b;
    len_out[s] = n;
  }
  if (ntile)
    ntile[s] = list_count(n, tile, over);
}
template <class R>
__global__ void k_list_tiles(R r, int32_t ns, int tile, bool first, const int32_t *ntile, const int32_t *toff,
                             int4 *tiles)
{
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  int c = 0, b = 0, n = 0, t0 = 0;
  if (s < ns)
  {
    c = ntile[s];
    t0 = toff[s];
    r(s, b, n);
  }
  list_write_wave(tiles, s, b, n, t0, c, tile, first);
}

// The walk's work items in subhalo size order: offsets iscan (iscan[ns] = total),
// the cleared chunk counters and the total for the host, in one block.
__global__ __launch_bounds__(LIST_THREADS) void k_items_one(SubArrays S, const int32_t *order, int32_t *iscan,
                                                            int32_t *wctr, int nctr, int32_t *total)
{
  __shared__ int32_t lds[LIST_ROWS * LIST_WAVES];
  for (int i = threadIdx.x; i < nctr; i += LIST_THREADS)
    wctr[i] = 0;
  int32_t carry = 0;
  for (int base = 0; base < S.nsub; base += LIST_STEP)
  {
    const int i0 = base + (int)threadIdx.x;
    int32_t v[LIST_ROWS];
#pragma unroll
    for (int k = 0; k < LIST_ROWS; k++)
      v[k] = order[min(i0 + k * LIST_THREADS, S.nsub - 1)];
#pragma unroll
    for (int k = 0; k < LIST_ROWS; k++)
      v[k] = S.nitems[v[k]];
#pragma unroll
    for (int k = 0; k < LIST_ROWS; k++)
      v[k] = (i0 + k * LIST_THREADS < S.nsub) ? v[k] : 0;
    const int32_t tot = list_excl_scan(v, lds);
#pragma unroll
    for (int k = 0; k < LIST_ROWS; k++)
      if (i0 + k * LIST_THREADS < S.nsub)
        iscan[i0 + k * LIST_THREADS] = carry + v[k];
    carry += tot;
  }
  if (threadIdx.x == 0)
  {
    iscan[S.nsub] = carry;
    *total = carry;
  }
}
// the many-block form's last step: counters cleared and the total for the host
__global__ void k_items_finish(const int32_t *iscan_end, int32_t *wctr, int nctr, int32_t *total)
{
  for (int i = threadIdx.x; i < nctr; i += blockDim.x)
    wctr[i] = 0;
  if (threadIdx.x == 0)
    *total = *iscan_end;
}

} // namespace hbtx
