// Post-unbinding properties of every subhalo's bound set, centred on its most
// bound particle (final slot 0, src/subhalo_unbind.cpp:754):
//   Subhalo_t::CalculateProfileProperties   src/subhalo.cpp:175-243
//     radii sorted, cumulative mass (double sums stored as float), radii below
//     the softening raised to it, v^2 ~ M(<r)/r: Rmax and Vmax at the first
//     maximum, RHalf = r[N/2], REnclose = r[N-1];
//   Snapshot_t::SphericalOverdensitySize    src/snapshot.cpp:258-282
//     outermost particle with M(<r) > rho_200 r^3;
//   Subhalo_t::CalculateShape               src/subhalo.cpp:245-309
//     plain and 1/r^2-weighted second moments over the bound particles but the
//     centre, float products summed in double, over Mbound.
// Every subhalo's bound particles are sorted by radius in one segmented sort;
// tiles of RED_TILE sorted slots then carry the cumulative mass (the tile offsets
// are scanned per subhalo, so no sum runs across subhaloes) and the per-tile
// candidates for the maxima and the shape sums, combined per subhalo at the end.
#pragma once
#include "common.h"
#include "unbind.h"

namespace hbtx
{
// per-tile slots of the reduction scratch (RED_NV doubles per tile)
enum
{
  PROF_SHAPE = 0,  // 12 shape sums: I {xx, xy, xz, yy, yz, zz}, then the weighted ones
  PROF_BESTV = 12, // largest v of the tile
  PROF_BESTQ = 13, // its slot (first of equal maxima)
  PROF_SOQ = 14,   // last slot meeting the overdensity, -1 if none
  PROF_TSUM = 15,  // mass of the tile
  PROF_TPRE = 16   // mass of the subhalo's earlier tiles
};

struct ProfArgs
{
  const int32_t *off;           // per subhalo first slot
  const int32_t *ford;          // final local order per slot
  const float4 *posm;
  const hbtx_sub_result *res;   // unbinding results (nbound, mbound, most bound position)
  const int32_t *seg_len;       // bound particles profiled per subhalo (0 when Nbound <= 1)
  const uint64_t *keys;         // radius bits per sorted slot
  const int32_t *vals;          // particle per sorted slot
  float *rc, *mc;               // per sorted slot: radius (softening floor), cumulative mass
  double *part;                 // per tile [RED_NV]
  DevParams P;
  float rho;                    // 200 rho_crit a^3 (float, src/snapshot.cpp:268-269)
  float vel_unit;               // G / a (float)
};

__global__ void k_prof_segments(int32_t nsub, const int32_t *off, const hbtx_sub_result *res, int32_t *seg_begin,
                                int32_t *seg_len)
{
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nsub)
    return;
  const int64_t nb = res[s].nbound;
  seg_begin[s] = off[s];
  seg_len[s] = (nb > 1 && !res[s].disrupted) ? (int32_t)nb : 0;
}

// PeriodicDistance(centre, x) (src/config_parser.h:220-233) as the sort key.
__global__ void k_prof_keys(ProfArgs A, int64_t n, const int32_t *sub_of, uint64_t *keys, int32_t *vals)
{
#pragma clang fp contract(off) // float expressions rounded as written, as on the host
  GRID_STRIDE(q, n)
  {
    const int s = sub_of[q];
    const int a = A.off[s];
    if (q - a >= A.seg_len[s])
      continue;
    const int p = a + A.ford[q];
    const float4 x = A.posm[p];
    const float *c = A.res[s].mostbound_pos;
    float dx = c[0] - x.x, dy = c[1] - x.y, dz = c[2] - x.z;
    if (A.P.periodic)
    {
      dx = nearest_f(dx, A.P.box, A.P.box_half);
      dy = nearest_f(dy, A.P.box, A.P.box_half);
      dz = nearest_f(dz, A.P.box, A.P.box_half);
    }
    keys[q] = (uint64_t)__float_as_uint(sqrtf(dx * dx + dy * dy + dz * dz));
    vals[q] = p;
  }
}

#define PROF_ITEMS (RED_TILE / RED_THREADS)
__global__ __launch_bounds__(RED_THREADS) void k_prof_tile_sum(ProfArgs A, const int4 *tiles, const int32_t *ntiles_p)
{
  __shared__ double lds[RED_THREADS / HBTX_WAVE];
  const int nt = *ntiles_p;
  for (int t = blockIdx.x; t < nt; t += gridDim.x)
  {
    const int4 tl = tiles[t];
    // (every load before the first sum: a thread's gathers are in flight together)
    float w[PROF_ITEMS];
    int p[PROF_ITEMS];
#pragma unroll
    for (int k = 0; k < PROF_ITEMS; k++)
      p[k] = A.vals[min(tl.y + (int)threadIdx.x + k * RED_THREADS, tl.z - 1)];
#pragma unroll
    for (int k = 0; k < PROF_ITEMS; k++)
      w[k] = A.posm[p[k]].w;
    double m = 0.;
#pragma unroll
    for (int k = 0; k < PROF_ITEMS; k++)
      if (tl.y + (int)threadIdx.x + k * RED_THREADS < tl.z)
        m += (double)w[k];
    double tot;
    block_excl_scan(m, lds, &tot);
    if (threadIdx.x == 0)
      A.part[(int64_t)t * RED_NV + PROF_TSUM] = tot;
  }
}

// one thread per subhalo: mass of the subhalo's earlier tiles, in tile order
__global__ void k_prof_tile_prefix(int32_t nsub, const int32_t *toff, const int32_t *ntile, double *part)
{
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nsub)
    return;
  // (eight tiles' sums loaded ahead: the additions are the only chain)
  double run = 0.;
  const int t1 = toff[s] + ntile[s];
  for (int t = toff[s]; t < t1; t += 8)
  {
    double x[8];
#pragma unroll
    for (int j = 0; j < 8; j++)
      x[j] = part[(int64_t)min(t + j, t1 - 1) * RED_NV + PROF_TSUM];
#pragma unroll
    for (int j = 0; j < 8; j++)
      if (t + j < t1)
      {
        part[(int64_t)(t + j) * RED_NV + PROF_TPRE] = run;
        run += x[j];
      }
  }
}

// Bound: the gather of the sorted slots' particles (a 64-byte line each, twice).  The
// tile's sorted arrays pass through LDS in whole lines (a thread sums 16 consecutive
// slots, so its own loads and stores touched a line a slot), PROF_AHEAD gathers are in
// flight together, and a tile of at most PROF_SHORT slots is one wave's, whose slots go to
// all of its threads.  3.0e6 slots in 5,000 subhaloes: 186 us, so 105 for the long tiles
// and 16 for the short ones.
#define PROF_AHEAD 4
#define PROF_SHORT 512
template <int THREADS> // 64: tiles of at most PROF_SHORT slots, 256: longer ones
__global__ __launch_bounds__(THREADS) void k_prof_tile_main(ProfArgs A, const int4 *tiles, const int32_t *ntiles_p)
{
#pragma clang fp contract(off) // float expressions rounded as written, as on the host
  constexpr int NW = THREADS / HBTX_WAVE;
  __shared__ double lds[NW];
  __shared__ double lsum[NW][12];
  __shared__ float lbv[NW];
  __shared__ int lbq[NW], lso[NW];
  // the tile's particles and radii, then its masses and radii (slot i at i + i / 16: a
  // thread's consecutive slots without bank conflicts)
  constexpr int CAP = (THREADS == HBTX_WAVE) ? PROF_SHORT : RED_TILE;
  __shared__ uint32_t lv[CAP + CAP / 16], lr[CAP + CAP / 16];
  auto at = [](int i) { return i + (i >> 4); };
  const int nt = *ntiles_p;
  const DevParams &P = A.P;
  const int w = threadIdx.x / HBTX_WAVE;
  for (int t = blockIdx.x; t < nt; t += gridDim.x)
  {
    const int4 tl = tiles[t];
    if ((tl.z - tl.y <= PROF_SHORT) != (THREADS == HBTX_WAVE))
      continue;
    const int s = tl.x;
    const int a = A.off[s];
    const int p0 = a + A.ford[a]; // the centre, left out of the shape sums (src/subhalo.cpp:262)
    const float *cen = A.res[s].mostbound_pos;
    const int len = tl.z - tl.y;
    for (int i = threadIdx.x; i < len; i += THREADS)
    {
      lv[at(i)] = (uint32_t)A.vals[tl.y + i];
      lr[at(i)] = (uint32_t)A.keys[tl.y + i];
    }
    __syncthreads();
    // consecutive slots, few a thread where the tile is short
    const int items = (len + THREADS - 1) / THREADS;
    const int i0 = items * threadIdx.x, i1 = min(i0 + items, len);
    double msum = 0.;
    for (int i = i0; i < i1; i += PROF_AHEAD)
    {
      float wk[PROF_AHEAD];
#pragma unroll
      for (int k = 0; k < PROF_AHEAD; k++)
        wk[k] = A.posm[lv[at(min(i + k, i1 - 1))]].w;
#pragma unroll
      for (int k = 0; k < PROF_AHEAD; k++)
        if (i + k < i1)
          msum += (double)wk[k];
    }
    double tot, before;
    if constexpr (THREADS == HBTX_WAVE)
      before = wave_incl_scan(msum) - msum;
    else
      before = block_excl_scan(msum, lds, &tot);
    double run = before + A.part[(int64_t)t * RED_NV + PROF_TPRE];
    double sh[12];
#pragma unroll
    for (int k = 0; k < 12; k++)
      sh[k] = 0.;
    float bv = -1.f;
    int bq = 0x7fffffff, so = -1;
    auto slot = [&](int i, int p, float4 x, uint32_t rbits) {
      const int q = tl.y + i;
      run += (double)x.w;
      const float m = (float)run;
      float r = __uint_as_float(rbits);
      if (r < P.eps)
        r = P.eps;
      const float v = __fdiv_rn(m, r);
      lr[at(i)] = __float_as_uint(r);
      lv[at(i)] = __float_as_uint(m);
      if (v > bv)
      {
        bv = v;
        bq = q;
      }
      if (m > A.rho * r * r * r)
        so = q;
      if (p != p0)
      {
        float d0 = x.x - cen[0], d1 = x.y - cen[1], d2 = x.z - cen[2];
        if (P.periodic)
        {
          d0 = nearest_f(d0, P.box, P.box_half);
          d1 = nearest_f(d1, P.box, P.box_half);
          d2 = nearest_f(d2, P.box, P.box_half);
        }
        const float pm = x.w;
        const float x2 = d0 * d0, y2 = d1 * d1, z2 = d2 * d2;
        sh[0] += (double)(x2 * pm);
        sh[1] += (double)(d0 * d1 * pm);
        sh[2] += (double)(d0 * d2 * pm);
        sh[3] += (double)(y2 * pm);
        sh[4] += (double)(d1 * d2 * pm);
        sh[5] += (double)(z2 * pm);
        const float dr2 = __fdiv_rn(x2 + y2 + z2, pm);
        sh[6] += (double)__fdiv_rn(x2, dr2);
        sh[7] += (double)__fdiv_rn(d0 * d1, dr2);
        sh[8] += (double)__fdiv_rn(d0 * d2, dr2);
        sh[9] += (double)__fdiv_rn(y2, dr2);
        sh[10] += (double)__fdiv_rn(d1 * d2, dr2);
        sh[11] += (double)__fdiv_rn(z2, dr2);
      }
    };
    for (int i = i0; i < i1; i += PROF_AHEAD)
    {
      int pk[PROF_AHEAD];
      uint32_t rk[PROF_AHEAD];
      float4 xk[PROF_AHEAD];
#pragma unroll
      for (int k = 0; k < PROF_AHEAD; k++)
      {
        pk[k] = (int)lv[at(min(i + k, i1 - 1))];
        rk[k] = lr[at(min(i + k, i1 - 1))];
      }
#pragma unroll
      for (int k = 0; k < PROF_AHEAD; k++)
        xk[k] = A.posm[pk[k]];
#pragma unroll
      for (int k = 0; k < PROF_AHEAD; k++)
        if (i + k < i1)
          slot(i + k, pk[k], xk[k], rk[k]);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < len; i += THREADS)
    {
      A.rc[tl.y + i] = __uint_as_float(lr[at(i)]);
      A.mc[tl.y + i] = __uint_as_float(lv[at(i)]);
    }
    // block: shape sums, the first largest v, the last overdense slot
#pragma unroll
    for (int k = 0; k < 12; k++)
      sh[k] = wave_sum_down(sh[k]);
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1)
    {
      const float ov = __shfl_down(bv, d, HBTX_WAVE);
      const int oq = __shfl_down(bq, d, HBTX_WAVE);
      if (ov > bv || (ov == bv && oq < bq))
      {
        bv = ov;
        bq = oq;
      }
      so = max(so, __shfl_down(so, d, HBTX_WAVE));
    }
    if (lane_id() == 0)
    {
#pragma unroll
      for (int k = 0; k < 12; k++)
        lsum[w][k] = sh[k];
      lbv[w] = bv;
      lbq[w] = bq;
      lso[w] = so;
    }
    __syncthreads();
    if (threadIdx.x == 0)
    {
      double *o = A.part + (int64_t)t * RED_NV;
      for (int k = 0; k < 12; k++)
      {
        double x = 0.;
        for (int ww = 0; ww < NW; ww++)
          x += lsum[ww][k];
        o[PROF_SHAPE + k] = x;
      }
      float v = lbv[0];
      int q = lbq[0], sq = lso[0];
      for (int ww = 1; ww < NW; ww++)
      {
        if (lbv[ww] > v || (lbv[ww] == v && lbq[ww] < q))
        {
          v = lbv[ww];
          q = lbq[ww];
        }
        sq = max(sq, lso[ww]);
      }
      o[PROF_BESTV] = (double)v;
      o[PROF_BESTQ] = (double)q;
      o[PROF_SOQ] = (double)sq;
    }
    __syncthreads();
  }
}

// one thread per subhalo: combine the tiles in order and write the properties
__global__ void k_prof_finish(ProfArgs A, int32_t nsub, const int32_t *toff, const int32_t *ntile,
                              hbtx_sub_profile *out)
{
#pragma clang fp contract(off) // float expressions rounded as written, as on the host
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nsub)
    return;
  hbtx_sub_profile o;
  float *f = &o.rmax_comoving;
  for (int k = 0; k < 18; k++)
    f[k] = 0.f;
  o.has_r200 = 0;
  o.reserved = 0;
  const int nb = A.seg_len[s];
  if (nb > 1)
  {
    const int a = A.off[s];
    double sh[12];
    for (int k = 0; k < 12; k++)
      sh[k] = 0.;
    float bv = -1.f;
    int bq = a, so = -1;
    // (four tiles' partials loaded ahead)
    const int t1 = toff[s] + ntile[s];
    for (int t = toff[s]; t < t1; t += 4)
    {
      double x[4][15];
#pragma unroll
      for (int j = 0; j < 4; j++)
      {
        const double *pt = A.part + (int64_t)min(t + j, t1 - 1) * RED_NV;
#pragma unroll
        for (int k = 0; k < 12; k++)
          x[j][k] = pt[PROF_SHAPE + k];
        x[j][12] = pt[PROF_BESTV];
        x[j][13] = pt[PROF_BESTQ];
        x[j][14] = pt[PROF_SOQ];
      }
#pragma unroll
      for (int j = 0; j < 4; j++)
      {
        if (t + j >= t1)
          break;
#pragma unroll
        for (int k = 0; k < 12; k++)
          sh[k] += x[j][k];
        const float v = (float)x[j][12];
        if (v > bv)
        {
          bv = v;
          bq = (int)x[j][13];
        }
        so = max(so, (int)x[j][14]);
      }
    }
    o.rmax_comoving = A.rc[bq];
    o.vmax_physical = sqrtf(bv * A.vel_unit);
    o.r_half_comoving = A.rc[a + nb / 2];
    o.r_enclose_comoving = A.rc[a + nb - 1];
    if (so >= 0)
    {
      const float m = A.mc[so];
      o.bound_m200_crit = m;
      o.bound_r200_crit_comoving = (float)pow((double)__fdiv_rn(m, A.rho), 1.0 / 3);
      o.has_r200 = 1;
    }
    const float mb = A.res[s].mbound;
    for (int k = 0; k < 6; k++)
    {
      o.inertial_tensor[k] = __fdiv_rn((float)sh[k], mb);
      o.inertial_tensor_weighted[k] = __fdiv_rn((float)sh[6 + k], mb);
    }
  }
  out[s] = o;
}

} // namespace hbtx
