// Potential at arbitrary points (GravityTree_t::EvaluatePotential on a batch of
// targets, src/gravity_tree.cpp:82-166) and the exact direct sum.
#pragma once
#include "walk.h"

namespace hbtx
{

struct PointArgs
{
  const float4 *tgt;       // target position + self mass (targetMass)
  const int32_t *tgt_order;// walk order of targets (spatially sorted) or null
  int32_t ntgt;
  int32_t eb, ee;          // walk-record unit range
  int32_t treemode;
  const double *cube;      // the tree's root cube (centre, half side)
  const uint2 *wt;         // walk records
  double *phi;             // specific potential, scattered to the target's input index
  int32_t *counter;        // work counters (ItemQueue), zeroed before launch
  int32_t chunks;          // item list split into this many contiguous chunks
  unsigned long long *stats;
  int32_t *overflow;       // set to WALK_STACK_OVERFLOW if the walk stack was full, or null
  DevParams P;
};

HBTX_DEV void store_potential(const PointArgs &A, float tgt_mass, const Kahan &acc, bool valid, int ti)
{
  if (!valid)
    return;
  const float self = tgt_mass / A.P.eps;
  A.phi[ti] = ((double)self + (double)acc.s - (double)acc.c) * A.P.G_over_a;
}

template <bool PERIODIC, bool STATS>
__global__ __launch_bounds__(WALK_WG_THREADS, 8) void k_points_potential(PointArgs A)
{
  const int lane = lane_id();
  __shared__ WalkLds wls[HBTX_WALK_WG_WAVES];
  WalkLds &wl = wls[threadIdx.x / HBTX_WAVE];
  unsigned long long st_steps = 0, st_visits = 0, st_accepts = 0, st_pairs = 0, st_near = 0;
  const int nitems = (A.ntgt + HBTX_WAVE - 1) / HBTX_WAVE;
  ItemQueue queue;
  queue.init(A.counter, A.chunks, nitems);
  for (;;)
  {
    const int it = queue.next();
    if (it < 0)
      break;
    const int t = it * HBTX_WAVE + lane;
    const bool valid = t < A.ntgt;
    const int ti = valid ? (A.tgt_order ? A.tgt_order[t] : t) : 0;
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
    if (valid)
      x = A.tgt[ti];
    Kahan acc;
    acc.init();
    WalkCounts wc = {0u, 0u, 0u, 0u};
    if (A.ee > A.eb)
    {
      if (A.treemode)
      {
        if (PERIODIC && cube_may_wrap(A.cube, valid, x.x, x.y, x.z, A.P))
          tree_walk_stack<PERIODIC, STATS>(A.wt, A.eb, A.ee, valid, x.x, x.y, x.z, A.P, acc, wc, wl, A.overflow);
        else
          tree_walk_stack<false, STATS>(A.wt, A.eb, A.ee, valid, x.x, x.y, x.z, A.P, acc, wc, wl, A.overflow);
      }
      else
      {
        if (PERIODIC &&
            records_may_wrap(A.wt + A.eb, lane, HBTX_WAVE, (A.ee - A.eb) / 2, valid, x.x, x.y, x.z, A.P))
          direct_sum<PERIODIC>(A.wt, A.eb, A.ee, x.x, x.y, x.z, A.P, acc, wc);
        else
          direct_sum<false>(A.wt, A.eb, A.ee, x.x, x.y, x.z, A.P, acc, wc);
        if (STATS)
          st_pairs += (unsigned long long)__popcll(wave_mask(valid)) * (unsigned long long)((A.ee - A.eb) / 2);
      }
    }
    if (STATS)
    {
      st_steps += wc.steps;
      st_visits += wc.visits;
      st_accepts += wc.accepts;
      st_near += wc.nnear;
    }
    store_potential(A, x.w, acc, valid, ti);
  }
  if (STATS && A.stats && lane == 0)
  {
    atomicAdd(A.stats + STAT_TREE_STEPS, st_steps);
    atomicAdd(A.stats + STAT_TREE_VISITS, st_visits);
    atomicAdd(A.stats + STAT_TREE_ACCEPT, st_accepts);
    atomicAdd(A.stats + STAT_DIRECT_PAIRS, st_pairs);
    atomicAdd(A.stats + STAT_NEAR, st_near);
  }
}

// The exact sum at few targets, several waves per 64 targets.  One wave alone
// leaves most of the chip idle (30,001 targets are 469 waves for 1024 SIMDs), but
// the compensated sum over the groups of four sources is a serial chain, and it
// has to stay that chain for the results to stay what they are.  So DS_WAVES waves
// form the groups' sums (about 52 issue cycles a pair) into LDS, DS_GROUPS each a
// stage, and one more wave adds them in order (four dependent operations a group,
// about an eighth of a group's work) while the others form the next stage's.
// 20,011 sources on 30,001 targets: 3104 us with one wave waiting for each group's
// records, 2087 us with the records loaded ahead (direct_groups), 227 us here (2.6e12
// pairs/s; the vector units alone allow about 3.0e12).  With 4 groups a wave and
// stage it took 241 us, and 192 instead of 158 us on 8,000 targets: a stage starts
// with its records not yet loaded, so longer stages wait less.
#define DS_WAVES 8
#define DS_GROUPS 8
#define DS_THREADS (HBTX_WAVE * (DS_WAVES + 1))
// Records from which on a block asks whether any of its pairs can wrap: the targets'
// bounds (36 lane exchanges) cost more than they can save on fewer.  2,000 periodic
// targets, asked and not: 10 sources away from the box faces 24.1 and 23.2 us (about a
// face 24.9 and 23.5), 32 sources 25.5 and 26.1, 200 sources 26.4 and 27.9.
#define DS_SCREEN_MIN 32
template <bool PERIODIC, bool STATS>
__global__ __launch_bounds__(DS_THREADS) void k_points_direct(PointArgs A)
{
  __shared__ float parts[2][DS_WAVES * DS_GROUPS][HBTX_WAVE];
  const int lane = lane_id();
  const int w = uniform(threadIdx.x / HBTX_WAVE);
  const int nitems = (A.ntgt + HBTX_WAVE - 1) / HBTX_WAVE;
  const uint2 *ent = A.wt + A.eb;
  const int ee = (A.ee - A.eb) / 2, ng = ee / 4;
  const int nstage = (ng + DS_WAVES * DS_GROUPS - 1) / (DS_WAVES * DS_GROUPS);
  unsigned long long st_pairs = 0;
  WalkCounts wc = {0u, 0u, 0u, 0u};
  for (int it = blockIdx.x; it < nitems; it += gridDim.x)
  {
    const int t = it * HBTX_WAVE + lane;
    const bool valid = t < A.ntgt;
    const int ti = valid ? (A.tgt_order ? A.tgt_order[t] : t) : 0;
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
    if (valid)
      x = A.tgt[ti];
    Kahan acc;
    acc.init();
    const bool wraps =
      PERIODIC && (ee < DS_SCREEN_MIN || __syncthreads_or(records_may_wrap(ent, threadIdx.x, DS_THREADS, ee, valid, x.x,
                                                                           x.y, x.z, A.P)));
    // stage st is formed in buffer st & 1 while stage st - 1 is added from the other
    for (int st = 0; st <= nstage; st++)
    {
      if (w < DS_WAVES)
      {
        const int g0 = (st * DS_WAVES + w) * DS_GROUPS;
        auto emit = [&](int g, float part) { parts[st & 1][w * DS_GROUPS + (g - g0)][lane] = part; };
        if (st < nstage && PERIODIC && wraps)
          direct_groups<PERIODIC, 2>(ent, g0, min(ng, g0 + DS_GROUPS), x.x, x.y, x.z, A.P, wc, emit);
        else if (st < nstage)
          direct_groups<false, 2>(ent, g0, min(ng, g0 + DS_GROUPS), x.x, x.y, x.z, A.P, wc, emit);
      }
      else if (st > 0)
      {
        const int n = min(DS_WAVES * DS_GROUPS, ng - (st - 1) * DS_WAVES * DS_GROUPS);
        const float(*b)[HBTX_WAVE] = parts[(st - 1) & 1];
        int k0 = 0;
        for (; k0 + 32 <= n; k0 += 32)
        {
          float v[32];
#pragma unroll
          for (int k = 0; k < 32; k++)
            v[k] = b[k0 + k][lane];
#pragma unroll
          for (int k = 0; k < 32; k++)
            acc.add(v[k]);
        }
        for (int k = k0; k < n; k++)
          acc.add(b[k][lane]);
      }
      __syncthreads();
    }
    if (w < DS_WAVES)
      continue;
    for (int i = ee & ~3; i < ee; i++)
    {
      bool nr = false;
      acc.add(direct_term<PERIODIC>(const_load_f4u(ent + 2 * i), x.x, x.y, x.z, A.P, nr));
    }
    if (STATS)
      st_pairs += (unsigned long long)__popcll(wave_mask(valid)) * (unsigned long long)ee;
    store_potential(A, x.w, acc, valid, ti);
  }
  if (STATS && A.stats && lane == 0)
  {
    atomicAdd(A.stats + STAT_DIRECT_PAIRS, st_pairs);
    atomicAdd(A.stats + STAT_NEAR, (unsigned long long)wc.nnear);
  }
}

// the walk's n_words counters (and overflow word) cleared, and one sort segment over the
// n targets
__global__ void k_points_begin(int32_t *counter, int n_words, int32_t *seg, int32_t n)
{
  for (int i = threadIdx.x; i < n_words; i += blockDim.x)
    counter[i] = 0;
  if (threadIdx.x < 2)
    seg[threadIdx.x] = (threadIdx.x == 0) ? 0 : n;
}

// keys of external target points in a tree's cube (walk order for coherence)
__global__ void k_point_keys(const float4 *tgt, int32_t n, const double *cube, uint64_t *keys, int32_t *vals)
{
  GRID_STRIDE(i, n)
  {
    const float4 x = tgt[i];
    keys[i] = octree_key(x.x, x.y, x.z, cube[0], cube[1], cube[2], cube[3]);
    vals[i] = (int32_t)i;
  }
}

// Caller-owned device arrays packed into the direct sum's records {x, y, z, m}
// (the layout the tree build emits for a direct-sum source set) and into the
// walk's target points {x, y, z, target mass}.
__global__ void k_pack_records(const float *pos, const float *mass, int32_t n, uint2 *wt)
{
  GRID_STRIDE(i, n)
  {
    wt[2 * i] = make_uint2(__float_as_uint(pos[3 * i]), __float_as_uint(pos[3 * i + 1]));
    wt[2 * i + 1] = make_uint2(__float_as_uint(pos[3 * i + 2]), __float_as_uint(mass[i]));
  }
}

__global__ void k_pack_points(const float *pos, const float *mass, int32_t n, float4 *out)
{
  GRID_STRIDE(i, n)
  out[i] = make_float4(pos[3 * i], pos[3 * i + 1], pos[3 * i + 2], mass ? mass[i] : 0.f);
}

} // namespace hbtx
