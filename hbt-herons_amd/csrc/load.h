// The caller's arrays, uploaded as they are, into the batch's device layout.
// (Interleaving them on one host thread took 60 ms for 8 million particles; these
// passes read 28 to 44 bytes and write 36 to 45 a particle, 0.2 ms.)
#pragma once
#include "common.h"

namespace hbtx
{

enum
{
  LOAD_BAD_MASS = 1,
  LOAD_BAD_TYPE = 2
};

// Positions and masses, velocities and internal energies, types; vel, u, type and
// id may be null (zero, zero, none, none).  bad: LOAD_* bits of what is out of range.
__global__ void k_load_particles(const float *__restrict__ pos, const float *__restrict__ vel,
                                 const float *__restrict__ mass, const float *__restrict__ u,
                                 const int32_t *__restrict__ type, const int64_t *__restrict__ id, int64_t n,
                                 float4 *__restrict__ posm, float4 *__restrict__ velu, int8_t *__restrict__ ptype,
                                 int64_t *__restrict__ ids, int32_t *bad)
{
  GRID_STRIDE(i, n)
  {
    const float m = mass[i];
    posm[i] = make_float4(pos[3 * i], pos[3 * i + 1], pos[3 * i + 2], m);
    velu[i] = vel ? make_float4(vel[3 * i], vel[3 * i + 1], vel[3 * i + 2], u ? u[i] : 0.f)
                  : make_float4(0.f, 0.f, 0.f, 0.f);
    int b = (m >= 0.f) ? 0 : LOAD_BAD_MASS;
    if (type)
    {
      const int t = type[i];
      ptype[i] = (int8_t)t;
      b |= (t >= 0 && t < 6) ? 0 : LOAD_BAD_TYPE;
    }
    if (id)
      ids[i] = id[i];
    if (b)
      atomicOr(bad, b);
  }
}

// Per-subhalo arrays: offsets, the (0, count) pairs of the one-subhalo views, the
// size order and the frames [6] (positions, then velocities; mb null: the frame).
__global__ void k_load_subs(const int32_t *__restrict__ off_in, const int32_t *__restrict__ order_in,
                            const float *__restrict__ ref_pos, const float *__restrict__ ref_vel,
                            const float *__restrict__ mb_pos, const float *__restrict__ mb_vel, int32_t nsub,
                            int32_t *__restrict__ off, int32_t *__restrict__ off_pairs, int32_t *__restrict__ order,
                            float *__restrict__ ref, float *__restrict__ mb)
{
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s > nsub)
    return;
  off[s] = off_in[s];
  off_pairs[2 * s] = 0;
  off_pairs[2 * s + 1] = (s < nsub) ? off_in[s + 1] - off_in[s] : 0;
  if (s == nsub)
    return;
  order[s] = order_in[s];
  for (int k = 0; k < 3; k++)
  {
    ref[6 * s + k] = ref_pos[3 * s + k];
    ref[6 * s + 3 + k] = ref_vel[3 * s + k];
    mb[6 * s + k] = mb_pos ? mb_pos[3 * s + k] : ref_pos[3 * s + k];
    mb[6 * s + 3 + k] = mb_vel ? mb_vel[3 * s + k] : ref_vel[3 * s + k];
  }
}

// Subhalo (and, if local is set, index inside it) of every slot.  A block takes
// LOAD_TILE consecutive slots: the subhaloes of its first and last slot bound every
// thread's search, which is over at once where one subhalo holds the tile.
#define LOAD_TILE 1024
HBTX_DEV int sub_search(const int32_t *off, int lo, int hi, int i)
{
  // the last s in [lo, hi] with off[s] <= i (off[lo] <= i): empty subhaloes are passed over
  while (lo < hi)
  {
    const int mid = (lo + hi + 1) >> 1;
    if (off[mid] <= i)
      lo = mid;
    else
      hi = mid - 1;
  }
  return lo;
}
__global__ __launch_bounds__(256) void k_load_sub_of(const int32_t *__restrict__ off, int32_t nsub, int64_t n,
                                                     int32_t *__restrict__ sub_of, int32_t *__restrict__ local)
{
  const int64_t ntile = (n + LOAD_TILE - 1) / LOAD_TILE;
  for (int64_t t = blockIdx.x; t < ntile; t += gridDim.x)
  {
    const int a = (int)(t * LOAD_TILE), e = (int)min((int64_t)n, (t + 1) * LOAD_TILE);
    const int lo = uniform(sub_search(off, 0, nsub - 1, a));
    const int hi = uniform(sub_search(off, lo, nsub - 1, e - 1));
    for (int i = a + threadIdx.x; i < e; i += 256)
    {
      const int s = sub_search(off, lo, hi, i);
      sub_of[i] = s;
      if (local)
        local[i] = i - off[s];
    }
  }
}

} // namespace hbtx
