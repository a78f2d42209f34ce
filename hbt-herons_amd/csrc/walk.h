// Potential + binding-energy kernel (one wave = 64 targets of one subhalo).
//
// Tree mode: each lane applies the reference's own opening test to its own
// target (open if len^2 > r^2 theta^2 with r to the cell's centre of mass,
// src/gravity_tree.cpp:139, stored as r^2 < crit2 = len^2/theta^2) over the
// depth-first walk records (16-byte particles, 24-byte cells), so that every lane
// accepts exactly the records its own walk accepts (src/gravity_tree.cpp:82-166),
// while the 64 lanes on spatially adjacent targets share one traversal: the
// batched stack walk below (tree_walk_stack).
//
// Direct mode: the entry list holds particles only and every pair is summed.
//
// The fused epilogue forms the binding energy of the full iteration
// (src/subhalo_unbind.cpp:602-616, src/gravity_tree.cpp:168-178) or the
// correction update (src/subhalo_unbind.cpp:577-589).
#pragma once
#include "common.h"
#include <type_traits>

namespace hbtx
{

enum
{
  STAT_TREE_STEPS = 0,    // wave steps of tree walks
  STAT_TREE_VISITS = 1,   // active lane-entry visits (opening test evaluated)
  STAT_TREE_ACCEPT = 2,   // accepted lane interactions (monopole or particle)
  STAT_DIRECT_PAIRS = 3,  // lane-pair evaluations in direct mode
  STAT_TARGETS = 4,       // targets processed
  STAT_ITEMS = 5,         // work items processed
  STAT_NEAR = 6,          // wave steps that evaluated the softening kernel
  NSTATS = 16
};

struct WalkArgs
{
  const int2 *items;        // (subhalo, first target) per work item
  const int32_t *nitems;    // number of items (device)
  int32_t *counter;         // work counters (ItemQueue), zeroed before launch
  int32_t nchunks;          // item list split into this many contiguous chunks
  const int32_t *cur;       // slot-layout target order
  const int32_t *off;       // per subhalo slot offset
  const int32_t *ntgt;
  const int32_t *mode;
  const int32_t *treemode;
  const double *cube;       // per subhalo: its tree's root cube (centre, half side), see cube_may_wrap
  const int32_t *ent_begin; // per subhalo: first walk-record unit of its tree
  const int32_t *ent_end;   // per subhalo: end unit
  const uint2 *wt;          // walk records (8-byte units, two spare units past the end)
  const float4 *posm;
  const float4 *velu;
  const float *selfm;       // target self mass (sources of a full iteration), else 0
  const float *ref;         // per subhalo frame [6]
  const float *oldref;      // per subhalo previous frame [6]
  float *energy;
  float *esl;               // the same energies by slot (off[s] + target index)
  float *eref;              // refinement energies (MODE_REFINE targets)
  unsigned long long *stats;
  int32_t *overflow;        // the round's overflow word (WALK_STACK_OVERFLOW)
  DevParams P;
};

HBTX_DEV uint64_t wave_mask(bool p)
{
  return __builtin_amdgcn_ballot_w64(p);
}

// Waves per walk workgroup.  Every wave walks on its own (its own items and its
// own LDS stack, no workgroup barrier); one, two and four waves a workgroup
// time the same, as a CU holds 32 one-wave workgroups with this LDS size.
#ifndef HBTX_WALK_WG_WAVES
#define HBTX_WALK_WG_WAVES 2
#endif
constexpr int WALK_WG_THREADS = HBTX_WAVE * HBTX_WALK_WG_WAVES;

// Work items 0 .. nit - 1 handed to the waves of a persistent kernel.  The list is cut
// into nch contiguous chunks with a counter each: workgroups go round the XCDs, so
// workgroup b drains chunk b % nch first (neighbouring items, which read the same part of
// a tree, stay on one XCD's L2), then helps with the others.  The wave that finds a chunk
// empty first sets its bit in the word after the counters, and a wave looking for
// another chunk reads that word before it touches a counter.  With a failed addition on
// every chunk's counter a wave, which are served one after the other, 8,192 waves spent
// longer on ending than a round of small items takes: walks (16 chunks, the tuned number)
// of 1.2e6 particles in subhaloes of at most 2,000, 0.89 ms, 0.47 so; in subhaloes up to a
// million, 2.1e6 particles 2.12 and 1.72 ms, 8e6 5.08 and 4.74.  (Several counters a chunk
// made it worse, 5.9 ms of 8e6: a wave that looks for work then reads them all, and they
// are what the others are adding to.)
#define QUEUE_STRIDE 32 // ints between counters: a cache line each
struct ItemQueue
{
  int32_t *ctr;
  int nch, q, r; // chunks, items a chunk (one more in the first r)
  int wq, wr;    // the same of the workgroups
  int cur;
  int first;     // this wave's number among its chunk's (-1 once it has taken that item)
  uint32_t done; // the chunks known to be empty

  HBTX_DEV void init(int32_t *counters, int chunks, int nit)
  {
    ctr = counters;
    nch = chunks;
    nit = uniform(nit);
    q = nit / nch;
    r = nit - q * nch;
    wq = gridDim.x / nch;
    wr = gridDim.x - wq * nch;
    const int g = blockIdx.x / nch;
    cur = blockIdx.x - g * nch;
    first = g * HBTX_WALK_WG_WAVES + uniform(threadIdx.x / HBTX_WAVE);
    done = 0u;
  }
  // the next item, or -1 (every wave ends: a turn that gives no item marks a chunk)
  HBTX_DEV int next()
  {
    for (;;)
    {
      // the chunk's first items go to its own waves by number, the rest by the counter
      const int size = q + (cur < r ? 1 : 0), waves = (wq + (cur < wr ? 1 : 0)) * HBTX_WALK_WG_WAVES;
      int got = first;
      if (first < 0)
      {
        got = 0;
        if (lane_id() == 0)
          got = atomicAdd(ctr + QUEUE_STRIDE * cur, 1);
        got = waves + uniform(got);
      }
      first = -1;
      if (got < size)
        return cur * q + min(cur, r) + got;
      done |= 1u << cur;
      if (nch == 1)
        return -1;
      uint32_t *word = reinterpret_cast<uint32_t *>(ctr + QUEUE_STRIDE * nch);
      if (got == max(size, waves) && lane_id() == 0)
        atomicOr(word, 1u << cur);
      done |= (uint32_t)uniform((int)__hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
      const uint32_t left = ~done & ((1u << nch) - 1u);
      if (left == 0u)
        return -1;
      const uint32_t after = left & ~((2u << cur) - 1u); // the next chunk, or the first
      cur = __ffs((int)(after ? after : left)) - 1;
    }
  }
};

// Squared distance with the fused multiply-adds written out, so that every kernel
// rounds alike: the x square first where XFIRST, else the y square.
template <bool PERIODIC, bool XFIRST>
HBTX_DEV float sep2(float ex, float ey, float ez, float px, float py, float pz, const DevParams &P)
{
#pragma clang fp contract(off)
  float dx, dy, dz;
  if (PERIODIC)
  {
    dx = nearest_diff_f(ex, px, P.box, P.box_half);
    dy = nearest_diff_f(ey, py, P.box, P.box_half);
    dz = nearest_diff_f(ez, pz, P.box, P.box_half);
  }
  else
  {
    dx = ex - px;
    dy = ey - py;
    dz = ez - pz;
  }
  return __builtin_fmaf(dz, dz, XFIRST ? __builtin_fmaf(dy, dy, dx * dx) : __builtin_fmaf(dx, dx, dy * dy));
}

// In a periodic box a pair's separation is wrapped only where one of its components
// is beyond half the box; elsewhere the wrapped separation and its rounding are those
// of a plain difference.  So a wave first asks whether any of its pairs can be: where
// none can (every subhalo that does not straddle the box edge), its targets take the
// non-periodic form, 3 vector instructions a pair for the separation instead of 33, and
// the same bits.  1e6 particles of periodic subhaloes: walks of five rounds 1.74 ms with
// every pair wrapped, 1.05 ms so.
//
// Of the targets against a tree: the particles lie in the root cube, the cells' centres
// of mass within rounding of it (the margin).
HBTX_DEV bool cube_may_wrap(const double *cube, bool valid, float px, float py, float pz, const DevParams &P)
{
  const double reach = 0.999 * (double)P.box_half - cube[3];
  const bool ok = fabs((double)px - cube[0]) <= reach && fabs((double)py - cube[1]) <= reach &&
                  fabs((double)pz - cube[2]) <= reach;
  return wave_mask(valid && !ok) != 0ull; // (NaN: wrapped)
}

// Of the targets against the particle records first, first + step, ... < n of this lane;
// the wave's answer covers all its lanes' records.
HBTX_DEV bool records_may_wrap(const uint2 *ent, int first, int step, int n, bool valid, float px, float py, float pz,
                               const DevParams &P)
{
  float lo[3] = {px, py, pz}, hi[3] = {px, py, pz};
#pragma unroll
  for (int k = 0; k < 3; k++)
  {
    lo[k] = valid ? lo[k] : INFINITY;
    hi[k] = valid ? hi[k] : -INFINITY;
#pragma unroll
    for (int d = 1; d < HBTX_WAVE; d <<= 1)
    {
      lo[k] = fminf(lo[k], __shfl_xor(lo[k], d, HBTX_WAVE));
      hi[k] = fmaxf(hi[k], __shfl_xor(hi[k], d, HBTX_WAVE));
    }
  }
  bool ok = true;
#pragma unroll 4
  for (int i = first; i < n; i += step)
  {
    const uint2 a = ent[2 * (int64_t)i], b = ent[2 * (int64_t)i + 1];
    const float r[3] = {__uint_as_float(a.x), __uint_as_float(a.y), __uint_as_float(b.x)};
#pragma unroll
    for (int k = 0; k < 3; k++)
      ok = ok && r[k] - lo[k] <= P.box_half && r[k] - hi[k] >= -P.box_half;
  }
  return wave_mask(!ok) != 0ull; // (NaN: wrapped)
}

// Per-wave work counters of one walk (uniform values, kept only in the stats
// instantiation; the walk is deterministic, so a stats run counts exactly the
// work of a timed run).
struct WalkCounts
{
  uint32_t steps, visits, accepts, nnear;
};

// Batched stack walk: lane-exact opening decisions, with the records a wave
// visits gathered 64 at a time instead of one dependent load per record.
//
// A stack entry (o, e, mask) stands for the sibling chain of records from byte
// offset o up to e, and mask holds the lanes that reached it (that opened every
// ancestor).  Processing record o: each reached lane applies its own opening
// test; a lane accepts the record (adds its term) unless it opens it; the chain's
// rest (o's skip, up to e) is pushed with the same mask, and an opened cell pushes
// its children's chain (o + 24, skip) with the mask of the lanes that opened it.
// A lane therefore accepts exactly the records its own walk accepts, and the wave
// visits exactly the records some lane reaches (the union of its lanes' walks);
// a batch pops up to 64 entries, loads their records together (one vector
// gather), stages them in LDS and then evaluates them back to back with no memory
// access on the chain between one record's test and the next.
//
// Capacity: a batch of B entries pushes at most 2 B, so B is cut to keep the stack
// WSTACK_HEADROOM below its capacity; once the room is gone single entries are
// popped, a depth-first descent that adds at most one entry per level (the
// chain's rest) plus the entry it stands on.  A tree has at most 22 cell levels
// (21-bit keys per axis under the root), so the stack never holds more than
// WSTACK_CAP - WSTACK_HEADROOM + 24 entries; a push beyond the capacity (never
// taken) raises the overflow word instead of writing.
constexpr int WSTACK_CAP = 160;
constexpr int WSTACK_HEADROOM = 32;

// m's bit for this lane ? a : b, with m a wave-uniform lane mask: one
// v_cndmask on the mask's SGPR pair, where a select on a per-lane bool would first
// turn the mask back into that bool with vector instructions.
HBTX_DEV float lane_select(uint64_t m, float a, float b)
{
  float r;
  asm("v_cndmask_b32_e64 %0, %1, %2, %3" : "=v"(r) : "v"(b), "v"(a), "s"(m));
  return r;
}

// acc = -a * b + acc on the lanes of the wave-uniform mask m, the others keeping
// acc: one FMA under a narrowed exec mask (restored in the same block), where a
// select would take a second vector instruction.
HBTX_DEV void fma_neg_on(uint64_t m, float &acc, float a, float b)
{
  uint64_t save;
  asm volatile("s_mov_b64 %1, exec\n\t"
               "s_and_b64 exec, exec, %4\n\t"
               "v_fma_f32 %0, -%2, %3, %0\n\t"
               "s_mov_b64 exec, %1"
               : "+v"(acc), "=&s"(save)
               : "v"(a), "v"(b), "s"(m)
               : "scc");
}

// acc -= m[k] * q[k] for k = 0..3 in order, each on the lanes of its wave-uniform
// mask only (a subset of exec): the sums of four records without a vector select, the
// exec mask saved and restored once.
HBTX_DEV void fma_neg_on4(const uint64_t on[4], float &acc, const float m[4], const float q[4])
{
  uint64_t save;
  asm volatile("s_mov_b64 %1, exec\n\t"
               "s_mov_b64 exec, %10\n\t"
               "v_fma_f32 %0, -%2, %6, %0\n\t"
               "s_mov_b64 exec, %11\n\t"
               "v_fma_f32 %0, -%3, %7, %0\n\t"
               "s_mov_b64 exec, %12\n\t"
               "v_fma_f32 %0, -%4, %8, %0\n\t"
               "s_mov_b64 exec, %13\n\t"
               "v_fma_f32 %0, -%5, %9, %0\n\t"
               "s_mov_b64 exec, %1"
               : "+v"(acc), "=&s"(save)
               : "v"(m[0]), "v"(m[1]), "v"(m[2]), "v"(m[3]), "v"(q[0]), "v"(q[1]), "v"(q[2]), "v"(q[3]), "s"(on[0]),
                 "s"(on[1]), "s"(on[2]), "s"(on[3]));
}

struct WalkLds
{
  int4 stk[WSTACK_CAP];  // (record offset, chain end, reached mask low, high word)
  float4 rec[HBTX_WAVE]; // a batch's records: x, y, z, m (then the lanes that opened each)
  float4 aux[HBTX_WAVE]; // crit2 (a cell only), mask low, crit2, mask high
};

#define WALK_STACK_OVERFLOW 4 // overflow-word bit: the walk stack was full (never expected)

template <bool PERIODIC, bool STATS>
HBTX_DEV void tree_walk_stack(const uint2 *wt, int ub, int ue, bool valid, float px, float py, float pz,
                              const DevParams &P, Kahan &acc, WalkCounts &wc, WalkLds &L, int32_t *overflow)
{
  const uint2 *tree = wt + ub;
  const int32_t span = 8 * (ue - ub);
  const int lane = lane_id();
  const uint64_t vmask = wave_mask(valid);
  if (vmask == 0ull)
    return;
  // lanes 0-31 read (crit2, mask low), lanes 32-63 (crit2, mask high) of a staged record
  const float2 *aw = reinterpret_cast<const float2 *>(L.aux) + (lane >> 5);
  // the staged records and open masks through VGPR base addresses (a zero the
  // compiler cannot see through), so that record j of an unrolled group is an
  // immediate offset instead of an address moved from an SGPR per record
  int vz;
  asm volatile("v_mov_b32 %0, 0" : "=v"(vz));
  const float4 *rec = L.rec + vz;
  uint2 *omw = reinterpret_cast<uint2 *>(L.rec) + vz;
  const uint32_t bit = 1u << (lane & 31);
  if (lane == 0)
    L.stk[0] = make_int4(0, span, (int)(uint32_t)vmask, (int)(uint32_t)(vmask >> 32));
  wave_lds_sync();
  int top = 1;
  float blk = 0.f;
  int nblk = 0;
  while (top > 0)
  {
    const int room = WSTACK_CAP - WSTACK_HEADROOM - top;
    const int nb = min(min(HBTX_WAVE, top), max(1, room));
    top -= nb;
    const uint64_t mine = ~0ull >> (HBTX_WAVE - nb); // the lanes with an entry of the batch
    // (a lane past them reads the last entry and stages it in the slot of its own number,
    // which is past the batch: no branch)
    const int src = top + min(lane, nb - 1);
    int32_t nx;
    int slot, ncell;
    uint64_t cmask;
    bool small_cells; // some cell's opening radius is below the softening length
    {
      const int4 it = L.stk[src];
      // 24 bytes whatever the record: a particle's last 8 are the next record's
      // (or the spare units past the records' end) and are not used, so that
      // both loads go out together
      const uint2 *rp = tree + (it.x >> 3);
      const uint2 u0 = rp[0], u1 = rp[1], u2 = rp[2];
      const float c2 = __uint_as_float(u2.x);
      // staged cells first, then particles (the order within a batch is free): a
      // particle is never opened, so its visit skips the opening test and mask
      cmask = __builtin_amdgcn_sicmp((int32_t)u1.y, 0, 40 /* < */) & mine;
      small_cells = (cmask & ~__builtin_amdgcn_fcmpf(c2, P.h2, 3 /* ordered >= */)) != 0ull;
      ncell = __popcll(cmask);
      const bool cell = (int32_t)u1.y < 0 && lane < nb;
      nx = cell ? (int32_t)u2.y : it.x + 16;
      const int before = mask_rank(cmask, 0);
      slot = cell ? before : ncell + lane - before;
      L.rec[slot] = make_float4(__uint_as_float(u0.x), __uint_as_float(u0.y), __uint_as_float(u1.x),
                                fabsf(__uint_as_float(u1.y)));
      L.aux[slot] = make_float4(c2, __int_as_float(it.z), c2, __int_as_float(it.w));
    }
    wave_lds_sync();
    // Records of the batch against every lane's target.  The lane predicates are
    // single compares whose masks the scalar unit combines: reached R, opened Lt
    // (r2 < crit2), near N (r2 < h2).  An accepted lane (R, not Lt) adds -m/r,
    // or the spline where N; the sum runs under the accepting lanes' exec mask,
    // so that a lane that does not accept never uses its 1/r (infinite where the
    // record is the target itself).  A cell's visit returns the lanes that opened it.
    using XF = std::true_type;
    using YF = std::false_type;
    using CELL = std::true_type;
    using PART = std::false_type;
    // (xf: the first of a group of four and the records past the last group square x
    // first, the others y)
    auto reached = [&](float mask_word) {
      return __builtin_amdgcn_uicmp(__float_as_uint(mask_word) & bit, 0u, 33 /* ne */);
    };
    auto near_terms = [&](uint64_t na, float r2, float rinv, float m) {
      if (STATS)
        wc.nnear++;
      // at zero distance (the target's own record, or a coincident source) the
      // spline is its value at u = 0, m hinv (-2.8), as spline_near forms it
      const uint64_t zm = __builtin_amdgcn_fcmpf(r2, 0.f, 1 /* ordered == */);
      const float tn = ((na & ~zm) == 0ull) ? (m * P.hinv) * -2.8f : spline_near(r2, rinv, m, P.hinv);
      blk += lane_select(na, tn, 0.f);
    };
    auto count = [&](uint64_t rm, uint64_t lm) {
      if (STATS)
      {
        wc.steps++;
        wc.visits += __popcll(rm);
        wc.accepts += __popcll(rm & ~lm);
      }
    };
    auto visit = [&](int j, auto is_cell, auto xf) -> uint64_t {
      const float4 r = rec[j];
      const float2 w = aw[2 * j];
      const float r2 = sep2<PERIODIC, decltype(xf)::value>(r.x, r.y, r.z, px, py, pz, P);
      const uint64_t rm = reached(w.y);
      const uint64_t lm = is_cell ? __builtin_amdgcn_fcmpf(r2, w.x, 4 /* ordered < */) : 0ull;
      const uint64_t nm = __builtin_amdgcn_fcmpf(r2, P.h2, 4 /* ordered < */);
      const float rinv = __builtin_amdgcn_rsqf(r2);
      fma_neg_on(rm & ~(lm | nm), blk, r.w, rinv);
      const uint64_t na = rm & nm & ~lm;
      if (na != 0ull)
        near_terms(na, r2, rinv, r.w);
      count(rm, lm);
      return rm & lm;
    };
    // Four records at once.  A cell no smaller than the softening (crit2 >= h2: all but
    // some 0.3% of the cells met) is opened by every lane it is near to, so it has no
    // near test; four particles share one branch on it.  Bound: the vector unit (some 16
    // instructions a record, 69% of its cycles) and, of a few waves, the latency of a
    // record's chain.  With a near test and branch a record: 8e6 particles, five rounds'
    // walks 5.33 ms, 5.16 so; a halo of 12,000 (two rounds of 188 waves) 0.394 and 0.366 ms.
    auto visit4 = [&](int j, auto is_cell, uint64_t opened[4]) {
      float m[4], r2[4], rinv[4];
      uint64_t rm[4], lm[4];
#pragma unroll
      for (int k = 0; k < 4; k++)
      {
        const float4 r = rec[j + k];
        const float2 w = aw[2 * (j + k)];
        r2[k] = (k == 0) ? sep2<PERIODIC, true>(r.x, r.y, r.z, px, py, pz, P)
                         : sep2<PERIODIC, false>(r.x, r.y, r.z, px, py, pz, P);
        m[k] = r.w;
        rm[k] = reached(w.y);
        // (opened by: a cell; near to: a particle)
        lm[k] = __builtin_amdgcn_fcmpf(r2[k], is_cell ? w.x : P.h2, 4 /* ordered < */);
        rinv[k] = __builtin_amdgcn_rsqf(r2[k]);
        count(rm[k], is_cell ? lm[k] : 0ull);
      }
      if (is_cell)
      {
#pragma unroll
        for (int k = 0; k < 4; k++)
        {
          opened[k] = rm[k] & lm[k];
          rm[k] &= ~lm[k];
        }
        fma_neg_on4(rm, blk, m, rinv);
      }
      else if (((rm[0] & lm[0]) | (rm[1] & lm[1]) | (rm[2] & lm[2]) | (rm[3] & lm[3])) == 0ull)
        fma_neg_on4(rm, blk, m, rinv);
      else
      {
#pragma unroll
        for (int k = 0; k < 4; k++)
        {
          fma_neg_on(rm[k] & ~lm[k], blk, m[k], rinv[k]);
          if ((rm[k] & lm[k]) != 0ull)
            near_terms(rm[k] & lm[k], r2[k], rinv[k], m[k]);
        }
      }
    };
    // plain FP32 sums over blocks of at least 16 records, Kahan-compensated
    // across blocks
    auto block_end = [&](int n) {
      nblk += n;
      if (nblk >= 16)
      {
        acc.add(blk);
        blk = 0.f;
        nblk = 0;
      }
    };
    // cells: the open masks go to the slots of records already read (record j's
    // first 8 bytes)
    int j = 0;
    for (; j + 4 <= ncell; j += 4)
    {
      uint64_t o[4];
      if (PERIODIC || small_cells) // (wrapped separations of four at once do not fit the registers)
      {
        o[0] = visit(j, CELL(), XF());
        o[1] = visit(j + 1, CELL(), YF());
        o[2] = visit(j + 2, CELL(), YF());
        o[3] = visit(j + 3, CELL(), YF());
      }
      else
        visit4(j, CELL(), o);
      if (lane == 0)
      {
#pragma unroll
        for (int k = 0; k < 4; k++)
          omw[2 * (j + k)] = make_uint2((uint32_t)o[k], (uint32_t)(o[k] >> 32));
      }
      block_end(4);
    }
    for (; j < ncell; j++)
    {
      const uint64_t o = visit(j, CELL(), XF());
      if (lane == 0)
        omw[2 * j] = make_uint2((uint32_t)o, (uint32_t)(o >> 32));
      block_end(1);
    }
    // particles
    for (; j + 4 <= nb; j += 4)
    {
      if (PERIODIC)
      {
        visit(j, PART(), XF());
        visit(j + 1, PART(), YF());
        visit(j + 2, PART(), YF());
        visit(j + 3, PART(), YF());
      }
      else
        visit4(j, PART(), nullptr);
      block_end(4);
    }
    for (; j < nb; j++)
    {
      visit(j, PART(), XF());
      block_end(1);
    }
    // push the chains' rests and the opened cells' children
    wave_lds_sync();
    // (the popped entries are still in place: nothing is pushed before this point)
    const int4 it = L.stk[src];
    const uint2 om = reinterpret_cast<const uint2 *>(L.rec)[2 * slot];
    const uint64_t msib = __builtin_amdgcn_sicmp(nx, it.y, 40 /* < */) & mine;
    const uint64_t mkid = __builtin_amdgcn_uicmp(om.x | om.y, 0u, 33 /* ne */) & cmask;
    int pos = mask_rank(mkid, mask_rank(msib, top));
    const int pushed = __popcll(msib) + __popcll(mkid);
    if (top + pushed > WSTACK_CAP)
    {
      if (lane == 0 && overflow)
        atomicOr(overflow, WALK_STACK_OVERFLOW);
      break;
    }
    if (nx < it.y && lane < nb)
      L.stk[pos++] = make_int4(nx, it.y, it.z, it.w);
    if ((om.x | om.y) != 0u && slot < ncell)
      L.stk[pos] = make_int4(it.x + 24, nx, (int)om.x, (int)om.y);
    top = uniform(top + pushed);
    wave_lds_sync();
  }
  acc.add(blk);
}

template <bool PERIODIC>
HBTX_DEV float direct_term(const float4 e, float px, float py, float pz, const DevParams &P, bool &near)
{
#pragma clang fp contract(off)
  const float r2 = sep2<PERIODIC, false>(e.x, e.y, e.z, px, py, pz, P);
  const float rinv = __builtin_amdgcn_rsqf(r2);
  float term = -e.w * rinv;
  const bool nr = r2 < P.h2;
  if (wave_mask(nr))
  {
    near = true;
    const float tn = spline_near(r2, rinv, e.w, P.hinv);
    term = nr ? tn : term;
  }
  return term;
}

// Four particle records (64 bytes at an 8-byte aligned unit) in one scalar load.
HBTX_DEV void const_load_4rec(const uint2 *p, float4 r[4])
{
  typedef int v16i __attribute__((ext_vector_type(16)));
  typedef const __attribute__((address_space(4))) v16i c16;
  const v16i a = *(const c16 *)(uintptr_t)p;
#pragma unroll
  for (int k = 0; k < 4; k++)
    r[k] = make_float4(__int_as_float(a[4 * k]), __int_as_float(a[4 * k + 1]), __int_as_float(a[4 * k + 2]),
                       __int_as_float(a[4 * k + 3]));
}

// One group of four records against every lane's target: their terms' sum.
template <bool PERIODIC>
HBTX_DEV float direct_group(const float4 r[4], float px, float py, float pz, const DevParams &P, bool &nr)
{
#pragma clang fp contract(off)
  float part = direct_term<PERIODIC>(r[0], px, py, pz, P, nr);
  part += direct_term<PERIODIC>(r[1], px, py, pz, P, nr);
  part += direct_term<PERIODIC>(r[2], px, py, pz, P, nr);
  part += direct_term<PERIODIC>(r[3], px, py, pz, P, nr);
  return part;
}

// The sums of groups [g0, g1) of a particle record list, in order, to emit(group,
// sum).  The records come through scalar loads, AHEAD groups (64 bytes each) ahead:
// a wave waits for its groups, sends the loads of the next ones and then evaluates
// (scalar loads return in any order, so a wait covers every load in flight: it
// has to come before the next ones go out).  Loading each group just before its use
// left a wave waiting for the L2 once per group.
template <bool PERIODIC, int AHEAD, class Emit>
HBTX_DEV void direct_groups(const uint2 *ent, int g0, int g1, float px, float py, float pz, const DevParams &P,
                            WalkCounts &wc, Emit emit)
{
  if (g0 >= g1)
    return;
  float4 a[AHEAD][4], b[AHEAD][4];
  auto load = [&](int g, float4(&u)[AHEAD][4]) {
#pragma unroll
    for (int k = 0; k < AHEAD; k++)
      const_load_4rec(ent + 8 * (int64_t)min(g + k, g1 - 1), u[k]); // (past the last group: the last again, unused)
  };
  auto arrived = [] {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xc07f); // lgkmcnt(0)
    __builtin_amdgcn_sched_barrier(0);
  };
  auto eval = [&](int g, float4(&u)[AHEAD][4]) {
#pragma unroll
    for (int k = 0; k < AHEAD; k++)
    {
      if (g + k >= g1)
        break;
      bool nr = false;
      emit(g + k, direct_group<PERIODIC>(u[k], px, py, pz, P, nr));
      wc.nnear += nr;
    }
  };
  load(g0, a);
  for (int g = g0; g < g1; g += 2 * AHEAD)
  {
    arrived();
    load(g + AHEAD, b);
    __builtin_amdgcn_sched_barrier(0);
    eval(g, a);
    if (g + AHEAD >= g1)
      break;
    arrived();
    load(g + 2 * AHEAD, a);
    __builtin_amdgcn_sched_barrier(0);
    eval(g + AHEAD, b);
  }
}

// Direct mode: the records are particles only (two units each), summed in
// groups of four, Kahan-compensated across groups.
template <bool PERIODIC>
HBTX_DEV void direct_sum(const uint2 *wt, int ub, int ue, float px, float py, float pz, const DevParams &P,
                         Kahan &acc, WalkCounts &wc)
{
  const uint2 *ent = wt + ub;
  const int ee = (ue - ub) / 2;
  direct_groups<PERIODIC, 1>(ent, 0, ee / 4, px, py, pz, P, wc, [&](int, float part) { acc.add(part); });
  for (int i = ee & ~3; i < ee; i++)
  {
    bool nr = false;
    acc.add(direct_term<PERIODIC>(const_load_f4u(ent + 2 * i), px, py, pz, P, nr));
  }
}

// Snapshot_t::RelativeVelocity in float (src/snapshot.h:135-148)
HBTX_DEV void rel_vel(const DevParams &P, float x0, float x1, float x2, float v0, float v1, float v2,
                      const float *rp, const float *rv, float dv[3])
{
  const float ha = P.hz * P.a;
  float dx[3] = {x0 - rp[0], x1 - rp[1], x2 - rp[2]};
  const float v[3] = {v0, v1, v2};
#pragma unroll
  for (int j = 0; j < 3; j++)
  {
    if (P.periodic)
      dx[j] = nearest_f(dx[j], P.box, P.box_half);
    dv[j] = v[j] - rv[j];
    dv[j] += ha * dx[j];
  }
}

template <bool PERIODIC, bool STATS>
__global__ __launch_bounds__(WALK_WG_THREADS, 8) void k_walk_energy(WalkArgs A)
{
  const DevParams &P = A.P;
  const int lane = lane_id();
  __shared__ WalkLds wls[HBTX_WALK_WG_WAVES];
  WalkLds &wl = wls[threadIdx.x / HBTX_WAVE];
  unsigned long long st_steps = 0, st_visits = 0, st_accepts = 0, st_pairs = 0, st_targets = 0, st_items = 0,
                     st_near = 0;
  ItemQueue queue;
  queue.init(A.counter, A.nchunks, *A.nitems);
  for (;;)
  {
    const int it = queue.next();
    if (it < 0)
      break;
    const int2 item = A.items[it];
    const int s = uniform(item.x);
    const int t = item.y + lane;
    const int nt = A.ntgt[s];
    const bool valid = t < nt;
    const int q = A.off[s] + t; // the target's slot
    const int p = valid ? A.cur[q] : 0;
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
    if (valid)
      x = A.posm[p];
    const int eb = uniform(A.ent_begin[s]), ee = uniform(A.ent_end[s]); // walk-record units
    Kahan acc;
    acc.init();
    WalkCounts wc = {0u, 0u, 0u, 0u};
    if (eb < ee)
    {
      if (A.treemode[s])
      {
        if (PERIODIC && cube_may_wrap(A.cube + 4 * (int64_t)s, valid, x.x, x.y, x.z, P))
          tree_walk_stack<PERIODIC, STATS>(A.wt, eb, ee, valid, x.x, x.y, x.z, P, acc, wc, wl, A.overflow);
        else
          tree_walk_stack<false, STATS>(A.wt, eb, ee, valid, x.x, x.y, x.z, P, acc, wc, wl, A.overflow);
      }
      else
      {
        if (PERIODIC && records_may_wrap(A.wt + eb, lane, HBTX_WAVE, (ee - eb) / 2, valid, x.x, x.y, x.z, P))
          direct_sum<PERIODIC>(A.wt, eb, ee, x.x, x.y, x.z, P, acc, wc);
        else
          direct_sum<false>(A.wt, eb, ee, x.x, x.y, x.z, P, acc, wc);
        if (STATS)
          st_pairs += (unsigned long long)__popcll(wave_mask(valid)) * (unsigned long long)((ee - eb) / 2);
      }
    }
    if (STATS)
    {
      st_steps += wc.steps;
      st_visits += wc.visits;
      st_accepts += wc.accepts;
      st_near += wc.nnear;
      st_targets += __popcll(wave_mask(valid));
      st_items += 1;
    }
    if (!valid)
      continue;
    const int md = A.mode[s];
    const float self = (md == MODE_FULL || md == MODE_REFINE || md == MODE_ADD) ? (A.selfm[p] / P.eps) : 0.f;
    const double phi = ((double)self + (double)acc.s - (double)acc.c) * P.G_over_a;
    const float4 v = A.velu[p];
    const float *rf = A.ref + 6 * s;
    if (md == MODE_FULL || md == MODE_REFINE)
    {
      float dv[3];
      rel_vel(P, x.x, x.y, x.z, v.x, v.y, v.z, rf, rf + 3, dv);
      const float k2 = dv[0] * dv[0] + dv[1] * dv[1] + dv[2] * dv[2];
      float E = (float)((double)k2 * 0.5 + phi);
      if (md == MODE_REFINE)
        A.eref[p] = E; // RefineBindingEnergyOrder: BindingEnergy with the true mass, no thermal term
      else
      {
        if (P.thermal)
          E += v.w;
        A.energy[p] = E;
        A.esl[q] = E;
      }
    }
    else if (md == MODE_ADD)
    {
      // potential of the bound particles from outside the proposal
      const float E = (float)((double)A.energy[p] + phi);
      A.energy[p] = E;
      A.esl[q] = E;
    }
    else
    {
      const float *of = A.oldref + 6 * s;
      float dV[3], ov[3];
      rel_vel(P, of[0], of[1], of[2], of[3], of[4], of[5], rf, rf + 3, dV);
      const float dK = (float)(0.5 * (double)(dV[0] * dV[0] + dV[1] * dV[1] + dV[2] * dV[2]));
      rel_vel(P, x.x, x.y, x.z, v.x, v.y, v.z, of, of + 3, ov);
      const float tkin = (ov[0] * dV[0] + ov[1] * dV[1] + ov[2] * dV[2]) + dK;
      const float E = (float)((double)A.energy[p] + ((double)tkin - phi));
      A.energy[p] = E;
      A.esl[q] = E;
    }
  }
  if (STATS && A.stats && lane == 0)
  {
    atomicAdd(A.stats + STAT_TREE_STEPS, st_steps);
    atomicAdd(A.stats + STAT_TREE_VISITS, st_visits);
    atomicAdd(A.stats + STAT_TREE_ACCEPT, st_accepts);
    atomicAdd(A.stats + STAT_DIRECT_PAIRS, st_pairs);
    atomicAdd(A.stats + STAT_TARGETS, st_targets);
    atomicAdd(A.stats + STAT_ITEMS, st_items);
    atomicAdd(A.stats + STAT_NEAR, st_near);
  }
}

} // namespace hbtx
