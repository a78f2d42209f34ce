// hbtx runtime: device buffers, the round pipeline, and the C-ABI entry points
// declared in include/hbtx.h.  All kernels live in the headers included below
// and are launched on the context's stream.
#include "hbtx.h"

#include "common.h"
#include "scan.h"
#include "sort.h"
#include "tree.h"
#include "walk.h"
#include "unbind.h"
#include "points.h"
#include "subsample.h"
#include "learn.h"
#include "tiles.h"
#include "lists.h"
#include "profile.h"
#include "reassign.h"
#include "load.h"
#include "transfer.h"

#define WALK_MAX_CHUNKS 16
#define WALK_COUNTERS ((WALK_MAX_CHUNKS + 1) * QUEUE_STRIDE) // ints
#define POINT_CHUNKS 8 // chunks of a point walk's items (one per XCD)
#define POINT_COUNTERS ((POINT_CHUNKS + 1) * QUEUE_STRIDE)
// entries whose walk records (at most 3 units each) keep unit offsets in int32
#define WREC_MAX_ENTRIES ((int64_t)0x7ffffff0 / 3 - 8)

#include <algorithm>
#include <atomic>
#include <cmath>
#include <dlfcn.h>
#include <fstream>
#include <sstream>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <numeric>
#include <stdexcept>
#include <string>
#include <vector>

using namespace hbtx;

namespace
{

struct Error : public std::runtime_error
{
  int code;
  Error(int c, const std::string &m) : std::runtime_error(m), code(c) {}
};

#define HIPCHK(x)                                                                                                    \
  do                                                                                                                 \
  {                                                                                                                  \
    hipError_t e_ = (x);                                                                                             \
    if (e_ != hipSuccess)                                                                                            \
      throw Error(HBTX_E_HIP, std::string(#x) + ": " + hipGetErrorString(e_) + " (" + __FILE__ + ":" +            \
                                  std::to_string(__LINE__) + ")");                                                   \
  } while (0)

#define REQUIRE(cond, code, msg)                                                                                     \
  do                                                                                                                 \
  {                                                                                                                  \
    if (!(cond))                                                                                                     \
      throw Error(code, msg);                                                                                        \
  } while (0)

// The array of hbtx_direct_potential_noalloc: packed source records, packed
// targets and the work counter, HBTX_NOALLOC_MAX_POINTS of each.  Every GPU holds
// its own copy at its own address until the process ends; all calls on one GPU
// share it (calls that overlap on one GPU race).
constexpr size_t kScratchTgt = 16 * (size_t)HBTX_NOALLOC_MAX_POINTS;
constexpr size_t kScratchCtr = 32 * (size_t)HBTX_NOALLOC_MAX_POINTS;
constexpr size_t kScratchBytes = kScratchCtr + 256;
__device__ __align__(256) unsigned char scratch[kScratchBytes];

// Device address of `scratch` on the current device, looked up once per device
// (host code never uses the array's name as an address).
void *scratch_address(int device)
{
  static std::mutex mu;
  static void *addr[256] = {};
  REQUIRE(device >= 0 && device < 256, HBTX_E_INVALID, "device index beyond 255");
  std::lock_guard<std::mutex> lock(mu);
  if (!addr[device])
  {
    void *p = nullptr;
    HIPCHK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    REQUIRE(p != nullptr, HBTX_E_HIP, "no device address for the scratch array");
    addr[device] = p;
  }
  return addr[device];
}

// Advanced by every device allocation and release: kernels captured in a graph
// hold buffer addresses, so a graph is valid only for the generation it was
// captured in.
std::atomic<uint64_t> g_alloc_gen{0};
std::atomic<int64_t> g_device_bytes{0}; // device memory the library's buffers hold, all contexts

template <class T>
struct DArr
{
  T *p = nullptr;
  size_t n = 0;
  void alloc(size_t count)
  {
    if (p && count <= n)
      return;
    release();
    g_alloc_gen++;
    size_t bytes = std::max<size_t>(count, 1) * sizeof(T);
    hipError_t e = hipMalloc((void **)&p, (bytes + 15) & ~(size_t)15); // (small transfers move whole words)
    if (e != hipSuccess)
    {
      p = nullptr;
      n = 0;
      throw Error(HBTX_E_ALLOC, "hipMalloc of " + std::to_string(bytes) + " bytes failed: " + hipGetErrorString(e));
    }
    n = count;
    g_device_bytes += (int64_t)bytes;
  }
  void release()
  {
    if (p)
    {
      (void)hipFree(p);
      g_alloc_gen++;
      g_device_bytes -= (int64_t)(std::max<size_t>(n, 1) * sizeof(T));
    }
    p = nullptr;
    n = 0;
  }
  ~DArr()
  {
    release();
  }
  DArr() = default;
  void swap(DArr &o)
  {
    std::swap(p, o.p);
    std::swap(n, o.n);
  }
  DArr(const DArr &) = delete;
  DArr &operator=(const DArr &) = delete;
};

inline int blocks_for(int64_t n, int threads = 256, int cap = 16384)
{
  int64_t b = (n + threads - 1) / threads;
  return (int)std::max<int64_t>(1, std::min<int64_t>(b, cap));
}

} // namespace

// ---------------------------------------------------------------------------
// Batch state
// ---------------------------------------------------------------------------
struct Batch
{
  int64_t n = 0;
  int32_t nsub = 0;
  int32_t max_count = 0;
  bool has_type = false;
  bool has_u = false;
  bool has_proposal = false;
  bool has_id = false;
  std::vector<int64_t> h_off;
  std::vector<int32_t> h_count;
  // particles
  DArr<float4> posm, velu;
  DArr<int8_t> ptype;
  DArr<int64_t> ids;     // particle ids (has_id), else a particle's id is its index in its subhalo
  DArr<char> raw;        // the upload, where the walk records' buffer is too small for it
  DArr<int32_t> load_bad;
  DArr<int32_t> sub_of, sub_zero, off, off_pairs, order, order_zero;
  DArr<int32_t> state, cur, cur2, src, src_sub, fvals, ford;
  DArr<float> energy, esl, selfm, fenergy, fpot, eref;
  DArr<uint8_t> proposal;
  DArr<int32_t> flag, crank, cnt, cscan;
  DArr<int64_t> flag64;
  DArr<uint64_t> keys;
  DArr<float4> ent;      // per entry (x, y, z, m): ent_cap + 1
  DArr<int32_t> eskip;   // per cell entry: skip
  DArr<int8_t> ent_depth;
  DArr<uint2> wt;        // walk records: 3 ent_cap + 4 units of 8 bytes
  DArr<int32_t> cell_u;  // per entry index: walk-record unit of a cell
  int32_t ent_cap = 0;
  int64_t ent_bound = 0; // entries of the largest trees the batch's subhaloes can make
  DArr<int2> items;
  DArr<int32_t> icnt, iscan;
  // subhaloes
  DArr<int32_t> status, corr, iters, mode, treemode, nlast, nbound, nrem, nuns, ntgt, nsrc, src_off, ent_begin,
    ent_end, nitems, bnd_cnt, bnd_tr, first_idx, seg_begin, seg_len, type_cnt, first_tracer, aux32;
  DArr<float> mlast, mbound, ref, oldref, mb, upscale, ref_in, mb_in, minit;
  DArr<int32_t> warm, npro, nadd, reset_;
  DArr<float> feat, logit;
  // 32-particle groups of the subhaloes of at least egroups_min particles (-1: none built)
  DArr<int32_t> egroups;
  int64_t egroups_n = 0, egroups_min = -1;
  bool feat_full = false;  // feat holds every particle's features (hbtx_batch_features)
  // active-slot tiles of the current round and their prefix sums
  DArr<int4> stiles;
  DArr<int32_t> stile_n, stile_off, tsum32, tpre32, sub_first32;
  DArr<int64_t> tsum64, tpre64, sub_total64;
  // previous snapshot's outputs for the learned warm start (same slot = same particle)
  DArr<int32_t> prev_rank;
  DArr<uint8_t> prev_bound;
  DArr<float> prev_energy, prev_com, prev_mb, prev_rs;
  bool has_prev = false;
  DArr<double> cube, len0, red, red2;
  DArr<uint32_t> bbox;
  DArr<int32_t> misc; // [0] active, [1] (unused), [2] overflow, [3] entry total, [4] max depth
  DArr<int32_t> wctr; // walk work counters
  int small_loads = 0; // loads in a row that the entry buffers are far too large for
  DArr<char2> lev;                // per dense source: the level pair of its tree
  DArr<int32_t> mom_slots;        // moment passes: per window / group, the cells that end beyond it
  DArr<hbtx_sub_result> dres;
  DArr<float> prof_r, prof_m; // profiles: sorted radii and cumulative masses
  DArr<hbtx_sub_profile> dprof;
  bool ran = false;
};

struct View
{
  int64_t n;
  int32_t nsub;
  int32_t max_count; // particles of the largest subhalo
  int64_t ent_bound; // entries of the largest trees its subhaloes can make
  SubArrays S;
  PartArrays Q;
  const int32_t *order;
  const int64_t *ids; // null: a particle's id is its index in its subhalo
  int64_t p0; // first particle of the view in the batch
  int32_t s0; // first subhalo of the view
  int32_t *ford;
  float *fenergy, *fpot;
  int32_t *fvals;
  hbtx_sub_result *dres;
  double *red, *red2;
  int32_t *type_cnt, *first_tracer;
};

struct TreeBufs
{
  DArr<float4> ent;
  DArr<int32_t> eskip;
  DArr<int8_t> ent_depth;
  DArr<uint2> wt; // walk records of the tree
  DArr<int32_t> src_of_entry;
  DArr<double> cube;
  size_t bytes() const
  {
    return ent.n * sizeof(float4) + (eskip.n + src_of_entry.n) * sizeof(int32_t) + ent_depth.n + wt.n * sizeof(uint2) +
           cube.n * sizeof(double);
  }
  void swap(TreeBufs &o)
  {
    ent.swap(o.ent);
    eskip.swap(o.eskip);
    ent_depth.swap(o.ent_depth);
    wt.swap(o.wt);
    src_of_entry.swap(o.src_of_entry);
    cube.swap(o.cube);
  }
};

// The buffers of the last tree freed, for a context's next one: a program that builds a
// tree, uses it and frees it spent 0.7 ms of a tree of 2e6 giving the buffers back and 0.3
// getting them again (a free above some 100 MB unmaps).  One tree's, TREE_SPARE_MAX bytes
// at most, given back with the context; a tree may be freed by any thread and after its
// context.  Nothing is in flight on a freed tree: the calls that read one wait for
// their results.
#define TREE_SPARE_MAX ((size_t)512 << 20)
struct TreeSpare
{
  std::mutex mu;
  bool open = true;
  TreeBufs bufs;

  void take(TreeBufs &to)
  {
    std::lock_guard<std::mutex> lock(mu);
    to.swap(bufs);
  }
  void give(TreeBufs &from)
  {
    if (from.bytes() > TREE_SPARE_MAX)
      return;
    std::lock_guard<std::mutex> lock(mu);
    if (open && from.bytes() > bufs.bytes())
      bufs.swap(from);
  }
  void close()
  {
    TreeBufs drop; // (freed after the lock)
    std::lock_guard<std::mutex> lock(mu);
    open = false;
    drop.swap(bufs);
  }
};

struct hbtx_tree : TreeBufs
{
  std::shared_ptr<TreeSpare> spare;
  int64_t n = 0;
  int32_t ne = 0;
  int64_t ncells = 0;
  DevParams P;
  int32_t nw = 0; // units of the walk records
  int32_t treemode = 1;
  ~hbtx_tree()
  {
    if (spare)
      spare->give(*this);
  }
};

struct hbtx_mlp
{
  DArr<float> master, m, v, wf, grad, partial;
  DArr<uint16_t> wb;
  DArr<double> lossp, loss;
  int64_t step = 0;
};

// What a segmented sort is made of, by its longest segment (seg_sort): each form sorts
// the segments of the ones before it too, none a longer segment.
enum SortForm
{
  SORT_FORM_WAVE,  // up to SORT_WAVE_MAX
  SORT_FORM_WAVE4, // up to SORT_WAVE4_MAX
  SORT_FORM_SMALL, // up to SORT_SMALL_MAX
  SORT_FORM_BLOCK, // up to SORT_BLOCK_MAX
  SORT_FORM_TILED
};
inline SortForm sort_form(int64_t max_len)
{
  return max_len <= SORT_WAVE_MAX    ? SORT_FORM_WAVE
         : max_len <= SORT_WAVE4_MAX ? SORT_FORM_WAVE4
         : max_len <= SORT_SMALL_MAX ? SORT_FORM_SMALL
         : max_len <= SORT_BLOCK_MAX ? SORT_FORM_BLOCK
                                     : SORT_FORM_TILED;
}

// What a captured round graph depends on besides buffer addresses: all that the host
// decides launches and arguments from.  (Buffers stay from load to load, so a batch of
// other subhaloes may meet the graphs of the one before.)
struct GraphKey
{
  uint64_t gen = ~0ull;
  int64_t p0 = -1, n = -1;
  int32_t s0 = -1, nsub = -1;
  int32_t sort = -1; // form of the source sort (SortForm of the largest subhalo)
  const void *ptype = nullptr, *proposal = nullptr;
  int32_t ent_cap = -1;
  DevParams P;
  bool operator==(const GraphKey &o) const
  {
    return gen == o.gen && p0 == o.p0 && n == o.n && s0 == o.s0 && nsub == o.nsub && sort == o.sort &&
           ptype == o.ptype && proposal == o.proposal && ent_cap == o.ent_cap && std::memcmp(&P, &o.P, sizeof(P)) == 0;
  }
};

// Workspaces of the calls that take host arrays, reused across calls.  Up to WS_KEEP_MAX
// bytes together they stay (20 million targets of a tree, 30 million samples of the
// classifier); a call that needed more gives them all back when it ends (WsUse).
#define WS_KEEP_MAX ((size_t)1 << 30)
struct Workspaces
{
  DArr<float> raw; // the arrays as uploaded
  DArr<float4> tgt, posm;
  DArr<double> phi;
  DArr<uint64_t> keys;
  DArr<int32_t> vals, seg, counter, off, sub_of, local;
  DArr<hbtx_sub_result> res;
  DArr<float> rc, mc, X;
  DArr<uint8_t> y;
  DArr<hbtx_sub_profile> prof;

  template <class F>
  void each(F &&f)
  {
    f(raw), f(tgt), f(posm), f(phi), f(keys), f(vals), f(seg), f(counter), f(off), f(sub_of), f(local), f(res), f(rc),
      f(mc), f(X), f(y), f(prof);
  }
  void bound()
  {
    size_t bytes = 0;
    each([&](auto &a) { bytes += a.n * sizeof(*a.p); });
    if (bytes > WS_KEEP_MAX)
      each([](auto &a) { a.release(); });
  }
};
struct WsUse // of one call
{
  Workspaces &ws;
  ~WsUse()
  {
    ws.bound();
  }
};

struct hbtx_ctx
{
  int device = 0;
  hipStream_t stream = nullptr;
  std::string err;
  int num_cu = 256;
  std::shared_ptr<TreeSpare> tree_spare;
  int walk_chunks = 8;          // item chunks of the walk (one per XCD)
  int64_t direct_cutoff = 1024; // sources at or below use the exact sum when params ask for the tuned value
  int walk_waves = 32;          // resident walk waves per CU (grid of the persistent walk)
  void *scratch = nullptr;      // this device's address of the no-allocation entry point's array
  std::string tune_source = "built-in defaults";
  // scratch
  DArr<int32_t> part32;
  DArr<int64_t> part64;
  DArr<uint64_t> kalt;
  DArr<int32_t> valt, sort_ntile, sort_toff, ghist, gchunk;
  DArr<int4> sort_tiles;
  DArr<int32_t> red_ntile, red_toff;
  DArr<int4> red_tiles;
  DArr<double> red_partial;
  DArr<unsigned long long> stats;
  Staging staging;
  int32_t *round_words = nullptr; // pinned: a round's words for the host
  hipEvent_t ev0 = nullptr, ev1 = nullptr, wev0 = nullptr, wev1 = nullptr;
  int64_t walk_items_hint = INT64_MAX; // work items of the previous round of the running view
  double walk_ms = 0.0;
  bool count_work = false;
  double stage_ms[8] = {0};
  int rounds = 0;
  // round graphs: head (plan, sources, octree, walk items) and tail (partition,
  // decision, frame), replayed around the directly launched walk
  hipGraphExec_t g_head[3] = {nullptr, nullptr, nullptr}, g_tail = nullptr; // head per round level
  GraphKey g_key;
  int graph_rounds = 0, graph_captures = 0;
  int64_t tree_entries = 0, tree_entries_first = 0; // octree entries built, all rounds / first round
  Batch B;
  Workspaces ws;
  // particle reassignment buffers (grow-only, reused across calls)
  struct
  {
    DArr<float> pos, radii;
    DArr<uint8_t> tracer;
    DArr<int32_t> sub, goff, gid, tflag, cnt, loff, qtiles, tval, qval, seg, out, tot;
    DArr<RsGroup> grp;
    DArr<uint32_t> bbox;
    DArr<uint64_t> tkey, qkey;
    DArr<float4> trec, nodes;
    DArr<int64_t> lbase;
    DArr<int4> tiles;
  } rs;
};

namespace
{

// ---------------------------------------------------------------------------
// primitives
// ---------------------------------------------------------------------------
template <class T>
void scan_excl(hbtx_ctx *c, const T *in, T *out, int64_t n, DArr<T> &part, const int32_t *n_dev = nullptr)
{
  if (n <= LIST_ONE_MAX)
  {
    k_scan_one<T><<<1, LIST_THREADS, 0, c->stream>>>(in, out, n, n_dev);
    HIPCHK(hipGetLastError());
    return;
  }
  const int64_t nb = std::max<int64_t>(1, (n + SCAN_TILE - 1) / SCAN_TILE);
  part.alloc(nb);
  k_scan_reduce<T><<<(unsigned)nb, SCAN_THREADS, 0, c->stream>>>(in, n, n_dev, part.p);
  k_scan_partials<T><<<1, SCAN_THREADS, 0, c->stream>>>(part.p, nb);
  k_scan_down<T><<<(unsigned)nb, SCAN_THREADS, 0, c->stream>>>(in, out, n, n_dev, part.p);
  HIPCHK(hipGetLastError());
}

void scan32(hbtx_ctx *c, const int32_t *in, int32_t *out, int64_t n)
{
  scan_excl<int32_t>(c, in, out, n, c->part32);
}
// length min(n_max, *n_dev), known on the device only; out[length] = total
void scan32_dev(hbtx_ctx *c, const int32_t *in, int32_t *out, int64_t n_max, const int32_t *n_dev)
{
  scan_excl<int32_t>(c, in, out, n_max, c->part32, n_dev);
}

// Tiles of `tile` slots over the ranges longer than `over` (lists.h); returns the
// device-side tile count.  begin_out / len_out (may be null) receive the ranges.
template <class R>
const int32_t *list_tiles(hbtx_ctx *c, const R &r, int32_t ns, int tile, int over, bool first, int32_t *ntile,
                          int32_t *toff, int4 *tiles, int32_t *begin_out = nullptr, int32_t *len_out = nullptr)
{
  const int gs = blocks_for(ns, 256, 1 << 24);
  const bool whole = ns <= LIST_THREADS;
  if (ns <= LIST_ONE_MAX)
    k_list_one<<<1, LIST_THREADS, 0, c->stream>>>(r, ns, tile, over, first, ntile, toff, whole ? tiles : nullptr,
                                                  begin_out, len_out);
  else
  {
    k_list_counts<<<gs, 256, 0, c->stream>>>(r, ns, tile, over, ntile, begin_out, len_out);
    scan32(c, ntile, toff, ns);
  }
  if (!whole)
    k_list_tiles<<<gs, 256, 0, c->stream>>>(r, ns, tile, first, ntile, toff, tiles);
  HIPCHK(hipGetLastError());
  return toff + ns;
}

// Radix tiles of a segmented sort over n elements in nseg segments: a segment
// longer than SORT_SMALL_MAX takes ceil(len / SORT_TILE) <= len / SORT_TILE + 1
// tiles, and at most n / (SORT_SMALL_MAX + 1) segments are that long.  (The block sort
// takes one tile a segment, so the same bound holds.)
int64_t sort_tile_bound(int64_t n, int64_t nseg)
{
  return n / SORT_TILE + std::min<int64_t>(nseg, n / (SORT_SMALL_MAX + 1)) + 2;
}

void reserve_sort(hbtx_ctx *c, int64_t n, int32_t nseg)
{
  c->kalt.alloc(n);
  c->valt.alloc(n);
  c->sort_ntile.alloc(nseg + 1);
  c->sort_toff.alloc(nseg + 1);
  const int64_t maxt = sort_tile_bound(n, nseg);
  c->sort_tiles.alloc(maxt);
  c->ghist.alloc(maxt * RADIX_MAX_BINS);
  c->gchunk.alloc(maxt * RADIX_MAX_BINS); // chunk totals and bases, stored at the chunks' head tiles
}

// Sort (keys, vals) within each segment, given by r and written to [seg_begin,
// seg_begin+seg_len) for the passes; keys use the low key_bits bits.
// max_len: no segment is longer (the passes for longer segments are left out).
template <class R>
void seg_sort(hbtx_ctx *c, uint64_t *keys, int32_t *vals, int32_t nseg, const R &r, int32_t *seg_begin,
              int32_t *seg_len, int64_t n_cap, int key_bits, int64_t max_len = INT64_MAX)
{
  reserve_sort(c, n_cap, nseg);
  // Above SORT_SMALL_MAX: a workgroup a segment where no segment is beyond one (a single
  // 12,000: 67 us, against 115 us in 32 launches through the tiled passes), else tiled
  // passes for all of them (with a larger segment's passes to be launched in any case,
  // those of 2,049 to 16,384 ride along: three sorts of 8e6 slots 960 us, and 1,160 with the
  // shorter segments in a workgroup each).
  const SortForm form = sort_form(max_len);
  const bool radix = form == SORT_FORM_TILED, block = form == SORT_FORM_BLOCK;
  if (radix || block)
    list_tiles(c, r, nseg, radix ? SORT_TILE : SORT_BLOCK_MAX, SORT_SMALL_MAX, false, c->sort_ntile.p, c->sort_toff.p,
               c->sort_tiles.p, seg_begin, seg_len);
  else
    k_list_counts<<<blocks_for(nseg, 256, 1 << 24), 256, 0, c->stream>>>(r, nseg, SORT_TILE, SORT_SMALL_MAX,
                                                                         (int32_t *)nullptr, seg_begin, seg_len);
  k_sort_wave<<<std::max(1, std::min((nseg + 3) / 4, 16384)), SORT_THREADS, 0, c->stream>>>(keys, vals, seg_begin,
                                                                                            seg_len, nseg);
  if (form > SORT_FORM_WAVE)
    k_sort_wave4<<<std::max(1, std::min((nseg + 3) / 4, 16384)), SORT_THREADS, 0, c->stream>>>(keys, vals, seg_begin,
                                                                                              seg_len, nseg);
  if (form > SORT_FORM_WAVE4)
    k_sort_small<<<std::max(1, std::min(nseg, 16384)), SORT_THREADS, 0, c->stream>>>(keys, vals, seg_begin, seg_len,
                                                                                      nseg);
  HIPCHK(hipGetLastError());
  const int32_t *ntiles_p = c->sort_toff.p + nseg;
  const int64_t maxt = sort_tile_bound(n_cap, nseg);
  if (block)
    k_sort_block<<<(int)std::min<int64_t>(maxt, c->num_cu), SORT_BLOCK_THREADS, sizeof(SortBlockLds), c->stream>>>(
        keys, vals, c->sort_tiles.p, ntiles_p, key_bits);
  HIPCHK(hipGetLastError());
  if (!radix)
    return;
  const int grid = (int)std::max<int64_t>(1, std::min<int64_t>(maxt, 4 * c->num_cu));
  // an even number of passes leaves the result in place; 9-bit digits where they save passes
  auto even_passes = [&](int rb) {
    const int p = (key_bits + rb - 1) / rb;
    return p + (p & 1);
  };
  const int rb = (even_passes(9) < even_passes(8)) ? 9 : 8;
  const int passes = even_passes(rb);
  for (int pass = 0; pass < passes; pass++)
  {
    const int shift = pass * rb;
    const uint64_t *kin = (pass & 1) ? c->kalt.p : keys;
    const int32_t *vin = (pass & 1) ? c->valt.p : vals;
    uint64_t *kout = (pass & 1) ? keys : c->kalt.p;
    int32_t *vout = (pass & 1) ? vals : c->valt.p;
    if (rb == 9)
    {
      k_radix_hist<9><<<grid, SORT_THREADS, 0, c->stream>>>(kin, c->sort_tiles.p, ntiles_p, shift, c->ghist.p);
      k_radix_chunk_scan<9><<<grid, SORT_THREADS, 0, c->stream>>>(c->sort_tiles.p, ntiles_p, c->sort_toff.p,
                                                                  c->sort_ntile.p, c->ghist.p, c->gchunk.p);
      k_radix_seg_scan<9><<<grid, SORT_THREADS, 0, c->stream>>>(seg_begin, c->sort_tiles.p, ntiles_p,
                                                                c->sort_toff.p, c->sort_ntile.p, c->gchunk.p);
      k_radix_scatter<9><<<grid, SORT_THREADS, 0, c->stream>>>(kin, vin, kout, vout, c->sort_tiles.p, ntiles_p,
                                                               shift, c->ghist.p, c->sort_toff.p, c->gchunk.p);
      continue;
    }
    k_radix_hist<8><<<grid, SORT_THREADS, 0, c->stream>>>(kin, c->sort_tiles.p, ntiles_p, shift, c->ghist.p);
    k_radix_chunk_scan<8><<<grid, SORT_THREADS, 0, c->stream>>>(c->sort_tiles.p, ntiles_p, c->sort_toff.p,
                                                                c->sort_ntile.p, c->ghist.p, c->gchunk.p);
    k_radix_seg_scan<8><<<grid, SORT_THREADS, 0, c->stream>>>(seg_begin, c->sort_tiles.p, ntiles_p, c->sort_toff.p,
                                                              c->sort_ntile.p, c->gchunk.p);
    k_radix_scatter<8><<<grid, SORT_THREADS, 0, c->stream>>>(kin, vin, kout, vout, c->sort_tiles.p, ntiles_p, shift,
                                                          c->ghist.p, c->sort_toff.p, c->gchunk.p);
  }
  HIPCHK(hipGetLastError());
}

// Tiles of RED_TILE slots over the ranges; returns device pointer to tile count.
template <class R>
const int32_t *red_tiles(hbtx_ctx *c, const R &r, int32_t nsub, int64_t n_cap)
{
  c->red_ntile.alloc(nsub + 1);
  c->red_toff.alloc(nsub + 1);
  const int64_t maxt = n_cap / RED_TILE + nsub + 1;
  c->red_tiles.alloc(maxt);
  c->red_partial.alloc(maxt * RED_NV);
  return list_tiles(c, r, nsub, RED_TILE, 0, false, c->red_ntile.p, c->red_toff.p, c->red_tiles.p);
}

int red_grid(hbtx_ctx *c, int64_t n_cap, int32_t nsub)
{
  return (int)std::max<int64_t>(1, std::min<int64_t>(n_cap / RED_TILE + nsub + 1, 8 * c->num_cu));
}

DevParams make_dev_params(const hbtx_params &p);

// Profiles and shapes of the bound sets described by A (positions, final order,
// results): sort by radius, tiled cumulative mass and candidates, per-subhalo
// combination into out (device).
void run_profiles(hbtx_ctx *c, const hbtx_params &prm, ProfArgs &A, int64_t n, int32_t nsub, const int32_t *sub_of,
                  int32_t *seg_begin, int32_t *seg_len, uint64_t *keys, int32_t *vals, hbtx_sub_profile *out,
                  int64_t max_len)
{
  hbtx_params p = prm;
  if (p.direct_cutoff < 0)
    p.direct_cutoff = c->direct_cutoff;
  A.P = make_dev_params(p);
  A.keys = keys;
  A.vals = vals;
  // as the reference types them: G, a, H and the factor 200 are floats (src/snapshot.cpp:268-269)
  const float G = (float)p.G, a = p.scale_factor;
  A.rho = (float)((double)(200.f * p.hz * p.hz) / 2.0 / (double)G * (double)a * (double)a * (double)a);
  A.vel_unit = G / a;
  hipStream_t st = c->stream;
  const int gs = blocks_for(nsub, 256, 1 << 20);
  const RangeArray ranges{seg_begin, seg_len};
  k_prof_segments<<<gs, 256, 0, st>>>(nsub, A.off, A.res, seg_begin, seg_len);
  k_prof_keys<<<blocks_for(n), 256, 0, st>>>(A, n, sub_of, keys, vals);
  seg_sort(c, keys, vals, nsub, ranges, seg_begin, seg_len, n, 32, max_len);
  const int32_t *nt = red_tiles(c, ranges, nsub, n);
  A.part = c->red_partial.p;
  const int rg = red_grid(c, n, nsub);
  k_prof_tile_sum<<<rg, RED_THREADS, 0, st>>>(A, c->red_tiles.p, nt);
  k_prof_tile_prefix<<<gs, 256, 0, st>>>(nsub, c->red_toff.p, c->red_ntile.p, c->red_partial.p);
  k_prof_tile_main<HBTX_WAVE><<<4 * rg, HBTX_WAVE, 0, st>>>(A, c->red_tiles.p, nt);
  k_prof_tile_main<RED_THREADS><<<rg, RED_THREADS, 0, st>>>(A, c->red_tiles.p, nt);
  k_prof_finish<<<gs, 256, 0, st>>>(A, nsub, c->red_toff.p, c->red_ntile.p, out);
  HIPCHK(hipGetLastError());
}

DevParams make_dev_params(const hbtx_params &p)
{
  REQUIRE(p.scale_factor > 0.f, HBTX_E_INVALID, "scale_factor must be positive");
  REQUIRE(p.softening > 0.f, HBTX_E_INVALID, "softening must be positive");
  REQUIRE(p.theta >= 0.f, HBTX_E_INVALID, "theta must be non-negative");
  REQUIRE(!p.periodic || p.box_size > 0.f, HBTX_E_INVALID, "box_size must be positive when periodic");
  DevParams P;
  std::memset(&P, 0, sizeof(P));
  const float eps = (p.max_phys_softening == -1.f) ? p.softening
                                                   : std::min(p.softening, p.max_phys_softening / p.scale_factor);
  P.G_over_a = p.G / (double)p.scale_factor;
  const float res = p.softening * 0.1f;
  P.res = res;
  P.eps = eps;
  P.h = (float)(2.8 * (double)eps);
  P.hinv = (float)(1.0 / (2.8 * (double)eps));
  P.h2 = P.h * P.h;
  P.theta2 = p.theta * p.theta;
  P.a = p.scale_factor;
  P.hz = p.hz;
  P.box = p.box_size;
  P.box_half = p.box_size / 2.f;
  P.prec = p.bound_mass_precision;
  P.core_factor = p.sub_core_size_factor;
  P.refine_frac = p.bound_fraction_center_refinement;
  P.periodic = p.periodic;
  P.thermal = p.dm_only ? 0 : p.thermal;
  P.dm_only = p.dm_only;
  P.tracer_mask = p.tracer_mask;
  P.donot_mask = p.donot_subsample_mask;
  P.per_type = p.upscale_per_type;
  P.refine = (p.max_sample_size > 0 && p.refine_most_bound) ? 1 : 0;
  P.mss = p.max_sample_size;
  P.min_part = p.min_num_part;
  P.min_tracer = p.min_num_tracer;
  P.core_min = p.sub_core_size_min;
  P.direct_cutoff = p.direct_cutoff;
  return P;
}

// default direct/tree cutoff when the caller asks for the tuned value
// ---------------------------------------------------------------------------
// Tuning: the direct/tree cutoff and the walk's item chunking.  Defaults are
// replaced by the autotuner's file (HBTX_TUNE_FILE, else hbtx_tune.json next to
// this library; written by hbt-herons_amd/autotune.py on the target GPU), then
// by the environment (HBTX_DIRECT_CUTOFF, HBTX_WALK_CHUNKS), then by
// hbtx_set_tuning.
// ---------------------------------------------------------------------------
bool json_int(const std::string &txt, const char *name, int64_t &out)
{
  const std::string key = std::string("\"") + name + "\"";
  const size_t k = txt.find(key);
  if (k == std::string::npos)
    return false;
  const size_t c = txt.find(':', k + key.size());
  if (c == std::string::npos)
    return false;
  char *end = nullptr;
  const long long v = strtoll(txt.c_str() + c + 1, &end, 10);
  if (end == txt.c_str() + c + 1)
    return false;
  out = v;
  return true;
}

std::string tune_file_path()
{
  if (const char *e = getenv("HBTX_TUNE_FILE"))
    return e;
  Dl_info info;
  if (dladdr((void *)&tune_file_path, &info) && info.dli_fname)
  {
    std::string lib = info.dli_fname;
    const size_t slash = lib.find_last_of('/');
    return (slash == std::string::npos ? std::string(".") : lib.substr(0, slash)) + "/hbtx_tune.json";
  }
  return "hbtx_tune.json";
}

// Most entries an octree over n sources can have: n particles, and at each of
// the key's depths 0..HBTX_KEY_LEVELS at most min(8^depth, n/2) cells (a cell
// holds >= 2 sources, and the cells of one depth are disjoint).  Every source
// set of a subhalo is a subset of its particles.
int64_t entry_bound(int64_t n)
{
  int64_t e = n, w = 1;
  if (n < 2)
    return e;
  int l = 0;
  for (; l <= HBTX_KEY_LEVELS && w < n / 2; l++, w *= 8)
    e += w;
  return e + (HBTX_KEY_LEVELS + 1 - l) * (n / 2);
}

void grow_entries(Batch &B, int64_t need, bool slack);

// Entry buffers (49 bytes an entry, some ten entries a particle where rounds are
// replayed) serve the batches that follow: made anew at each load they cost a program of
// large batches gigabytes of allocations and frees a call.  They are given back once ENTRY_SMALL_LOADS loads in
// a row could do with an eighth of them, so that a small batch between large ones does
// not cost the large ones theirs.
#define ENTRY_SMALL_LOADS 16
#define ENTRY_KEEP ((size_t)1 << 20) // entries that are kept in any case
void bound_entries(Batch &B)
{
  const size_t need = (size_t)std::max<int64_t>(3 * B.n + 64, B.ent_bound);
  const bool small = B.ent.n > ENTRY_KEEP && B.ent.n / 8 > need;
  B.small_loads = small ? B.small_loads + 1 : 0;
  if (B.small_loads < ENTRY_SMALL_LOADS)
    return;
  B.small_loads = 0;
  B.ent.release();
  B.eskip.release();
  B.ent_depth.release();
  B.wt.release();
  B.cell_u.release();
}

void batch_reserve(hbtx_ctx *c, Batch &B)
{
  const int64_t n = B.n;
  const int32_t ns = B.nsub;
  B.posm.alloc(n);
  B.velu.alloc(n);
  B.ptype.alloc(n);
  if (B.has_id)
    B.ids.alloc(n);
  B.load_bad.alloc(1);
  B.sub_of.alloc(n);
  B.sub_zero.alloc(std::max<int64_t>(B.max_count, 1));
  B.off.alloc(ns + 1);
  B.off_pairs.alloc(2 * (int64_t)ns + 2);
  B.order.alloc(ns + 1);
  B.order_zero.alloc(1);
  B.state.alloc(n);
  B.cur.alloc(n);
  B.cur2.alloc(n);
  B.src.alloc(n);
  B.src_sub.alloc(n);
  B.fvals.alloc(n);
  B.ford.alloc(n);
  B.energy.alloc(n);
  B.esl.alloc(n);
  B.selfm.alloc(n);
  B.fenergy.alloc(n);
  B.fpot.alloc(n);
  B.eref.alloc(n);
  B.proposal.alloc(n);
  B.flag.alloc(n + 1);
  B.crank.alloc(n + 1);
  B.cnt.alloc(n + 1);
  B.cscan.alloc(n + 1);
  B.flag64.alloc(n + 1);
  B.keys.alloc(n);
  B.lev.alloc(n + 1);
  bound_entries(B);
  grow_entries(B, std::min<int64_t>(3 * n + 64, WREC_MAX_ENTRIES), false);
  B.items.alloc(n / HBTX_WAVE + ns + 1);
  B.icnt.alloc(ns + 1);
  B.iscan.alloc(ns + 1);
  DArr<int32_t> *i32s[] = {&B.status, &B.corr, &B.iters, &B.mode, &B.treemode, &B.nlast, &B.nbound, &B.nrem,
                           &B.nuns, &B.ntgt, &B.nsrc, &B.src_off, &B.ent_begin, &B.ent_end, &B.nitems, &B.bnd_cnt,
                           &B.bnd_tr, &B.first_idx, &B.seg_begin, &B.seg_len, &B.first_tracer,
                           &B.aux32};
  for (auto *a : i32s)
    a->alloc(ns + 1);
  B.type_cnt.alloc(6 * (int64_t)ns + 6);
  DArr<int32_t> *w3[] = {&B.warm, &B.npro, &B.nadd, &B.reset_};
  for (auto *a : w3)
    a->alloc(ns + 1);
  DArr<float> *f1[] = {&B.mlast, &B.mbound, &B.minit};
  for (auto *a : f1)
    a->alloc(ns + 1);
  DArr<float> *f6[] = {&B.ref, &B.oldref, &B.mb, &B.upscale, &B.ref_in, &B.mb_in};
  for (auto *a : f6)
    a->alloc(6 * (int64_t)ns + 6);
  B.cube.alloc(4 * (int64_t)ns + 4);
  B.len0.alloc(ns + 1);
  B.red.alloc((int64_t)RED_NV * ns + RED_NV);
  B.red2.alloc((int64_t)RED_NV * ns + RED_NV);
  B.bbox.alloc(6 * (int64_t)ns + 6);
  B.misc.alloc(8);
  B.wctr.alloc(WALK_COUNTERS);
  B.dres.alloc(ns + 1);
  c->stats.alloc(NSTATS);
  {
    const int64_t maxt = n / SLOT_TILE + ns + 2;
    B.stiles.alloc(maxt);
    B.stile_n.alloc(ns + 1);
    B.stile_off.alloc(ns + 1);
    B.tsum32.alloc(maxt + 1);
    B.tpre32.alloc(maxt + 1);
    B.tsum64.alloc(maxt + 1);
    B.tpre64.alloc(maxt + 1);
    B.sub_first32.alloc(ns + 1);
    B.sub_total64.alloc(ns + 1);
  }
  reserve_sort(c, n, ns);
}

View make_view(Batch &B, int64_t p0, int64_t n, int32_t s0, int32_t nsub, bool whole)
{
  View V;
  V.n = n;
  V.nsub = nsub;
  V.max_count = whole ? B.max_count : (int32_t)n;
  V.ent_bound = whole ? B.ent_bound : entry_bound(n);
  V.p0 = p0;
  V.s0 = s0;
  SubArrays &S = V.S;
  S.nsub = nsub;
  S.off = whole ? B.off.p : B.off_pairs.p + 2 * s0;
  S.sub_of = whole ? B.sub_of.p : B.sub_zero.p;
  S.status = B.status.p + s0;
  S.corr = B.corr.p + s0;
  S.iters = B.iters.p + s0;
  S.mode = B.mode.p + s0;
  S.treemode = B.treemode.p + s0;
  S.nlast = B.nlast.p + s0;
  S.nbound = B.nbound.p + s0;
  S.nrem = B.nrem.p + s0;
  S.nuns = B.nuns.p + s0;
  S.ntgt = B.ntgt.p + s0;
  S.nsrc = B.nsrc.p + s0;
  S.mlast = B.mlast.p + s0;
  S.mbound = B.mbound.p + s0;
  S.ref = B.ref.p + 6 * s0;
  S.oldref = B.oldref.p + 6 * s0;
  S.mb = B.mb.p + 6 * s0;
  S.upscale = B.upscale.p + 6 * s0;
  S.src_off = B.src_off.p + s0;
  S.ent_begin = B.ent_begin.p + s0;
  S.ent_end = B.ent_end.p + s0;
  S.nitems = B.nitems.p + s0;
  S.cube = B.cube.p + 4 * s0;
  S.len0 = B.len0.p + s0;
  S.bbox = B.bbox.p + 6 * s0;
  S.bnd_cnt = B.bnd_cnt.p + s0;
  S.bnd_tr = B.bnd_tr.p + s0;
  S.first_idx = B.first_idx.p + s0;
  S.active_count = B.misc.p + 0;
  S.max_active_n = B.misc.p + 6;
  S.warm = B.warm.p + s0;
  S.npro = B.npro.p + s0;
  S.nadd = B.nadd.p + s0;
  S.reset = B.reset_.p + s0;
  S.minit = B.minit.p + s0;
  PartArrays &Q = V.Q;
  Q.posm = B.posm.p + p0;
  Q.velu = B.velu.p + p0;
  Q.ptype = B.has_type ? B.ptype.p + p0 : nullptr;
  Q.state = B.state.p + p0;
  Q.energy = B.energy.p + p0;
  Q.esl = B.esl.p + p0;
  Q.selfm = B.selfm.p + p0;
  Q.cur = B.cur.p + p0;
  Q.cur2 = B.cur2.p + p0;
  Q.proposal = B.has_proposal ? B.proposal.p + p0 : nullptr;
  V.order = whole ? B.order.p : B.order_zero.p;
  V.ids = B.has_id ? B.ids.p + p0 : nullptr;
  V.ford = B.ford.p + p0;
  V.fenergy = B.fenergy.p + p0;
  V.fpot = B.fpot.p + p0;
  V.fvals = B.fvals.p + p0;
  V.dres = B.dres.p + s0;
  V.red = B.red.p + (int64_t)RED_NV * s0;
  V.red2 = B.red2.p + (int64_t)RED_NV * s0;
  V.type_cnt = B.type_cnt.p + 6 * s0;
  V.first_tracer = B.first_tracer.p + s0;
  return V;
}

TreeArgs tree_args(Batch &B, View &V, const DevParams &P)
{
  TreeArgs T;
  T.src = B.src.p;
  T.keys = B.keys.p;
  T.src_sub = B.src_sub.p;
  T.src_off = V.S.src_off;
  T.nsrc = V.S.nsrc;
  T.treemode = V.S.treemode;
  T.mode = V.S.mode;
  T.len0 = V.S.len0;
  T.posm = V.Q.posm;
  T.ptype = V.Q.ptype;
  T.upscale = V.S.upscale;
  T.cnt = B.cnt.p;
  T.cscan = B.cscan.p;
  T.s_total = B.tpre32.p + (V.n / SLOT_TILE + V.nsub + 1); // grand total of the source tile scan
  T.ent = B.ent.p;
  T.eskip = B.eskip.p;
  T.ent_depth = B.ent_depth.p;
  T.wt = B.wt.p;
  T.cell_u = B.cell_u.p;
  T.lev = B.lev.p;
  T.cap = B.ent_cap;
  T.overflow = B.misc.p + 2;
  T.P = P;
  return T;
}

void build_sources_tree(hbtx_ctx *c, Batch &B, View &V, const DevParams &P, const int32_t *nt, bool graph,
                        int level, bool tsum_ready);
// device round counter (1 in the first round), advanced by k_round_begin
int32_t *round_ptr(Batch &B)
{
  return B.misc.p + 5;
}

// entry buffers for at least `need` entries (slack: a quarter more, for the next
// rounds); buffers that are large enough already stay
void grow_entries(Batch &B, int64_t need, bool slack)
{
  const int64_t cap = std::min<int64_t>(slack ? need + need / 4 + 64 : need, WREC_MAX_ENTRIES);
  REQUIRE(cap >= need, HBTX_E_CAPACITY, "tree entry count exceeds the walk-record range");
  B.ent.alloc(cap + 1);
  B.eskip.alloc(cap + 1);
  B.ent_depth.alloc((cap + 16) & ~(int64_t)15);
  B.wt.alloc(3 * cap + 4);
  B.cell_u.alloc(cap + 1);
  B.ent_cap = (int32_t)cap;
}

int64_t slot_tile_cap(const View &V)
{
  return V.n / SLOT_TILE + V.nsub + 1; // (tree_args reads the source total at tpre32[this])
}
int tile_grid(hbtx_ctx *c, const View &V)
{
  return (int)std::max<int64_t>(1, std::min<int64_t>(slot_tile_cap(V), 16 * c->num_cu));
}

// Tiles over the slot ranges of the view's active subhaloes (mode set by the
// round's plan); returns the device-side tile count.
const int32_t *build_slot_tiles(hbtx_ctx *c, Batch &B, View &V)
{
  return list_tiles(c, RangeActive{V.S}, V.nsub, SLOT_TILE, 0, true, B.stile_n.p, B.stile_off.p, B.stiles.p);
}

// Sources of the round -> dense list, then (tree-mode subhaloes) the octree.
void round_sources_and_tree(hbtx_ctx *c, Batch &B, View &V, const DevParams &P, bool graph, int level)
{
  hipStream_t st = c->stream;
  const int64_t n = V.n;
  const int gb = blocks_for(n);
  const int gs = blocks_for(V.nsub, 256, 1 << 20);
  const int32_t *nt = build_slot_tiles(c, B, V);
  if (P.mss > 0)
  {
    // candidate ranks in E-list order and the mass upscale factors (:290-391)
    k_mark_candidates<<<gb, 256, 0, st>>>(V.S, V.Q, n, B.flag.p);
    scan32(c, B.flag.p, B.crank.p, n);
    const int32_t *nt = red_tiles(c, RangeUpscale{V.S}, V.nsub, n);
    k_upscale_tiles<<<red_grid(c, n, V.nsub), 256, 0, st>>>(V.S, V.Q, P, c->red_tiles.p, nt, B.crank.p,
                                                            c->red_partial.p);
    k_red_finalize<<<red_finalize_blocks(V.nsub), 256, 0, st>>>(c->red_toff.p, c->red_ntile.p, V.nsub, c->red_partial.p, V.red2);
    k_upscale_finish<<<gs, 256, 0, st>>>(V.S, P, V.red2);
  }
  // (without subsampling the candidate rank is irrelevant: every candidate is a source)
  k_mark_sources<<<tile_grid(c, V), SCAN_THREADS, 0, st>>>(V.S, V.Q, P, B.stiles.p, nt, round_ptr(B),
                                                           P.mss > 0 ? B.crank.p : nullptr, B.flag.p, B.tsum32.p,
                                                           (int32_t)slot_tile_cap(V));
  build_sources_tree(c, B, V, P, nt, graph, level, true);
}

// Flags in B.flag (on the slots of the active tiles) -> dense source list, tree
// cube, keys, sort, octree entries.  tsum_ready: the flag producer already wrote
// the tile totals into B.tsum32.
void build_sources_tree(hbtx_ctx *c, Batch &B, View &V, const DevParams &P, const int32_t *nt, bool graph,
                        int level, bool tsum_ready)
{
  hipStream_t st = c->stream;
  const int64_t n = V.n;
  const int gb = blocks_for(n);
  const int gs = blocks_for(V.nsub, 256, 1 << 20);
  const int64_t maxt = slot_tile_cap(V);
  if (!tsum_ready)
    k_tile_sum<int32_t><<<tile_grid(c, V), SLOT_THREADS, 0, st>>>(B.stiles.p, nt, (int32_t)maxt, B.flag.p,
                                                                  B.tsum32.p);
  scan_excl<int32_t>(c, B.tsum32.p, B.tpre32.p, maxt, c->part32);
  const int32_t *s_total = B.tpre32.p + maxt;
  k_scatter_sources<<<tile_grid(c, V), SLOT_THREADS, 0, st>>>(V.S, B.stiles.p, nt, B.flag.p, B.tpre32.p, B.src.p,
                                                              B.src_sub.p, B.sub_first32.p);
  if (level >= 2)
  {
    // direct sums only: the sources' records, in the dense list's order
    TreeArgs T = tree_args(B, V, P);
    k_sub_src_direct<<<gs, 256, 0, st>>>(V.S, B.sub_first32.p, s_total, B.misc.p + 3);
    k_emit_direct<<<blocks_for(n, 256, 8 * 1024), 256, 0, st>>>(T);
    HIPCHK(hipGetLastError());
    return;
  }
  k_sub_src<<<gs, 256, 0, st>>>(V.S, B.sub_first32.p);
  const int32_t *nbt = red_tiles(c, RangeTreeSrc{V.S}, V.nsub, n);
  k_bbox_tiles<<<red_grid(c, n, V.nsub), 256, 0, st>>>(V.S, V.Q.posm, B.src.p, c->red_tiles.p, nbt);
  k_cube<<<gs, 256, 0, st>>>(V.S);
  k_keys<<<gb, 256, 0, st>>>(V.S, P, V.Q.posm, B.src.p, B.src_sub.p, s_total, B.keys.p);
  seg_sort(c, B.keys.p, B.src.p, V.nsub, RangeTreeSrc{V.S}, B.seg_begin.p, B.seg_len.p, n, 63,
           level >= 1 ? SORT_SMALL_MAX : V.max_count);
  k_targets_from_sources<<<gb, 256, 0, st>>>(V.S, V.Q, B.src.p, B.src_sub.p, s_total);
  TreeArgs T = tree_args(B, V, P);
  k_tree_count<<<blocks_for(n, 256, 8 * 1024), 256, 0, st>>>(T, B.cnt.p);
  scan32_dev(c, B.cnt.p, B.cscan.p, n, s_total);
  if (!graph && B.ent_cap < V.ent_bound)
  {
    // exact entry count and depth of this round's trees; grow the entry buffers if needed
    k_entry_total<<<1, 1, 0, st>>>(s_total, B.cscan.p, B.misc.p + 3, 0x7fffffff, B.misc.p + 2);
    int32_t etot = 0;
    HIPCHK(hipMemcpyAsync(&etot, B.misc.p + 3, sizeof(int32_t), hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    REQUIRE(etot >= 0, HBTX_E_CAPACITY, "tree entry count overflows int32");
    if (etot > B.ent_cap)
    {
      grow_entries(B, etot, true);
      T = tree_args(B, V, P);
    }
  }
  // (buffers that hold the largest trees the view can make need no count; a captured
  // round, which cannot wait for one, always has them)
  k_tree_emit<<<blocks_for(n, EMIT_TILE, 8 * 1024), EMIT_TILE, 0, st>>>(T);
  k_sub_entries<<<gs, 256, 0, st>>>(V.S, B.cscan.p, B.ent_cap, B.misc.p + 2);
  k_entry_total<<<1, 1, 0, st>>>(s_total, B.cscan.p, B.misc.p + 3, B.ent_cap, B.misc.p + 2);
  // moments bottom-up: LDS-staged windows, then one pass per level of window
  // groups (levels sized for the entry capacity; each pass reads the entry total)
  std::vector<int64_t> units{(std::max<int64_t>(B.ent_cap, 1) + MOM_WIN - 1) / MOM_WIN};
  while (units.back() > 1)
    units.push_back((units.back() + MOM_GROUP - 1) / MOM_GROUP);
  int64_t nslots = 0;
  for (int64_t u : units)
    nslots += u;
  B.mom_slots.alloc(nslots * MOM_SLOTS);
  int32_t *sl = B.mom_slots.p;
  k_moments_windows<<<(int)std::min<int64_t>(units[0], 4096), MOM_THREADS, 0, st>>>(T, B.misc.p + 3, sl);
  int64_t span = MOM_WIN;
  for (size_t k = 1; k < units.size(); k++)
  {
    int32_t *up = sl + units[k - 1] * MOM_SLOTS;
    k_moments_groups<<<(int)std::min<int64_t>(units[k], 4096), MOM_GROUP, 0, st>>>(T, B.misc.p + 3, span, sl, up);
    sl = up;
    span *= MOM_GROUP;
  }
  HIPCHK(hipGetLastError());
}

WalkArgs walk_args(hbtx_ctx *c, Batch &B, View &V, const DevParams &P)
{
  WalkArgs W;
  W.items = B.items.p;
  W.nitems = B.iscan.p + V.nsub;
  W.counter = B.wctr.p;
  W.nchunks = c->walk_chunks;
  W.cur = V.Q.cur;
  W.off = V.S.off;
  W.ntgt = V.S.ntgt;
  W.mode = V.S.mode;
  W.treemode = V.S.treemode;
  W.cube = V.S.cube;
  W.ent_begin = V.S.ent_begin;
  W.ent_end = V.S.ent_end;
  W.wt = B.wt.p;
  W.posm = V.Q.posm;
  W.velu = V.Q.velu;
  W.selfm = V.Q.selfm;
  W.ref = V.S.ref;
  W.oldref = V.S.oldref;
  W.energy = V.Q.energy;
  W.esl = V.Q.esl;
  W.eref = B.eref.p + V.p0;
  W.stats = c->stats.p;
  W.overflow = B.misc.p + 2;
  W.P = P;
  return W;
}

// the walk's work items (largest subhaloes first) and its cleared chunk counters
void round_items(hbtx_ctx *c, Batch &B, View &V)
{
  hipStream_t st = c->stream;
  const int gs = blocks_for(V.nsub, 256, 1 << 20);
  int32_t *total = B.misc.p + 7; // read after the round
  if (V.nsub <= LIST_ONE_MAX)
    k_items_one<<<1, LIST_THREADS, 0, st>>>(V.S, V.order, B.iscan.p, B.wctr.p, WALK_COUNTERS, total);
  else
  {
    k_items_count<<<gs, 256, 0, st>>>(V.S, V.order, B.icnt.p);
    scan32(c, B.icnt.p, B.iscan.p, V.nsub);
    k_items_finish<<<1, 256, 0, st>>>(B.iscan.p + V.nsub, B.wctr.p, WALK_COUNTERS, total);
  }
  k_items_emit<<<blocks_for((int64_t)V.nsub * HBTX_WAVE, 256, 1 << 24), 256, 0, st>>>(V.S, V.order, B.iscan.p,
                                                                                       B.items.p);
  HIPCHK(hipGetLastError());
}

// the persistent walk over the round's items, timed by the walk events
void round_walk_launch(hbtx_ctx *c, Batch &B, View &V, const DevParams &P)
{
  hipStream_t st = c->stream;
  WalkArgs W = walk_args(c, B, V, P);
  // (the persistent walk needs no more waves than items; a round has no more
  // items than the round before it, as every subhalo's target count only shrinks)
  const int64_t maxitems = std::min<int64_t>(V.n / HBTX_WAVE + V.nsub + 1, c->walk_items_hint);
  const int waves = (int)std::max<int64_t>(1, std::min<int64_t>(maxitems, (int64_t)c->walk_waves * c->num_cu));
  const int grid = (waves + HBTX_WALK_WG_WAVES - 1) / HBTX_WALK_WG_WAVES;
  HIPCHK(hipEventRecord(c->wev0, st));
  if (P.periodic)
  {
    if (c->count_work)
      k_walk_energy<true, true><<<grid, WALK_WG_THREADS, 0, st>>>(W);
    else
      k_walk_energy<true, false><<<grid, WALK_WG_THREADS, 0, st>>>(W);
  }
  else
  {
    if (c->count_work)
      k_walk_energy<false, true><<<grid, WALK_WG_THREADS, 0, st>>>(W);
    else
      k_walk_energy<false, false><<<grid, WALK_WG_THREADS, 0, st>>>(W);
  }
  HIPCHK(hipEventRecord(c->wev1, st));
  HIPCHK(hipGetLastError());
}

void round_walk(hbtx_ctx *c, Batch &B, View &V, const DevParams &P)
{
  round_items(c, B, V);
  round_walk_launch(c, B, V, P);
}

void round_partition(hbtx_ctx *c, Batch &B, View &V, const DevParams &P, bool warm_round)
{
  hipStream_t st = c->stream;
  const int64_t n = V.n;
  const int gb = blocks_for(n);
  const int gs = blocks_for(V.nsub, 256, 1 << 20);
  // the round's active tiles (built from the plan at the start of the round)
  const int32_t *nt = B.stile_off.p + V.nsub;
  const int tg = tile_grid(c, V);
  if (warm_round)
    k_fill_i32<<<gs, 256, 0, st>>>(B.aux32.p, V.nsub, 0);
  const int64_t maxt = slot_tile_cap(V);
  k_partition_flags<<<tg, SCAN_THREADS, 0, st>>>(V.S, V.Q, P, B.stiles.p, nt, B.flag64.p,
                                                 warm_round ? B.aux32.p : nullptr, B.tsum64.p, (int32_t)maxt);
  scan_excl<int64_t>(c, B.tsum64.p, B.tpre64.p, maxt, c->part64);
  k_partition_scatter<<<tg, SLOT_THREADS, 0, st>>>(V.S, V.Q, B.stiles.p, nt, round_ptr(B), B.flag64.p, B.tpre64.p,
                                                   B.sub_total64.p);
  k_copy_cur<<<tg, 256, 0, st>>>(V.S, V.Q, B.stiles.p, nt, B.sub_total64.p, P.periodic);
  if (P.mss > 0)
  {
    k_fill_i32<<<gs, 256, 0, st>>>(B.aux32.p, V.nsub, 0);
    k_count_unsampled<<<gb, 256, 0, st>>>(V.S, V.Q, P, n, B.aux32.p);
    k_set_unsampled<<<gs, 256, 0, st>>>(V.S, B.aux32.p);
  }
  k_round_decide<<<gs, 256, 0, st>>>(V.S, P, B.sub_total64.p, warm_round ? B.aux32.p : nullptr);
  const int32_t *ntiles = red_tiles(c, RangeCom{V.S}, V.nsub, n);
  k_red_tile<ComOp><<<red_grid(c, n, V.nsub), RED_THREADS, 0, st>>>(V.S, V.Q, P, c->red_tiles.p, ntiles,
                                                                     c->red_partial.p);
  k_red_finalize<<<red_finalize_blocks(V.nsub), 256, 0, st>>>(c->red_toff.p, c->red_ntile.p, V.nsub, c->red_partial.p, V.red);
  k_round_finish<<<gs, 256, 0, st>>>(V.S, P, V.red);
  if (P.periodic)
    k_round_finish_periodic<<<gs, 256, 0, st>>>(V.S, V.Q, P, V.red);
  if (warm_round)
  {
    k_warm_reset_particles<<<gb, 256, 0, st>>>(V.S, V.Q, n);
    k_warm_reset_subs<<<gs, 256, 0, st>>>(V.S, B.ref_in.p + 6 * V.s0);
  }
  HIPCHK(hipGetLastError());
}

__global__ void k_final_local(SubArrays S, int64_t n, const int32_t *vals, const float *energy, int32_t *ford,
                              float *fenergy)
{
  GRID_STRIDE(q, n)
  {
    const int s = S.sub_of[q];
    const int p = vals[q];
    ford[q] = p - S.off[s];
    fenergy[q] = energy[p];
  }
}

__global__ void k_final_sub(SubArrays S, PartArrays Q, DevParams P, const int32_t *vals, const double *kin,
                            const double *core, const int32_t *first_tracer, const float *ref_in,
                            const int64_t *ids, hbtx_sub_result *out)
{
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= S.nsub)
    return;
  hbtx_sub_result R = {};
  const int n = S.off[s + 1] - S.off[s];
  const int st = S.status[s];
  R.iterations = S.iters[s];
  R.mostbound_id = -1;
  const float *mb = S.mb + 6 * s;
  if (n == 0)
  {
    // orphan early exit (src/subhalo_unbind.cpp:472-489): frame unchanged, core = most-bound
    for (int k = 0; k < 3; k++)
    {
      R.com_pos[k] = ref_in[6 * s + k];
      R.com_vel[k] = ref_in[6 * s + 3 + k];
      R.mostbound_pos[k] = mb[k];
      R.mostbound_vel[k] = mb[3 + k];
      R.core_pos[k] = mb[k];
      R.core_vel[k] = mb[3 + k];
    }
    out[s] = R;
    return;
  }
  const float *rf = S.ref + 6 * s;
  for (int k = 0; k < 3; k++)
  {
    R.com_pos[k] = rf[k];
    R.com_vel[k] = rf[3 + k];
  }
  if (st != ST_CONVERGED)
  {
    R.disrupted = 1;
    for (int k = 0; k < 3; k++)
    {
      R.mostbound_pos[k] = mb[k];
      R.mostbound_vel[k] = mb[3 + k];
      R.core_pos[k] = mb[k];
      R.core_vel[k] = mb[3 + k];
    }
    out[s] = R;
    return;
  }
  const int nb = S.nbound[s];
  R.nbound = nb;
  R.mbound = S.mbound[s];
  const int p0 = vals[S.off[s]];
  const float4 x0 = Q.posm[p0];
  const float4 v0 = Q.velu[p0];
  R.mostbound_pos[0] = x0.x;
  R.mostbound_pos[1] = x0.y;
  R.mostbound_pos[2] = x0.z;
  R.mostbound_vel[0] = v0.x;
  R.mostbound_vel[1] = v0.y;
  R.mostbound_vel[2] = v0.z;
  const double *v = kin + (int64_t)RED_NV * s;
  if (nb > 1)
  {
    const double M = v[6];
    double E = v[0] - v[1];
    E /= M;
    double K = v[2] * (0.5 / M);
    R.spec_pot = (float)(E - K);
    R.spec_kin = (float)K;
    R.spec_am[0] = (float)(v[3] / M);
    R.spec_am[1] = (float)(v[4] / M);
    R.spec_am[2] = (float)(v[5] / M);
  }
  if (!P.dm_only)
  {
    for (int k = 0; k < 6; k++)
    {
      R.nbound_type[k] = (int64_t)v[13 + k];
      R.mbound_type[k] = (float)v[7 + k];
    }
    const int ft = first_tracer[s];
    R.tracer_index = (ft == 0x7fffffff) ? 0 : ft;
  }
  else
    R.tracer_index = 0;
  if (nb > 0)
  {
    const int p = vals[S.off[s] + (int)R.tracer_index];
    R.mostbound_id = ids ? ids[p] : (int64_t)(p - S.off[s]);
  }
  const double *c = core + (int64_t)RED_NV * s;
  const double msum = c[0];
  double s2r = 0., s2v = 0.;
  for (int d = 0; d < 3; d++)
  {
    const double pos = c[1 + d] / msum;
    const double pos2 = c[4 + d] / msum - pos * pos;
    const double vel = c[7 + d] / msum;
    const double vel2 = c[10 + d] / msum - vel * vel;
    float cp = (float)pos;
    if (P.periodic)
      cp = (float)(pos + (double)x0.x * (d == 0) + (double)x0.y * (d == 1) + (double)x0.z * (d == 2));
    R.core_pos[d] = cp;
    R.core_vel[d] = (float)vel;
    s2r += pos2;
    s2v += vel2;
  }
  R.core_sigma_r = (float)sqrt(s2r);
  R.core_sigma_v = (float)sqrt(s2v);
  out[s] = R;
}

void run_final(hbtx_ctx *c, Batch &B, View &V, const DevParams &P, bool want_pot, int rounds)
{
  hipStream_t st = c->stream;
  const int64_t n = V.n;
  const int gb = blocks_for(n);
  const int gs = blocks_for(V.nsub, 256, 1 << 20);
  k_final_keys<<<gb, 256, 0, st>>>(V.S, V.Q, n, rounds, B.keys.p, V.fvals);
  int gbits = 0;
  while ((1 << gbits) <= rounds)
    gbits++;
  seg_sort(c, B.keys.p, V.fvals, V.nsub, RangeConverged{V.S}, B.seg_begin.p, B.seg_len.p, n, 32 + gbits, V.max_count);
  if (P.refine)
  {
    // RefineBindingEnergyOrder (:395-425): tree over the most bound particles, true masses
    k_refine_plan<<<gs, 256, 0, st>>>(V.S, P);
    const int32_t *nt = build_slot_tiles(c, B, V);
    k_slot_of<<<gb, 256, 0, st>>>(V.S, n, V.fvals, V.Q.cur2);
    k_mark_refine<<<gb, 256, 0, st>>>(V.S, V.Q, n, V.Q.cur2, B.flag.p);
    build_sources_tree(c, B, V, P, nt, false, 0, false);
    c->walk_items_hint = INT64_MAX; // (other targets than the rounds')
    round_walk(c, B, V, P);
    k_refine_keys<<<gb, 256, 0, st>>>(V.S, n, V.fvals, B.eref.p + V.p0, B.keys.p);
    seg_sort(c, B.keys.p, V.fvals, V.nsub, RangeRefine{V.S}, B.seg_begin.p, B.seg_len.p, n, 32, V.max_count);
  }
  k_final_local<<<gb, 256, 0, st>>>(V.S, n, V.fvals, V.Q.energy, V.ford, V.fenergy);
  // kinematics / types over the bound particles (input order)
  const int32_t *ntiles = red_tiles(c, RangeConverged{V.S}, V.nsub, n);
  if (V.Q.ptype)
    k_final_tile<true><<<red_grid(c, n, V.nsub), RED_THREADS, 0, st>>>(V.S, V.Q, P, c->red_tiles.p, ntiles,
                                                                      c->red_partial.p);
  else
    k_final_tile<false><<<red_grid(c, n, V.nsub), RED_THREADS, 0, st>>>(V.S, V.Q, P, c->red_tiles.p, ntiles,
                                                                       c->red_partial.p);
  k_red_finalize<<<red_finalize_blocks(V.nsub), 256, 0, st>>>(c->red_toff.p, c->red_ntile.p, V.nsub, c->red_partial.p, V.red);
  const int gw = blocks_for((int64_t)V.nsub * HBTX_WAVE, 256, 1 << 24);
  k_first_tracer<<<gw, 256, 0, st>>>(V.S, V.Q, P, V.fvals, V.first_tracer);
  k_core_wave<<<gw, 256, 0, st>>>(V.S, V.Q, P, V.fvals, V.red2);
  k_final_sub<<<gs, 256, 0, st>>>(V.S, V.Q, P, V.fvals, V.red, V.red2, V.first_tracer, B.ref_in.p + 6 * V.s0,
                                  V.ids, V.dres);
  if (want_pot)
    k_potential_energy<<<gb, 256, 0, st>>>(V.S, V.Q, P, n, V.fvals, V.fpot);
  HIPCHK(hipGetLastError());
}

// Iterate one view to convergence. Returns rounds used.
// Per-view state at the start of the unbinding: particles, frames, the initial
// Mbound (:537-541) and the leading do-not-subsample run (:522-524).
void init_view(hbtx_ctx *c, Batch &B, View &V, const DevParams &P, bool warm)
{
  hipStream_t st = c->stream;
  const int gb = blocks_for(V.n);
  const int gs = blocks_for(V.nsub, 256, 1 << 20);
  k_init_particles<<<gb, 256, 0, st>>>(V.S, V.Q, V.n);
  k_init_subs<<<gs, 256, 0, st>>>(V.S, B.ref_in.p + 6 * V.s0, B.mb_in.p + 6 * V.s0, nullptr);
  k_fill_i32<<<1, 64, 0, st>>>(B.misc.p, 8, 0);
  const int32_t *nt = red_tiles(c, RangeAll{V.S}, V.nsub, V.n);
  k_fill_i32<<<gs, 256, 0, st>>>(B.aux32.p, V.nsub, 0x7fffffff);
  k_fill_i32<<<gs, 256, 0, st>>>(V.S.first_idx, V.nsub, 0x7fffffff);
  if (warm && P.periodic)
    k_first_proposed<<<gb, 256, 0, st>>>(V.S, V.Q, V.n);
  if (P.periodic)
    k_init_mass_tiles<true><<<red_grid(c, V.n, V.nsub), 256, 0, st>>>(V.S, V.Q, P, c->red_tiles.p, nt, c->red_partial.p,
                                                                B.aux32.p);
  else
    k_init_mass_tiles<false><<<red_grid(c, V.n, V.nsub), 256, 0, st>>>(V.S, V.Q, P, c->red_tiles.p, nt, c->red_partial.p,
                                                                B.aux32.p);
  k_red_finalize<<<red_finalize_blocks(V.nsub), 256, 0, st>>>(c->red_toff.p, c->red_ntile.p, V.nsub, c->red_partial.p, V.red);
  k_init_mass_finish<<<gs, 256, 0, st>>>(V.S, V.Q, P, V.red, B.aux32.p, warm ? 1 : 0);
  HIPCHK(hipGetLastError());
}

// First part of a round, up to the walk: plan, sources, octrees, work items.
// graph: no host synchronisation (the part is being captured).  level (from the
// largest source count of the round, which the host has from the round before): 0
// any; 1 every subhalo's sources fit the LDS sort (no radix passes); 2 every subhalo
// takes the direct sum (no keys, sorts, cells or moments).
void round_head(hbtx_ctx *c, Batch &B, View &V, const DevParams &P, bool graph, bool warm_round, int level = 0)
{
  hipStream_t st = c->stream;
  const int gs = blocks_for(V.nsub, 256, 1 << 20);
  k_round_begin<<<1, 64, 0, st>>>(V.S.active_count, round_ptr(B), V.S.max_active_n);
  k_plan<<<gs, 256, 0, st>>>(V.S, P, round_ptr(B));
  round_sources_and_tree(c, B, V, P, graph, level);
  if (warm_round && level < 2)
  {
    // warm round: every target, in Hilbert order of its cell in the proposal's tree cube
    k_warm_keys<<<blocks_for(V.n), 256, 0, st>>>(V.S, V.Q, V.n, B.keys.p);
    seg_sort(c, B.keys.p, V.Q.cur, V.nsub, RangeWarm{V.S}, B.seg_begin.p, B.seg_len.p, V.n, 30, V.max_count);
  }
  round_items(c, B, V);
}

void drop_graphs(hbtx_ctx *c)
{
  for (auto &g : c->g_head)
  {
    if (g)
      (void)hipGraphExecDestroy(g);
    g = nullptr;
  }
  if (c->g_tail)
    (void)hipGraphExecDestroy(c->g_tail);
  c->g_tail = nullptr;
  c->g_key = GraphKey();
}

template <class F>
hipGraphExec_t capture(hbtx_ctx *c, F &&record)
{
  hipStream_t st = c->stream;
  HIPCHK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
  try
  {
    record();
  }
  catch (...)
  {
    hipGraph_t g = nullptr;
    (void)hipStreamEndCapture(st, &g);
    if (g)
      (void)hipGraphDestroy(g);
    (void)hipGetLastError();
    throw;
  }
  hipGraph_t g = nullptr;
  HIPCHK(hipStreamEndCapture(st, &g));
  hipGraphExec_t ex = nullptr;
  const hipError_t e = hipGraphInstantiate(&ex, g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  HIPCHK(e);
  return ex;
}

// Round graphs for this view, captured again when a buffer moved or the view or
// the parameters changed.  Capture only records: every buffer the round touches
// already has its size from the first (direct) round.  Returns false (rounds
// then run directly) if the capture could not be made.
bool ensure_round_graphs(hbtx_ctx *c, Batch &B, View &V, const DevParams &P, int level)
{
  GraphKey k;
  k.p0 = V.p0;
  k.n = V.n;
  k.s0 = V.s0;
  k.nsub = V.nsub;
  k.sort = sort_form(V.max_count);
  k.ptype = V.Q.ptype;
  k.proposal = V.Q.proposal;
  k.ent_cap = B.ent_cap;
  k.P = P;
  k.gen = g_alloc_gen.load();
  if (c->g_head[level] && c->g_tail && k == c->g_key)
    return true;
  if (!(k == c->g_key))
    drop_graphs(c);
  try
  {
    c->g_head[level] = capture(c, [&] { round_head(c, B, V, P, true, false, level); });
    if (!c->g_tail)
      c->g_tail = capture(c, [&] { round_partition(c, B, V, P, false); });
  }
  catch (const Error &)
  {
    drop_graphs(c);
    return false;
  }
  if (g_alloc_gen.load() != k.gen)
  {
    drop_graphs(c);
    return false;
  }
  c->g_key = k;
  c->graph_captures++;
  return true;
}

// The overflow word of a round: bit 1 the entry buffers were too small, bit 2 a
// tree's records exceed the walk's int32 byte offsets, bit 4 a walk stack was full
// (not reachable for trees of at most 22 cell levels).
void check_overflow(int32_t ov)
{
  REQUIRE(!(ov & WALK_STACK_OVERFLOW), HBTX_E_CAPACITY, "tree walk stack capacity exceeded");
  REQUIRE(!(ov & 2), HBTX_E_CAPACITY,
          "a subhalo's octree exceeds the walk's 2 GiB record span (int32 byte offsets)");
  REQUIRE(ov == 0, HBTX_E_CAPACITY, "tree entry capacity exceeded");
}

// Iterate one view to convergence. Returns rounds used.  graphs: rounds after
// the first replay the captured head and tail around the walk.
int run_view(hbtx_ctx *c, Batch &B, View &V, const DevParams &P, bool want_pot, bool warm, bool graphs)
{
  hipStream_t st = c->stream;
  if (graphs)
  {
    // replayed rounds need entry buffers for the largest trees the view can make
    if (B.ent_bound > WREC_MAX_ENTRIES)
      graphs = false;
    else if (B.ent_cap < B.ent_bound)
      grow_entries(B, B.ent_bound, false);
  }
  init_view(c, B, V, P, warm);
  c->walk_items_hint = INT64_MAX;
  // (the first round's sources: at most every particle)
  auto level_of = [&](int64_t max_src) { return (max_src <= P.direct_cutoff) ? 2 : (max_src <= SORT_SMALL_MAX ? 1 : 0); };
  int round = 0, level = level_of(V.max_count);
  const int max_rounds = 2000;
  if (!c->round_words)
    HIPCHK(hipHostMalloc((void **)&c->round_words, 8 * sizeof(int32_t), hipHostMallocDefault));
  while (true)
  {
    REQUIRE(round < max_rounds, HBTX_E_INVALID, "unbinding did not converge within the round limit");
    round++;
    const bool replay = graphs && round >= 2 && ensure_round_graphs(c, B, V, P, level);
    if (replay)
    {
      HIPCHK(hipGraphLaunch(c->g_head[level], st));
      round_walk_launch(c, B, V, P);
      HIPCHK(hipGraphLaunch(c->g_tail, st));
      c->graph_rounds++;
    }
    else
    {
      round_head(c, B, V, P, false, warm && round == 1, level);
      round_walk_launch(c, B, V, P);
      round_partition(c, B, V, P, warm && round == 1);
    }
    // the round's words straight into pinned host memory (a copy of 32 bytes costs more
    // than the wait itself)
    k_publish<<<1, 64, 0, st>>>(B.misc.p, c->round_words, 8);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(st));
    const int32_t *h_misc = c->round_words;
    float wms = 0.f;
    HIPCHK(hipEventElapsedTime(&wms, c->wev0, c->wev1));
    c->walk_ms += wms;
    c->walk_items_hint = std::max(h_misc[7], 1);
    c->tree_entries += h_misc[3];
    if (round == 1)
      c->tree_entries_first += h_misc[3];
    level = level_of(h_misc[6]);
    check_overflow(h_misc[2]);
    if (h_misc[0] == 0)
      break;
  }
  run_final(c, B, V, P, want_pot, round);
  return round;
}

// The batch layout limits, checked before anything touches the device:
// particle slots and subhalo indices are int32, and the walk addresses one
// subhalo's records by int32 byte offsets, so a subhalo's tree (16 bytes a
// particle, 24 a cell) must stay below 2 GiB.  Particles alone fix the bound
// below; the cells are counted on the device once the tree exists (the span
// check of k_sub_entries).
void check_layout(int64_t n, int64_t nsub, const int64_t *offsets)
{
  REQUIRE(n >= 0 && nsub >= 1, HBTX_E_INVALID, "need n >= 0 and nsub >= 1");
  REQUIRE(n < (int64_t)0x20000000, HBTX_E_INVALID, "at most 2^29 particles per batch");
  REQUIRE(nsub < (int64_t)0x7fffffff, HBTX_E_INVALID, "too many subhaloes");
  REQUIRE(offsets, HBTX_E_INVALID, "null offsets");
  REQUIRE(offsets[0] == 0 && offsets[nsub] == n, HBTX_E_INVALID, "offsets must start at 0 and end at n");
  for (int64_t s = 0; s < nsub; s++)
  {
    REQUIRE(offsets[s + 1] >= offsets[s], HBTX_E_INVALID, "offsets must be non-decreasing");
    REQUIRE(offsets[s + 1] - offsets[s] <= HBTX_MAX_SUBHALO_PARTICLES, HBTX_E_CAPACITY,
            "subhalo " + std::to_string(s) + " has " + std::to_string(offsets[s + 1] - offsets[s]) +
              " particles: its octree would exceed the walk's 2 GiB record span (at most " +
              std::to_string((long long)HBTX_MAX_SUBHALO_PARTICLES) + " particles per subhalo)");
  }
}

// Subhaloes by particle count, largest first, equal counts in input order (three
// counting passes over the 27 bits of a count).
void size_order(const std::vector<int32_t> &count, std::vector<int32_t> &order)
{
  const size_t n = count.size();
  std::vector<int32_t> tmp(n);
  order.resize(n);
  std::iota(order.begin(), order.end(), 0);
  for (int pass = 0; pass < 3; pass++)
  {
    auto digit = [&](int32_t s) { return 511 - ((count[s] >> (9 * pass)) & 511); };
    size_t start[513] = {0};
    for (size_t i = 0; i < n; i++)
      start[digit((int32_t)i) + 1]++;
    for (int d = 0; d < 512; d++)
      start[d + 1] += start[d];
    for (size_t i = 0; i < n; i++)
      tmp[start[digit(order[i])]++] = order[i];
    order.swap(tmp);
  }
}

// The caller's arrays as they are through pinned staging (transfer.h) into one
// device block, and from there into the batch's layout (load.h).  vel, u, type, id,
// mb_pos and mb_vel may be null.
void upload_batch(hbtx_ctx *c, Batch &B, int64_t n, const float *pos, const float *vel, const float *mass,
                  const float *u, const int32_t *type, const int64_t *id, int64_t nsub, const int64_t *offsets,
                  const float *ref_pos, const float *ref_vel, const float *mb_pos, const float *mb_vel)
{
  check_layout(n, nsub, offsets);
  REQUIRE(pos && mass && ref_pos && ref_vel, HBTX_E_INVALID, "null input array");
  B.n = n;
  B.nsub = (int32_t)nsub;
  B.has_type = type != nullptr;
  B.has_u = u != nullptr;
  B.has_id = id != nullptr;
  B.has_proposal = false;
  B.has_prev = false;
  B.egroups_min = -1;
  B.feat_full = false;
  B.ran = false;
  B.h_off.assign(offsets, offsets + nsub + 1);
  B.h_count.resize(nsub);
  B.max_count = 0;
  B.ent_bound = 0;
  for (int64_t s = 0; s < nsub; s++)
  {
    B.h_count[s] = (int32_t)(offsets[s + 1] - offsets[s]);
    B.max_count = std::max(B.max_count, B.h_count[s]);
    B.ent_bound += entry_bound(B.h_count[s]);
  }
  batch_reserve(c, B);
  std::vector<int32_t> horder;
  size_order(B.h_count, horder);

  std::vector<XferPart> parts;
  size_t end = 0;
  auto place = [&](size_t bytes) {
    const size_t at = end;
    end = (at + bytes + 15) & ~(size_t)15;
    return at;
  };
  auto array = [&](const void *src, size_t bytes) {
    const size_t at = place(src ? bytes : 0);
    if (src && bytes)
      parts.push_back(xfer_from(at, src, bytes));
    return at;
  };
  const size_t a_off = place((nsub + 1) * sizeof(int32_t));
  parts.push_back({a_off, nullptr, (nsub + 1) * sizeof(int32_t), [offsets](char *slot, size_t off, size_t len) {
                     for (size_t i = 0; i < len / 4; i++)
                       ((int32_t *)slot)[i] = (int32_t)offsets[off / 4 + i];
                   }});
  const size_t a_order = array(horder.data(), nsub * sizeof(int32_t));
  const size_t a_rp = array(ref_pos, 3 * nsub * sizeof(float)), a_rv = array(ref_vel, 3 * nsub * sizeof(float));
  const size_t a_mp = array(mb_pos, 3 * nsub * sizeof(float)), a_mv = array(mb_vel, 3 * nsub * sizeof(float));
  const size_t a_mass = array(mass, n * sizeof(float)), a_pos = array(pos, 3 * n * sizeof(float));
  const size_t a_vel = array(vel, 3 * n * sizeof(float)), a_u = array(u, n * sizeof(float));
  const size_t a_type = array(type, n * sizeof(int32_t)), a_id = array(id, n * sizeof(int64_t));
  // the walk records' buffer (72 bytes a particle, idle between runs) takes the block
  char *raw = (char *)B.wt.p;
  if (end > B.wt.n * sizeof(uint2))
  {
    B.raw.alloc(end);
    raw = B.raw.p;
  }
  hipStream_t st = c->stream;
  HIPCHK(c->staging.up(c->device, st, raw, parts));
  auto dev = [&](const void *given, size_t at) { return given ? (const float *)(raw + at) : nullptr; };
  k_fill_i32<<<1, 64, 0, st>>>(B.load_bad.p, 1, 0);
  k_fill_i32<<<blocks_for(B.max_count), 256, 0, st>>>(B.sub_zero.p, std::max<int64_t>(B.max_count, 1), 0);
  k_fill_i32<<<1, 64, 0, st>>>(B.order_zero.p, 1, 0);
  k_load_subs<<<blocks_for(nsub + 1, 256, 1 << 24), 256, 0, st>>>(
    (const int32_t *)(raw + a_off), (const int32_t *)(raw + a_order), dev(ref_pos, a_rp), dev(ref_vel, a_rv),
    dev(mb_pos, a_mp), dev(mb_vel, a_mv), (int32_t)nsub, B.off.p, B.off_pairs.p, B.order.p, B.ref_in.p, B.mb_in.p);
  k_load_particles<<<blocks_for(n), 256, 0, st>>>(dev(pos, a_pos), dev(vel, a_vel), dev(mass, a_mass), dev(u, a_u),
                                                  (const int32_t *)dev(type, a_type), (const int64_t *)dev(id, a_id), n,
                                                  B.posm.p, B.velu.p, B.ptype.p, B.ids.p, B.load_bad.p);
  k_load_sub_of<<<blocks_for((n + 3) / 4), 256, 0, st>>>(B.off.p, (int32_t)nsub, n, B.sub_of.p, nullptr);
  HIPCHK(hipGetLastError());
  int32_t bad = 0;
  HIPCHK(c->staging.down(c->device, st, {xfer_to(&bad, B.load_bad.p, sizeof(bad))}));
  B.raw.release();
  if (bad)
    B.n = B.nsub = 0; // nothing is loaded
  // (the walk records mark cells by the sign bit of the mass)
  REQUIRE(!(bad & LOAD_BAD_MASS), HBTX_E_INVALID, "particle masses must be non-negative");
  REQUIRE(!(bad & LOAD_BAD_TYPE), HBTX_E_INVALID, "particle type out of range [0,6)");
}

void run_batch(hbtx_ctx *c, const hbtx_params &prm, uint32_t flags, double *elapsed_ms)
{
  Batch &B = c->B;
  REQUIRE(B.n > 0 || B.nsub > 0, HBTX_E_INVALID, "no batch loaded");
  hbtx_params p = prm;
  if (p.direct_cutoff < 0)
    p.direct_cutoff = c->direct_cutoff;
  REQUIRE(p.max_sample_size >= 0, HBTX_E_INVALID, "MaxSampleSizeOfPotentialEstimate must be >= 0");
  const bool warm = (flags & HBTX_WARMSTART) != 0;
  REQUIRE(!warm || B.has_proposal, HBTX_E_INVALID, "warm start needs a proposal (hbtx_batch_set_proposal / propose)");
  REQUIRE(!warm || p.max_sample_size == 0, HBTX_E_INVALID, "warm start is exclusive with subsampling");
  const DevParams P = make_dev_params(p);
  hipStream_t st = c->stream;
  HIPCHK(hipMemsetAsync(c->stats.p, 0, NSTATS * sizeof(unsigned long long), st));
  c->walk_ms = 0.0;
  c->rounds = 0;
  c->graph_rounds = 0;
  c->graph_captures = 0;
  c->tree_entries = c->tree_entries_first = 0;
  HIPCHK(hipEventRecord(c->ev0, st));
  const bool want_pot = (flags & HBTX_SAVE_POTENTIAL) != 0;
  c->count_work = (flags & HBTX_COUNT) != 0;
  if (flags & HBTX_PLAIN)
  {
    for (int32_t s = 0; s < B.nsub; s++)
    {
      View V = make_view(B, B.h_off[s], B.h_count[s], s, 1, false);
      c->rounds += run_view(c, B, V, P, want_pot, warm, false);
    }
  }
  else
  {
    View V = make_view(B, 0, B.n, 0, B.nsub, true);
    c->rounds = run_view(c, B, V, P, want_pot, warm, (flags & HBTX_NO_GRAPH) == 0);
  }
  HIPCHK(hipEventRecord(c->ev1, st));
  HIPCHK(hipEventSynchronize(c->ev1));
  float ms = 0.f;
  HIPCHK(hipEventElapsedTime(&ms, c->ev0, c->ev1));
  if (elapsed_ms)
    *elapsed_ms = ms;
  B.ran = true;
}

void fetch_batch(hbtx_ctx *c, int64_t *out_order, float *out_energy, float *out_potential,
                 hbtx_sub_result *out_res)
{
  Batch &B = c->B;
  REQUIRE(B.ran, HBTX_E_INVALID, "batch has not been run");
  const int64_t n = B.n;
  std::vector<XferPart> parts;
  if (out_order)
    parts.push_back({0, B.ford.p, n * sizeof(int32_t), [out_order](char *slot, size_t off, size_t len) {
                       const int32_t *v = (const int32_t *)slot;
                       int64_t *o = out_order + off / 4;
                       for (size_t i = 0; i < len / 4; i++)
                         o[i] = v[i];
                     }});
  if (out_energy)
    parts.push_back(xfer_to(out_energy, B.fenergy.p, n * sizeof(float)));
  if (out_potential)
    parts.push_back(xfer_to(out_potential, B.fpot.p, n * sizeof(float)));
  if (out_res)
    parts.push_back(xfer_to(out_res, B.dres.p, B.nsub * sizeof(hbtx_sub_result)));
  HIPCHK(c->staging.down(c->device, c->stream, parts));
}

// ---------------------------------------------------------------------------
// tree API
// ---------------------------------------------------------------------------
void build_tree(hbtx_ctx *c, const hbtx_params &prm, int64_t n, const float *pos, const float *mass, hbtx_tree *T,
                int treemode)
{
  REQUIRE(n >= 1, HBTX_E_INVALID, "a tree needs at least one source");
  Batch &B = c->B;
  const int64_t off[2] = {0, n};
  float zero3[3] = {0.f, 0.f, 0.f};
  upload_batch(c, B, n, pos, nullptr, mass, nullptr, nullptr, nullptr, 1, off, zero3, zero3, nullptr, nullptr);
  hbtx_params p = prm;
  p.direct_cutoff = treemode ? 0 : ((int64_t)1 << 40);
  p.max_sample_size = 0;
  const DevParams P = make_dev_params(p);
  View V = make_view(B, 0, n, 0, 1, true);
  hipStream_t st = c->stream;
  k_init_particles<<<blocks_for(n), 256, 0, st>>>(V.S, V.Q, n);
  k_init_subs<<<1, 64, 0, st>>>(V.S, B.ref_in.p, B.mb_in.p, nullptr);
  k_fill_i32<<<1, 64, 0, st>>>(B.misc.p, 8, 0);
  k_round_begin<<<1, 64, 0, st>>>(V.S.active_count, round_ptr(B), V.S.max_active_n);
  k_plan<<<1, 64, 0, st>>>(V.S, P, round_ptr(B));
  round_sources_and_tree(c, B, V, P, false, 0);
  int32_t h_misc[4];
  HIPCHK(hipMemcpyAsync(h_misc, B.misc.p, sizeof(h_misc), hipMemcpyDeviceToHost, st));
  HIPCHK(hipStreamSynchronize(st));
  check_overflow(h_misc[2]);
  const int32_t ne = h_misc[3];
  T->spare = c->tree_spare;
  T->spare->take(*T);
  T->n = n;
  T->ne = ne;
  T->ncells = ne - n;
  T->P = P;
  T->treemode = treemode;
  T->ent.alloc((int64_t)ne + 1);
  T->eskip.alloc((int64_t)ne + 1);
  T->ent_depth.alloc(ne);
  T->src_of_entry.alloc(n);
  T->cube.alloc(4);
  // walk records: 2 units per particle, 3 per cell, and two spare units
  T->nw = (int32_t)(2 * n + 3 * ((int64_t)ne - n));
  T->wt.alloc((int64_t)T->nw + 2);
  HIPCHK(hipMemcpyAsync(T->wt.p, B.wt.p, ((int64_t)T->nw + 2) * sizeof(uint2), hipMemcpyDeviceToDevice, st));
  HIPCHK(hipMemcpyAsync(T->ent.p, B.ent.p, ((int64_t)ne + 1) * sizeof(float4), hipMemcpyDeviceToDevice, st));
  HIPCHK(hipMemcpyAsync(T->eskip.p, B.eskip.p, ((int64_t)ne + 1) * sizeof(int32_t), hipMemcpyDeviceToDevice, st));
  HIPCHK(hipMemcpyAsync(T->ent_depth.p, B.ent_depth.p, ne, hipMemcpyDeviceToDevice, st));
  HIPCHK(hipMemcpyAsync(T->src_of_entry.p, B.src.p, n * sizeof(int32_t), hipMemcpyDeviceToDevice, st));
  HIPCHK(hipMemcpyAsync(T->cube.p, B.cube.p, 4 * sizeof(double), hipMemcpyDeviceToDevice, st));
  HIPCHK(hipStreamSynchronize(st));
  B.ran = false;
}

// Potentials at A's targets: the tree walk, or the exact sum over the records.
// The exact sum takes several waves per 64 targets up to DS_ITEMS_PER_CU times 64
// targets a CU (196,608 on 256 CUs); beyond that one wave per 64 targets keeps the chip as
// full, without the exchange.  One wave against several, us:
//   targets            30,001      131,072      196,608      262,144      400,000
//   500 sources       71,   29     72,   56     85,   72     97,   87    122,  121
//   2,000            233,   45    170,  126    180,  173    216,  221    289,  322
//   20,011          2131,  241   1368,  968   1560, 1393   1781, 1834   2400, 2743
// (30,001 targets are 469 waves' worth for 468 waves: one of them takes two.)
#define DS_ITEMS_PER_CU 12
template <bool PERIODIC, bool STATS>
void launch_points(hbtx_ctx *c, const PointArgs &A)
{
  const int64_t nt = A.ntgt;
  const int64_t items = (nt + HBTX_WAVE - 1) / HBTX_WAVE;
  if (!A.treemode && items <= (int64_t)DS_ITEMS_PER_CU * c->num_cu)
  {
    k_points_direct<PERIODIC, STATS>
      <<<(unsigned)std::max<int64_t>(1, items), DS_THREADS, 0, c->stream>>>(A);
    return;
  }
  const int grid = (int)std::max<int64_t>(1, std::min<int64_t>(nt / HBTX_WAVE + 1, 32 * c->num_cu) / HBTX_WALK_WG_WAVES);
  k_points_potential<PERIODIC, STATS><<<grid, WALK_WG_THREADS, 0, c->stream>>>(A);
}

void tree_points(hbtx_ctx *c, hbtx_tree *T, int64_t nt, const float *tpos, const float *tmass, double *out)
{
  REQUIRE(nt >= 0 && nt < (int64_t)0x20000000, HBTX_E_INVALID, "bad target count");
  if (nt == 0)
    return;
  hipStream_t st = c->stream;
  auto &W = c->ws;
  WsUse use{W};
  W.raw.alloc(4 * nt);
  W.tgt.alloc(nt);
  W.phi.alloc(nt);
  W.keys.alloc(nt);
  W.vals.alloc(nt);
  W.seg.alloc(4); // the range, and the sort's copy of it
  W.counter.alloc(POINT_COUNTERS + 1); // work counters, then the overflow word
  std::vector<XferPart> parts{xfer_from(0, tpos, 3 * nt * sizeof(float))};
  if (tmass)
    parts.push_back(xfer_from(3 * nt * sizeof(float), tmass, nt * sizeof(float)));
  HIPCHK(c->staging.up(c->device, st, W.raw.p, parts));
  k_pack_points<<<blocks_for(nt), 256, 0, st>>>(W.raw.p, tmass ? W.raw.p + 3 * nt : nullptr, (int32_t)nt, W.tgt.p);
  k_points_begin<<<1, 256, 0, st>>>(W.counter.p, POINT_COUNTERS + 1, W.seg.p, (int32_t)nt);
  // walk order: targets sorted by their key in the tree cube
  k_point_keys<<<blocks_for(nt), 256, 0, st>>>(W.tgt.p, (int32_t)nt, T->cube.p, W.keys.p, W.vals.p);
  if (T->treemode)
    seg_sort(c, W.keys.p, W.vals.p, 1, RangeArray{W.seg.p, W.seg.p + 1}, W.seg.p + 2, W.seg.p + 3, nt, 63, nt);
  PointArgs A;
  A.tgt = W.tgt.p;
  A.tgt_order = W.vals.p;
  A.ntgt = (int32_t)nt;
  A.eb = 0;
  A.ee = T->nw;
  A.treemode = T->treemode;
  A.cube = T->cube.p;
  A.wt = T->wt.p;
  A.phi = W.phi.p;
  A.counter = W.counter.p;
  A.chunks = POINT_CHUNKS;
  A.stats = c->stats.p;
  A.overflow = W.counter.p + POINT_COUNTERS;
  A.P = T->P;
  HIPCHK(hipMemsetAsync(c->stats.p, 0, NSTATS * sizeof(unsigned long long), st));
  HIPCHK(hipEventRecord(c->wev0, st));
  if (T->P.periodic)
    c->count_work ? launch_points<true, true>(c, A) : launch_points<true, false>(c, A);
  else
    c->count_work ? launch_points<false, true>(c, A) : launch_points<false, false>(c, A);
  HIPCHK(hipEventRecord(c->wev1, st));
  HIPCHK(hipGetLastError());
  int32_t ov = 0;
  HIPCHK(c->staging.down(c->device, st, {xfer_to(out, W.phi.p, nt * sizeof(double)), xfer_to(&ov, W.counter.p + POINT_COUNTERS, 4)}));
  REQUIRE(ov == 0, HBTX_E_CAPACITY, "tree walk stack capacity exceeded");
  float wms = 0.f;
  HIPCHK(hipEventElapsedTime(&wms, c->wev0, c->wev1));
  c->walk_ms = wms;
}

int fail(hbtx_ctx *c, int code, const std::string &msg)
{
  if (c)
    c->err = msg;
  return code;
}

} // namespace

#define API_GUARD(ctx, ...)                                                                                          \
  try                                                                                                                \
  {                                                                                                                  \
    __VA_ARGS__;                                                                                                     \
    return HBTX_OK;                                                                                                  \
  }                                                                                                                  \
  catch (const Error &e)                                                                                             \
  {                                                                                                                  \
    return fail(ctx, e.code, e.what());                                                                              \
  }                                                                                                                  \
  catch (const std::exception &e)                                                                                    \
  {                                                                                                                  \
    return fail(ctx, HBTX_E_INVALID, e.what());                                                                      \
  }

extern "C" {

void hbtx_default_params(hbtx_params *p)
{
  if (!p)
    return;
  std::memset(p, 0, sizeof(*p));
  p->G = 43.0071;
  p->scale_factor = 1.f;
  p->hz = 0.f;
  p->softening = 0.001f;
  p->max_phys_softening = -1.f;
  p->theta = 0.45f;
  p->bound_mass_precision = 0.995f;
  p->max_sample_size = 1000;
  p->refine_most_bound = 1;
  p->bound_fraction_center_refinement = 0.1f;
  p->min_num_part = 20;
  p->min_num_tracer = 10;
  p->tracer_mask = (1 << 1) | (1 << 4);
  p->donot_subsample_mask = (1 << 5);
  p->periodic = 1;
  p->box_size = 0.f;
  p->thermal = 0;
  p->dm_only = 1;
  p->upscale_per_type = 1;
  p->sub_core_size_factor = 0.f;
  p->sub_core_size_min = 20;
  p->direct_cutoff = -1;
}

} // extern "C"

void load_tuning(hbtx_ctx *c)
{
  const std::string path = tune_file_path();
  std::ifstream f(path);
  if (f)
  {
    std::stringstream ss;
    ss << f.rdbuf();
    const std::string txt = ss.str();
    int64_t v;
    if (json_int(txt, "direct_cutoff", v) && v >= 0)
      c->direct_cutoff = v;
    if (json_int(txt, "walk_chunks", v) && v >= 1)
      c->walk_chunks = (int)std::min<int64_t>(WALK_MAX_CHUNKS, v);
    if (json_int(txt, "walk_waves", v) && v >= 1)
      c->walk_waves = (int)std::min<int64_t>(64, v);
    c->tune_source = path;
  }
  if (const char *e = getenv("HBTX_DIRECT_CUTOFF"))
  {
    c->direct_cutoff = std::max<int64_t>(0, atoll(e));
    c->tune_source = "environment";
  }
  if (const char *e = getenv("HBTX_WALK_CHUNKS"))
  {
    c->walk_chunks = std::min(WALK_MAX_CHUNKS, std::max(1, atoi(e)));
    c->tune_source = "environment";
  }
  if (const char *e = getenv("HBTX_WALK_WAVES"))
  {
    c->walk_waves = std::min(64, std::max(1, atoi(e)));
    c->tune_source = "environment";
  }
}

extern "C" {

int hbtx_create(hbtx_ctx **out, int device)
{
  if (!out)
    return HBTX_E_INVALID;
  *out = nullptr;
  hbtx_ctx *c = new (std::nothrow) hbtx_ctx();
  if (!c)
    return HBTX_E_ALLOC;
  try
  {
    int ndev = 0;
    HIPCHK(hipGetDeviceCount(&ndev));
    REQUIRE(device >= 0 && device < ndev, HBTX_E_INVALID, "no such HIP device");
    c->device = device;
    HIPCHK(hipSetDevice(device));
    hipDeviceProp_t prop;
    HIPCHK(hipGetDeviceProperties(&prop, device));
    c->num_cu = std::max(1, prop.multiProcessorCount);
    c->scratch = scratch_address(device);
    // (more than the 64 KiB a kernel gets unasked)
    HIPCHK(hipFuncSetAttribute((const void *)k_sort_block, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)sizeof(SortBlockLds)));
    load_tuning(c);
    HIPCHK(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
    HIPCHK(hipEventCreate(&c->ev0));
    HIPCHK(hipEventCreate(&c->ev1));
    HIPCHK(hipEventCreate(&c->wev0));
    HIPCHK(hipEventCreate(&c->wev1));
    c->stats.alloc(NSTATS);
    c->tree_spare = std::make_shared<TreeSpare>();
  }
  catch (const Error &e)
  {
    int code = e.code;
    delete c;
    return code;
  }
  catch (const std::bad_alloc &)
  {
    delete c;
    return HBTX_E_ALLOC;
  }
  *out = c;
  return HBTX_OK;
}

void hbtx_destroy(hbtx_ctx *c)
{
  if (!c)
    return;
  (void)hipSetDevice(c->device);
  if (c->stream)
    (void)hipStreamSynchronize(c->stream);
  c->tree_spare->close();
  if (c->ev0)
    (void)hipEventDestroy(c->ev0);
  if (c->ev1)
    (void)hipEventDestroy(c->ev1);
  if (c->wev0)
    (void)hipEventDestroy(c->wev0);
  if (c->wev1)
    (void)hipEventDestroy(c->wev1);
  drop_graphs(c);
  if (c->round_words)
    (void)hipHostFree(c->round_words);
  hipStream_t st = c->stream;
  delete c;
  if (st)
    (void)hipStreamDestroy(st);
}

const char *hbtx_last_error(const hbtx_ctx *c)
{
  return c ? c->err.c_str() : "null context";
}

int hbtx_device_sync(hbtx_ctx *c)
{
  if (!c)
    return HBTX_E_INVALID;
  API_GUARD(c, HIPCHK(hipStreamSynchronize(c->stream)));
}

int hbtx_check_layout(int64_t n, int64_t nsub, const int64_t *offsets, char *msg, int32_t msg_len)
{
  std::string m;
  int rc = HBTX_OK;
  try
  {
    check_layout(n, nsub, offsets);
  }
  catch (const Error &e)
  {
    rc = e.code;
    m = e.what();
  }
  if (msg && msg_len > 0)
  {
    const size_t k = std::min<size_t>(m.size(), (size_t)msg_len - 1);
    std::memcpy(msg, m.data(), k);
    msg[k] = 0;
  }
  return rc;
}

int hbtx_batch_load(hbtx_ctx *c, int64_t n, const float *pos, const float *vel, const float *mass, const float *u,
                    const int32_t *type, const int64_t *id, int64_t nsub, const int64_t *offsets,
                    const float *ref_pos, const float *ref_vel, const float *mb_pos, const float *mb_vel)
{
  if (!c)
    return HBTX_E_INVALID;
  API_GUARD(c, {
    HIPCHK(hipSetDevice(c->device));
    check_layout(n, nsub, offsets);
    REQUIRE(vel, HBTX_E_INVALID, "null input array");
    upload_batch(c, c->B, n, pos, vel, mass, u, type, id, nsub, offsets, ref_pos, ref_vel, mb_pos, mb_vel);
  });
}

int hbtx_batch_set_proposal(hbtx_ctx *c, const uint8_t *proposal)
{
  if (!c)
    return HBTX_E_INVALID;
  API_GUARD(c, {
    REQUIRE(proposal, HBTX_E_INVALID, "null proposal");
    HIPCHK(hipSetDevice(c->device));
    HIPCHK(c->staging.up(c->device, c->stream, c->B.proposal.p, {xfer_from(0, proposal, c->B.n)}));
    c->B.has_proposal = true;
  });
}

int hbtx_batch_run(hbtx_ctx *c, const hbtx_params *prm, uint32_t flags, double *elapsed_ms)
{
  if (!c || !prm)
    return HBTX_E_INVALID;
  API_GUARD(c, {
    HIPCHK(hipSetDevice(c->device));
    run_batch(c, *prm, flags, elapsed_ms);
  });
}

int hbtx_batch_fetch(hbtx_ctx *c, int64_t *out_order, float *out_energy, float *out_potential,
                     hbtx_sub_result *out_res)
{
  if (!c)
    return HBTX_E_INVALID;
  API_GUARD(c, fetch_batch(c, out_order, out_energy, out_potential, out_res));
}

static const char *kStatNames[NSTATS] = {"tree_wave_steps", "tree_lane_visits", "tree_lane_accepts",
                                         "direct_lane_pairs", "targets", "work_items", "near_interactions",
                                         "tree_entries", "tree_entries_first", "unused9", "unused10", "unused11",
                                         "walk_ms",
                                         "rounds", "graph_rounds", "graph_captures"};

int hbtx_batch_stats(hbtx_ctx *c, double *stats, int nstats)
{
  if (!c || !stats)
    return HBTX_E_INVALID;
  API_GUARD(c, {
    unsigned long long h[NSTATS];
    HIPCHK(hipMemcpy(h, c->stats.p, sizeof(h), hipMemcpyDeviceToHost));
    for (int i = 0; i < nstats && i < NSTATS; i++)
      stats[i] = (double)h[i];
    if (nstats > 7)
      stats[7] = (double)c->tree_entries;
    if (nstats > 8)
      stats[8] = (double)c->tree_entries_first;
    if (nstats > 12)
      stats[12] = c->walk_ms;
    if (nstats > 13)
      stats[13] = c->rounds;
    if (nstats > 14)
      stats[14] = c->graph_rounds;
    if (nstats > 15)
      stats[15] = c->graph_captures;
  });
}

int hbtx_device_bytes(int64_t *bytes)
{
  if (!bytes)
    return HBTX_E_INVALID;
  *bytes = g_device_bytes.load();
  return 0;
}

const char *hbtx_stat_name(int i)
{
  return (i >= 0 && i < NSTATS) ? kStatNames[i] : "";
}

int hbtx_unbind_batch(hbtx_ctx *c, const hbtx_params *prm, int64_t n, const float *pos, const float *vel,
                      const float *mass, const float *u, const int32_t *type, const int64_t *id, int64_t nsub,
                      const int64_t *offsets, const float *ref_pos, const float *ref_vel, const float *mb_pos,
                      const float *mb_vel, uint32_t flags, int64_t *out_order, float *out_energy,
                      float *out_potential, hbtx_sub_result *out_res)
{
  if (!c || !prm)
    return HBTX_E_INVALID;
  API_GUARD(c, {
    HIPCHK(hipSetDevice(c->device));
    check_layout(n, nsub, offsets);
    REQUIRE(vel, HBTX_E_INVALID, "null input array");
    upload_batch(c, c->B, n, pos, vel, mass, u, type, id, nsub, offsets, ref_pos, ref_vel, mb_pos, mb_vel);
    run_batch(c, *prm, flags, nullptr);
    fetch_batch(c, out_order, out_energy, out_potential, out_res);
  });
}

int hbtx_tree_build(hbtx_ctx *c, const hbtx_params *prm, int64_t n, const float *pos, const float *mass,
                    hbtx_tree **tree, int64_t *ncells)
{
  if (!c || !prm || !tree || !pos || !mass)
    return HBTX_E_INVALID;
  *tree = nullptr;
  hbtx_tree *T = new (std::nothrow) hbtx_tree();
  if (!T)
    return HBTX_E_ALLOC;
  try
  {
    HIPCHK(hipSetDevice(c->device));
    build_tree(c, *prm, n, pos, mass, T, 1);
  }
  catch (const Error &e)
  {
    delete T;
    return fail(c, e.code, e.what());
  }
  *tree = T;
  if (ncells)
    *ncells = T->ncells;
  return HBTX_OK;
}

int hbtx_tree_potential(hbtx_ctx *c, hbtx_tree *T, int64_t n_tgt, const float *tgt_pos, const float *tgt_mass,
                        double *out_pot)
{
  if (!c || !T || (n_tgt > 0 && (!tgt_pos || !out_pot)))
    return HBTX_E_INVALID;
  API_GUARD(c, {
    HIPCHK(hipSetDevice(c->device));
    tree_points(c, T, n_tgt, tgt_pos, tgt_mass, out_pot);
  });
}

int hbtx_tree_binding_energy(hbtx_ctx *c, hbtx_tree *T, int64_t n_tgt, const float *tgt_pos, const float *tgt_vel,
                             const float *ref_pos, const float *ref_vel, const float *tgt_mass, double *out_energy)
{
  if (!c || !T || (n_tgt > 0 && (!tgt_pos || !tgt_vel || !ref_pos || !ref_vel || !out_energy)))
    return HBTX_E_INVALID;
  API_GUARD(c, {
    HIPCHK(hipSetDevice(c->device));
    tree_points(c, T, n_tgt, tgt_pos, tgt_mass, out_energy);
    const float ha = T->P.hz * T->P.a;
    for (int64_t i = 0; i < n_tgt; i++)
    {
      // Snapshot_t::RelativeVelocity in float, then VecNorm * 0.5 + pot
      float k2 = 0.f;
      for (int j = 0; j < 3; j++)
      {
        float dx = tgt_pos[3 * i + j] - ref_pos[j];
        if (T->P.periodic)
          dx = (dx > T->P.box_half) ? dx - T->P.box : ((dx < -T->P.box_half) ? dx + T->P.box : dx);
        float dv = tgt_vel[3 * i + j] - ref_vel[j];
        dv += ha * dx;
        k2 += dv * dv;
      }
      out_energy[i] = (double)k2 * 0.5 + out_energy[i];
    }
  });
}

int hbtx_tree_export(hbtx_ctx *c, hbtx_tree *T, int64_t cap, int32_t *kind, int64_t *pidx, float *mass, float *com,
                     float *len, int64_t *skip, int32_t *depth, int64_t *nentries)
{
  if (!c || !T)
    return HBTX_E_INVALID;
  API_GUARD(c, {
    HIPCHK(hipSetDevice(c->device));
    const int32_t ne = T->ne;
    if (nentries)
      *nentries = ne;
    REQUIRE(cap >= ne, HBTX_E_CAPACITY, "export capacity too small");
    std::vector<float4> en(ne);
    std::vector<int32_t> esk(ne);
    std::vector<int8_t> dep(ne);
    std::vector<int32_t> src(T->n);
    double cube[4];
    HIPCHK(hipMemcpy(en.data(), T->ent.p, ne * sizeof(float4), hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(esk.data(), T->eskip.p, ne * sizeof(int32_t), hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(cube, T->cube.p, sizeof(cube), hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(dep.data(), T->ent_depth.p, ne, hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(src.data(), T->src_of_entry.p, T->n * sizeof(int32_t), hipMemcpyDeviceToHost));
    int64_t pi = 0;
    for (int32_t q = 0; q < ne; q++)
    {
      const bool part = dep[q] < 0;
      if (kind)
        kind[q] = part ? 0 : 1;
      if (pidx)
        pidx[q] = part ? (int64_t)src[pi] : -1;
      if (part)
        pi++;
      if (mass)
        mass[q] = en[q].w;
      if (com)
      {
        com[3 * q] = en[q].x;
        com[3 * q + 1] = en[q].y;
        com[3 * q + 2] = en[q].z;
      }
      if (len)
      {
        // the cell's side: the root cube's, halved per level while not below the
        // resolution (the same rule and float rounding as the build)
        double L = 2.0 * cube[3];
        for (int l = 0; l < dep[q]; l++)
          L = (L >= T->P.res) ? L * 0.5 : L;
        const float lf = (float)L;
        len[q] = part ? 0.f : std::sqrt(lf * lf);
      }
      if (skip)
        skip[q] = part ? q + 1 : esk[q];
      if (depth)
        depth[q] = dep[q];
    }
  });
}

void hbtx_tree_free(hbtx_tree *T)
{
  delete T;
}

int hbtx_direct_potential(hbtx_ctx *c, const hbtx_params *prm, int64_t n_src, const float *src_pos,
                          const float *src_mass, int64_t n_tgt, const float *tgt_pos, const float *tgt_mass,
                          double *out_pot)
{
  if (!c || !prm)
    return HBTX_E_INVALID;
  hbtx_tree T;
  API_GUARD(c, {
    HIPCHK(hipSetDevice(c->device));
    build_tree(c, *prm, n_src, src_pos, src_mass, &T, 0);
    tree_points(c, &T, n_tgt, tgt_pos, tgt_mass, out_pot);
  });
}

int hbtx_direct_potential_noalloc(hbtx_ctx *c, const hbtx_params *prm, int64_t n_src, const float *d_src_pos,
                                  const float *d_src_mass, int64_t n_tgt, const float *d_tgt_pos,
                                  const float *d_tgt_mass, double *d_out_pot)
{
  if (!c || !prm)
    return HBTX_E_INVALID;
  API_GUARD(c, {
    REQUIRE(n_src >= 1 && n_tgt >= 0, HBTX_E_INVALID, "need at least one source and n_tgt >= 0");
    REQUIRE(n_src <= HBTX_NOALLOC_MAX_POINTS && n_tgt <= HBTX_NOALLOC_MAX_POINTS, HBTX_E_CAPACITY,
            "hbtx_direct_potential_noalloc takes at most HBTX_NOALLOC_MAX_POINTS (" +
              std::to_string(HBTX_NOALLOC_MAX_POINTS) + ") sources and targets; got " + std::to_string(n_src) +
              " and " + std::to_string(n_tgt));
    REQUIRE(d_src_pos && d_src_mass, HBTX_E_INVALID, "null source array");
    REQUIRE(n_tgt == 0 || (d_tgt_pos && d_out_pot), HBTX_E_INVALID, "null target or output array");
    REQUIRE(c->scratch, HBTX_E_HIP, "the scratch array has no device address");
    HIPCHK(hipSetDevice(c->device));
    hbtx_params p = *prm;
    p.direct_cutoff = (int64_t)1 << 40;
    p.max_sample_size = 0;
    const DevParams P = make_dev_params(p);
    hipStream_t st = c->stream;
    unsigned char *base = static_cast<unsigned char *>(c->scratch);
    uint2 *wt = reinterpret_cast<uint2 *>(base);
    float4 *tgt = reinterpret_cast<float4 *>(base + kScratchTgt);
    int32_t *counter = reinterpret_cast<int32_t *>(base + kScratchCtr);
    k_pack_records<<<blocks_for(n_src), 256, 0, st>>>(d_src_pos, d_src_mass, (int32_t)n_src, wt);
    if (n_tgt > 0)
    {
      k_pack_points<<<blocks_for(n_tgt), 256, 0, st>>>(d_tgt_pos, d_tgt_mass, (int32_t)n_tgt, tgt);
      k_fill_i32<<<1, 64, 0, st>>>(counter, 1, 0); // the previous call's count stays in the array
      PointArgs A;
      A.tgt = tgt;
      A.tgt_order = nullptr;
      A.ntgt = (int32_t)n_tgt;
      A.eb = 0;
      A.ee = (int32_t)(2 * n_src);
      A.treemode = 0;
      A.cube = nullptr;
      A.wt = wt;
      A.phi = d_out_pot;
      A.counter = counter; // (the scratch array holds one)
      A.chunks = 1;
      A.stats = nullptr;
      A.overflow = nullptr; // direct sums only
      A.P = P;
      P.periodic ? launch_points<true, false>(c, A) : launch_points<false, false>(c, A);
    }
    HIPCHK(hipGetLastError());
  });
}

int hbtx_batch_profiles(hbtx_ctx *c, const hbtx_params *prm, hbtx_sub_profile *out)
{
  if (!c || !prm || !out)
    return HBTX_E_INVALID;
  API_GUARD(c, {
    HIPCHK(hipSetDevice(c->device));
    Batch &B = c->B;
    REQUIRE(B.ran, HBTX_E_INVALID, "batch has not been run");
    B.prof_r.alloc(std::max<int64_t>(B.n, 1));
    B.prof_m.alloc(std::max<int64_t>(B.n, 1));
    B.dprof.alloc(std::max<int32_t>(B.nsub, 1));
    ProfArgs A;
    A.off = B.off.p;
    A.ford = B.ford.p;
    A.posm = B.posm.p;
    A.res = B.dres.p;
    A.seg_len = B.seg_len.p;
    A.rc = B.prof_r.p;
    A.mc = B.prof_m.p;
    run_profiles(c, *prm, A, B.n, B.nsub, B.sub_of.p, B.seg_begin.p, B.seg_len.p, B.keys.p, B.src.p, B.dprof.p,
                 B.max_count);
    HIPCHK(c->staging.down(c->device, c->stream, {xfer_to(out, B.dprof.p, B.nsub * sizeof(hbtx_sub_profile))}));
  });
}

int hbtx_profiles(hbtx_ctx *c, const hbtx_params *prm, int64_t n, const float *pos, const float *mass, int64_t nsub,
                  const int64_t *offsets, const int64_t *nbound, const float *mbound, hbtx_sub_profile *out)
{
  if (!c || !prm || !out || (n > 0 && (!pos || !mass)) || !offsets || !nbound || !mbound || nsub < 1)
    return HBTX_E_INVALID;
  API_GUARD(c, {
    HIPCHK(hipSetDevice(c->device));
    REQUIRE(n < (int64_t)0x20000000 && nsub < (int64_t)0x7fffffff, HBTX_E_INVALID, "too large");
    REQUIRE(offsets[0] == 0 && offsets[nsub] == n, HBTX_E_INVALID, "offsets must start at 0 and end at n");
    hipStream_t st = c->stream;
    std::vector<int32_t> hoff(nsub + 1);
    std::vector<hbtx_sub_result> hres(nsub);
    int64_t max_len = 0;
    for (int64_t s = 0; s < nsub; s++)
    {
      const int64_t a = offsets[s], e = offsets[s + 1];
      REQUIRE(a <= e && e <= n && nbound[s] >= 0 && nbound[s] <= e - a, HBTX_E_INVALID,
              "bound sets must lie inside ascending subhalo ranges");
      hoff[s] = (int32_t)a;
      hbtx_sub_result &R = hres[s];
      std::memset(&R, 0, sizeof(R));
      R.nbound = nbound[s];
      R.mbound = mbound[s];
      max_len = std::max(max_len, nbound[s]);
      if (nbound[s] > 0)
        for (int k = 0; k < 3; k++)
          R.mostbound_pos[k] = pos[3 * a + k];
    }
    hoff[nsub] = (int32_t)n;
    auto &W = c->ws;
    WsUse use{W};
    const int64_t n1 = std::max<int64_t>(n, 1);
    W.raw.alloc(4 * n1);
    W.posm.alloc(n1);
    W.off.alloc(nsub + 1);
    W.sub_of.alloc(n1);
    W.local.alloc(n1);
    W.seg.alloc(2 * (nsub + 1));
    W.vals.alloc(n1);
    W.keys.alloc(n1);
    W.res.alloc(nsub);
    W.rc.alloc(n1);
    W.mc.alloc(n1);
    W.prof.alloc(nsub);
    HIPCHK(c->staging.up(c->device, st, W.raw.p,
                         {xfer_from(0, pos, 3 * n * sizeof(float)), xfer_from(3 * n * sizeof(float), mass, n * sizeof(float))}));
    HIPCHK(c->staging.up(c->device, st, W.off.p, {xfer_from(0, hoff.data(), (nsub + 1) * sizeof(int32_t))}));
    HIPCHK(c->staging.up(c->device, st, W.res.p, {xfer_from(0, hres.data(), nsub * sizeof(hbtx_sub_result))}));
    if (n > 0)
      k_pack_points<<<blocks_for(n), 256, 0, st>>>(W.raw.p, W.raw.p + 3 * n, (int32_t)n, W.posm.p);
    k_load_sub_of<<<blocks_for((n + 3) / 4), 256, 0, st>>>(W.off.p, (int32_t)nsub, n, W.sub_of.p, W.local.p);
    ProfArgs A;
    A.off = W.off.p;
    A.ford = W.local.p;
    A.posm = W.posm.p;
    A.res = W.res.p;
    A.seg_len = W.seg.p + nsub + 1;
    A.rc = W.rc.p;
    A.mc = W.mc.p;
    run_profiles(c, *prm, A, n, (int32_t)nsub, W.sub_of.p, W.seg.p, W.seg.p + nsub + 1, W.keys.p, W.vals.p, W.prof.p,
                 max_len);
    HIPCHK(c->staging.down(c->device, st, {xfer_to(out, W.prof.p, nsub * sizeof(hbtx_sub_profile))}));
  });
}

// ---------------------------------------------------------------------------
// particle reassignment
// ---------------------------------------------------------------------------
int hbtx_reassign_targets(hbtx_ctx *c, const hbtx_params *prm, int64_t n, const float *pos, const uint8_t *is_tracer,
                          const int32_t *sub, int64_t ngroups, const int64_t *group_offsets, int32_t k, float rguess,
                          int32_t *out_target, double *elapsed_ms)
{
  if (!c || !prm || !group_offsets || ngroups < 1 || (n > 0 && (!pos || !is_tracer || !sub || !out_target)))
    return HBTX_E_INVALID;
  API_GUARD(c, {
    HIPCHK(hipSetDevice(c->device));
    REQUIRE(n < (int64_t)0x20000000 && ngroups < (int64_t)0x20000000, HBTX_E_INVALID, "too large");
    REQUIRE(k >= 1 && k <= 32, HBTX_E_INVALID, "k (NumNeighboursForReassignment) must lie in 1..32");
    REQUIRE(group_offsets[0] == 0 && group_offsets[ngroups] == n, HBTX_E_INVALID,
            "group offsets must start at 0 and end at n");
    int64_t max_group = 0;
    for (int64_t g = 0; g < ngroups; g++)
    {
      REQUIRE(group_offsets[g] <= group_offsets[g + 1], HBTX_E_INVALID, "group offsets must ascend");
      max_group = std::max(max_group, group_offsets[g + 1] - group_offsets[g]);
    }
    // GeoTree_t::NearestNeighbours(centre, k, SofteningHalo * 0.1) (src/subhalo_reassign_gas.cpp:144)
    const float r0 = (rguess > 0.f) ? rguess : (float)(prm->softening * 0.1);
    REQUIRE(r0 > 0.f && std::isfinite(r0), HBTX_E_INVALID, "the first search radius must be positive");
    std::vector<float> rad(RS_RADII);
    rad[0] = r0;
    for (int j = 1; j < RS_RADII; j++)
      rad[j] = (float)((double)rad[j - 1] * 1.26); // rguess *= 1.26 (src/geometric_tree.cpp:127)
    REQUIRE(rad[RS_RADII - 1] >= 1e30f, HBTX_E_INVALID, "the first search radius is too small");
    if (elapsed_ms)
      *elapsed_ms = 0.0;
    if (n == 0)
      return HBTX_OK;
    auto &R = c->rs;
    const int32_t G = (int32_t)ngroups;
    std::vector<int32_t> hoff(G + 1);
    for (int32_t g = 0; g <= G; g++)
      hoff[g] = (int32_t)group_offsets[g];
    R.pos.alloc(3 * n);
    R.radii.alloc(RS_RADII);
    R.tracer.alloc(n);
    R.sub.alloc(n);
    R.goff.alloc(G + 1);
    R.gid.alloc(n);
    R.tflag.alloc(n + 1);
    R.cnt.alloc((int64_t)RS_LEVELS * G);
    R.loff.alloc((int64_t)RS_LEVELS * (G + 1));
    R.qtiles.alloc(G + 1);
    R.tval.alloc(n);
    R.qval.alloc(n);
    R.tkey.alloc(n);
    R.qkey.alloc(n);
    R.seg.alloc(6 * (int64_t)G);
    R.out.alloc(n);
    R.tot.alloc(RS_LEVELS + 2);
    R.grp.alloc(G);
    R.bbox.alloc(7 * (int64_t)G);
    R.trec.alloc(n);
    R.lbase.alloc(RS_LEVELS);
    hipStream_t st = c->stream;
    HIPCHK(c->staging.up(c->device, st, R.pos.p, {xfer_from(0, pos, 3 * n * sizeof(float))}));
    HIPCHK(c->staging.up(c->device, st, R.tracer.p, {xfer_from(0, is_tracer, n)}));
    HIPCHK(c->staging.up(c->device, st, R.sub.p, {xfer_from(0, sub, n * sizeof(int32_t))}));
    HIPCHK(c->staging.up(c->device, st, R.goff.p, {xfer_from(0, hoff.data(), (G + 1) * sizeof(int32_t))}));
    HIPCHK(c->staging.up(c->device, st, R.radii.p, {xfer_from(0, rad.data(), RS_RADII * sizeof(float))}));
    RsArgs A;
    A.n = (int32_t)n;
    A.ngroups = G;
    A.pos = R.pos.p;
    A.tracer = R.tracer.p;
    A.sub = R.sub.p;
    A.goff = R.goff.p;
    A.box = prm->box_size;
    A.half = prm->box_size / 2;
    A.periodic = prm->periodic ? 1 : 0;
    A.k = k;
    A.gid = R.gid.p;
    A.tflag = R.tflag.p;
    A.grp = R.grp.p;
    A.bbox = R.bbox.p;
    A.cnt = R.cnt.p;
    A.loff = R.loff.p;
    A.qtiles_n = R.qtiles.p;
    A.tkey = R.tkey.p;
    A.qkey = R.qkey.p;
    A.tval = R.tval.p;
    A.qval = R.qval.p;
    A.seg = R.seg.p;
    A.trec = R.trec.p;
    A.nodes = nullptr;
    A.lbase = R.lbase.p;
    A.out = R.out.p;
    HIPCHK(hipEventRecord(c->ev0, st));
    k_rs_flags<<<blocks_for(n), 256, 0, st>>>(A);
    scan32(c, R.tflag.p, R.tflag.p, n);
    k_rs_groups<<<blocks_for(G, 256, 1 << 20), 256, 0, st>>>(A);
    k_rs_scatter<<<blocks_for(n, RS_CHUNK), RS_THREADS, 0, st>>>(A);
    for (int l = 0; l < RS_LEVELS; l++)
      scan32(c, R.cnt.p + (int64_t)l * G, R.loff.p + (int64_t)l * (G + 1), G);
    scan32(c, R.qtiles.p, R.qtiles.p, G);
    k_rs_totals<<<1, 64, 0, st>>>(A, R.tot.p);
    int32_t tot[RS_LEVELS + 2];
    HIPCHK(hipMemcpyAsync(tot, R.tot.p, sizeof(tot), hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    const int32_t NT = tot[RS_LEVELS], ntiles = tot[RS_LEVELS + 1];
    int64_t lb[RS_LEVELS], nodes = 0;
    for (int l = 0; l < RS_LEVELS; l++)
    {
      lb[l] = nodes;
      nodes += tot[l];
    }
    R.nodes.alloc(2 * std::max<int64_t>(nodes, 1));
    R.tiles.alloc(std::max<int32_t>(ntiles, 1));
    A.nodes = R.nodes.p;
    HIPCHK(hipMemcpyAsync(R.lbase.p, lb, sizeof(lb), hipMemcpyHostToDevice, st));
    k_rs_keys<<<blocks_for(n), 256, 0, st>>>(A, NT);
    k_rs_group_finish<<<blocks_for(G, 256, 1 << 20), 256, 0, st>>>(A);
    int32_t *sort_b = R.seg.p + 4 * (int64_t)G, *sort_l = R.seg.p + 5 * (int64_t)G;
    seg_sort(c, R.tkey.p, R.tval.p, G, RangeArray{R.seg.p, R.seg.p + G}, sort_b, sort_l, std::max<int32_t>(NT, 1),
             3 * RS_KEY_BITS, max_group);
    seg_sort(c, R.qkey.p, R.qval.p, G, RangeArray{R.seg.p + 2 * (int64_t)G, R.seg.p + 3 * (int64_t)G}, sort_b, sort_l,
             std::max<int64_t>(n - NT, 1), 3 * RS_KEY_BITS, max_group);
    if (NT > 0)
      k_rs_records<<<blocks_for(NT), 256, 0, st>>>(A, NT);
    for (int l = 0; l < RS_LEVELS; l++)
      if (tot[l] > 0)
        k_rs_level<<<blocks_for(tot[l]), 256, 0, st>>>(A, l, tot[l]);
    if (ntiles > 0)
    {
      k_rs_tiles<<<blocks_for(ntiles), 256, 0, st>>>(A, R.tiles.p, ntiles);
      const int wpb = RS_THREADS / HBTX_WAVE;
      const int grid = (int)std::min<int64_t>((ntiles + wpb - 1) / wpb, 1 << 20);
      if (k <= 8)
        k_rs_knn<8><<<grid, RS_THREADS, 0, st>>>(A, R.tiles.p, ntiles, R.radii.p);
      else if (k <= 10) // the reference's default NumNeighboursForReassignment
        k_rs_knn<10><<<grid, RS_THREADS, 0, st>>>(A, R.tiles.p, ntiles, R.radii.p);
      else if (k <= 16)
        k_rs_knn<16><<<grid, RS_THREADS, 0, st>>>(A, R.tiles.p, ntiles, R.radii.p);
      else
        k_rs_knn<32><<<grid, RS_THREADS, 0, st>>>(A, R.tiles.p, ntiles, R.radii.p);
    }
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventRecord(c->ev1, st));
    HIPCHK(c->staging.down(c->device, st, {xfer_to(out_target, R.out.p, n * sizeof(int32_t))}));
    if (elapsed_ms)
    {
      float ms = 0.f;
      HIPCHK(hipEventElapsedTime(&ms, c->ev0, c->ev1));
      *elapsed_ms = ms;
    }
  });
}

int hbtx_segmented_sort(hbtx_ctx *c, int64_t n, uint64_t *keys, int32_t *vals, int64_t nseg,
                        const int64_t *seg_offsets)
{
  if (!c || (n > 0 && (!keys || !vals)) || !seg_offsets)
    return HBTX_E_INVALID;
  API_GUARD(c, {
    HIPCHK(hipSetDevice(c->device));
    REQUIRE(n < (int64_t)0x40000000 && nseg < (int64_t)0x7fffffff, HBTX_E_INVALID, "too large");
    hipStream_t st = c->stream;
    DArr<uint64_t> dk;
    DArr<int32_t> dv, sb, sl, sb2, sl2;
    int64_t max_len = 0;
    sb2.alloc(nseg);
    sl2.alloc(nseg);
    dk.alloc(n);
    dv.alloc(n);
    sb.alloc(nseg);
    sl.alloc(nseg);
    std::vector<int32_t> hb(nseg), hl(nseg);
    for (int64_t s = 0; s < nseg; s++)
    {
      REQUIRE(seg_offsets[s + 1] >= seg_offsets[s], HBTX_E_INVALID, "bad segments");
      hb[s] = (int32_t)seg_offsets[s];
      hl[s] = (int32_t)(seg_offsets[s + 1] - seg_offsets[s]);
      max_len = std::max<int64_t>(max_len, hl[s]);
    }
    HIPCHK(c->staging.up(c->device, st, dk.p, {xfer_from(0, keys, n * 8)}));
    HIPCHK(c->staging.up(c->device, st, dv.p, {xfer_from(0, vals, n * 4)}));
    HIPCHK(hipMemcpyAsync(sb.p, hb.data(), nseg * 4, hipMemcpyHostToDevice, st));
    HIPCHK(hipMemcpyAsync(sl.p, hl.data(), nseg * 4, hipMemcpyHostToDevice, st));
    // digit passes only over the bits the keys use
    uint64_t any = 0;
    for (int64_t i = 0; i < n; i++)
      any |= keys[i];
    int bits = 1;
    while (bits < 64 && (any >> bits) != 0)
      bits++;
    seg_sort(c, dk.p, dv.p, (int32_t)nseg, RangeArray{sb.p, sl.p}, sb2.p, sl2.p, n, bits, max_len);
    HIPCHK(c->staging.down(c->device, st, {xfer_to(keys, dk.p, n * 8), xfer_to(vals, dv.p, n * 4)}));
  });
}

} // extern "C"

namespace
{
uint64_t splitmix(uint64_t &x)
{
  uint64_t z = (x += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
double urand(uint64_t &x)
{
  return (double)(splitmix(x) >> 11) * (1.0 / 9007199254740992.0);
}

void mlp_alloc(hbtx_mlp *M)
{
  M->master.alloc(MLP_NPAR);
  M->m.alloc(MLP_NPAR);
  M->v.alloc(MLP_NPAR);
  M->wf.alloc(MLP_NPAR);
  M->grad.alloc(MLP_NPAR);
  M->wb.alloc(MLP_NPAR);
  M->loss.alloc(1);
}

void mlp_upload(hbtx_ctx *c, hbtx_mlp *M, const float *master)
{
  hipStream_t st = c->stream;
  HIPCHK(hipMemcpyAsync(M->master.p, master, MLP_NPAR * sizeof(float), hipMemcpyHostToDevice, st));
  HIPCHK(hipMemsetAsync(M->m.p, 0, MLP_NPAR * sizeof(float), st));
  HIPCHK(hipMemsetAsync(M->v.p, 0, MLP_NPAR * sizeof(float), st));
  k_mlp_round<<<(MLP_NPAR + 255) / 256, 256, 0, st>>>(M->master.p, M->wf.p, M->wb.p);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(st));
  M->step = 0;
}

// proposed particles of the loaded batch
int64_t count_proposed(hbtx_ctx *c, Batch &B)
{
  hipStream_t st = c->stream;
  c->ws.counter.alloc(2);
  k_fill_i32<<<1, 64, 0, st>>>(c->ws.counter.p, 1, 0);
  k_count_flags<<<blocks_for((B.n + 15) / 16, 256, 1024), 256, 0, st>>>(B.proposal.p, B.n, c->ws.counter.p);
  HIPCHK(hipGetLastError());
  int32_t cnt = 0;
  HIPCHK(c->staging.down(c->device, st, {xfer_to(&cnt, c->ws.counter.p, sizeof(cnt))}));
  return cnt;
}

// samples of a call (labels may be null) into the context's workspace
void mlp_samples(hbtx_ctx *c, int64_t n, const float *X, const uint8_t *y)
{
  auto &W = c->ws;
  W.X.alloc(n * MLP_IN);
  HIPCHK(c->staging.up(c->device, c->stream, W.X.p, {xfer_from(0, X, n * MLP_IN * sizeof(float))}));
  if (!y)
    return;
  W.y.alloc(n);
  HIPCHK(c->staging.up(c->device, c->stream, W.y.p, {xfer_from(0, y, n)}));
}

// forward+backward of nb samples (rows idx[0..nb) of dX, or rows 0..nb) -> M->grad, M->loss
void mlp_grad_device(hbtx_ctx *c, hbtx_mlp *M, const float *dX, const uint8_t *dy, const int32_t *idx, int64_t nb)
{
  hipStream_t st = c->stream;
  const int nblk = mlp_grad_blocks(nb, c->num_cu);
  M->partial.alloc((int64_t)nblk * MLP_NPAR);
  M->lossp.alloc(nblk);
  k_mlp_grad<<<nblk, MLP_BLOCK, 0, st>>>(M->wf.p, dX, dy, idx, nb, 1.f / (float)nb, M->partial.p, M->lossp.p);
  k_mlp_reduce<<<(MLP_NPAR + HBTX_WAVE - 1) / HBTX_WAVE, 256, 0, st>>>(M->partial.p, nblk, M->grad.p, M->lossp.p, M->loss.p);
  HIPCHK(hipGetLastError());
}
} // namespace

extern "C" {

int hbtx_mlp_create(hbtx_ctx *c, uint64_t seed, hbtx_mlp **out)
{
  if (!c || !out)
    return HBTX_E_INVALID;
  *out = nullptr;
  hbtx_mlp *M = new (std::nothrow) hbtx_mlp();
  if (!M)
    return HBTX_E_ALLOC;
  try
  {
    HIPCHK(hipSetDevice(c->device));
    mlp_alloc(M);
    std::vector<float> w(MLP_NPAR, 0.f);
    uint64_t x = seed;
    const double l1 = std::sqrt(6.0 / MLP_IN), l2 = std::sqrt(6.0 / MLP_H), l3 = std::sqrt(3.0 / MLP_H);
    for (int i = 0; i < MLP_H * MLP_IN; i++)
      w[MLP_OFF_W1 + i] = (float)((2.0 * urand(x) - 1.0) * l1);
    for (int i = 0; i < MLP_H * MLP_H; i++)
      w[MLP_OFF_W2 + i] = (float)((2.0 * urand(x) - 1.0) * l2);
    for (int i = 0; i < MLP_H; i++)
      w[MLP_OFF_W3 + i] = (float)((2.0 * urand(x) - 1.0) * l3);
    mlp_upload(c, M, w.data());
  }
  catch (const Error &e)
  {
    delete M;
    return fail(c, e.code, e.what());
  }
  *out = M;
  return HBTX_OK;
}

void hbtx_mlp_free(hbtx_mlp *M)
{
  delete M;
}

int hbtx_mlp_get_weights(hbtx_ctx *c, hbtx_mlp *M, float *master, uint16_t *bf16)
{
  if (!c || !M)
    return HBTX_E_INVALID;
  API_GUARD(c, {
    HIPCHK(hipSetDevice(c->device));
    HIPCHK(hipStreamSynchronize(c->stream));
    if (master)
      HIPCHK(hipMemcpy(master, M->master.p, MLP_NPAR * sizeof(float), hipMemcpyDeviceToHost));
    if (bf16)
      HIPCHK(hipMemcpy(bf16, M->wb.p, MLP_NPAR * sizeof(uint16_t), hipMemcpyDeviceToHost));
  });
}

int hbtx_mlp_set_weights(hbtx_ctx *c, hbtx_mlp *M, const float *master)
{
  if (!c || !M || !master)
    return HBTX_E_INVALID;
  API_GUARD(c, {
    HIPCHK(hipSetDevice(c->device));
    mlp_upload(c, M, master);
  });
}

int hbtx_mlp_gradient(hbtx_ctx *c, hbtx_mlp *M, int64_t n, const float *X, const uint8_t *y, float *grad,
                      double *loss)
{
  if (!c || !M || n <= 0 || !X || !y)
    return HBTX_E_INVALID;
  API_GUARD(c, {
    HIPCHK(hipSetDevice(c->device));
    hipStream_t st = c->stream;
    WsUse use{c->ws};
    mlp_samples(c, n, X, y);
    auto &dX = c->ws.X;
    auto &dy = c->ws.y;
    mlp_grad_device(c, M, dX.p, dy.p, nullptr, n);
    double l = 0.0;
    std::vector<XferPart> parts{xfer_to(&l, M->loss.p, sizeof(double))};
    if (grad)
      parts.push_back(xfer_to(grad, M->grad.p, MLP_NPAR * sizeof(float)));
    HIPCHK(c->staging.down(c->device, st, parts));
    if (loss)
      *loss = l / (double)n;
  });
}

int hbtx_mlp_train(hbtx_ctx *c, hbtx_mlp *M, int64_t n, const float *X, const uint8_t *y, int32_t epochs,
                   int32_t batch, float lr, uint64_t seed, double *mean_loss)
{
  if (!c || !M || n <= 0 || !X || !y || epochs <= 0 || batch <= 0)
    return HBTX_E_INVALID;
  API_GUARD(c, {
    HIPCHK(hipSetDevice(c->device));
    REQUIRE(n < (int64_t)0x7fffffff, HBTX_E_INVALID, "too many training samples");
    hipStream_t st = c->stream;
    WsUse use{c->ws};
    mlp_samples(c, n, X, y);
    auto &dX = c->ws.X;
    auto &dy = c->ws.y;
    DArr<int32_t> didx;
    didx.alloc(n);
    std::vector<int32_t> perm(n);
    uint64_t rs = seed;
    const float b1 = 0.9f, b2 = 0.999f;
    double last = 0.0;
    std::vector<double> lbatch;
    for (int ep = 0; ep < epochs; ep++)
    {
      std::iota(perm.begin(), perm.end(), 0);
      for (int64_t i = n - 1; i > 0; i--)
      {
        const int64_t j = (int64_t)(splitmix(rs) % (uint64_t)(i + 1));
        std::swap(perm[i], perm[j]);
      }
      HIPCHK(hipMemcpyAsync(didx.p, perm.data(), n * sizeof(int32_t), hipMemcpyHostToDevice, st));
      DArr<double> losses;
      const int64_t nsteps = (n + batch - 1) / batch;
      losses.alloc(nsteps);
      for (int64_t k = 0; k < nsteps; k++)
      {
        const int64_t b0 = k * batch, nb = std::min<int64_t>(batch, n - b0);
        mlp_grad_device(c, M, dX.p, dy.p, didx.p + b0, nb);
        M->step++;
        const float c1 = 1.f - std::pow(b1, (float)M->step), c2 = 1.f - std::pow(b2, (float)M->step);
        k_mlp_adam<<<(MLP_NPAR + 255) / 256, 256, 0, st>>>(M->master.p, M->m.p, M->v.p, M->grad.p, M->wf.p,
                                                            M->wb.p, lr, b1, b2, 1e-8f, c1, c2);
        HIPCHK(hipMemcpyAsync(losses.p + k, M->loss.p, sizeof(double), hipMemcpyDeviceToDevice, st));
      }
      lbatch.resize(nsteps);
      HIPCHK(hipMemcpyAsync(lbatch.data(), losses.p, nsteps * sizeof(double), hipMemcpyDeviceToHost, st));
      HIPCHK(hipStreamSynchronize(st));
      double tot = 0.0;
      for (double v : lbatch)
        tot += v;
      last = tot / (double)n;
    }
    if (mean_loss)
      *mean_loss = last;
  });
}

int hbtx_mlp_predict(hbtx_ctx *c, hbtx_mlp *M, int64_t n, const float *X, float *logit)
{
  if (!c || !M || n < 0 || (n > 0 && (!X || !logit)))
    return HBTX_E_INVALID;
  API_GUARD(c, {
    HIPCHK(hipSetDevice(c->device));
    if (n == 0)
      return HBTX_OK;
    hipStream_t st = c->stream;
    WsUse use{c->ws};
    mlp_samples(c, n, X, nullptr);
    auto &dX = c->ws.X;
    auto &dl = c->ws.rc;
    dl.alloc(n);
    k_mlp_forward<<<mlp_forward_blocks(n), 256, 0, st>>>(M->wf.p, M->wb.p, dX.p, n, dl.p, nullptr, 0);
    HIPCHK(hipGetLastError());
    HIPCHK(c->staging.down(c->device, st, {xfer_to(logit, dl.p, n * sizeof(float))}));
  });
}

int hbtx_batch_set_previous(hbtx_ctx *c, const int32_t *prev_rank, const uint8_t *prev_bound,
                            const float *prev_energy, const float *prev_com_pos, const float *prev_com_vel,
                            const float *prev_mbound, const float *prev_rscale)
{
  if (!c || !prev_rank || !prev_bound || !prev_energy || !prev_com_pos || !prev_com_vel || !prev_mbound ||
      !prev_rscale)
    return HBTX_E_INVALID;
  API_GUARD(c, {
    HIPCHK(hipSetDevice(c->device));
    Batch &B = c->B;
    REQUIRE(B.n > 0, HBTX_E_INVALID, "no batch loaded");
    hipStream_t st = c->stream;
    const int64_t n = B.n, ns = B.nsub;
    B.prev_rank.alloc(n);
    B.prev_bound.alloc(n);
    B.prev_energy.alloc(n);
    B.prev_com.alloc(6 * ns);
    B.prev_mb.alloc(ns);
    B.prev_rs.alloc(ns);
    std::vector<float> com(6 * ns);
    for (int64_t s = 0; s < ns; s++)
      for (int k = 0; k < 3; k++)
      {
        com[6 * s + k] = prev_com_pos[3 * s + k];
        com[6 * s + 3 + k] = prev_com_vel[3 * s + k];
      }
    auto up = [&](void *dst, const void *src, size_t bytes) {
      HIPCHK(c->staging.up(c->device, st, dst, {xfer_from(0, src, bytes)}));
    };
    up(B.prev_rank.p, prev_rank, n * sizeof(int32_t));
    up(B.prev_bound.p, prev_bound, n);
    up(B.prev_energy.p, prev_energy, n * sizeof(float));
    up(B.prev_com.p, com.data(), 6 * ns * sizeof(float));
    up(B.prev_mb.p, prev_mbound, ns * sizeof(float));
    up(B.prev_rs.p, prev_rscale, ns * sizeof(float));
    B.has_prev = true;
    B.feat_full = false;  // the features depend on the previous outputs
  });
}

int hbtx_batch_features(hbtx_ctx *c, const hbtx_params *prm, float *out_features)
{
  if (!c || !prm)
    return HBTX_E_INVALID;
  API_GUARD(c, {
    HIPCHK(hipSetDevice(c->device));
    Batch &B = c->B;
    REQUIRE(B.n > 0 && B.has_prev, HBTX_E_INVALID, "load a batch and its previous-snapshot outputs first");
    const DevParams P = make_dev_params(*prm);
    hipStream_t st = c->stream;
    const int64_t n = B.n;
    B.feat.alloc(n * MLP_IN);
    View V = make_view(B, 0, n, 0, B.nsub, true);
    PrevArrays A{B.prev_rank.p, B.prev_bound.p, B.prev_energy.p, B.prev_com.p, B.prev_mb.p, B.prev_rs.p};
    k_features<<<blocks_for(n), 256, 0, st>>>(V.S, V.Q, P, A, n, B.feat.p, nullptr, 0);
    HIPCHK(hipGetLastError());
    B.feat_full = true;
    if (out_features)
    {
      HIPCHK(hipMemcpyAsync(out_features, B.feat.p, n * MLP_IN * sizeof(float), hipMemcpyDeviceToHost, st));
      HIPCHK(hipStreamSynchronize(st));
    }
  });
}

int hbtx_batch_get_proposal(hbtx_ctx *c, uint8_t *proposal)
{
  if (!c || !proposal)
    return HBTX_E_INVALID;
  API_GUARD(c, {
    HIPCHK(hipSetDevice(c->device));
    Batch &B = c->B;
    REQUIRE(B.n > 0 && B.has_proposal, HBTX_E_INVALID, "no proposal on the device");
    HIPCHK(hipStreamSynchronize(c->stream));
    HIPCHK(hipMemcpy(proposal, B.proposal.p, B.n, hipMemcpyDeviceToHost));
  });
}

int hbtx_batch_propose(hbtx_ctx *c, hbtx_mlp *M, float threshold, int64_t min_particles, int64_t *nproposed,
                       double *elapsed_ms)
{
  if (!c || !M || !(threshold > 0.f && threshold < 1.f) || min_particles < 0)
    return HBTX_E_INVALID;
  API_GUARD(c, {
    HIPCHK(hipSetDevice(c->device));
    Batch &B = c->B;
    REQUIRE(B.n > 0 && B.feat.p && B.feat_full, HBTX_E_INVALID, "compute the batch features first");
    hipStream_t st = c->stream;
    const int64_t n = B.n;
    B.logit.alloc(n);
    HIPCHK(hipEventRecord(c->wev0, st));
    k_mlp_forward<<<mlp_forward_blocks(n), 256, 0, st>>>(M->wf.p, M->wb.p, B.feat.p, n, B.logit.p, nullptr, 0);
    k_proposal_from_logit<<<blocks_for(n), 256, 0, st>>>(B.logit.p, n, std::log(threshold / (1.f - threshold)),
                                                          B.sub_of.p, B.off.p, min_particles, B.proposal.p);
    HIPCHK(hipEventRecord(c->wev1, st));
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventSynchronize(c->wev1));
    float ms = 0.f;
    HIPCHK(hipEventElapsedTime(&ms, c->wev0, c->wev1));
    if (elapsed_ms)
      *elapsed_ms = ms;
    B.has_proposal = true;
    if (nproposed)
    {
      *nproposed = count_proposed(c, B);
    }
  });
}

int hbtx_batch_warm_proposal(hbtx_ctx *c, const hbtx_params *prm, hbtx_mlp *M, float threshold,
                             int64_t min_particles, int64_t *nproposed, double *elapsed_ms)
{
  if (!c || !prm || !M || !(threshold > 0.f && threshold < 1.f) || min_particles < 0)
    return HBTX_E_INVALID;
  API_GUARD(c, {
    HIPCHK(hipSetDevice(c->device));
    Batch &B = c->B;
    REQUIRE(B.n > 0 && B.has_prev, HBTX_E_INVALID, "load a batch and its previous-snapshot outputs first");
    const DevParams P = make_dev_params(*prm);
    hipStream_t st = c->stream;
    const int64_t n = B.n;
    if (B.egroups_min != min_particles)
    {
      // the 32-particle groups that hold a particle of a subhalo of at least
      // min_particles particles (subhaloes are contiguous, so the list ascends)
      std::vector<int32_t> g;
      int64_t last = -1;
      for (int32_t s = 0; s < B.nsub; s++)
      {
        const int64_t a = B.h_off[s], e = B.h_off[s + 1];
        if (e - a < std::max<int64_t>(min_particles, 1))
          continue;
        for (int64_t q = std::max<int64_t>(a / 32, last + 1); q <= (e - 1) / 32; q++)
          g.push_back((int32_t)q);
        last = (e - 1) / 32;
      }
      B.egroups.alloc(std::max<size_t>(g.size(), 1));
      if (!g.empty())
        HIPCHK(hipMemcpyAsync(B.egroups.p, g.data(), g.size() * sizeof(int32_t), hipMemcpyHostToDevice, st));
      HIPCHK(hipStreamSynchronize(st));
      B.egroups_n = (int64_t)g.size();
      B.egroups_min = min_particles;
    }
    B.feat.alloc(n * MLP_IN);
    B.logit.alloc(n);
    B.feat_full = false;  // only the listed groups' features are written
    View V = make_view(B, 0, n, 0, B.nsub, true);
    PrevArrays A{B.prev_rank.p, B.prev_bound.p, B.prev_energy.p, B.prev_com.p, B.prev_mb.p, B.prev_rs.p};
    HIPCHK(hipEventRecord(c->wev0, st));
    if (B.egroups_n > 0)
    {
      k_features<<<blocks_for(32 * B.egroups_n), 256, 0, st>>>(V.S, V.Q, P, A, n, B.feat.p, B.egroups.p,
                                                               B.egroups_n);
      k_mlp_forward<<<mlp_forward_blocks(32 * B.egroups_n), 256, 0, st>>>(M->wf.p, M->wb.p, B.feat.p, n,
                                                                          B.logit.p, B.egroups.p, B.egroups_n);
    }
    k_proposal_from_logit<<<blocks_for(n), 256, 0, st>>>(B.logit.p, n, std::log(threshold / (1.f - threshold)),
                                                          B.sub_of.p, B.off.p, std::max<int64_t>(min_particles, 1),
                                                          B.proposal.p);
    HIPCHK(hipEventRecord(c->wev1, st));
    HIPCHK(hipGetLastError());
    B.has_proposal = true;
    if (elapsed_ms || nproposed)
      HIPCHK(hipEventSynchronize(c->wev1));
    if (elapsed_ms)
    {
      float ms = 0.f;
      HIPCHK(hipEventElapsedTime(&ms, c->wev0, c->wev1));
      *elapsed_ms = ms;
    }
    if (nproposed)
    {
      *nproposed = count_proposed(c, B);
    }
  });
}

} // extern "C"

extern "C" {

int hbtx_get_tuning(hbtx_ctx *c, int64_t *direct_cutoff, int32_t *walk_chunks)
{
  if (!c)
    return HBTX_E_INVALID;
  if (direct_cutoff)
    *direct_cutoff = c->direct_cutoff;
  if (walk_chunks)
    *walk_chunks = c->walk_chunks;
  return HBTX_OK;
}

int hbtx_set_tuning(hbtx_ctx *c, int64_t direct_cutoff, int32_t walk_chunks)
{
  if (!c || direct_cutoff < 0 || walk_chunks < 1 || walk_chunks > WALK_MAX_CHUNKS)
    return HBTX_E_INVALID;
  c->direct_cutoff = direct_cutoff;
  c->walk_chunks = walk_chunks;
  c->tune_source = "hbtx_set_tuning";
  return HBTX_OK;
}

} // extern "C"
