// Copies of the caller's (pageable) arrays to and from the device through pinned
// staging.
//
// The runtime copies pageable memory through staging of its own on one thread: 26
// to 33 GB/s up and 11 to 17 GB/s down on the MI355X host (down, page faults of the
// output arrays add to it), where the link carries 57 GB/s each way.  Here a few
// threads take chunks of the transfer: each fills (or empties) pinned slots of its
// own while its other slots are on the link.  The threads live for one transfer;
// small transfers stay on the calling thread.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <functional>
#include <thread>
#include <vector>

namespace hbtx
{

// A copy costs about 11 us beside its bytes, so chunks are large: 352 MB went up in
// 9.7 ms by 1 MiB chunks, 7.7 ms by 2 MiB and 7.0 ms by 4 MiB (6.2 ms at the link's
// rate); 8 MiB and six or eight threads gave nothing more.
constexpr size_t XFER_CHUNK = 4 << 20; // bytes a slot holds
constexpr int XFER_THREADS = 4;
constexpr int XFER_SLOTS = 2 * XFER_THREADS; // 32 MiB pinned
constexpr size_t XFER_SMALL = 2 << 20;       // at or below: the calling thread alone

// A piece of a transfer: bytes at dev (up: an offset in the destination block),
// and what bytes [off, off + len) of it are on the host: a plain copy, or a
// conversion element by element (off and len are multiples of 4 then).
struct XferPart
{
  size_t at;   // up: offset in the block
  void *dev;   // down: source
  size_t bytes;
  std::function<void(char *slot, size_t off, size_t len)> host;
};

inline XferPart xfer_from(size_t at, const void *src, size_t bytes)
{
  return {at, nullptr, bytes,
          [src](char *slot, size_t off, size_t len) { std::memcpy(slot, (const char *)src + off, len); }};
}
inline XferPart xfer_to(void *dst, const void *dev, size_t bytes)
{
  return {0, const_cast<void *>(dev), bytes,
          [dst](char *slot, size_t off, size_t len) { std::memcpy((char *)dst + off, slot, len); }};
}

// Small transfers as one kernel that reads or writes the pinned slot itself over the
// link (a copy of its own costs about 11 us, and waiting for it as much again).
struct XferSmall
{
  static constexpr int MAX_PARTS = 6;
  static constexpr size_t MAX_BYTES = 128 << 10;
  int nparts;
  uint32_t *dst[MAX_PARTS];
  const uint32_t *src[MAX_PARTS];
  uint32_t words[MAX_PARTS];
};
__global__ void k_xfer_small(XferSmall X)
{
  for (int k = 0; k < X.nparts; k++)
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < X.words[k]; i += gridDim.x * blockDim.x)
      X.dst[k][i] = X.src[k][i];
}

// The pinned slots of one context, made at the first transfer and released with the
// context.  One transfer at a time (a context serves one host thread).
struct Staging
{
  char *pinned = nullptr;
  hipEvent_t ev[XFER_SLOTS] = {};
  unsigned small_slot = 0;

  hipError_t init()
  {
    if (pinned)
      return hipSuccess;
    hipError_t e = hipHostMalloc((void **)&pinned, XFER_CHUNK * XFER_SLOTS, hipHostMallocDefault);
    for (int k = 0; e == hipSuccess && k < XFER_SLOTS; k++)
      e = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
    if (e != hipSuccess)
      release();
    return e;
  }
  void release()
  {
    for (auto &x : ev)
    {
      if (x)
        (void)hipEventDestroy(x);
      x = nullptr;
    }
    if (pinned)
      (void)hipHostFree(pinned);
    pinned = nullptr;
  }
  ~Staging()
  {
    release();
  }

  char *slot(int s) const
  {
    return pinned + XFER_CHUNK * (size_t)s;
  }
  static int threads_for(size_t bytes, size_t nchunks)
  {
    const size_t hw = std::max(1u, std::thread::hardware_concurrency());
    return (bytes <= XFER_SMALL) ? 1 : (int)std::min({(size_t)XFER_THREADS, hw, nchunks});
  }
  // work(t) on nt threads (this one is t = 0); fewer if no more can be made
  template <class F>
  static void on_threads(int nt, F &&work)
  {
    std::vector<std::thread> th;
    th.reserve(nt);
    try
    {
      for (int t = 1; t < nt; t++)
        th.emplace_back(work, t);
    }
    catch (...)
    {
      // (the threads that are there take all the chunks)
    }
    work(0);
    for (auto &x : th)
      x.join();
  }

  // Fills the device block dev from the parts (ascending offsets; the gaps between
  // them stay undefined).  Returns once every part has been read and its copies are
  // enqueued on the stream; a slot is reused only when its copy has ended.
  hipError_t up(int device, hipStream_t stream, void *dev, const std::vector<XferPart> &parts)
  {
    hipError_t e0 = init();
    if (e0 != hipSuccess || parts.empty())
      return e0;
    const size_t total = parts.back().at + parts.back().bytes;
    if (total <= XferSmall::MAX_BYTES)
    {
      const int s = small_slot++ % XFER_SLOTS;
      hipError_t e = hipEventSynchronize(ev[s]);
      if (e != hipSuccess)
        return e;
      for (const XferPart &p : parts)
        p.host(slot(s) + p.at, 0, p.bytes);
      XferSmall X;
      X.nparts = 1;
      X.dst[0] = (uint32_t *)dev;
      X.src[0] = (const uint32_t *)slot(s);
      X.words[0] = (uint32_t)((total + 3) / 4); // (device blocks are whole words long)
      k_xfer_small<<<std::max(1u, (X.words[0] + 1023) / 1024), 256, 0, stream>>>(X);
      e = hipGetLastError();
      return (e == hipSuccess) ? hipEventRecord(ev[s], stream) : e;
    }
    const size_t nc = (total + XFER_CHUNK - 1) / XFER_CHUNK;
    const int nt = threads_for(total, nc);
    std::atomic<size_t> next{0};
    std::atomic<int> err{(int)hipSuccess};
    on_threads(nt, [&](int t) {
      hipError_t e = hipSetDevice(device);
      int s = t; // this thread's slots: t, t + nt, ...
      while (e == hipSuccess && err.load() == (int)hipSuccess)
      {
        const size_t k = next.fetch_add(1);
        if (k >= nc)
          break;
        const size_t a = k * XFER_CHUNK, b = std::min(total, a + XFER_CHUNK);
        e = hipEventSynchronize(ev[s]); // (its last copy; an event never recorded is over)
        if (e != hipSuccess)
          break;
        for (const XferPart &p : parts)
        {
          const size_t lo = std::max(a, p.at), hi = std::min(b, p.at + p.bytes);
          if (lo < hi)
            p.host(slot(s) + (lo - a), lo - p.at, hi - lo);
        }
        e = hipMemcpyAsync((char *)dev + a, slot(s), b - a, hipMemcpyHostToDevice, stream);
        if (e == hipSuccess)
          e = hipEventRecord(ev[s], stream);
        s = (s + nt < XFER_SLOTS) ? s + nt : t;
      }
      if (e != hipSuccess)
        err.store((int)e);
    });
    const hipError_t e = (hipError_t)err.load();
    if (e != hipSuccess)
      (void)hipStreamSynchronize(stream);
    return e;
  }

  // Brings every part to the host, after the stream's earlier work; returns once the
  // host arrays are written.
  hipError_t down(int device, hipStream_t stream, const std::vector<XferPart> &parts)
  {
    hipError_t e0 = init();
    if (e0 != hipSuccess)
      return e0;
    struct Chunk
    {
      const XferPart *p;
      size_t off, len;
    };
    std::vector<Chunk> chunks;
    size_t total = 0;
    for (const XferPart &p : parts)
      for (size_t o = 0; o < p.bytes; o += XFER_CHUNK)
      {
        chunks.push_back({&p, o, std::min(XFER_CHUNK, p.bytes - o)});
        total += chunks.back().len;
      }
    bool words = parts.size() <= XferSmall::MAX_PARTS;
    for (const XferPart &p : parts)
      words = words && (p.bytes & 3) == 0;
    if (total <= XferSmall::MAX_BYTES && words)
    {
      const int s = small_slot++ % XFER_SLOTS;
      hipError_t e = hipEventSynchronize(ev[s]);
      if (e != hipSuccess)
        return e;
      XferSmall X;
      X.nparts = (int)parts.size();
      size_t at = 0;
      for (int k = 0; k < X.nparts; k++)
      {
        X.dst[k] = (uint32_t *)(slot(s) + at);
        X.src[k] = (const uint32_t *)parts[k].dev;
        X.words[k] = (uint32_t)(parts[k].bytes / 4);
        at += parts[k].bytes;
      }
      k_xfer_small<<<std::max<size_t>(1, (total + 4095) / 4096), 256, 0, stream>>>(X);
      e = hipGetLastError();
      if (e == hipSuccess)
        e = hipStreamSynchronize(stream);
      if (e == hipSuccess)
        for (int k = 0; k < X.nparts; k++)
          parts[k].host((char *)X.dst[k], 0, parts[k].bytes);
      return e;
    }
    const size_t nc = chunks.size();
    const int nt = threads_for(total, nc);
    std::atomic<size_t> next{0};
    std::atomic<int> err{(int)hipSuccess};
    on_threads(nt, [&](int t) {
      hipError_t e = hipSetDevice(device);
      // this thread's slots in turn, with the chunk each one's copy carries
      const int mine = (XFER_SLOTS - t + nt - 1) / nt;
      size_t chunk_of[XFER_SLOTS];
      int head = 0, flying = 0; // oldest of the copies in flight, and their number
      bool more = true;
      while (e == hipSuccess && err.load() == (int)hipSuccess)
      {
        while (more && flying < mine && e == hipSuccess)
        {
          const size_t k = next.fetch_add(1);
          if (k >= nc)
          {
            more = false;
            break;
          }
          const int i = (head + flying) % mine, s = t + i * nt;
          e = hipEventSynchronize(ev[s]); // (an earlier transfer's copy)
          if (e == hipSuccess)
            e = hipMemcpyAsync(slot(s), (char *)chunks[k].p->dev + chunks[k].off, chunks[k].len,
                               hipMemcpyDeviceToHost, stream);
          if (e == hipSuccess)
            e = hipEventRecord(ev[s], stream);
          chunk_of[i] = k;
          flying++;
        }
        if (e != hipSuccess || flying == 0)
          break;
        const int s = t + head * nt;
        e = hipEventSynchronize(ev[s]);
        if (e != hipSuccess)
          break;
        const Chunk &c = chunks[chunk_of[head]];
        c.p->host(slot(s), c.off, c.len);
        head = (head + 1) % mine;
        flying--;
      }
      if (e != hipSuccess)
        err.store((int)e);
    });
    const hipError_t e = (hipError_t)err.load();
    if (e != hipSuccess)
      (void)hipStreamSynchronize(stream); // no copy may still be writing a slot
    return e;
  }
};

} // namespace hbtx
