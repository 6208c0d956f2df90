// kmi_xfer.hip — host transfers through pinned buffers kept by the context.
//
// A copy between the device and ordinary (pageable) host memory runs at a fraction of the
// link: the runtime stages it on one thread, and a result array the host has just allocated
// takes a page fault per page on the way (134 MB to the host: 2.4 ms into pinned memory,
// 7.3 ms into touched pages, 12 ms into a new array).  Here a kernel stores into a ring of
// pinned chunks while a few host threads move the chunks that have arrived to their
// destination, first touch included (2.7 ms and 3.4 ms), or for uploads the threads fill chunks
// that the runtime copies to the device.
#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include "kmi_internal.h"

namespace kmi {

namespace {
constexpr size_t kChunk = 2u << 20;      // bytes of a pinned chunk
constexpr int kSlots = 12;               // chunks in the ring: 24 MB
constexpr size_t kAlone = 1u << 20;      // transfers up to this run on the calling thread
constexpr unsigned kHelpers = 5;         // beside the calling thread; six copy faster than the link

// A piece costs a few µs besides its 18 µs per MB, so small transfers are cut little; pieces start
// on 256 bytes.
inline size_t piece_bytes(size_t total) {
  if (total <= kAlone) return kAlone;
  if (total <= (4u << 20)) return ((total + 1) / 2 + 255) / 256 * 256;
  return std::min(kChunk, (total / 4 + 255) / 256 * 256);
}

struct Piece {
  char* dev;
  size_t bytes;
  size_t at;  // offset in the host arrays, laid end to end
};

inline void relax() { __builtin_ia32_pause(); }

// Between the device and a chunk of the ring, 16 bytes a lane, by loads or stores across the link.
// To the host 55 GB/s; the runtime's copy leaves the choice of a copy engine to what is idle at that
// moment, and on some of them a stream stays at 11 GB/s for all its copies: 17.6 MB 490 or 1,520 µs,
// here always 420.  From the host the loads run at 40 GB/s, the runtime's copies at 44, but a single
// piece arrives sooner (256 KB 23.3 → 20.2 µs a call).
__global__ void __launch_bounds__(256) k_ring_copy(const char* __restrict__ src, char* __restrict__ dst, unsigned bytes) {
  const unsigned n = bytes / 16;
  for (unsigned i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256)
    reinterpret_cast<uint4*>(dst)[i] = reinterpret_cast<const uint4*>(src)[i];
  if (blockIdx.x == 0 && threadIdx.x < bytes % 16) dst[n * 16 + threadIdx.x] = src[n * 16 + threadIdx.x];
}

// dev: the side on the device (the chunk is aligned).
hipError_t ring_copy(char* dst, const char* src, const char* dev, size_t bytes, hipStream_t stream) {
  if (reinterpret_cast<uintptr_t>(dev) % 16) return hipMemcpyAsync(dst, src, bytes, hipMemcpyDefault, stream);
  const unsigned groups = unsigned(std::min<size_t>(512, (bytes + 4095) / 4096));
  hipLaunchKernelGGL(k_ring_copy, dim3(groups), dim3(256), 0, stream, src, dst, unsigned(bytes));
  return hipGetLastError();
}
}  // namespace

struct HostCopier {
  std::mutex call;   // one transfer at a time per context
  std::mutex setup;
  char* ring = nullptr;
  hipEvent_t ev[kSlots] = {};
  bool pending[kSlots] = {};  // ev[k] guards a device copy out of slot k

  // the transfer in progress, shared with the helpers
  std::vector<Piece> pieces;
  const HostSeg* seg = nullptr;
  std::vector<size_t> start;  // offset of each host array, and the total
  bool to_host = true;
  std::atomic<size_t> ready{0};  // pieces [0, ready) may be moved
  std::atomic<size_t> next{0};   // next piece to take
  std::vector<std::atomic<unsigned char>> moved;
  std::atomic<bool> stop{false};  // the transfer is over
  std::atomic<unsigned> inside{0};  // helpers that may still read the fields above

  std::mutex m;
  std::condition_variable wake;
  uint64_t round = 0;
  bool quit = false;
  std::vector<std::thread> helpers;

  char* slot(size_t k) { return ring + (k % kSlots) * kChunk; }

  // Moves one piece that is ready; false when none is.
  bool move_one() {
    size_t k = next.load(std::memory_order_relaxed);
    do {
      if (k >= ready.load(std::memory_order_acquire)) return false;
    } while (!next.compare_exchange_weak(k, k + 1, std::memory_order_acq_rel));
    const Piece& p = pieces[k];
    size_t i = size_t(std::upper_bound(start.begin(), start.end(), p.at) - start.begin()) - 1;
    for (size_t o = 0; o < p.bytes; ++i) {  // a piece may span host arrays
      const size_t in = p.at + o - start[i], n = std::min(p.bytes - o, start[i + 1] - start[i] - in);
      char* const host = static_cast<char*>(seg[i].host) + in;
      if (to_host) std::memcpy(host, slot(k) + o, n);
      else std::memcpy(slot(k) + o, host, n);
      o += n;
    }
    moved[k].store(1, std::memory_order_release);
    return true;
  }

  void help() {
    uint64_t seen = 0;
    std::unique_lock<std::mutex> lock(m);
    for (;;) {
      wake.wait(lock, [&] { return quit || round != seen; });
      if (quit) return;
      seen = round;
      if (stop.load(std::memory_order_acquire)) continue;  // woken after the transfer ended
      inside.fetch_add(1, std::memory_order_acq_rel);
      lock.unlock();
      while (!stop.load(std::memory_order_acquire))
        if (!move_one()) relax();
      inside.fetch_sub(1, std::memory_order_acq_rel);
      lock.lock();
    }
  }

  hipError_t prepare() {
    std::lock_guard<std::mutex> lock(setup);
    if (ring) return hipSuccess;
    hipError_t e = hipHostMalloc(reinterpret_cast<void**>(&ring), kSlots * kChunk, hipHostMallocDefault);
    for (int k = 0; k < kSlots && e == hipSuccess; ++k)
      if (!ev[k]) e = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
    if (e != hipSuccess) {
      if (ring) (void)hipHostFree(ring);
      ring = nullptr;
    }
    return e;
  }

  void start_helpers() {
    if (!helpers.empty()) return;
    const unsigned n = std::min(kHelpers, std::max(1u, std::thread::hardware_concurrency()) - 1u);
    try {
      for (unsigned k = 0; k < n; ++k) helpers.emplace_back([this] { help(); });
    } catch (...) {
      // fewer helpers (or none): the calling thread moves what they do not
    }
  }

  hipError_t free_slot(size_t k) {
    const int q = int(k % kSlots);
    if (!pending[q]) return hipSuccess;
    pending[q] = false;
    return hipEventSynchronize(ev[q]);
  }

  // The pieces in order; `stream` carries the device side.
  hipError_t pump(hipStream_t stream) {
    const size_t n = pieces.size();
    hipError_t e = hipSuccess;
    size_t issued = 0;
    auto wait_moved = [&](size_t k) {
      while (!moved[k].load(std::memory_order_acquire))
        if (!move_one()) relax();
    };
    if (to_host) {
      auto issue = [&]() -> hipError_t {
        const size_t k = issued;
        if (hipError_t x = free_slot(k); x != hipSuccess) return x;
        hipError_t x = ring_copy(slot(k), pieces[k].dev, pieces[k].dev, pieces[k].bytes, stream);
        if (x == hipSuccess && n > 1) x = hipEventRecord(ev[k % kSlots], stream);
        if (x == hipSuccess) ++issued;
        return x;
      };
      while (issued < n && issued < size_t(kSlots) && e == hipSuccess) e = issue();
      size_t arrived = 0;
      if (n == 1 && e == hipSuccess) {  // one piece: the stream is waited for, not an event
        e = hipStreamSynchronize(stream);
        if (e == hipSuccess) ready.store(arrived = 1, std::memory_order_release);
      }
      while (arrived < n && e == hipSuccess) {
        e = hipEventSynchronize(ev[arrived % kSlots]);
        if (e != hipSuccess) break;
        ready.store(++arrived, std::memory_order_release);
        while (issued < n && issued - (kSlots - 1) <= arrived && e == hipSuccess) {
          if (!moved[issued - kSlots].load(std::memory_order_acquire)) {
            if (arrived < issued) break;  // more is on its way: the slot frees meanwhile
            wait_moved(issued - kSlots);
          }
          e = issue();
        }
      }
      if (e == hipSuccess)
        for (size_t k = 0; k < n; ++k) wait_moved(k);
      else
        (void)hipStreamSynchronize(stream);  // no copy into the ring stays in flight
    } else {
      size_t open = 0;  // pieces the helpers may fill
      while (issued < n && e == hipSuccess) {
        while (open < n && open < issued + kSlots && e == hipSuccess) {
          // a slot whose device copy is still running is opened only when it is the next
          // one needed, so that the others go on
          if (pending[open % kSlots] && open > issued) {
            const hipError_t q = hipEventQuery(ev[open % kSlots]);
            if (q == hipErrorNotReady) break;
            if (q != hipSuccess) { e = q; break; }
          }
          e = free_slot(open);
          if (e == hipSuccess) ready.store(++open, std::memory_order_release);
        }
        if (e != hipSuccess) break;
        wait_moved(issued);
        const size_t k = issued;
        e = n == 1 ? ring_copy(pieces[k].dev, slot(k), pieces[k].dev, pieces[k].bytes, stream)
                   : hipMemcpyAsync(pieces[k].dev, slot(k), pieces[k].bytes, hipMemcpyHostToDevice, stream);
        if (e == hipSuccess) e = hipEventRecord(ev[k % kSlots], stream);
        if (e == hipSuccess) pending[k % kSlots] = true, ++issued;
      }
    }
    return e;
  }

  hipError_t transfer(hipStream_t stream, const HostSeg* segs, int count, bool down) {
    std::lock_guard<std::mutex> one(call);
    seg = segs;
    start.assign(1, 0);
    for (int i = 0; i < count; ++i) start.push_back(start.back() + segs[i].bytes);
    const size_t total = start.back();
    if (total == 0) return down ? hipStreamSynchronize(stream) : hipSuccess;
    hipError_t e = hipSuccess;
    pieces.clear();
    for (int i = 0; i < count;) {  // runs of arrays that lie end to end on the device
      int j = i + 1;
      while (j < count && static_cast<char*>(segs[j].dev) == static_cast<char*>(segs[j - 1].dev) + segs[j - 1].bytes) ++j;
      const size_t run = start[j] - start[i], piece = piece_bytes(run);
      for (size_t o = 0; o < run; o += piece)
        pieces.push_back(Piece{static_cast<char*>(segs[i].dev) + o, std::min(piece, run - o), start[i] + o});
      i = j;
    }
    to_host = down;
    std::vector<std::atomic<unsigned char>> flags(pieces.size());
    for (auto& f : flags) f.store(0, std::memory_order_relaxed);
    moved.swap(flags);
    ready.store(0, std::memory_order_relaxed);
    next.store(0, std::memory_order_relaxed);
    const bool alone = total <= kAlone;
    if (!alone) {
      start_helpers();
      {
        std::lock_guard<std::mutex> lock(m);
        stop.store(false, std::memory_order_release);
        ++round;
      }
      wake.notify_all();
    }
    e = pump(stream);
    if (!alone) {
      {
        std::lock_guard<std::mutex> lock(m);  // a helper that wakes from here on sees stop
        stop.store(true, std::memory_order_release);
      }
      while (inside.load(std::memory_order_acquire)) relax();
    }
    return e;
  }

  ~HostCopier() {
    {
      std::lock_guard<std::mutex> lock(m);
      quit = true;
    }
    wake.notify_all();
    for (auto& t : helpers) t.join();
    for (int k = 0; k < kSlots; ++k) {
      if (pending[k]) (void)hipEventSynchronize(ev[k]);
      if (ev[k]) (void)hipEventDestroy(ev[k]);
    }
    if (ring) (void)hipHostFree(ring);
  }
};

HostCopier* host_copier_create() { return new (std::nothrow) HostCopier(); }
void host_copier_destroy(HostCopier* c) { delete c; }

// The runtime's own path.
static hipError_t plain_copy(hipStream_t stream, const HostSeg* seg, int count, bool down) {
  hipError_t e = hipSuccess;
  for (int s = 0; s < count && e == hipSuccess; ++s)
    if (seg[s].bytes)
      e = down ? hipMemcpyAsync(seg[s].host, seg[s].dev, seg[s].bytes, hipMemcpyDeviceToHost, stream)
               : hipMemcpyAsync(seg[s].dev, seg[s].host, seg[s].bytes, hipMemcpyHostToDevice, stream);
  if (!down) return e;
  const hipError_t w = hipStreamSynchronize(stream);
  return e != hipSuccess ? e : w;
}

// Uploads that the ring makes faster.  The runtime stages small arrays at 2.3 GB/s, now and then up to
// 1 MB, and larger ones it pins and copies from at 37 GB/s, which the ring's extra pass reaches once that
// drops to 31 (µs plain / ring: 64 KB 33 / 15, 256 KB 17 or 107 / 20, 1 MB 43 / 52, 2 MB 71 / 98, 16 MB
// 450 / 514, 48 MB 1,570 / 1,340, 128 MB 4,270 / 3,390).
static bool ring_uploads(const HostSeg* seg, int count) {
  size_t total = 0;
  for (int s = 0; s < count; ++s) total += seg[s].bytes;
  return total <= kAlone || total > (32u << 20);
}

static hipError_t copy(kmi_ctx* ctx, const HostSeg* seg, int count, bool down) {
  if (!down && !ring_uploads(seg, count)) return plain_copy(ctx->stream, seg, count, down);
  try {
    if (ctx->copier && ctx->copier->prepare() == hipSuccess)
      return ctx->copier->transfer(ctx->stream, seg, count, down);
  } catch (...) {  // host memory: nothing has been queued yet
  }
  (void)hipGetLastError();  // no pinned memory left
  return plain_copy(ctx->stream, seg, count, down);
}

hipError_t copy_to_host(kmi_ctx* ctx, const HostSeg* seg, int count) { return copy(ctx, seg, count, true); }
hipError_t copy_to_device(kmi_ctx* ctx, const HostSeg* seg, int count) { return copy(ctx, seg, count, false); }

}  // namespace kmi
