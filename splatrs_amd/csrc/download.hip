// Models from device planes to records in host memory: a transposing kernel writes chunks of
// records over the bus into a small ring of pinned memory, and the calling thread and a few more
// copy them from there, while later chunks are written, to where the caller wants them.  Bound by
// those copies, mostly the first touch of the caller's pages (4 KB each): 236 MB (a million
// Gaussians) to new pages take one thread 18 ms, two 10 ms, four 7.5 ms and eight 5 ms, the bus
// 4.4 ms; the runtime's own copy into pageable memory, from records staged in device memory,
// took 24 ms (15 ms to pages touched before).  40 steps of a million Gaussians at
// 1920x1080 with the download: 72.9 -> 56.8 ms.
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>

#include "internal.hpp"

namespace splat {

namespace {

constexpr size_t kChunkRows = 4096;  // 0.97 MB
// A further thread per this many chunks, and at most kCopiers: starting one takes about 20 us.
constexpr size_t kChunksPerCopier = 4;
constexpr size_t kCopiers = 7;

struct Chunk {
  const float* planes;
  size_t rows, stride;
  float* out;
};

// The chunks' progress.  Slots are used in turn; a chunk is issued (its kernel and event are on
// the stream) once the one that had its slot before is copied.
struct Progress {
  std::mutex mutex;
  std::condition_variable changed;
  const std::vector<Chunk>& chunks;
  HostRing& ring;
  size_t issued = 0, taken = 0;
  bool closed = false;
  std::vector<char> copied;
  hipError_t error = hipSuccess;

  // Copy the next issued chunk, if there is one (the lock is held on entry and exit).
  bool copy_one(std::unique_lock<std::mutex>& lock) {
    if (taken == issued) return false;
    const size_t c = taken++;
    lock.unlock();
    const size_t slot = c % kHostRingSlots;
    const hipError_t e = hipEventSynchronize(ring.ready[slot]);
    if (e == hipSuccess)
      std::memcpy(chunks[c].out, ring.slot(slot), chunks[c].rows * kParams * sizeof(float));
    lock.lock();
    if (e != hipSuccess) error = e;
    copied[c] = 1;
    changed.notify_all();
    return true;
  }

  void work(int device) {
    (void)hipSetDevice(device);
    std::unique_lock<std::mutex> lock(mutex);
    while (true) {
      if (copy_one(lock)) continue;
      if (closed) return;
      changed.wait(lock);
    }
  }
};

// Ends and joins the threads, also where an exception leaves the issuing loop.
struct Copiers {
  Progress& p;
  std::vector<std::thread> threads;
  ~Copiers() {
    {
      std::lock_guard<std::mutex> lock(p.mutex);
      p.closed = true;
    }
    p.changed.notify_all();
    for (auto& t : threads) t.join();
  }
};

bool on_device(const void* p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();  // not known to the runtime: ordinary memory
    return false;
  }
  return a.type == hipMemoryTypeDevice;
}

}  // namespace

HostRing::~HostRing() {
  for (hipEvent_t e : ready)
    if (e) (void)hipEventDestroy(e);
  if (ptr) (void)hipHostFree(ptr);
}

void HostRing::reserve() {
  for (hipEvent_t& e : ready)
    if (!e) SPLAT_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  if (!ptr)
    SPLAT_HIP(hipHostMalloc(&ptr, kHostRingSlots * kChunkRows * kParams * sizeof(float),
                            hipHostMallocMapped | hipHostMallocCoherent));
}

float* HostRing::slot(size_t k) const {
  return static_cast<float*>(ptr) + k * kChunkRows * kParams;
}

void planes_to_host(splat_ctx* ctx, const HostRecords* arrays, size_t count) {
  std::vector<Chunk> chunks;
  for (size_t k = 0; k < count; k++) {
    const HostRecords& a = arrays[k];
    if (!a.out || a.n == 0) continue;
    if (on_device(a.out)) {  // the runtime checks the range and knows other devices' memory
      DevBuf staging;
      const size_t bytes = a.n * kParams * sizeof(float);
      planes_to_aos(ctx, a.planes, a.n, a.stride, (float*)staging.reserve(bytes));
      SPLAT_HIP(hipMemcpyAsync(a.out, staging.ptr, bytes, hipMemcpyDeviceToHost, ctx->stream));
      SPLAT_HIP(hipStreamSynchronize(ctx->stream));
      continue;
    }
    for (size_t r = 0; r < a.n; r += kChunkRows)
      chunks.push_back({a.planes + r, std::min(kChunkRows, a.n - r), a.stride,
                        a.out + r * kParams});
  }
  HostRing& ring = ctx->ring;
  if (!chunks.empty()) ring.reserve();
  Progress p{.chunks = chunks, .ring = ring, .copied = std::vector<char>(chunks.size(), 0)};
  {
    Copiers copiers{p, {}};
    const size_t want = std::min(kCopiers, chunks.size() / kChunksPerCopier);
    try {
      for (size_t k = 0; k < want; k++)
        copiers.threads.emplace_back([&p, ctx] { p.work(ctx->device); });
    } catch (const std::system_error&) {
      // no more threads to be had: those there are, and this one, do the copies
    }
    std::unique_lock<std::mutex> lock(p.mutex);
    for (size_t c = 0; c < chunks.size(); c++) {
      while (c >= kHostRingSlots && !p.copied[c - kHostRingSlots])
        if (!p.copy_one(lock)) p.changed.wait(lock);
      lock.unlock();
      planes_to_aos(ctx, chunks[c].planes, chunks[c].rows, chunks[c].stride,
                    ring.slot(c % kHostRingSlots));
      SPLAT_HIP(hipEventRecord(ring.ready[c % kHostRingSlots], ctx->stream));
      lock.lock();
      p.issued = c + 1;
      p.changed.notify_one();
    }
    while (p.copy_one(lock)) {
    }
  }
  SPLAT_HIP(p.error);
  SPLAT_HIP(hipStreamSynchronize(ctx->stream));
}

}  // namespace splat
