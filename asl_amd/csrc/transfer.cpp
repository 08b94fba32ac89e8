// Copies between device memory and ordinary (pageable) host memory through
// pinned buffers: the runtime's own path for pageable memory copies to and
// from its staging buffer in turn with the DMA (18 GB/s to the host, 32 GB/s
// from it; 2.5 GB/s for a process's first 17 MB), while pinned memory moves at 56
// GB/s and one core copies 35 to 80 GB/s (5 GB/s into memory that was never
// touched: the first write of a page faults, which only more cores make up for).
// So chunks go through a ring of pinned buffers, the DMA of one beside the host
// copy of others, and larger transfers take a few threads.  Before and after:
// restart of a 120 x 70 x 66 D3Q19 lattice (populations in, 10 steps,
// populations, rho and u out, 100 MB) 7.4 -> 3.4 ms; 100 steps of a 300 x 50 x 50
// D3Q15 duct with rho and u read (13 MB) 2.74 -> 2.50 ms; 20 steps on 160 x 72 x
// 60 with a surface force and u (17 MB) 1.70 -> 1.29 ms.
//
// Which way a transfer goes, us, runtime / ring with events (memory touched
// before, after the process's first ones):
//   to the host     70 KB 11.1 / 17.9, 512 KB 29 / 35, 1 MB 59 / 66, 2 MB 118 /
//                   115, 3 MB 178 / 153, 8 MB 465 / 315, 32 MB 1890 / 930
//   to the device   70 KB 10.5 / 17.8, 1 MB 51 / 59, 4 MB 131 / 183, 8 MB 240 /
//                   315, 24 MB 680 / 708, 32 MB 910 / 905, 48 MB 1757 / 1323; writes of
//                   the populations of three lattices in turn: 10.7 MB 345 / 425,
//                   15.5 MB 566 / 540, 25.5 MB 920 / 805
// - memory that the runtime knows (pinned, on a device): its own path; 3.4 MB
//   into pinned memory take 69 us there and 157 through the ring;
// - to the host, one chunk or less: one buffer and a wait for the stream in
//   place of an event (23 KB 9.5, 70 KB 12, 443 KB 26), unless the host has not
//   waited for more launches than WAIT_STREAM, which makes such a wait dear.  16^3
//   steps and a read of rho, stream / event: 1 step 23.8 / 31.2, 6 steps 39 / 46, 8
//   steps 70 / 53, 40 steps 190 / 165;
// - to the device, less than RING_FROM: the runtime's path.
//
// One ring for the process (RING buffers of CHUNK bytes), held while some
// lattice or trainer exists; a second thread that transfers meanwhile takes
// the runtime's path.
#include "transfer.hpp"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>

namespace aslhip {
namespace {

constexpr size_t CHUNK = 2u << 20;
constexpr int RING = 8;                      // buffers: chunks in flight and chunks being copied
constexpr int COPIERS = 4;                   // copy threads
constexpr size_t THREADS_FROM = 4u << 20;    // smaller transfers end before a thread would pay
constexpr int WAIT_STREAM = 6;               // launches up to which waiting for the stream beats an event
constexpr size_t RING_FROM = 14u << 20;      // to the device: smaller transfers take the runtime's path
constexpr int MAX_DEVICES = 64;

std::mutex ring_mu;   // held during a transfer
int holders = 0;
char *ring = nullptr;
hipEvent_t ring_ev[MAX_DEVICES][RING] = {};

void release_ring() {
  for (auto &dev : ring_ev)
    for (auto &e : dev)
      if (e) {
        (void)hipEventDestroy(e);
        e = nullptr;
      }
  if (ring) (void)hipHostFree(ring);
  ring = nullptr;
}

// Ordinary host memory, nothing that the runtime allocated or registered.
bool pageable(const void *p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
  (void)hipGetLastError();
  return true;
}

// The ring and the current device's events (null: use the runtime's path, also
// for a stream of another device, on which they cannot be recorded).
hipEvent_t *ring_ready(hipStream_t s) {
  int dev = 0, of = 0;
  if (hipGetDevice(&dev) != hipSuccess || hipStreamGetDevice(s, &of) != hipSuccess || of != dev || dev < 0 ||
      dev >= MAX_DEVICES)
    return nullptr;
  if (!ring && hipHostMalloc(&ring, RING * CHUNK, hipHostMallocPortable) != hipSuccess) {
    (void)hipGetLastError();
    ring = nullptr;
    return nullptr;
  }
  for (auto &e : ring_ev[dev])
    if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
      (void)hipGetLastError();
      e = nullptr;
      return nullptr;
    }
  return ring_ev[dev];
}

// The host side of a transfer: copies chunks between the ring and the host's
// memory.  Thread w takes chunks w, w + COPIERS, ..., each once it is allowed;
// without threads the caller copies.
struct Copiers {
  char *host;
  size_t n;
  bool to_ring;
  std::atomic<long> allowed[COPIERS], done[COPIERS];  // last chunk of each thread
  std::atomic<bool> stop{false};
  std::thread th[COPIERS];
  bool running = false;

  Copiers(char *h, size_t bytes, bool in) : host(h), n(bytes), to_ring(in) {
    for (int w = 0; w < COPIERS; ++w) {
      allowed[w] = -1;
      done[w] = -1;
    }
    if (n < THREADS_FROM || std::thread::hardware_concurrency() < 2 * COPIERS) return;
    try {
      for (int w = 0; w < COPIERS; ++w) th[w] = std::thread([this, w] { work(w); });
      running = true;
    } catch (const std::exception &) {  // no thread, or no memory for one, to be had
      finish();
    }
  }
  ~Copiers() { finish(); }
  Copiers(const Copiers &) = delete;
  Copiers &operator=(const Copiers &) = delete;

  void copy(long k) const {
    char *b = ring + (k % RING) * CHUNK, *h = host + k * CHUNK;
    const size_t m = std::min(CHUNK, n - k * CHUNK);
    if (to_ring)
      std::memcpy(b, h, m);
    else
      std::memcpy(h, b, m);
  }
  void work(int w) {
    for (long k = w; static_cast<size_t>(k) * CHUNK < n; k += COPIERS) {
      while (allowed[w].load(std::memory_order_acquire) < k) {
        if (stop.load(std::memory_order_relaxed)) return;
        std::this_thread::yield();
      }
      copy(k);
      done[w].store(k, std::memory_order_release);
    }
  }
  // Chunk k may be copied (each chunk once, in order).
  void allow(long k) {
    if (running)
      allowed[k % COPIERS].store(k, std::memory_order_release);
    else
      copy(k);
  }
  // Until chunk k, which has been allowed, is copied.
  void wait(long k) const {
    if (!running) return;
    while (done[k % COPIERS].load(std::memory_order_acquire) < k) std::this_thread::yield();
  }
  void finish() {
    stop = true;
    for (auto &t : th)
      if (t.joinable()) t.join();
    running = false;
  }
};

}  // namespace

void transfer_hold() {
  std::lock_guard<std::mutex> lock(ring_mu);
  ++holders;
}

void transfer_drop() {
  std::lock_guard<std::mutex> lock(ring_mu);
  if (--holders == 0) release_ring();
}

hipError_t to_host(void *dst, const void *src, size_t n, hipStream_t s, int *launches) {
  if (n == 0) return hipStreamSynchronize(s);
  std::unique_lock<std::mutex> lock(ring_mu, std::defer_lock);
  hipEvent_t *ev = pageable(dst) && lock.try_lock() ? ring_ready(s) : nullptr;
  if (!ev) {
    const hipError_t e = hipStreamSynchronize(s);
    return e != hipSuccess ? e : hipMemcpy(dst, src, n, hipMemcpyDeviceToHost);
  }
  if (n <= CHUNK) {
    hipError_t e = hipMemcpyAsync(ring, src, n, hipMemcpyDeviceToHost, s);
    const bool event = launches && *launches > WAIT_STREAM;
    if (e == hipSuccess && event) e = hipEventRecord(ev[0], s);
    const hipError_t w = e == hipSuccess && event ? hipEventSynchronize(ev[0]) : hipStreamSynchronize(s);
    if (launches && !event) *launches = 0;
    if (e == hipSuccess) e = w;
    if (e == hipSuccess) std::memcpy(dst, ring, n);
    return e;
  }
  const long chunks = static_cast<long>((n + CHUNK - 1) / CHUNK);
  hipError_t e = hipSuccess;
  auto issue = [&](long k) {
    const size_t o = k * CHUNK;
    e = hipMemcpyAsync(ring + (k % RING) * CHUNK, static_cast<const char *>(src) + o, std::min(CHUNK, n - o),
                       hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipEventRecord(ev[k % RING], s);
  };
  Copiers c(static_cast<char *>(dst), n, false);
  // at chunk k: k .. k + DEPTH - 1 in flight, the copies of k - RING + DEPTH and later ones still at work
  constexpr long DEPTH = RING - COPIERS;
  long sent = 0;
  for (long k = 0; k < chunks && e == hipSuccess; ++k) {
    for (; sent < chunks && sent < k + DEPTH && e == hipSuccess; ++sent) {
      if (sent >= RING) c.wait(sent - RING);  // its buffer
      issue(sent);
    }
    if (e == hipSuccess) e = hipEventSynchronize(ev[k % RING]);
    if (e == hipSuccess) c.allow(k);
  }
  if (e != hipSuccess) {
    (void)hipStreamSynchronize(s);  // nothing may still write to the ring
    return e;
  }
  for (long k = std::max(0L, chunks - COPIERS); k < chunks; ++k) c.wait(k);
  return hipSuccess;
}

hipError_t to_device(void *dst, const void *src, size_t n, hipStream_t s, bool wait) {
  if (n == 0) return hipSuccess;
  std::unique_lock<std::mutex> lock(ring_mu, std::defer_lock);
  hipEvent_t *ev = n >= RING_FROM && pageable(src) && lock.try_lock() ? ring_ready(s) : nullptr;
  if (!ev) {
    const hipError_t e = hipMemcpyAsync(dst, src, n, hipMemcpyHostToDevice, s);
    return e != hipSuccess || !wait ? e : hipStreamSynchronize(s);
  }
  const long chunks = static_cast<long>((n + CHUNK - 1) / CHUNK);
  hipError_t e = hipSuccess;
  Copiers c(const_cast<char *>(static_cast<const char *>(src)), n, true);
  long given = 0;  // chunks whose buffer the copiers have been given
  for (long k = 0; k < chunks && e == hipSuccess; ++k) {
    for (; given < chunks && given < k + (c.running ? COPIERS : 1) && e == hipSuccess; ++given) {
      if (given >= RING) e = hipEventSynchronize(ev[given % RING]);  // its last DMA
      if (e == hipSuccess) c.allow(given);
    }
    if (e != hipSuccess) break;
    c.wait(k);
    const size_t o = k * CHUNK;
    e = hipMemcpyAsync(static_cast<char *>(dst) + o, ring + (k % RING) * CHUNK, std::min(CHUNK, n - o),
                       hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipEventRecord(ev[k % RING], s);
  }
  // the ring is another transfer's next
  const hipError_t w = hipStreamSynchronize(s);
  return e != hipSuccess ? e : w;
}

}  // namespace aslhip
