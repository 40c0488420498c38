// Staged copies of large pageable host vectors.
//
// A pageable hipMemcpyAsync moves the data through the runtime's own staging
// buffer with one host thread: 12-15 GB/s, and a vector that the caller has
// just allocated is page-faulted in by that thread as well.  Here up to 8
// threads copy 2 MiB chunks to and from pinned buffers (two each, so a
// thread's host copy runs beside the DMA of its other buffer).
//
// Domain-wall M^dag M of 16^3x32, Ls 16, on host vectors (201 MB each way, a
// fresh output array): 27.5 -> 12.4 ms; a 12-source Wilson propagator (302 MB
// out) 168 -> 145 ms.
#include "hostcopy.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

namespace cpship {

namespace {

struct Ring {
  char* pinned = nullptr;   // WORKERS * BUFS chunks
  hipEvent_t done[HostStager::WORKERS * HostStager::BUFS] = {};
  int device = 0;
  ~Ring() {
    for (hipEvent_t e : done)
      if (e) (void)hipEventDestroy(e);
    if (pinned) (void)hipHostFree(pinned);
  }
};

constexpr size_t MAX_IDLE = 2;
std::mutex pool_mu;
// (never destroyed: at exit the runtime may be gone before it)
std::vector<std::unique_ptr<Ring>>& idle = *new std::vector<std::unique_ptr<Ring>>;
int owners = 0;

// a ring of the current device, or nullptr
std::unique_ptr<Ring> take_ring() {
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return nullptr;
  {
    std::lock_guard<std::mutex> lk(pool_mu);
    for (size_t k = 0; k < idle.size(); k++)
      if (idle[k]->device == device) {
        std::unique_ptr<Ring> r = std::move(idle[k]);
        idle.erase(idle.begin() + (long)k);
        return r;
      }
  }
  std::unique_ptr<Ring> r(new (std::nothrow) Ring);
  if (!r) return nullptr;
  r->device = device;
  for (hipEvent_t& e : r->done)
    if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
      e = nullptr;
      (void)hipGetLastError();
      return nullptr;
    }
  void* p = nullptr;
  if (hipHostMalloc(&p, HostStager::WORKERS * HostStager::BUFS * HostStager::CHUNK, hipHostMallocDefault) !=
      hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  r->pinned = static_cast<char*>(p);
  return r;
}

// (one that the pool does not keep is freed on return)
void give_ring(std::unique_ptr<Ring> r) {
  std::lock_guard<std::mutex> lk(pool_mu);
  if (owners > 0 && idle.size() < MAX_IDLE) idle.push_back(std::move(r));   // capacity reserved by the first owner
}

// Every chunk is taken by one worker; a worker's failure stops the others and
// is returned.
hipError_t run(Ring& ring, char* dev, char* host, size_t bytes, hipStream_t st, bool up) {
  constexpr int WORKERS = HostStager::WORKERS, BUFS = HostStager::BUFS;
  constexpr size_t CHUNK = HostStager::CHUNK;
  const size_t nchunk = (bytes + CHUNK - 1) / CHUNK;
  const int device = ring.device;
  std::atomic<size_t> next{0};
  std::atomic<int> failed{(int)hipSuccess};
  auto work = [&](int w) {
    auto check = [&](hipError_t e) {
      if (e != hipSuccess) failed.store((int)e);
      return e == hipSuccess;
    };
    if (!check(hipSetDevice(device))) return;
    char* buf[BUFS];
    hipEvent_t ev[BUFS];
    size_t at[BUFS], len[BUFS] = {};   // chunk in flight in each buffer (len 0: none)
    for (int b = 0; b < BUFS; b++) {
      buf[b] = ring.pinned + (size_t)(w * BUFS + b) * CHUNK;
      ev[b] = ring.done[w * BUFS + b];
    }
    auto settle = [&](int b) {
      if (!len[b]) return true;
      const bool ok = check(hipEventSynchronize(ev[b]));
      if (ok && !up) std::memcpy(host + at[b], buf[b], len[b]);
      len[b] = 0;
      return ok;
    };
    int b = 0;
    for (;; b = (b + 1) % BUFS) {
      if (!settle(b) || failed.load() != (int)hipSuccess) break;
      const size_t c = next.fetch_add(1);
      if (c >= nchunk) break;
      const size_t off = c * CHUNK, n = std::min(CHUNK, bytes - off);
      if (up) std::memcpy(buf[b], host + off, n);
      if (!check(up ? hipMemcpyAsync(dev + off, buf[b], n, hipMemcpyHostToDevice, st)
                    : hipMemcpyAsync(buf[b], dev + off, n, hipMemcpyDeviceToHost, st)) ||
          !check(hipEventRecord(ev[b], st))) {
        (void)hipStreamSynchronize(st);   // a copy may be under way without its event
        break;
      }
      at[b] = off;
      len[b] = n;
    }
    // the buffers are free again when the call returns, also after a failure
    for (int k = 0; k < BUFS; k++) settle((b + k) % BUFS);
  };
  const int workers = (int)std::min<size_t>({(size_t)WORKERS, nchunk, std::max(1u, std::thread::hardware_concurrency())});
  std::vector<std::thread> pool;
  try {
    pool.reserve(workers - 1);
    for (int w = 1; w < workers; w++) pool.emplace_back(work, w);
  } catch (...) {   // fewer threads: the others take their chunks
  }
  work(0);
  for (std::thread& t : pool) t.join();
  return (hipError_t)failed.load();
}

// Vectors below 16 MiB, and host memory that the runtime knows (pinned, so
// that the DMA reads it directly), take a plain copy.
bool worth_staging(const void* host, size_t bytes) {
  if (bytes < 8 * HostStager::CHUNK) return false;
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, host) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return a.type == hipMemoryTypeUnregistered;
}

// the staged copy, if it is worth it and a ring is there
bool staged(void* dev, void* host, size_t bytes, hipStream_t st, bool up, hipError_t* rc) {
  if (!worth_staging(host, bytes)) return false;
  std::unique_ptr<Ring> r = take_ring();
  if (!r) return false;
  *rc = run(*r, static_cast<char*>(dev), static_cast<char*>(host), bytes, st, up);
  give_ring(std::move(r));
  return true;
}

}  // namespace

HostStager::HostStager() {
  std::lock_guard<std::mutex> lk(pool_mu);
  idle.reserve(MAX_IDLE);
  owners++;
}

HostStager::~HostStager() {
  std::lock_guard<std::mutex> lk(pool_mu);
  if (--owners == 0) idle.clear();
}

hipError_t HostStager::to_device(void* dev, const void* host, size_t bytes, hipStream_t st) {
  hipError_t rc;
  if (staged(dev, const_cast<void*>(host), bytes, st, true, &rc)) return rc;
  return hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, st);
}

hipError_t HostStager::to_host(void* host, const void* dev, size_t bytes, hipStream_t st) {
  hipError_t rc;
  if (!staged(const_cast<void*>(dev), host, bytes, st, false, &rc))
    rc = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, st);
  return rc == hipSuccess ? hipStreamSynchronize(st) : rc;
}

}  // namespace cpship
