// Downloads into the caller's pageable host memory.
//
// A plain hipMemcpy into fresh pageable memory runs at about 11 GB/s: one
// thread takes the page faults and copies out of the runtime's staging buffer.
// A large download is instead cut into slices, one per thread; each slice goes
// through two pinned chunks, the device filling one while the thread copies the
// other to its place.
#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>

#include "solver.hpp"

namespace dgk {

namespace {

constexpr int kLanes = 8;                       // threads of one download
constexpr int kStreams = 2;                     // copy streams they share
constexpr int64_t kChunk = (int64_t)1 << 20;    // bytes of a pinned chunk
// Below this a plain copy is as fast as starting the threads (16.8 MB: 1.2 ->
// 0.8 ms, 134 MB: 12.8 -> 4.2 ms, the caller's pages fresh in both).
constexpr int64_t kSliced = (int64_t)4 << 20;
// Making the pool takes 7-8 ms with its streams' first use, of which a first plain
// copy pays most as well: a first download of 57 MB 16.5 ms sliced, 17.2 plain, of
// 134 MB 18.9 and 24.8.  Below this many bytes a program is left with plain copies.
constexpr int64_t kWorthPool = (int64_t)48 << 20;

// The pinned chunks, streams and events of one download at a time, shared by
// every handle of the process (16 MiB): made once kWorthPool bytes have been
// asked for, given back when the last handle is destroyed.  `mu` guards the
// counts and `busy` and is held for no longer than they take to change; who has
// set `busy` owns the rest.
struct Pool {
  std::mutex mu;
  int refs = 0;
  bool busy = false;   // a download is using or making the chunks
  int device = -1;     // -1: not made
  int64_t plain = 0;   // bytes of large downloads so far, while not made
  char *pinned = nullptr;
  hipStream_t stream[kStreams] = {};
  hipEvent_t event[kLanes][2] = {};
};
Pool g_pool;

void free_pool(Pool &p) {
  for (int l = 0; l < kLanes; ++l) {
    for (int b = 0; b < 2; ++b)
      if (p.event[l][b]) (void)hipEventDestroy(p.event[l][b]);
    p.event[l][0] = p.event[l][1] = nullptr;
  }
  for (hipStream_t &s : p.stream) {
    if (s) (void)hipStreamDestroy(s);
    s = nullptr;
  }
  if (p.pinned) (void)hipHostFree(p.pinned);
  p.pinned = nullptr;
  p.device = -1;
  p.plain = 0;
}

bool make_pool(Pool &p, int device) {
  bool ok = hipHostMalloc((void **)&p.pinned, 2 * kLanes * kChunk, hipHostMallocDefault) == hipSuccess;
  for (int k = 0; k < kStreams && ok; ++k)
    ok = hipStreamCreateWithFlags(&p.stream[k], hipStreamNonBlocking) == hipSuccess;
  for (int l = 0; l < kLanes && ok; ++l) {
    for (int b = 0; b < 2 && ok; ++b)
      ok = hipEventCreateWithFlags(&p.event[l][b], hipEventDisableTiming) == hipSuccess;
  }
  if (!ok) {
    (void)hipGetLastError();
    free_pool(p);
    return false;
  }
  p.device = device;
  return true;
}

// One slice: bytes [0, n) of src to dst through lane l's two chunks.
hipError_t copy_slice(const Pool &p, int l, char *dst, const char *src, int64_t n) {
  hipError_t e = hipSetDevice(p.device);
  if (e != hipSuccess) return e;
  const hipStream_t stream = p.stream[l % kStreams];
  char *buf[2] = {p.pinned + 2 * l * kChunk, p.pinned + (2 * l + 1) * kChunk};
  const int64_t chunks = (n + kChunk - 1) / kChunk;
  auto issue = [&](int64_t c) {
    const int64_t off = c * kChunk, len = n - off < kChunk ? n - off : kChunk;
    hipError_t r = hipMemcpyAsync(buf[c & 1], src + off, len, hipMemcpyDeviceToHost, stream);
    if (r == hipSuccess) r = hipEventRecord(p.event[l][c & 1], stream);
    return r;
  };
  e = issue(0);
  for (int64_t c = 0; c < chunks && e == hipSuccess; ++c) {
    if (c + 1 < chunks) e = issue(c + 1);  // its chunk was emptied a turn ago
    if (e == hipSuccess) e = hipEventSynchronize(p.event[l][c & 1]);
    if (e != hipSuccess) break;
    const int64_t off = c * kChunk, len = n - off < kChunk ? n - off : kChunk;
    std::memcpy(dst + off, buf[c & 1], len);
  }
  if (e != hipSuccess) (void)hipStreamSynchronize(stream);  // nothing writes the chunks
  return e;
}

hipMemoryType memory_type(const void *p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return hipMemoryTypeUnregistered;
  }
  return a.type;
}

// Ordinary pageable memory, the only kind the slices are for: the runtime
// copies straight into pinned memory at the link's rate, and a thread cannot
// write device memory.
bool pageable(const void *p) { return memory_type(p) == hipMemoryTypeUnregistered; }

}  // namespace

bool device_memory(const void *p) { return memory_type(p) == hipMemoryTypeDevice; }

void transfer_retain() {
  std::lock_guard<std::mutex> lk(g_pool.mu);
  ++g_pool.refs;
}

void transfer_release() {
  std::lock_guard<std::mutex> lk(g_pool.mu);
  if (--g_pool.refs == 0 && !g_pool.busy) free_pool(g_pool);  // and the count starts anew
}

namespace {

// The pool for one download, if no other has it, it is worth making and it
// belongs to this device; given back at the end of the scope.
class Lease {
 public:
  Lease(int64_t bytes, int device) {
    {
      std::lock_guard<std::mutex> lk(g_pool.mu);
      if (g_pool.busy || g_pool.refs < 1) return;
      if (g_pool.device < 0) {
        g_pool.plain += bytes;
        if (g_pool.plain < kWorthPool) return;
      } else if (g_pool.device != device) {
        return;
      }
      g_pool.busy = held_ = true;
    }
    usable_ = g_pool.device == device || make_pool(g_pool, device);
  }
  ~Lease() {
    if (!held_) return;
    std::lock_guard<std::mutex> lk(g_pool.mu);
    g_pool.busy = false;
    if (g_pool.refs == 0) free_pool(g_pool);
  }
  Lease(const Lease &) = delete;
  Lease &operator=(const Lease &) = delete;
  explicit operator bool() const { return usable_; }

 private:
  bool held_ = false, usable_ = false;
};

int download_sliced(void *dst, const void *src, int64_t bytes) {
  int64_t slice = (bytes + kLanes - 1) / kLanes;
  slice = (slice + 4095) / 4096 * 4096;
  std::atomic<int> failed{0};
  auto work = [&](int l) {
    const int64_t at = l * slice, n = bytes - at < slice ? bytes - at : slice;
    if (n <= 0) return;
    const hipError_t e = copy_slice(g_pool, l, (char *)dst + at, (const char *)src + at, n);
    if (e != hipSuccess) failed.store((int)e);
  };
  std::thread t[kLanes];
  for (int l = 1; l < kLanes; ++l) {
    try {
      t[l] = std::thread(work, l);
    } catch (...) {  // no thread: this one does its slice
    }
  }
  work(0);
  for (int l = 1; l < kLanes; ++l) {
    if (t[l].joinable()) t[l].join();
    else work(l);
  }
  if (const int e = failed.load())
    return set_error(DGK_ERR_DEVICE,
                     std::string("download: ") + hipGetErrorString((hipError_t)e));
  return DGK_OK;
}

}  // namespace

int download(void *dst, const void *src, int64_t bytes, int device, hipStream_t s) {
  if (bytes >= kSliced && pageable(dst)) {
    // the steps queued before it are waited for with nothing held: other
    // threads' handles and downloads do not wait for them
    DGK_HIP(hipStreamSynchronize(s));
    Lease lease(bytes, device);
    if (lease) return download_sliced(dst, src, bytes);
  }
  DGK_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s));
  DGK_HIP(hipStreamSynchronize(s));
  return DGK_OK;
}

}  // namespace dgk
