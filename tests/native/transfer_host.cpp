// csrc/transfer.cpp on the host, with the HIP calls that it makes replaced by
// these: device memory is host memory, a copy is a memcpy, and a stream's
// queued work is a gate that the test opens.  One scenario per run, named on the
// command line; exit status 0 when it holds.
#include <algorithm>
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <future>
#include <mutex>
#include <set>
#include <string>
#include <vector>

#include "solver.hpp"

namespace dgk {
int set_error(int code, const std::string &) { return code; }
}  // namespace dgk

namespace {

std::mutex mu;
std::condition_variable cv;
bool gate_open = true;         // queued work of stream kBusy has finished
int waiting = 0;               // callers in hipStreamSynchronize(kBusy)
hipStream_t const kBusy = (hipStream_t)0x10;
int pinned_allocs = 0, pinned_frees = 0, copies = 0;
long fail_copy = -1;           // this copy fails
std::set<const void *> not_pageable;

void open_gate() {
  std::lock_guard<std::mutex> lk(mu);
  gate_open = true;
  cv.notify_all();
}

}  // namespace

extern "C" {
hipError_t hipStreamSynchronize(hipStream_t s) {
  std::unique_lock<std::mutex> lk(mu);
  if (s != kBusy) return hipSuccess;
  ++waiting;
  cv.notify_all();
  cv.wait(lk, [] { return gate_open; });
  --waiting;
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  {
    std::lock_guard<std::mutex> lk(mu);
    if (copies++ == fail_copy) return hipErrorUnknown;
  }
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  std::lock_guard<std::mutex> lk(mu);
  ++pinned_allocs;
  *p = std::malloc(n);
  return hipSuccess;
}
hipError_t hipHostFree(void *p) {
  std::lock_guard<std::mutex> lk(mu);
  ++pinned_frees;
  std::free(p);
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t)0x20; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = (hipEvent_t)0x30; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipMalloc(void **, size_t) { return hipErrorOutOfMemory; }
const char *hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
  std::memset(a, 0, sizeof(*a));
  a->type = not_pageable.count(p) ? hipMemoryTypeDevice : hipMemoryTypeUnregistered;
  return hipSuccess;
}
}

namespace {

using dgk::download;
using std::chrono::seconds;
constexpr int64_t MiB = 1 << 20;

struct Field {
  std::vector<char> src, dst;
  explicit Field(int64_t n) : src(n), dst(n, 0) {
    for (int64_t k = 0; k < n; ++k) src[k] = (char)(k * 131 + (k >> 12));
  }
  int get(hipStream_t s = nullptr) {
    std::fill(dst.begin(), dst.end(), 0);
    return download(dst.data(), src.data(), (int64_t)src.size(), 0, s);
  }
  bool same() const { return src == dst; }
};

int fails(const char *what) {
  std::fprintf(stderr, "%s\n", what);
  return 1;
}

// a download whose stream still has steps queued, in a thread of its own, up to
// its wait
struct Waiting {
  Field f{8 * MiB};
  std::thread t;
  Waiting() {
    gate_open = false;
    t = std::thread([this] { f.get(kBusy); });
    std::unique_lock<std::mutex> lk(mu);
    cv.wait(lk, [] { return waiting > 0; });
  }
  ~Waiting() {
    open_gate();
    t.join();
  }
};

void make_pool() {
  dgk::transfer_retain();
  Field f(64 * MiB);
  f.get();
}

// another thread's handles come and go
int handles_while_waiting() {
  make_pool();
  Waiting w;
  auto other = std::async(std::launch::async, [] {
    dgk::transfer_retain();
    dgk::transfer_release();
  });
  const bool free = other.wait_for(seconds(5)) == std::future_status::ready;
  open_gate();
  return free ? 0 : fails("creating a handle waits for another handle's steps");
}

// another thread's large download goes through the idle chunks
int download_while_waiting() {
  make_pool();
  Waiting w;
  Field f(8 * MiB);
  const int before = copies;
  f.get();
  const int n = copies - before;
  open_gate();
  return n == 8 && f.same() ? 0 : fails("a download was copied plainly though no chunk was in use");
}

// The bytes asked for are counted while a handle lives: a program that makes
// and destroys its handles starts anew with each.
int plain_count_ends_with_handles() {
  Field f(20 * MiB);
  for (int k = 0; k < 3; ++k) {
    dgk::transfer_retain();
    f.get();
    dgk::transfer_release();
  }
  return pinned_allocs == 0 ? 0 : fails("bytes of destroyed handles made the pool");
}

// Sliced downloads at the sizes where chunks and slices change: every byte, in
// the number of copies that the slices and chunks make.
int sliced_sizes() {
  make_pool();
  for (int64_t n : {4 * MiB, 4 * MiB + 1, 4 * MiB + 512, 8 * MiB - 1, 8 * MiB, 8 * MiB + 4096,
                    8 * MiB + 4097, 16 * MiB + 8, 33 * MiB + 77}) {
    Field f(n);
    const int before = copies;
    if (f.get() != 0 || !f.same()) return fails("bytes differ");
    const int64_t slice = ((n + 7) / 8 + 4095) / 4096 * 4096;
    int64_t want = 0;
    for (int64_t at = 0; at < n; at += slice) want += (std::min(slice, n - at) + MiB - 1) / MiB;
    if (copies - before != want) return fails("not the sliced way");
  }
  Field f(4 * MiB - 8);
  const int before = copies;
  if (f.get() != 0 || !f.same() || copies - before != 1) return fails("below 4 MiB: one copy");
  return 0;
}

// Destinations that are not pageable take one copy; a copy that fails is
// reported and leaves the pool usable.
int plain_destinations_and_failures() {
  make_pool();
  Field f(8 * MiB);
  not_pageable.insert(f.dst.data());
  const int before = copies;
  if (f.get() != 0 || !f.same() || copies - before != 1) return fails("not one plain copy");
  not_pageable.clear();
  fail_copy = copies + 5;
  if (f.get() == 0) return fails("a failed copy was not reported");
  fail_copy = -1;
  if (f.get() != 0 || !f.same()) return fails("no download after a failed one");
  dgk::transfer_release();
  return pinned_allocs == 1 && pinned_frees == 1 ? 0 : fails("the pool was not given back");
}

}  // namespace

int main(int, char **argv) {
  const std::string s = argv[1];
  if (s == "handles_while_waiting") return handles_while_waiting();
  if (s == "download_while_waiting") return download_while_waiting();
  if (s == "plain_count_ends_with_handles") return plain_count_ends_with_handles();
  if (s == "sliced_sizes") return sliced_sizes();
  if (s == "plain_destinations_and_failures") return plain_destinations_and_failures();
  return 2;
}
