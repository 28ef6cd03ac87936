// kept_buffers.cpp against a runtime of two devices of 8 MiB that records
// every call (see test_kept_buffers.py).  A buffer with work queued on it must
// not be kept before its own device has been waited for.
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <map>
#include <mutex>
#include <set>
#include <thread>
#include <vector>

#include "kept_buffers.hpp"

namespace {
int current = 0;
bool capturing = false;           // hipDeviceSynchronize is refused
std::set<int> busy;               // devices with work in flight
struct Block {
  size_t bytes;
  int dev;
};
std::map<void*, Block> live;
size_t used[2] = {0, 0};
const size_t kTotal = 8u << 20;
std::mutex mu;
}  // namespace

extern "C" {
hipError_t hipGetDevice(int* d) { *d = current; return hipSuccess; }
hipError_t hipSetDevice(int d) { current = d; return hipSuccess; }
hipError_t hipDeviceSynchronize() {
  if (capturing) return hipErrorStreamCaptureUnsupported;
  std::lock_guard<std::mutex> l(mu);
  busy.erase(current);
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipMemGetInfo(size_t* f, size_t* t) { *f = kTotal - used[current]; *t = kTotal; return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) {
  std::lock_guard<std::mutex> l(mu);
  if (used[current] + n > kTotal) return hipErrorOutOfMemory;
  *p = std::malloc(16);
  live[*p] = Block{n, current};
  used[current] += n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {  // waits for the device that owns p
  std::lock_guard<std::mutex> l(mu);
  auto it = live.find(p);
  if (it == live.end()) std::abort();
  busy.erase(it->second.dev);
  used[it->second.dev] -= it->second.bytes;
  live.erase(it);
  std::free(p);
  return hipSuccess;
}
}

#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); std::exit(1); } } while (0)

using namespace hmx;

int main() {
  int e = 0;
  // work on device 0's buffer, given up while device 1 is current
  TakenBuffer a = take_buffer(1000, &e);
  CHECK(e == 0 && a.dev == 0 && a.bytes >= 1000);
  busy.insert(0);
  current = 1;
  give_buffer(a);
  CHECK(busy.empty() && current == 1 && kept_memory(0) == a.bytes && kept_memory(1) == 0);
  // device 1 gets memory of its own, device 0 the kept buffer
  TakenBuffer b = take_buffer(1000, &e);
  CHECK(e == 0 && b.dev == 1 && b.p != a.p);
  current = 0;
  TakenBuffer c = take_buffer(1000, &e);
  CHECK(c.p == a.p && c.dev == 0 && kept_memory(0) == 0);
  // a refused wait (stream capture): the buffer is not kept
  capturing = true;
  give_buffer(c);
  capturing = false;
  CHECK(kept_memory(0) == 0 && used[0] == 0);
  // the bound is one device's own: an eighth of it, the oldest go first
  std::vector<TakenBuffer> v;
  for (int d = 0; d < 2; ++d) {
    current = d;
    for (int i = 0; i < 5; ++i) v.push_back(take_buffer(300u << 10, &e));
  }
  current = 0;
  for (const TakenBuffer& t : v) give_buffer(t);
  CHECK(kept_memory(0) == 3 * v[0].bytes && kept_memory(1) == 3 * v[0].bytes && current == 0);
  CHECK(take_buffer(300u << 10, &e).p == v[2].p);
  give_buffer(v[2]);
  // a buffer above the bound goes back at once
  give_buffer(take_buffer(2u << 20, &e));
  CHECK(used[0] == kept_memory(0));
  // an allocation without room empties this device's list and no other's
  TakenBuffer big = take_buffer(kTotal - (256u << 10), &e);
  CHECK(e == 0 && kept_memory(0) == 0 && kept_memory(1) == 3 * v[0].bytes);
  TakenBuffer none = take_buffer(kTotal, &e);
  CHECK(e != 0 && none.p == nullptr);
  give_buffer(none);
  give_buffer(big);
  give_buffer(b);
  release_kept_memory();
  CHECK(kept_memory(0) == 0 && kept_memory(1) == 0 && used[0] == 0 && used[1] == 0 && live.empty());
  // several threads
  std::vector<std::thread> th;
  for (int t = 0; t < 4; ++t)
    th.emplace_back([] {
      int err = 0;
      for (int i = 0; i < 2000; ++i) give_buffer(take_buffer(1 + (i * 977) % 100000, &err));
    });
  for (auto& t : th) t.join();
  release_kept_memory();
  CHECK(used[0] == 0 && live.empty());
  std::printf("ok\n");
  return 0;
}
