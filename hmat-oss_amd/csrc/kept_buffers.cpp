#include "kept_buffers.hpp"

#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <list>
#include <map>
#include <mutex>

namespace hmx {

namespace {
struct Kept {
  std::list<TakenBuffer> buffers;  // oldest first
  size_t bytes = 0, limit = 0;
};
std::mutex kept_mutex;
std::map<int, Kept>& kept_on() {  // by device; never destroyed (the runtime may end before it)
  static auto* m = new std::map<int, Kept>;
  return *m;
}

// sizes are rounded up to an eighth of their power of two, so that buffers of
// similar objects fit each other
size_t rounded_size(size_t n) {
  size_t step = 256;
  while (step * 16 <= n) step *= 2;
  return (n + step - 1) / step * step;
}

void release_device(Kept& k) {
  for (const TakenBuffer& b : k.buffers) (void)hipFree(b.p);
  k.buffers.clear();
  k.bytes = 0;
}

// Makes 'dev' current and the caller's device again at the end.
struct OnDevice {
  int before = -1;
  bool ok;
  explicit OnDevice(int dev) {
    ok = hipGetDevice(&before) == hipSuccess;
    if (ok && before == dev)
      before = -1;
    else if (ok)
      ok = hipSetDevice(dev) == hipSuccess;
  }
  ~OnDevice() {
    if (before >= 0) (void)hipSetDevice(before);
  }
};
}  // namespace

namespace {
bool keep(const TakenBuffer& b) {
  try {
    std::lock_guard<std::mutex> lock(kept_mutex);
    Kept& k = kept_on()[b.dev];
    if (k.limit == 0) {
      size_t freeb = 0, total = 0;
      if (hipMemGetInfo(&freeb, &total) == hipSuccess) k.limit = total / 8;
    }
    if (b.bytes > k.limit) return false;
    k.buffers.push_back(b);
    k.bytes += b.bytes;
    while (k.bytes > k.limit) {
      (void)hipFree(k.buffers.front().p);
      k.bytes -= k.buffers.front().bytes;
      k.buffers.pop_front();
    }
    return true;
  } catch (...) {  // no host memory for the record
    return false;
  }
}
}  // namespace

void release_kept_memory() {
  std::lock_guard<std::mutex> lock(kept_mutex);
  for (auto& k : kept_on()) release_device(k.second);
}

size_t kept_memory(int dev) {
  std::lock_guard<std::mutex> lock(kept_mutex);
  auto it = kept_on().find(dev);
  return it == kept_on().end() ? 0 : it->second.bytes;
}

void give_buffer(const TakenBuffer& b) {
  if (!b.p) return;
  {
    OnDevice on(b.dev);
    if (on.ok && hipDeviceSynchronize() == hipSuccess) {
      if (keep(b)) return;
    } else {
      (void)hipGetLastError();
    }
  }
  (void)hipFree(b.p);
}

TakenBuffer take_buffer(size_t bytes, int* error) {
  const size_t want = rounded_size(std::max<size_t>(bytes, 1));
  TakenBuffer b{nullptr, 0, 0};
  *error = (int)hipGetDevice(&b.dev);
  if (*error != (int)hipSuccess) return b;
  {
    std::lock_guard<std::mutex> lock(kept_mutex);
    Kept& k = kept_on()[b.dev];
    auto best = k.buffers.end();
    for (auto it = k.buffers.begin(); it != k.buffers.end(); ++it)
      if (it->bytes >= want && it->bytes <= want + want / 4 && (best == k.buffers.end() || it->bytes < best->bytes))
        best = it;
    if (best != k.buffers.end()) {
      b = *best;
      k.bytes -= b.bytes;
      k.buffers.erase(best);
      return b;
    }
  }
  hipError_t e = hipMalloc(&b.p, want);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    {
      std::lock_guard<std::mutex> lock(kept_mutex);
      release_device(kept_on()[b.dev]);
    }
    e = hipMalloc(&b.p, want);
  }
  *error = (int)e;
  if (e != hipSuccess)
    b.p = nullptr;
  else
    b.bytes = want;
  return b;
}

}  // namespace hmx
