// Device memory kept between objects (host code, HIP runtime calls only).
//
// A buffer given up by a DevBuf is kept for the next one of its size instead
// of going back to the driver, which clears device memory before it hands it
// out again: a program that builds, factorises and drops one matrix after the
// other (a likelihood per hyperparameter, a batch of systems) spent most of
// its time there (N = 50,000: assembly 12 ms of kernels, 474 ms a pass; an
// 8,000-point likelihood and gradient 107 ms with clean memory at hand, 204 ms
// without).  At most an eighth of a device's memory is kept on it, the oldest
// buffers go first.  All of a device's kept buffers go back when an allocation
// on it fails, all of every device's in release_kept_memory().
#pragma once
#include <cstddef>

namespace hmx {

struct TakenBuffer {
  void* p;
  size_t bytes;
  int dev;
};

// At least 'bytes' bytes on the current device, content undefined.  p is null
// and 'error' the hipError_t where the device has no room.
TakenBuffer take_buffer(size_t bytes, int* error);

// Gives up a buffer of take_buffer.  Waits for the buffer's device first, as
// hipFree does, whichever device is current: a kept buffer has no work of any
// stream left on it.
void give_buffer(const TakenBuffer& b);

// Gives the kept buffers back to the driver.
void release_kept_memory();

// Bytes kept on a device.
size_t kept_memory(int dev);

}  // namespace hmx
