// Copies between pageable host arrays and the device through pinned slots and
// several host threads, and cached device blocks (mpcx_stage.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <vector>

namespace mpcx {
struct HostCopy {
  void* host;           // null: skipped
  void* dev;
  size_t bytes;         // on the device
  bool widen = false;   // copy_out: int32 on the device to int64 on the host
};
// Both are complete when they return (the stream is drained); they order after
// the work already on st.
int copy_out(const std::vector<HostCopy>& v, hipStream_t st);
int copy_in(const std::vector<HostCopy>& v, hipStream_t st);
inline HostCopy upload(void* dev, const void* host, size_t bytes) { return HostCopy{const_cast<void*>(host), dev, bytes, false}; }
// hipMalloc that gives back the device blocks kept between calls when memory
// runs out, and tries once more
hipError_t device_alloc_bytes(void** p, size_t n);
template <typename T>
inline hipError_t device_alloc(T** p, size_t n) { return device_alloc_bytes((void**)p, n); }
// device blocks kept between calls (bounded; released by mpcx_shutdown, and by
// device_alloc when it finds no memory)
void* block_get(size_t n, size_t* got);
void block_put(void* p, size_t n);
void blocks_release();
void stage_release();
}  // namespace mpcx
