// main_amd/csrc/mpcx_stage.hip on the host, with the HIP calls of
// hip/hip_runtime.h beside this file; driven by tests/test_stage_host.py.
#include <stdio.h>
#include <stdlib.h>
#include <map>
#include <mutex>
#include <atomic>
#include <new>
#include "../../main_amd/csrc/mpcx_stage.hip"

static std::atomic<long> g_fail_at{-1};   // the allocation that fails (counted down; below 0: none)
static bool fails() {
  return g_fail_at.load() >= 0 && g_fail_at.fetch_sub(1) == 0;
}
void* operator new(size_t n) {
  void* p = fails() ? nullptr : malloc(n ? n : 1);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }

struct Copy {
  void* dst;
  const void* src;
  size_t n;
};
struct StubStream {
  int dev = 0;
  Copy q[4096];   // copies done .. queued are not yet made
  size_t done = 0, queued = 0;
};
struct StubEvent {
  StubStream* st = nullptr;
  size_t at = 0;   // copies of the stream before it
  int dev = 0;
};

static std::recursive_mutex g_mu;
static StubStream g_null;
static int g_dev = 0;
static size_t g_heap = ~(size_t)0, g_used = 0, g_mallocs = 0, g_frees = 0, g_host_mallocs = 0, g_events = 0;
static std::map<char*, size_t> g_device, g_pinned;
static size_t g_direct = 0;   // bytes copied from or to pinned memory of the caller's

static StubStream* stream(hipStream_t st) { return st ? st : &g_null; }
static bool within(const std::map<char*, size_t>& m, const void* p) {
  auto it = m.upper_bound((char*)p);
  return it != m.begin() && (char*)p < std::prev(it)->first + std::prev(it)->second;
}
static void run_to(StubStream* s, size_t at) {
  for (; s->done < at; s->done++) {
    const Copy& c = s->q[s->done % 4096];
    memcpy(c.dst, c.src, c.n);
  }
}
#define LOCK std::lock_guard<std::recursive_mutex> lock(g_mu)
hipError_t hipGetDevice(int* dev) { LOCK; *dev = g_dev; return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t st, int* dev) { LOCK; *dev = stream(st)->dev; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t st) { LOCK; run_to(stream(st), stream(st)->queued); return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) {
  LOCK;
  if (n > g_heap - g_used) return hipErrorOutOfMemory;
  *p = malloc(n ? n : 1);
  g_device[(char*)*p] = n;
  g_used += n;
  g_mallocs++;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  LOCK;
  auto it = g_device.find((char*)p);
  if (it == g_device.end()) return hipErrorInvalidValue;
  g_used -= it->second;
  g_frees++;
  g_device.erase(it);
  free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  LOCK;
  *p = malloc(n);
  memset(*p, 0xee, n);
  g_host_mallocs++;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  LOCK;
  *e = new (malloc(sizeof(StubEvent))) StubEvent();   // (the stand-in's own memory does not fail)
  (*e)->dev = g_dev;
  g_events++;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { LOCK; free(e); g_events--; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t st) {
  LOCK;
  if (e->dev != stream(st)->dev) return hipErrorInvalidValue;
  e->st = stream(st);
  e->at = e->st->queued;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) { LOCK; if (e->st) run_to(e->st, e->at); return hipSuccess; }
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind kind, hipStream_t st) {
  LOCK;
  if (within(g_pinned, kind == hipMemcpyDeviceToHost ? dst : src)) g_direct += n;
  if (stream(st)->queued - stream(st)->done >= 4096) return hipErrorUnknown;
  stream(st)->q[stream(st)->queued++ % 4096] = Copy{dst, src, n};
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  LOCK;
  *a = hipPointerAttribute_t{within(g_pinned, p) ? hipMemoryTypeHost : hipMemoryTypeUnregistered, 0, nullptr, nullptr, 0, 0};
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stub error"; }
namespace mpcx {
int set_error(int code, const char*) { return code; }
}

extern "C" {
void t_reset(size_t heap) {
  mpcx::blocks_release();
  mpcx::stage_release();
  while (!g_device.empty()) (void)hipFree(g_device.begin()->first);
  g_heap = heap;
  g_mallocs = g_frees = g_host_mallocs = g_direct = 0;
  g_pinned.clear();
  g_dev = 0;
  g_null.dev = 0;
}
void t_device(int dev) { g_dev = g_null.dev = dev; }
size_t t_used() { return g_used; }
size_t t_mallocs() { return g_mallocs; }
size_t t_frees() { return g_frees; }
size_t t_host_mallocs() { return g_host_mallocs; }
size_t t_events() { return g_events; }
size_t t_direct() { return g_direct; }
void t_pin(void* p, size_t n) { g_pinned[(char*)p] = n; }
void* t_block_get(size_t n, size_t* got) { return mpcx::block_get(n, got); }
void t_block_put(void* p, size_t n) { mpcx::block_put(p, n); }
void* t_alloc(size_t n) {
  void* p = nullptr;
  return mpcx::device_alloc(&p, n) == hipSuccess ? p : nullptr;
}
void t_free(void* p) { (void)hipFree(p); }
// n arrays between the host and "device" memory (here host memory too); the
// result plus 1000 if the allocation to fail came up
int t_copy(int n, void** host, void** dev, const size_t* bytes, const int* widen, int out, long fail_at) {
  std::vector<mpcx::HostCopy> v;
  for (int i = 0; i < n; i++) v.push_back(mpcx::HostCopy{host[i], dev[i], bytes[i], widen[i] != 0});
  g_fail_at = fail_at;
  const int rc = out ? mpcx::copy_out(v, nullptr) : mpcx::copy_in(v, nullptr);
  const bool failed = fail_at >= 0 && g_fail_at < 0;
  g_fail_at = -1;
  return failed ? 1000 + rc : rc;
}
}
