// The few calls of the HIP runtime that main_amd/csrc/mpcx_stage.hip makes, on
// host memory (tests/stage/stage_host.cpp implements them): a device heap of a
// set size, and streams that run a copy as late as their user may rely on --
// when an event after it or the stream is waited for.
#pragma once
#include <stddef.h>
#include <stdint.h>

typedef int hipError_t;
enum { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1, hipMemoryTypeDevice = 2 };
enum { hipHostMallocDefault = 0, hipHostMallocPortable = 1, hipEventDisableTiming = 2 };
struct StubStream;
struct StubEvent;
typedef StubStream* hipStream_t;
typedef StubEvent* hipEvent_t;
struct hipPointerAttribute_t {
  hipMemoryType type;
  int device;
  void *devicePointer, *hostPointer;
  int isManaged;
  unsigned allocationFlags;
};

hipError_t hipGetDevice(int* dev);
hipError_t hipStreamGetDevice(hipStream_t st, int* dev);
hipError_t hipStreamSynchronize(hipStream_t st);
hipError_t hipMalloc(void** p, size_t n);
hipError_t hipFree(void* p);
hipError_t hipHostMalloc(void** p, size_t n, unsigned flags);
hipError_t hipHostFree(void* p);
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned flags);
hipError_t hipEventDestroy(hipEvent_t e);
hipError_t hipEventRecord(hipEvent_t e, hipStream_t st);
hipError_t hipEventSynchronize(hipEvent_t e);
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind kind, hipStream_t st);
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p);
hipError_t hipGetLastError();
const char* hipGetErrorString(hipError_t e);
