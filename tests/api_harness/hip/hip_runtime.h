// Test double of the HIP runtime for the host code of wahgpu_api.hip, compiled
// for the CPU: everything runs at once on the calling thread, device memory is
// host memory, and a stream that captures refuses what a capture refuses.
#pragma once

#include <stddef.h>
#include <stdint.h>

#define __host__
#define __device__
#define __align__(n) __attribute__((aligned(n)))

enum hipError_t {
  hipSuccess = 0,
  hipErrorInvalidValue = 1,
  hipErrorOutOfMemory = 2,
  hipErrorInvalidDevice = 101,
  hipErrorStreamCaptureUnsupported = 900,
};
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
enum hipStreamCaptureStatus { hipStreamCaptureStatusNone = 0, hipStreamCaptureStatusActive = 1 };
enum hipStreamCaptureMode { hipStreamCaptureModeThreadLocal = 1 };

struct FakeStream {
  bool capturing = false;
};
struct FakeEvent {
  uint64_t at = 0;  // what was recorded when
};
struct FakeGraph {
  int unused;
};
typedef FakeStream* hipStream_t;
typedef FakeEvent* hipEvent_t;
typedef FakeGraph* hipGraph_t;
typedef FakeGraph* hipGraphExec_t;
struct hipDeviceProp_t {
  char name[256];
  char gcnArchName[256];
  int multiProcessorCount;
};

constexpr unsigned hipEventDisableTiming = 2, hipHostMallocDefault = 0, hipStreamDefault = 0;

const char* hipGetErrorString(hipError_t e);
hipError_t hipGetLastError();
hipError_t hipGetDeviceCount(int* n);
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int device);
hipError_t hipSetDevice(int device);
hipError_t hipMallocBytes(void** p, size_t bytes);
hipError_t hipFree(void* p);
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned flags);
hipError_t hipHostFree(void* p);
hipError_t hipMemcpy(void* dst, const void* src, size_t bytes, hipMemcpyKind kind);
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind kind,
                          hipStream_t s);
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned flags);
hipError_t hipStreamDestroy(hipStream_t s);
hipError_t hipStreamSynchronize(hipStream_t s);
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned flags);
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st);
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode mode);
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g);
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, void*, void*, size_t);
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t s);
hipError_t hipGraphDestroy(hipGraph_t g);
hipError_t hipGraphExecDestroy(hipGraphExec_t e);
hipError_t hipEventCreate(hipEvent_t* e);
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned flags);
hipError_t hipEventDestroy(hipEvent_t e);
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s);
hipError_t hipEventSynchronize(hipEvent_t e);
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b);

template <class T>
hipError_t hipMalloc(T** p, size_t bytes) {
  return hipMallocBytes(reinterpret_cast<void**>(p), bytes);
}
template <class T>
hipError_t hipGetSymbolAddress(void** p, T& symbol) {
  *p = &symbol;
  return hipSuccess;
}
#define HIP_SYMBOL(x) x
