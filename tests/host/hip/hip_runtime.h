// The part of the HIP host interface that the library's copies use, on host
// memory: what is queued runs as late as a wait allows, and memory from
// hipHostMalloc lies between guards that every access is held to.
#pragma once
#include <cstddef>

typedef int hipError_t;
constexpr hipError_t hipSuccess = 0, hipErrorInvalidValue = 1;
typedef struct FakeStream* hipStream_t;
typedef struct FakeEvent* hipEvent_t;
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1 };
struct hipPointerAttribute_t {
  hipMemoryType type;
};
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2;

const char* hipGetErrorString(hipError_t);
hipError_t hipGetLastError();
hipError_t hipMalloc(void**, size_t);
hipError_t hipFree(void*);
hipError_t hipHostMalloc(void**, size_t, unsigned);
hipError_t hipHostFree(void*);
hipError_t hipPointerGetAttributes(hipPointerAttribute_t*, const void*);
hipError_t hipGetDevice(int*);
hipError_t hipSetDevice(int);
hipError_t hipStreamGetDevice(hipStream_t, int*);
hipError_t hipEventCreate(hipEvent_t*);
hipError_t hipEventCreateWithFlags(hipEvent_t*, unsigned);
hipError_t hipEventDestroy(hipEvent_t);
hipError_t hipEventRecord(hipEvent_t, hipStream_t);
hipError_t hipEventSynchronize(hipEvent_t);
hipError_t hipStreamSynchronize(hipStream_t);
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t);
hipError_t hipMemcpy2DAsync(void*, size_t, const void*, size_t, size_t, size_t, hipMemcpyKind, hipStream_t);
