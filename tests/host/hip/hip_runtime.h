// A host-only stand-in for the HIP calls of pools.cpp: memory is malloc's, work
// is done at once, a failed call leaves its error for hipGetLastError as the
// runtime's do, and calls after the end of main are counted.
#pragma once
#include <cstddef>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
typedef struct fake_event *hipEvent_t;
typedef struct fake_stream *hipStream_t;
constexpr unsigned hipEventDisableTiming = 2, hipStreamNonBlocking = 1;

hipError_t hipGetLastError();
hipError_t hipGetDevice(int *dev);
hipError_t hipMalloc(void **p, size_t bytes);
hipError_t hipFree(void *p);
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned flags = 0);
hipError_t hipHostFree(void *p);
hipError_t hipMemcpy(void *dst, const void *src, size_t bytes, hipMemcpyKind kind);
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned flags);
hipError_t hipEventDestroy(hipEvent_t e);
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s);
hipError_t hipEventSynchronize(hipEvent_t e);
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned flags);
hipError_t hipStreamDestroy(hipStream_t s);
hipError_t hipStreamSynchronize(hipStream_t s);
