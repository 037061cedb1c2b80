// The part of the HIP runtime's interface that staged transfers use, for a host program of its own
// (host_stage.cpp, which defines the functions).
#pragma once
#include <cstddef>
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
typedef int hipStream_t;
typedef int hipEvent_t;
enum { hipHostMallocDefault = 0, hipEventDisableTiming = 2 };
hipError_t hipHostMalloc(void** p, size_t n, unsigned flags);
hipError_t hipHostFree(void* p);
hipError_t hipMalloc(void** p, size_t n);
hipError_t hipFree(void* p);
hipError_t hipGetLastError();
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind kind, hipStream_t stream);
hipError_t hipStreamSynchronize(hipStream_t stream);
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned flags);
hipError_t hipEventDestroy(hipEvent_t e);
hipError_t hipEventRecord(hipEvent_t e, hipStream_t stream);
hipError_t hipEventSynchronize(hipEvent_t e);
