// The runtime calls of lbm_hostcopy.cpp on the CPU: two devices, streams and
// events that belong to one, errors that stay with the thread until read, and
// counts of what is held.
#pragma once
#include <cstddef>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorInvalidHandle = 400 };
enum hipMemcpyKind { hipMemcpyDeviceToHost = 2 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1, hipMemoryTypeDevice = 2 };
struct hipPointerAttribute_t { hipMemoryType type; };
constexpr unsigned hipHostMallocPortable = 1, hipEventDisableTiming = 2;

struct FakeStream { int dev; };
struct FakeEvent { int dev; };
typedef FakeStream* hipStream_t;
typedef FakeEvent* hipEvent_t;

hipError_t hipGetLastError();
hipError_t hipGetDevice(int* dev);
hipError_t hipSetDevice(int dev);
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned flags);
hipError_t hipHostFree(void* p);
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p);
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned flags);
hipError_t hipEventDestroy(hipEvent_t e);
hipError_t hipEventRecord(hipEvent_t e, hipStream_t st);
hipError_t hipEventSynchronize(hipEvent_t e);
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind kind, hipStream_t st);
hipError_t hipStreamSynchronize(hipStream_t st);
