// The host calls that device_buffer.hpp and device_pool.cpp make, for a test
// program that defines them itself (no device).
#pragma once
#include <cstddef>
#include <cstdint>

#define __host__
#define __device__
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };
constexpr hipError_t hipErrorMemoryAllocation = hipErrorOutOfMemory;
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
using hipStream_t = void*;

hipError_t hipMalloc(void** p, size_t bytes);
hipError_t hipFree(void* p);
hipError_t hipGetDevice(int* device);
hipError_t hipGetLastError();
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t);
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t);
inline const char* hipGetErrorString(hipError_t) { return "fake"; }
