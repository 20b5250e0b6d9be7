/* The few declarations of the HIP runtime that bsx_internal.h and bsx_mem.hip
 * name, for a build of the memory code without a GPU; memory_check.cpp defines
 * the allocator behind them. */
#pragma once
#include <stddef.h>

typedef enum { hipSuccess = 0, hipErrorOutOfMemory = 2 } hipError_t;
typedef struct ihipStream* hipStream_t;
typedef struct { float x, y; } float2;
#define hipHostMallocDefault 0

extern "C" {
hipError_t hipMalloc(void** p, size_t bytes);
hipError_t hipFree(void* p);
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned flags);
hipError_t hipHostFree(void* p);
hipError_t hipGetDevice(int* dev);
hipError_t hipDeviceSynchronize(void);
hipError_t hipGetLastError(void);
const char* hipGetErrorString(hipError_t e);
}
