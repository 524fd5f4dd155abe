// The few HIP calls of workspace.cpp over host memory with a budget, for a host
// test of the pool.
#pragma once
#include <stddef.h>
#include <stdlib.h>

#include <map>

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };
enum { hipHostMallocMapped = 2, hipHostMallocCoherent = 0x40000000 };

inline size_t g_budget = 0, g_used = 0;  // device bytes
inline int g_blocks = 0;                 // device and host blocks held
inline std::map<void*, size_t> g_size;

inline hipError_t hipMalloc(void** p, size_t n)
{
    if (g_used + n > g_budget) return hipErrorOutOfMemory;
    *p = malloc(n);
    g_size[*p] = n;
    g_used += n;
    ++g_blocks;
    return hipSuccess;
}
inline hipError_t hipFree(void* p)
{
    g_used -= g_size[p];
    g_size.erase(p);
    --g_blocks;
    free(p);
    return hipSuccess;
}
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    *p = malloc(n);
    ++g_blocks;
    return hipSuccess;
}
inline hipError_t hipHostFree(void* p)
{
    --g_blocks;
    free(p);
    return hipSuccess;
}
inline hipError_t hipHostGetDevicePointer(void** d, void* p, unsigned)
{
    *d = p;
    return hipSuccess;
}
inline hipError_t hipGetLastError() { return hipSuccess; }
