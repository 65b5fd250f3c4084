// Device memory for host programs: a budget of bytes instead of a GPU.
#pragma once

#include <cstdarg>
#include <map>

#include "bh_internal.h"

namespace stub {
inline size_t budget = size_t(1) << 40, live_bytes = 0;
inline std::map<void *, size_t> live;
inline char *next = (char *)4096;   // addresses are numbers only
}  // namespace stub

extern "C" hipError_t hipMalloc(void **p, size_t bytes)
{
    if (stub::live_bytes + bytes > stub::budget) return hipErrorOutOfMemory;
    *p = stub::next;
    stub::next += (bytes + 4095) / 4096 * 4096;
    stub::live[*p] = bytes;
    stub::live_bytes += bytes;
    return hipSuccess;
}
extern "C" hipError_t hipFree(void *p)
{
    if (!p) return hipSuccess;
    if (!stub::live.count(p)) return hipErrorInvalidValue;
    stub::live_bytes -= stub::live[p];
    stub::live.erase(p);
    return hipSuccess;
}
extern "C" hipError_t hipGetDevice(int *device) { return *device = 0, hipSuccess; }
extern "C" hipError_t hipGetLastError() { return hipSuccess; }
extern "C" const char *hipGetErrorString(hipError_t) { return "stub"; }
namespace bh {
void set_error(const char *, ...) {}
}  // namespace bh
