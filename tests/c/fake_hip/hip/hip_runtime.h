// The few HIP runtime calls of device_memory.cpp over host memory that is never touched, for a test
// of the pool's rules on a machine without a GPU: one device of `fake_total` bytes.
#pragma once

#include <cstddef>
#include <map>

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };

inline size_t fake_total = size_t(256) << 30;
inline std::map<void*, size_t> fake_blocks;
inline size_t fake_next = 1 << 20, fake_used = 0, fake_foreign = 0;  // foreign: held by others
inline int fake_syncs = 0, fake_mallocs = 0;

inline hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipDeviceSynchronize() { ++fake_syncs; return hipSuccess; }
inline hipError_t hipMemGetInfo(size_t* free, size_t* total)
{
  *total = fake_total;
  *free  = fake_total - fake_used - fake_foreign;
  return hipSuccess;
}
inline hipError_t hipMalloc(void** p, size_t n)
{
  if (fake_used + fake_foreign + n > fake_total) { return hipErrorOutOfMemory; }
  *p = reinterpret_cast<void*>(fake_next);
  fake_next += n;
  fake_blocks[*p] = n;
  fake_used += n;
  ++fake_mallocs;
  return hipSuccess;
}
inline hipError_t hipFree(void* p)
{
  fake_used -= fake_blocks.at(p);
  fake_blocks.erase(p);
  return hipSuccess;
}
