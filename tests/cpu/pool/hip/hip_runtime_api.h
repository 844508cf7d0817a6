// Host-only stand-in for <hip/hip_runtime_api.h> with two devices of limited
// memory, for tests/cpu/pool_check.cpp: every allocation is host memory booked
// on the thread's current device.
#pragma once
#include <cstddef>
#include <cstdlib>
#include <map>
#include <mutex>

typedef int hipError_t;
typedef void* hipStream_t;
constexpr hipError_t hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2;

struct FakeHip
{
  std::mutex mx;
  size_t capacity[2] = {0, 0}, used[2] = {0, 0};
  struct Block
  {
    int device;
    size_t bytes;
  };
  std::map<void*, Block> blocks;
  int mallocs = 0, frees = 0;
};
inline FakeHip g_hip;
inline thread_local int t_device = 0;

inline hipError_t hipGetDevice(int* d)
{
  *d = t_device;
  return hipSuccess;
}
inline hipError_t hipSetDevice(int d)
{
  t_device = d;
  return hipSuccess;
}
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipDeviceSynchronize() { return hipSuccess; }
inline hipError_t hipMalloc(void** p, size_t n)
{
  std::lock_guard<std::mutex> lk(g_hip.mx);
  if (g_hip.used[t_device] + n > g_hip.capacity[t_device])
    return hipErrorOutOfMemory;
  g_hip.used[t_device] += n;
  *p = std::malloc(n);
  g_hip.blocks[*p] = {t_device, n};
  ++g_hip.mallocs;
  return hipSuccess;
}
inline hipError_t hipFree(void* p)
{
  std::lock_guard<std::mutex> lk(g_hip.mx);
  auto it = g_hip.blocks.find(p);
  if (it == g_hip.blocks.end())
    return hipErrorInvalidValue;
  g_hip.used[it->second.device] -= it->second.bytes;
  g_hip.blocks.erase(it);
  std::free(p);
  ++g_hip.frees;
  return hipSuccess;
}
