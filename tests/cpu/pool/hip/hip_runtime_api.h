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
// every stream is being captured while this is set
inline bool g_capturing = false;
enum hipStreamCaptureStatus { hipStreamCaptureStatusNone, hipStreamCaptureStatusActive };
inline hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s)
{
  *s = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
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
template <typename T>
hipError_t hipMalloc(T** p, size_t n)
{
  return hipMalloc((void**)p, n);
}

// the rest of what dgx_api.cpp calls: streams do nothing, copies are immediate
#include <cstring>
typedef int* hipEvent_t;
enum hipMemcpyKind
{
  hipMemcpyHostToDevice,
  hipMemcpyDeviceToHost,
  hipMemcpyDeviceToDevice,
  hipMemcpyDefault
};
constexpr unsigned hipStreamNonBlocking = 1;
constexpr unsigned hipHostMallocPortable = 1;
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
  *p = std::malloc(n);
  return hipSuccess;
}
inline const char* hipGetErrorString(hipError_t e)
{
  return e == hipErrorOutOfMemory ? "out of memory" : "error";
}
inline hipError_t hipGetDeviceCount(int* n)
{
  *n = 2;
  return hipSuccess;
}
inline hipError_t hipMemGetInfo(size_t* free, size_t* total)
{
  std::lock_guard<std::mutex> lk(g_hip.mx);
  *total = g_hip.capacity[t_device];
  *free  = *total - g_hip.used[t_device];
  return hipSuccess;
}
inline hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind)
{
  std::memcpy(d, s, n);
  return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t)
{
  return hipMemcpy(d, s, n, k);
}
inline hipError_t hipMemset(void* d, int v, size_t n)
{
  std::memset(d, v, n);
  return hipSuccess;
}
inline hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return hipMemset(d, v, n); }
inline hipError_t hipStreamCreateWithFlags(hipStream_t*, unsigned) { return hipSuccess; }
inline hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
inline hipError_t hipEventCreate(hipEvent_t*) { return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventElapsedTime(float* t, hipEvent_t, hipEvent_t)
{
  *t = 1.0f;
  return hipSuccess;
}
