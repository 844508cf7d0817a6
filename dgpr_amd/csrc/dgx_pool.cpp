// dgx_pool.cpp -- see dgx_pool.hpp (no counterpart in the reference, which
// allocates what it needs once, solve_cuda.cu:1180-1234).
#include "dgx_pool.hpp"

#include <algorithm>
#include <mutex>
#include <vector>

namespace dgx
{

static std::mutex g_mutex;
static std::vector<dgx_ctx*> g_contexts;

OnDevice::OnDevice(int device) : prev_(-1)
{
  int cur = -1;
  if (hipGetDevice(&cur) == hipSuccess && cur != device && hipSetDevice(device) == hipSuccess)
    prev_ = cur;
}

OnDevice::~OnDevice()
{
  if (prev_ >= 0)
    (void)hipSetDevice(prev_);
}

// adj_busy: 1 while a call or a reclaim has the workspace
static bool claim(int* flag)
{
  int idle = 0;
  return __atomic_compare_exchange_n(flag, &idle, 1, false, __ATOMIC_ACQUIRE, __ATOMIC_RELAXED);
}

static void unclaim(int* flag)
{
  __atomic_store_n(flag, 0, __ATOMIC_RELEASE);
}

// the claimed workspace's memory; whether there was any
static bool free_workspace(dgx_ctx* c)
{
  const bool any = c->adj_ws != nullptr;
  if (any)
  {
    OnDevice on(c->device);
    (void)hipStreamSynchronize(c->stream);
    (void)hipFree(c->adj_ws);
  }
  c->adj_ws       = nullptr;
  c->adj_ws_bytes = 0;
  return any;
}

void pool_add(dgx_ctx* c)
{
  std::lock_guard<std::mutex> lk(g_mutex);
  g_contexts.push_back(c);
}

void pool_remove(dgx_ctx* c)
{
  std::lock_guard<std::mutex> lk(g_mutex);
  g_contexts.erase(std::remove(g_contexts.begin(), g_contexts.end(), c), g_contexts.end());
}

bool pool_reclaim(int device)
{
  std::lock_guard<std::mutex> lk(g_mutex);
  bool any = false;
  for (dgx_ctx* c : g_contexts)
  {
    if (c->device != device)
      continue;
    if (claim(&c->adj_busy))
    {
      any = free_workspace(c) || any;
      unclaim(&c->adj_busy);
    }
    any = geometry_release(c) || any;
  }
  return any;
}

hipError_t pool_malloc(void** p, size_t bytes, int device)
{
  OnDevice on(device);
  hipError_t e = hipMalloc(p, bytes);
  if (e != hipSuccess)
  {
    (void)hipGetLastError();
    *p = nullptr;
    if (pool_reclaim(device) && (e = hipMalloc(p, bytes)) != hipSuccess)
    {
      (void)hipGetLastError();
      *p = nullptr;
    }
  }
  return e;
}

hipError_t Workspace::open(size_t ndouble)
{
  const size_t need = ndouble * sizeof(double);
  held_ = claim(&c_->adj_busy);
  if (!held_)
  {
    const hipError_t e = pool_malloc((void**)&own_, need, c_->device);
    next_ = own_;
    return e;
  }
  if (c_->adj_ws_bytes < need)
  {
    free_workspace(c_);
    const hipError_t e = pool_malloc((void**)&c_->adj_ws, need, c_->device);
    if (e != hipSuccess)
      return e;
    c_->adj_ws_bytes = need;
  }
  next_ = c_->adj_ws;
  return hipSuccess;
}

Workspace::~Workspace()
{
  if (own_)
  {
    OnDevice on(c_->device);
    (void)hipStreamSynchronize(c_->stream);
    (void)hipFree(own_);
  }
  if (held_)
  {
    if (c_->adj_ws_bytes > WORKSPACE_KEEP)
      free_workspace(c_);
    unclaim(&c_->adj_busy);
  }
}

MeshLease::MeshLease(const MeshArgs& m, dgx_ctx* c) : MeshArgs(m), c_(nullptr)
{
  geov = geof = nullptr;
  int n = __atomic_load_n(&c->geo_users, __ATOMIC_RELAXED);
  while (n >= 0 && !__atomic_compare_exchange_n(&c->geo_users, &n, n + 1, true, __ATOMIC_ACQUIRE,
                                                __ATOMIC_RELAXED))
    ;
  if (n < 0)
    return;
  geov = c->geo;
  geof = c->geo + (size_t)c->nelem * GEOV * c->nbf;
  hipStreamCaptureStatus s = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(c->stream, &s) == hipSuccess && s == hipStreamCaptureStatusNone)
    c_ = c;
}

MeshLease::~MeshLease()
{
  if (c_)
    __atomic_fetch_sub(&c_->geo_users, 1, __ATOMIC_RELEASE);
}

bool geometry_release(dgx_ctx* c)
{
  int idle = 0;
  if (!__atomic_compare_exchange_n(&c->geo_users, &idle, -1, false, __ATOMIC_ACQUIRE,
                                   __ATOMIC_RELAXED))
    return false;
  OnDevice on(c->device);
  // kernels of returned calls may still read it, on any stream
  if (hipDeviceSynchronize() != hipSuccess)
  {
    (void)hipGetLastError();
    __atomic_store_n(&c->geo_users, 0, __ATOMIC_RELEASE);
    return false;
  }
  (void)hipFree(c->geo);
  c->geo       = nullptr;
  c->geo_bytes = 0;
  return true;
}

void workspace_release(dgx_ctx* c)
{
  if (claim(&c->adj_busy))
  {
    free_workspace(c);
    unclaim(&c->adj_busy);
  }
}

}  // namespace dgx
