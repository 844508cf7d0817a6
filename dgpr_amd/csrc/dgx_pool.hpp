// dgx_pool.hpp -- device memory that a context keeps to be faster and can do
// without: the workspace of the adjoint calls and the stored geometry.  What no
// call is using of it is freed when an allocation of the library fails, so that
// whatever fits into the device's memory without it still does.
#pragma once

#include "dgx_ctx.hpp"

namespace dgx
{

// Makes `device` the current one until it goes out of scope.
class OnDevice
{
 public:
  explicit OnDevice(int device);
  ~OnDevice();
  OnDevice(const OnDevice&) = delete;
  OnDevice& operator=(const OnDevice&) = delete;

 private:
  int prev_;
};

// Contexts whose spare memory may be taken (from dgx_create to dgx_destroy).
void pool_add(dgx_ctx* c);
void pool_remove(dgx_ctx* c);
// Frees the spare memory of idle contexts on `device`; whether there was any.
bool pool_reclaim(int device);
// hipMalloc on `device`, after a reclaim when the first attempt fails.
hipError_t pool_malloc(void** p, size_t bytes, int device);

// The temporaries of one adjoint call, cut from the context's workspace.  It
// stays with the context (grown when a call needs more, at most
// WORKSPACE_KEEP) until dgx_adjoint_release, dgx_destroy or a reclaim:
// allocating and freeing a dozen buffers took 1-3 ms a call, more than the
// kernels of a small residual adjoint.  A call that finds it in use by another
// thread has memory of its own.
constexpr size_t WORKSPACE_KEEP = (size_t)1 << 30;
class Workspace
{
 public:
  explicit Workspace(dgx_ctx* c) : c_(c) {}
  ~Workspace();
  Workspace(const Workspace&) = delete;
  Workspace& operator=(const Workspace&) = delete;
  hipError_t open(size_t ndouble);
  // n doubles, at a multiple of 256 bytes (open() asks for `padded` sizes)
  double* take(size_t n)
  {
    double* p = next_;
    next_ += padded(n);
    return p;
  }
  static size_t padded(size_t n) { return (n + 31) & ~(size_t)31; }

 private:
  dgx_ctx* c_;
  double* next_ = nullptr;
  double* own_  = nullptr;  // memory of this call only
  bool held_    = false;    // the context's workspace is this call's
};

// Frees the context's workspace unless a call is using it.
void workspace_release(dgx_ctx* c);

// The context's mesh for one launch.  While it exists the stored geometry that
// it points to is not freed; a launch recorded into a graph (the context's
// stream is being captured), and keep(), hold it as long as the context lives.
class MeshLease : public MeshArgs
{
 public:
  MeshLease(const MeshArgs& m, dgx_ctx* c);
  ~MeshLease();
  MeshLease(const MeshLease&) = delete;
  MeshLease& operator=(const MeshLease&) = delete;
  MeshArgs keep()
  {
    c_ = nullptr;
    return *this;
  }

 private:
  dgx_ctx* c_;  // whose geometry goes back at the end
};
MeshLease mesh_args(const dgx_ctx* c);

// Frees the context's stored geometry unless a launch or a graph may read it;
// whether it did.
bool geometry_release(dgx_ctx* c);

}  // namespace dgx
