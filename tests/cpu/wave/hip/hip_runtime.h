// Host-only stand-in for <hip/hip_runtime.h> that runs one 64-lane workgroup of
// libdgx's stage bodies on the CPU, every lane a fiber (tests/cpu/wave_check.cpp).
// A lane runs alone until it meets the others: at __syncthreads, or at an
// instruction that takes values of other lanes (matrix instruction, shuffle,
// vote), which exchanges those values and nothing else.
//   * shared: all lanes use one LDS image, and what a lane writes is there at
//     once for those that run after it (lanes in ascending or descending order);
//   * own: every lane has its own image, and its writes reach the others at the
//     next __syncthreads only.
// A body whose lanes exchange data through LDS without a barrier between the
// write and the read (or the read and the next write) differs between these.
#pragma once
#include <ucontext.h>

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <vector>

#define __device__
#define __host__
#define __global__
#define __constant__
#define __shared__ static
#define __launch_bounds__(n)
#define amdgpu_waves_per_eu(w) unused
#define __forceinline__ inline

typedef int hipError_t;
typedef void* hipStream_t;
using std::fabs;
using std::max;
using std::min;
using std::sqrt;

struct WaveIndex
{
  int x;
};
inline WaveIndex threadIdx, blockIdx;

struct Wave
{
  enum Mode { SHARED_UP, SHARED_DOWN, OWN };
  static constexpr int L = 64;
  Mode mode;
  ucontext_t home, lane[L];
  std::vector<unsigned char> stack[L], image[L], base;
  int at[L];        // what the lane waits at: 0 nothing, 1 barrier, 2 exchange, 3 end
  unsigned ops[L];  // exchanges so far: two buffers suffice, no lane is two ahead
  double ex[2][2][L];
  int conflicts = 0;  // words two lanes wrote differently between two barriers
  std::function<void(unsigned char*)> body;

  void wait(int what)
  {
    const int me = threadIdx.x;
    at[me]       = what;
    swapcontext(&lane[me], &home);
  }
  void merge()
  {
    if (mode != OWN)
      return;
    std::vector<unsigned char> next = base;
    for (size_t o = 0; o < base.size(); o += 4)
      for (int l = 0; l < L; ++l)
        if (std::memcmp(&image[l][o], &base[o], 4) != 0)
        {
          if (std::memcmp(&next[o], &base[o], 4) != 0 &&
              std::memcmp(&next[o], &image[l][o], 4) != 0)
            ++conflicts;
          std::memcpy(&next[o], &image[l][o], 4);
        }
    base = next;
    for (auto& i : image)
      i = base;
  }
  void run(Mode m, size_t lds, std::function<void(unsigned char*)> f);
};
inline Wave* g_wave;

inline void wave_entry()
{
  Wave* w = g_wave;
  w->body(w->image[w->mode == Wave::OWN ? threadIdx.x : 0].data());
  w->wait(3);
}

inline void Wave::run(Mode m, size_t lds, std::function<void(unsigned char*)> f)
{
  g_wave = this;
  mode   = m;
  body   = f;
  // 16-byte aligned by the allocator; every word a NaN until it is written
  base.assign((lds + 15) / 16 * 16, 0xff);
  for (int l = 0; l < L; ++l)
  {
    image[l] = base;
    at[l]    = 0;
    ops[l]   = 0;
    stack[l].resize(512 << 10);
    getcontext(&lane[l]);
    lane[l].uc_stack.ss_sp   = stack[l].data();
    lane[l].uc_stack.ss_size = stack[l].size();
    lane[l].uc_link          = &home;
    makecontext(&lane[l], wave_entry, 0);
  }
  for (;;)
  {
    for (int k = 0; k < L; ++k)
    {
      threadIdx.x = (m == SHARED_DOWN) ? L - 1 - k : k;
      swapcontext(&home, &lane[threadIdx.x]);
    }
    for (int l = 1; l < L; ++l)
      if (at[l] != at[0])
      {
        std::fprintf(stderr, "lanes 0 and %d wait at different things\n", l);
        std::exit(2);
      }
    if (at[0] == 3)
      return;
    if (at[0] == 1)
      merge();
  }
}

inline void __syncthreads() { g_wave->wait(1); }

// publishes a and b of this lane; afterwards every lane's are in the result
inline const double (*wave_exchange(double a, double b))[Wave::L]
{
  Wave& w      = *g_wave;
  const int me = threadIdx.x, k = w.ops[me]++ & 1;
  w.ex[k][0][me] = a;
  w.ex[k][1][me] = b;
  w.wait(2);
  return w.ex[k];
}

// lane j + 4 b + 16 k holds A[b][j][k], B[b][k][j], C[b][k][j]
inline double __builtin_amdgcn_mfma_f64_4x4x4f64(double a, double x, double c, int, int, int)
{
  const double (*e)[Wave::L] = wave_exchange(a, x);
  const int l = threadIdx.x, j = l & 3, b = (l >> 2) & 3, i = l >> 4;
  for (int k = 0; k < 4; ++k)
    c += e[0][i + 4 * b + 16 * k] * e[1][j + 4 * b + 16 * k];
  return c;
}

inline int __any(int p)
{
  const double (*e)[Wave::L] = wave_exchange(p != 0, 0.0);
  for (int l = 0; l < Wave::L; ++l)
    if (e[0][l] != 0.0)
      return 1;
  return 0;
}

inline double __shfl_xor(double v, int m, int)
{
  const double (*e)[Wave::L] = wave_exchange(v, 0.0);
  return e[0][threadIdx.x ^ m];
}

inline int atomicOr(int* p, int v)
{
  const int o = *p;
  *p |= v;
  return o;
}

inline double __builtin_amdgcn_rcp(double x) { return 1.0 / x; }
inline void __builtin_amdgcn_sched_barrier(int) {}
// used by the FP32 bodies only, which are not run here
typedef float wave_f4 __attribute__((ext_vector_type(4)));
inline int __float_as_int(float) { std::abort(); }
inline float __int_as_float(int) { std::abort(); }
inline unsigned __float_as_uint(float) { std::abort(); }
inline float __uint_as_float(unsigned) { std::abort(); }
inline int __builtin_amdgcn_ds_bpermute(int, int) { std::abort(); }
template <typename... T>
wave_f4 __builtin_amdgcn_mfma_f32_4x4x1f32(T...) { std::abort(); }
template <typename... T>
wave_f4 __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(T...) { std::abort(); }
