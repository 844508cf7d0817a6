// dgx_tile_kernels.hip -- the tiled stage kernel of q = 1 meshes (dgx_tile.hpp)
// and the boundary states it starts from, with their host launch helpers.
#include "dgx_stage.hpp"

#include <type_traits>

namespace dgx
{

// Boundary states (bound_states.cpp:24-130) of every domain-boundary face
// point of the Gauss-nodal state V, into the boundary section of a trace
// record set: what a tiled stage reads besides V itself, after V was set from
// outside.  One thread per boundary face point (sides in the order of
// bface_index); the points of periodic sides are not read and not written.
template <int P, bool AFF>
__global__ __launch_bounds__(64) void dgx_boundary_kernel(MeshArgs mesh, Phys ph,
                                                          const double* __restrict__ V,
                                                          double* __restrict__ Tout, int* status)
{
  constexpr int N = P + 1, NF = N * N, NB = N * N * N;
  const size_t t = (size_t)blockIdx.x * 64 + threadIdx.x;
  if (t >= boundary_faces(mesh.nx, mesh.ny, mesh.nz) * NF)
    return;
  const int fpt = (int)(t % NF), bf = (int)(t / NF);
  const int sx = mesh.ny * mesh.nz, sy = mesh.nx * mesh.nz, sz = mesh.nx * mesh.ny;
  const int nd = bf < 2 * sx ? 0 : (bf < 2 * (sx + sy) ? 1 : 2);
  const int in = bf - (nd == 0 ? 0 : (nd == 1 ? 2 * sx : 2 * (sx + sy)));
  const int s  = nd == 0 ? sx : (nd == 1 ? sy : sz);
  const int hi = in >= s, c = in - hi * s, f = 2 * nd + hi;
  const int n1 = nd == 0 ? mesh.ny : mesh.nx;  // first tangential element count
  const int i1 = c % n1, i2 = c / n1;
  const int far = (nd == 0 ? mesh.nx : (nd == 1 ? mesh.ny : mesh.nz)) - 1;
  const int i0 = hi ? far : 0;
  const int ci = nd == 0 ? i0 : i1, cj = nd == 1 ? i0 : (nd == 0 ? i1 : i2), ck = nd == 2 ? i0 : i2;
  int bt;
  if (neighbour(mesh, ci, cj, ck, f, &bt) >= 0)
    return;
  const size_t e = ((size_t)ck * mesh.ny + cj) * mesh.nx + ci;
  const PTab& pt = c_ptab[P - 1];
  const int a = fpt % N, b = fpt / N;
  double U[5];
#pragma unroll
  for (int r = 0; r < 5; ++r)
  {
    double v = 0.0;
#pragma unroll
    for (int m = 0; m < N; ++m)
      v += pt.L[hi][m] * V[(e * 5 + r) * NB + line_node<N>(nd, m, a, b)];
    U[r] = v;
  }
  double Ji[3][3], nv[3], Ub[5];
  const int gi0 = (nd == 0) ? 0 : a;
  const int gi1 = (nd == 1) ? 0 : ((nd == 0) ? a : b);
  const int gi2 = (nd == 2) ? 0 : b;
  face_geometry<1, AFF, true>(c_qtab[P - 1][0], mesh.nodes + e * 24, AFF ? mesh.arec + e * GREC : nullptr,
                        nd, hi, gi0, gi1, gi2, Ji, nv);
  if (!boundary_state(bt, U, nv, ph, Ub))
    atomicOr(status, 1);
  double* B = Tout + (size_t)mesh.nelem * 6 * 8 * NF + (size_t)bf * 5 * NF + fpt;
#pragma unroll
  for (int r = 0; r < 5; ++r)
    B[r * NF] = Ub[r];
}

template <int P>
static hipError_t launch_boundary(const MeshArgs& m, const Phys& ph, const double* V, double* Tout,
                                  int* status, hipStream_t st)
{
  const size_t n = boundary_faces(m.nx, m.ny, m.nz) * (size_t)((P + 1) * (P + 1));
  const dim3 grid((unsigned)((n + 63) / 64)), block(64);
  if (m.affine)
    hipLaunchKernelGGL((dgx_boundary_kernel<P, true>), grid, block, 0, st, m, ph, V, Tout, status);
  else
    hipLaunchKernelGGL((dgx_boundary_kernel<P, false>), grid, block, 0, st, m, ph, V, Tout, status);
  return hipGetLastError();
}

hipError_t boundary_dispatch(int p, const MeshArgs& m, const Phys& ph, const double* V,
                             double* Tout, int* status, hipStream_t st)
{
  bool any = false;
  for (int i = 0; i < 6; ++i)
    any = any || characteristic_bc(m.bounds[i]);
  if (!any)
    return hipSuccess;
  switch (p)
  {
    case 1: return launch_boundary<1>(m, ph, V, Tout, status, st);
    case 2: return launch_boundary<2>(m, ph, V, Tout, status, st);
    case 3: return launch_boundary<3>(m, ph, V, Tout, status, st);
  }
  return hipErrorInvalidValue;
}

// One thread per element and direction: the element's high face against the low
// face of the element across it, corner differences to a few roundings of the
// coordinates.
__global__ __launch_bounds__(256) void dgx_matched_kernel(MeshArgs mesh, int* flag)
{
  const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= (size_t)mesh.nelem * 3)
    return;
  const int e = (int)(t / 3), d = (int)(t % 3);
  const int ci = e % mesh.nx, cj = (e / mesh.nx) % mesh.ny, ck = e / (mesh.nx * mesh.ny);
  int bt;
  const int nb = neighbour(mesh, ci, cj, ck, 2 * d + 1, &bt);
  if (nb < 0)
    return;
  // node strides along the face and across it
  const int s1 = d == 0 ? 6 : 3, s2 = d == 2 ? 6 : 12;
  const double* A = mesh.nodes + (size_t)e * 24 + (3 << d);
  const double* B = mesh.nodes + (size_t)nb * 24;
  double diff = 0.0, mag = 0.0;
  bool same = true;
  for (int c = 0; c < 4; ++c)
  {
    const int o = (c & 1) * s1 + (c >> 1) * s2;
    for (int i = 0; i < 3; ++i)
    {
      const double x = (A[o + i] - A[i]) - (B[o + i] - B[i]);
      same = same && x == x;
      diff = fmax(diff, fabs(x));
      mag  = fmax(mag, fmax(fabs(A[o + i]), fabs(B[o + i])));
    }
  }
  if (!same || !(diff <= 8.0 * 2.220446049250313e-16 * mag))
    *flag = 1;
}

hipError_t matched_dispatch(const MeshArgs& m, int* flag, hipStream_t st)
{
  hipLaunchKernelGGL(dgx_matched_kernel, dim3((unsigned)(((size_t)m.nelem * 3 + 255) / 256)),
                     dim3(256), 0, st, m, flag);
  return hipGetLastError();
}

// the record-reading body in FP64 (meshes whose faces do not match)
template <int P>
static hipError_t launch_tile_rec(const MeshArgs& m, const Phys& ph, const StageArgs& sa,
                                  const double* lam, int* status, int waves, hipStream_t st)
{
  constexpr int R = tile_rows(P);
  const dim3 grid(tile_blocks(P, m.nelem, true)), block(64);
  const bool norm = sa.normp != nullptr;
  if (waves == 2 && norm)
    hipLaunchKernelGGL((dgx_tile_stage_kernel<P, 1, R, 2, double, false, 0, true, true>), grid, block,
                       0, st, m, ph, sa, lam, status);
  else if (waves == 2)
    hipLaunchKernelGGL((dgx_tile_stage_kernel<P, 1, R, 2, double, false, 0, false, true>), grid, block,
                       0, st, m, ph, sa, lam, status);
  else if (waves == 3 && norm)
    hipLaunchKernelGGL((dgx_tile_stage_kernel<P, 1, R, 3, double, false, 0, true, true>), grid, block,
                       0, st, m, ph, sa, lam, status);
  else if (waves == 3)
    hipLaunchKernelGGL((dgx_tile_stage_kernel<P, 1, R, 3, double, false, 0, false, true>), grid, block,
                       0, st, m, ph, sa, lam, status);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

template <int P, int Q, int W, typename TT, bool AFF, int CT, bool NORM>
static void launch_tile_w(const MeshArgs& m, const Phys& ph, const StageArgs& sa, const double* lam,
                          int* status, hipStream_t st)
{
  constexpr bool FP64 = sizeof(TT) == sizeof(double);
  const dim3 grid(tile_blocks(P, m.nelem, !FP64));
  if constexpr (FP64 && line_order(P))
    if (line_tiled(P, m.nelem))
    {
      hipLaunchKernelGGL((dgx_line_stage_kernel<P, W, AFF, NORM>), grid, dim3(64), 0, st, m, ph, sa,
                         lam, status);
      return;
    }
  if constexpr (!FP64 || P != 2)
    hipLaunchKernelGGL((dgx_tile_stage_kernel<P, Q, tile_rows(P), W, TT, AFF, CT, NORM>), grid,
                       dim3(64), 0, st, m, ph, sa, lam, status);
}

template <int P, int Q, typename TT, bool AFF, int CT>
static hipError_t launch_tile_ct(const MeshArgs& m, const Phys& ph, const StageArgs& sa,
                                 const double* lam, int* status, int waves, hipStream_t st)
{
  if (waves != 2 && waves != 3)
    return hipErrorInvalidValue;
  // a target of 3 runs the 2-wave instance of the state-reading bodies at p = 2
  // and 3: with a third of the registers less they spill.  Per stage at 2 and at 3
  // waves: 32^3 p = 2 90 / 220 us, 16^3 p = 3 23 / 41, 64^3 p = 3 978 / 2554,
  // 48x24x24 p = 3 curved 128 / 253 (p = 1: 64^3 247 / 234)
  constexpr bool FP64 = sizeof(TT) == sizeof(double);
  constexpr int W3    = FP64 && P != 1 ? 2 : 3;
  const bool norm     = sa.normp != nullptr;
  if (waves == 2 && norm)
    launch_tile_w<P, Q, 2, TT, AFF, CT, true>(m, ph, sa, lam, status, st);
  else if (waves == 2)
    launch_tile_w<P, Q, 2, TT, AFF, CT, false>(m, ph, sa, lam, status, st);
  else if (norm)
    launch_tile_w<P, Q, W3, TT, AFF, CT, true>(m, ph, sa, lam, status, st);
  else
    launch_tile_w<P, Q, W3, TT, AFF, CT, false>(m, ph, sa, lam, status, st);
  return hipGetLastError();
}

// the matrix-core contraction forms exist for p = 3 with FP32 trace records
template <int P, int Q, typename TT, bool AFF>
static hipError_t launch_tile_t(const MeshArgs& m, const Phys& ph, const StageArgs& sa,
                         const double* lam, int* status, int waves, hipStream_t st)
{
  if constexpr (P == 3 && std::is_same<TT, float>::value)
  {
    if (sa.ctype == 1)
      return launch_tile_ct<P, Q, TT, AFF, 1>(m, ph, sa, lam, status, waves, st);
    if (sa.ctype == 2)
      return launch_tile_ct<P, Q, TT, AFF, 2>(m, ph, sa, lam, status, waves, st);
  }
  return launch_tile_ct<P, Q, TT, AFF, 0>(m, ph, sa, lam, status, waves, st);
}

template <int P>
static hipError_t launch_tile(const MeshArgs& m, const Phys& ph, const StageArgs& sa,
                              const double* lam, int* status, int waves, hipStream_t st)
{
  if (sa.trace32)
    return m.affine ? launch_tile_t<P, 1, float, true>(m, ph, sa, lam, status, waves, st)
                    : launch_tile_t<P, 1, float, false>(m, ph, sa, lam, status, waves, st);
  if (!m.matched)
    return launch_tile_rec<P>(m, ph, sa, lam, status, waves, st);
  return m.affine ? launch_tile_t<P, 1, double, true>(m, ph, sa, lam, status, waves, st)
                  : launch_tile_t<P, 1, double, false>(m, ph, sa, lam, status, waves, st);
}

hipError_t tile_rhs_dispatch(int p, const MeshArgs& m, const Phys& ph, const StageArgs& sa,
                             const double* lam, int* status, int waves, hipStream_t st)
{
  switch (p)
  {
    case 1: return launch_tile<1>(m, ph, sa, lam, status, waves, st);
    case 2: return launch_tile<2>(m, ph, sa, lam, status, waves, st);
    case 3: return launch_tile<3>(m, ph, sa, lam, status, waves, st);
  }
  return hipErrorInvalidValue;
}

hipError_t upload_tables_tile(const PTab* pt, const QTab* qt)
{
  hipError_t e = hipMemcpyToSymbol(HIP_SYMBOL(c_ptab), pt, sizeof(PTab) * 3);
  if (e != hipSuccess)
    return e;
  return hipMemcpyToSymbol(HIP_SYMBOL(c_qtab), qt, sizeof(QTab) * 9);
}

}  // namespace dgx
