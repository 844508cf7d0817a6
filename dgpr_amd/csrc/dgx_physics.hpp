// dgx_physics.hpp -- pointwise physics of the stage kernel written once for
// a generic scalar type T: double in the residual kernels, forward-mode dual
// numbers (local Jacobians) in the discrete adjoint.  Arguments that the
// adjoint's dual passes hold fixed (reference-space gradients, gradient
// tractions) have their own type G / V, so a pass over the state carries no
// zero derivatives for them.
#pragma once

#include "dgx_device.hpp"

namespace dgx
{

// ---- viscous flux in velocity-gradient form ---------------------------------
// The Newtonian flux A(s, grad s) of flux.cpp:156-202 depends on the
// conserved-variable gradient only through the velocity gradient
//   Lv[i][d] = d u_i / d x_d = (d m_i/dx_d - u_i d rho/dx_d) / rho
// (there is no heat flux), and every BR2 / dual-consistency argument is a
// jump times the normal, whose velocity gradient is rank one:
//   (U_jump (x) n)  ->  dm (x) n,   dm_i = (jump_m_i - u_i jump_rho) / rho.
// tau(X) = mu (X + X^T) - 2/3 mu tr(X) I;  the energy row is u . tau.

// w = tau(X) n for X with X n = xn, X^T n = xtn, tr X = tr
template <typename T>
__device__ __forceinline__ void tau_n(double mu, const T* xn, const T* xtn, T tr, const double* n,
                                      T* w)
{
  T lt = -(2.0 / 3.0) * mu * tr;
#pragma unroll
  for (int i = 0; i < 3; ++i)
    w[i] = mu * (xn[i] + xtn[i]) + lt * n[i];
}

// velocity gradient from reference-space derivatives gr[c][0..3] of
// (rho, m) and the inverse Jacobian Ji[c][d]
template <typename T, typename G>
__device__ __forceinline__ void vel_grad(const G gr[3][4], const T* u, T ir, const double Ji[3][3],
                                         T Lv[3][3])
{
  T dv[3][3];  // dv[c][i] = d u_i / d xi_c
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int i = 0; i < 3; ++i)
      dv[c][i] = (gr[c][1 + i] - gr[c][0] * u[i]) * ir;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int d = 0; d < 3; ++d)
      Lv[i][d] = dv[0][i] * Ji[0][d] + dv[1][i] * Ji[1][d] + dv[2][i] * Ji[2][d];
}

// One face point seen from the own side: outputs G = F - QH.n (5) and the
// physical dual-consistency flux dcQ as a symmetric stress S (6: xx yy zz
// xy xz yz) whose energy row is u_L . S.
//
// Interior (solve.cpp:393-626):
//   F   = roe(UL, UR, n)
//   dcQ = A(UL, (UL - (UL+UR)/2) n)            = tau(dmL/2 (x) n)
//   QH  = (A(UL,gL) + A(UR,gR))/2 - eta (dL + dR)/2,
//   dL  = lamL/2 A(UL, (UL-UR) n),  dR = lamR/2 A(UR, (UL-UR) n)
// so QH.n = tau(Lv_L/2 - cL dmL(x)n) n + tau(Lv_R/2 - cR dmR(x)n) n with
// c = eta lam / 4, plus the energy rows u_L.(...) and u_R.(...).
// Boundary (solve.cpp:628-794): Ub = boundary state, F = F(Ub).n,
//   dcQ = tau(dm (x) n) with jump UL - Ub,  QH.n = A(UL, gL).n - eta lamL A(Ub, (UL-Ub) n).n
template <typename T>
struct FacePointT
{
  T G[5];
  T S[6];
};
using FacePoint = FacePointT<double>;

// Gradient traction tau(grad u).n of one side, from the reference-space
// derivatives gr[c][0..3] of (rho, m), the inverse Jacobian Ji and the normal:
// with dv[c][i] = d u_i/d xi_c,  (L n)_i = sum_c dv[c][i] (Ji n)_c,
// (L^T n)_d = sum_c Ji[c][d] (dv[c] . n),  tr L = sum_c dv[c] . Ji[c].
template <typename T, typename G>
__device__ __forceinline__ void grad_traction(const G gr[3][4], const T* U, const double Ji[3][3],
                                              const double* n, double mu, T* vg)
{
  T ir = rcp(U[0]);
  T u[3] = {U[1] * ir, U[2] * ir, U[3] * ir};
  T Ln[3] = {0.0, 0.0, 0.0}, LTn[3] = {0.0, 0.0, 0.0}, tr = 0.0;
#pragma unroll
  for (int c = 0; c < 3; ++c)
  {
    T dv0 = (gr[c][1] - gr[c][0] * u[0]) * ir;
    T dv1 = (gr[c][2] - gr[c][0] * u[1]) * ir;
    T dv2 = (gr[c][3] - gr[c][0] * u[2]) * ir;
    double mc = Ji[c][0] * n[0] + Ji[c][1] * n[1] + Ji[c][2] * n[2];
    T kc = dv0 * n[0] + dv1 * n[1] + dv2 * n[2];
    Ln[0] += dv0 * mc;
    Ln[1] += dv1 * mc;
    Ln[2] += dv2 * mc;
    LTn[0] += Ji[c][0] * kc;
    LTn[1] += Ji[c][1] * kc;
    LTn[2] += Ji[c][2] * kc;
    tr += dv0 * Ji[c][0] + dv1 * Ji[c][1] + dv2 * Ji[c][2];
  }
  tau_n(mu, Ln, LTn, tr, n, vg);
}

// vgL, vgR: gradient tractions tau(grad u).n of the own and neighbour traces
// (vgR unused on boundary faces).  tau(a (x) n).n = mu a + mu/3 (a.n) n.
// Ub is the neighbour trace (interior) or the boundary state (boundary).
template <typename T, typename V>
__device__ __forceinline__ void face_point_physics(bool interior, const T* UL, const T* Ub,
                                                   const V* vgL, const V* vgR, const double* n,
                                                   double lamL, double lamR, const Phys& ph,
                                                   FacePointT<T>& out)
{
  const double mu = ph.mu;
  T irL = rcp(UL[0]);
  T uL[3] = {UL[1] * irL, UL[2] * irL, UL[3] * irL};
  if (interior)
    roe_flux(UL, Ub, n, ph.gamma, out.G);
  else
    euler_flux_n(Ub, ph.gamma, n, out.G);
  T irB = rcp(Ub[0]);
  T uB[3] = {Ub[1] * irB, Ub[2] * irB, Ub[3] * irB};
  T jr = UL[0] - Ub[0];
  T dmL[3], dmB[3];
#pragma unroll
  for (int i = 0; i < 3; ++i)
  {
    T jm = UL[1 + i] - Ub[1 + i];
    dmL[i] = (jm - jr * uL[i]) * irL;
    dmB[i] = (jm - jr * uB[i]) * irB;
  }
  T dnL = dmL[0] * n[0] + dmL[1] * n[1] + dmL[2] * n[2];
  T dnB = dmB[0] * n[0] + dmB[1] * n[1] + dmB[2] * n[2];

  // own side: hL tau(grad u_L).n - cL tau(dmL (x) n).n (interior: halved,
  // with the penalty; boundary: the full gradient traction)
  double hL = interior ? 0.5 : 1.0;
  double cL = interior ? 0.25 * ph.eta * lamL : 0.0;
  T w[3];
#pragma unroll
  for (int i = 0; i < 3; ++i)
    w[i] = hL * vgL[i] - cL * mu * (dmL[i] + (1.0 / 3.0) * dnL * n[i]);
  T q[4] = {w[0], w[1], w[2], uL[0] * w[0] + uL[1] * w[1] + uL[2] * w[2]};

  // other side: neighbour (interior) or boundary penalty at the boundary state
  double cB = interior ? 0.25 * ph.eta * lamR : ph.eta * lamL;
  double hB = interior ? 0.5 : 0.0;
#pragma unroll
  for (int i = 0; i < 3; ++i)
    w[i] = hB * vgR[i] - cB * mu * (dmB[i] + (1.0 / 3.0) * dnB * n[i]);
  q[0] += w[0];
  q[1] += w[1];
  q[2] += w[2];
  q[3] += uB[0] * w[0] + uB[1] * w[1] + uB[2] * w[2];
#pragma unroll
  for (int i = 0; i < 3; ++i)
    out.G[1 + i] -= q[i];
  out.G[4] -= q[3];

  // dual-consistency stress tau(s dmL (x) n), s = 1/2 (interior) or 1
  double s = interior ? 0.5 : 1.0;
  T a0 = s * dmL[0], a1 = s * dmL[1], a2 = s * dmL[2];
  T lt = -(2.0 / 3.0) * mu * s * dnL;
  out.S[0] = 2.0 * mu * a0 * n[0] + lt;
  out.S[1] = 2.0 * mu * a1 * n[1] + lt;
  out.S[2] = 2.0 * mu * a2 * n[2] + lt;
  out.S[3] = mu * (a0 * n[1] + a1 * n[0]);
  out.S[4] = mu * (a0 * n[2] + a2 * n[0]);
  out.S[5] = mu * (a1 * n[2] + a2 * n[1]);
}


// One face point of the FP64 kernels: face_point_physics and what follows it,
// with fewer operations (FP64 issue bounds the state-reading kernel: 64^3 p = 3
// cube 1312 -> 1290 us per stage with a mean of 1.03x over the q = 1 cases; 1-2 %
// on the record-reading kernels).  From both traces with their velocities u and
// reciprocal densities ir, the gradient tractions, the own inverse Jacobian
// Ji with its normal products mc[c] = Ji[c] . n, and the quadrature factor sc:
//   G[r]     sc (F - QH.n)
//   hc[c][r] sc Ji[c] . dcQ, the contravariant dual-consistency flux, whose
//            stress tau(a (x) n) gives  mu ((Ji[c].a) n + mc a - 2/3 (a.n) Ji[c])
//            with a = s dmL, without forming the stress.
// D >= 0: the face is known to be normal to reference direction D, whose
// Ji[D] = mc[D] n (the row itself is not read).
template <int D = -1>
__device__ __forceinline__ void face_point_fp64(bool interior, const double* UL, const double* uL,
                                                double irL, const double* Ub, const double* uB,
                                                double irB, const double* vgL, const double* vgR,
                                                const double* n, const double Ji[3][3],
                                                const double* mc, double lamL, double lamR,
                                                double sc, const Phys& ph, double* G,
                                                double hc[3][4])
{
  const double mu = ph.mu;
  double d[5];  // Ub - UL
  if (interior)
    roe_flux_fp64(UL, uL, irL, Ub, uB, irB, n, ph.gamma, G, d);
  else
  {
    euler_flux_n(Ub, ph.gamma, n, G);
#pragma unroll
    for (int r = 0; r < 4; ++r)
      d[r] = Ub[r] - UL[r];
  }
  // velocity jumps at the two states, UL - Ub: dm = -(d_m - d_rho u) / rho
  double dmL[3], dmB[3];
#pragma unroll
  for (int i = 0; i < 3; ++i)
  {
    dmL[i] = (d[0] * uL[i] - d[1 + i]) * irL;
    dmB[i] = (d[0] * uB[i] - d[1 + i]) * irB;
  }
  const double dnL = dmL[0] * n[0] + dmL[1] * n[1] + dmL[2] * n[2];
  const double dnB = dmB[0] * n[0] + dmB[1] * n[1] + dmB[2] * n[2];
  // h tau(grad u).n - c tau(dm (x) n).n of both sides (see face_point_physics)
  const double em = ph.eta * mu;
  const double hL = interior ? 0.5 : 1.0, cL = interior ? 0.25 * em * lamL : 0.0;
  const double hB = interior ? 0.5 : 0.0, cB = interior ? 0.25 * em * lamR : em * lamL;
  const double tL = cL * (1.0 / 3.0) * dnL, tB = cB * (1.0 / 3.0) * dnB;
  double qE = 0.0;
#pragma unroll
  for (int i = 0; i < 3; ++i)
  {
    const double wL = hL * vgL[i] - cL * dmL[i] - tL * n[i];
    const double wB = hB * vgR[i] - cB * dmB[i] - tB * n[i];
    G[1 + i] = sc * (G[1 + i] - (wL + wB));
    qE += uL[i] * wL + uB[i] * wB;
  }
  G[0] *= sc;
  G[4] = sc * (G[4] - qE);
  // dual-consistency flux
  const double al = (interior ? 0.5 : 1.0) * mu * sc;
  const double a[3] = {al * dmL[0], al * dmL[1], al * dmL[2]};
  const double t = (2.0 / 3.0) * al * dnL;
#pragma unroll
  for (int c = 0; c < 3; ++c)
  {
    if (c == D)
    {
      const double k = (1.0 / 3.0) * al * dnL;
#pragma unroll
      for (int i = 0; i < 3; ++i)
        hc[c][i] = mc[c] * (a[i] + k * n[i]);
    }
    else
    {
      const double k = Ji[c][0] * a[0] + Ji[c][1] * a[1] + Ji[c][2] * a[2];
#pragma unroll
      for (int i = 0; i < 3; ++i)
        hc[c][i] = k * n[i] + mc[c] * a[i] - t * Ji[c][i];
    }
    hc[c][3] = uL[0] * hc[c][0] + uL[1] * hc[c][1] + uL[2] * hc[c][2];
  }
}

// One face point of the record-reading kernels: G scaled by sc and the
// contravariant dual-consistency flux hc, by face_point_fp64 (FAST) or, in the
// mixed forms, by face_point_physics.
template <bool FAST>
__device__ __forceinline__ void face_point(bool interior, const double* UL, const double* Ub,
                                           const double* vgL, const double* vgR, const double* n,
                                           const double Ji[3][3], double lamL, double lamR,
                                           double sc, const Phys& ph, double* G, double hc[3][4])
{
  const double irL  = rcp(UL[0]);
  const double uL[3] = {UL[1] * irL, UL[2] * irL, UL[3] * irL};
  if constexpr (FAST)
  {
    const double irB   = rcp(Ub[0]);
    const double uB[3] = {Ub[1] * irB, Ub[2] * irB, Ub[3] * irB};
    const double mc[3] = {Ji[0][0] * n[0] + Ji[0][1] * n[1] + Ji[0][2] * n[2],
                          Ji[1][0] * n[0] + Ji[1][1] * n[1] + Ji[1][2] * n[2],
                          Ji[2][0] * n[0] + Ji[2][1] * n[1] + Ji[2][2] * n[2]};
    face_point_fp64(interior, UL, uL, irL, Ub, uB, irB, vgL, vgR, n, Ji, mc, lamL, lamR, sc, ph, G,
                    hc);
  }
  else
  {
    FacePoint fpo;
    face_point_physics(interior, UL, Ub, vgL, vgR, n, lamL, lamR, ph, fpo);
    // contravariant dual-consistency flux h_c = Ji[c] . dcQ (rows 1-4)
    const double* S       = fpo.S;
    const double Sm[3][3] = {{S[0], S[3], S[4]}, {S[3], S[1], S[5]}, {S[4], S[5], S[2]}};
#pragma unroll
    for (int c = 0; c < 3; ++c)
    {
#pragma unroll
      for (int i = 0; i < 3; ++i)
        hc[c][i] = sc * (Ji[c][0] * Sm[0][i] + Ji[c][1] * Sm[1][i] + Ji[c][2] * Sm[2][i]);
      hc[c][3] = uL[0] * hc[c][0] + uL[1] * hc[c][1] + uL[2] * hc[c][2];
    }
#pragma unroll
    for (int r = 0; r < 5; ++r)
      G[r] = fpo.G[r] * sc;
  }
}

// Volume flux H = Q - F (flux.cpp:24-48 Euler, flux.cpp:156-202 Newtonian
// viscous, no heat flux) at a Gauss node, in velocity-gradient form, from the
// node state Vq and the reference-space derivatives gr[c][0..3] of (rho, m).
template <typename T, typename G>
__device__ __forceinline__ void volume_flux(const T* Vq, const G gr[3][4], const double Ji[3][3],
                                            double gamma, double mu, T H[3][5])
{
  T ir = rcp(Vq[0]);
  T u[3] = {Vq[1] * ir, Vq[2] * ir, Vq[3] * ir};
  T Lv[3][3];
  vel_grad(gr, u, ir, Ji, Lv);
  T p  = (gamma - 1.0) * (Vq[4] - 0.5 * Vq[0] * (u[0] * u[0] + u[1] * u[1] + u[2] * u[2]));
  T Ht = (Vq[4] + p) * ir;
  T lt = -(2.0 / 3.0) * mu * (Lv[0][0] + Lv[1][1] + Lv[2][2]);
#pragma unroll
  for (int d = 0; d < 3; ++d)
  {
    T tau[3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
    {
      tau[i] = mu * (Lv[d][i] + Lv[i][d]);
      if (i == d)
        tau[i] += lt;
    }
    T md    = Vq[1 + d];
    H[d][0] = -md;
#pragma unroll
    for (int i = 0; i < 3; ++i)
    {
      H[d][1 + i] = tau[i] - md * u[i];
      if (i == d)
        H[d][1 + i] -= p;
    }
    H[d][4] = u[0] * tau[0] + u[1] * tau[1] + u[2] * tau[2] - md * Ht;
  }
}

// Geometry of a Gauss node for volume_flux_fp64, from J^-1 and w det J or from J
// (w: the node's quadrature weight).
struct NodeGeo
{
  double B[3][3], A[3][3], kv, wJ;
  __device__ __forceinline__ void inverse(const double* Ji, double wdet, double mu)
  {
    wJ = wdet;
    kv = mu;
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int d = 0; d < 3; ++d)
      {
        B[c][d] = Ji[3 * c + d];
        A[c][d] = wJ * B[c][d];
      }
  }
  __device__ __forceinline__ void curved(const double J[3][3], double w, double mu)
  {
    // rows of det J Ji: cross products of the columns of J
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int d = 0; d < 3; ++d)
      {
        const int c1 = (c + 1) % 3, c2 = (c + 2) % 3, d1 = (d + 1) % 3, d2 = (d + 2) % 3;
        B[c][d] = J[d1][c1] * J[d2][c2] - J[d2][c1] * J[d1][c2];
        A[c][d] = w * B[c][d];
      }
    const double det = J[0][0] * B[0][0] + J[1][0] * B[0][1] + J[2][0] * B[0][2];
    wJ = w * det;
    kv = mu * rcp(det);
  }
};

// Contravariant volume flux F[c] = A[c] . H (H of volume_flux) of the FP64
// state-reading kernels: A[c] = w det J Ji[c], and the gradient is formed with
// rows B = Ji (kv = mu) or the adjugate det J Ji (kv = mu / det J):
//   A.(tau - u m - p) = S A - (A.m) u  with  S = tau - p I,  and the energy row
//   u.(S A) - (E/rho) (A.m)
// (VISC false: the inviscid part, tau = 0, gr and B not read),
// 130 operations where H, then A H, take 175 (64^3 p = 3 cube 1161 -> 1150 us per
// RK4 stage with the factor n of Ji[D] taken out in face_traction and
// face_point_fp64: 3 % fewer FP64 operations; general-order kernel 20^3 p = 5 223.6 ->
// 220.5 us).
template <bool VISC = true>
__device__ __forceinline__ void volume_flux_fp64(const double* Vq, const double gr[3][4],
                                                 const double B[3][3], double kv,
                                                 const double A[3][3], double gamma,
                                                 double F[3][5])
{
  const double ir = rcp(Vq[0]);
  const double u[3] = {Vq[1] * ir, Vq[2] * ir, Vq[3] * ir};
  const double p = (gamma - 1.0) *
                   (Vq[4] - 0.5 * (Vq[1] * u[0] + Vq[2] * u[1] + Vq[3] * u[2]));
  double S[6] = {-p, -p, -p, 0.0, 0.0, 0.0};
  if constexpr (VISC)
  {
    double L[3][3];  // rho d u_i / d x_d
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int i = 0; i < 3; ++i)
      {
        const double dv = gr[c][1 + i] - gr[c][0] * u[i];
#pragma unroll
        for (int d = 0; d < 3; ++d)
          L[d][i] = (c == 0) ? B[c][d] * dv : L[d][i] + B[c][d] * dv;
      }
    const double k = kv * ir, k2 = 2.0 * k;
    const double t = -(2.0 / 3.0) * k * (L[0][0] + L[1][1] + L[2][2]) - p;
    S[0] = k2 * L[0][0] + t;
    S[1] = k2 * L[1][1] + t;
    S[2] = k2 * L[2][2] + t;
    S[3] = k * (L[0][1] + L[1][0]);
    S[4] = k * (L[0][2] + L[2][0]);
    S[5] = k * (L[1][2] + L[2][1]);
  }
  const double e = Vq[4] * ir;
#pragma unroll
  for (int c = 0; c < 3; ++c)
  {
    const double* a = A[c];
    const double m  = a[0] * Vq[1] + a[1] * Vq[2] + a[2] * Vq[3];
    const double s0 = VISC ? S[0] * a[0] + S[3] * a[1] + S[4] * a[2] : S[0] * a[0];
    const double s1 = VISC ? S[3] * a[0] + S[1] * a[1] + S[5] * a[2] : S[1] * a[1];
    const double s2 = VISC ? S[4] * a[0] + S[5] * a[1] + S[2] * a[2] : S[2] * a[2];
    F[c][0] = -m;
    F[c][1] = s0 - m * u[0];
    F[c][2] = s1 - m * u[1];
    F[c][3] = s2 - m * u[2];
    F[c][4] = u[0] * s0 + u[1] * s1 + u[2] * s2 - m * e;
  }
}

// Inviscid part of volume_flux (H = -F, the Euler flux): the values
// volume_flux gives with mu = 0, whose viscous terms are exact zeros.
template <typename T>
__device__ __forceinline__ void euler_volume_flux(const T* Vq, double gamma, T H[3][5])
{
  T ir = rcp(Vq[0]);
  T u[3] = {Vq[1] * ir, Vq[2] * ir, Vq[3] * ir};
  T p  = (gamma - 1.0) * (Vq[4] - 0.5 * Vq[0] * (u[0] * u[0] + u[1] * u[1] + u[2] * u[2]));
  T Ht = (Vq[4] + p) * ir;
#pragma unroll
  for (int d = 0; d < 3; ++d)
  {
    T md    = Vq[1 + d];
    H[d][0] = -md;
#pragma unroll
    for (int i = 0; i < 3; ++i)
    {
      H[d][1 + i] = -(md * u[i]);
      if (i == d)
        H[d][1 + i] -= p;
    }
    H[d][4] = -(md * Ht);
  }
}

}  // namespace dgx
