// dgx_tile_state.hpp -- the FP64 tiled stage: tiles and face subpasses as in
// dgx_tile.hpp, but both traces of a face point and their gradient tractions
// are formed from the element states instead of read from trace records.
//
// What bounds the record-reading kernel is its traffic: at p = 3 a stage moves
// 458 B per degree of freedom, 288 of them trace records (written once, read
// by the own and the neighbour side), at the rate of a large copy.  Reading
// the neighbour's 4 nodes behind each face point instead (L2 and Infinity
// Cache hits mostly: every element is read once as own and six times as a
// neighbour) leaves the state arrays; the traces of the new state need not be
// produced, only the states of inflow and outflow boundary faces.  What bounds
// this kernel is FP64 issue (about 2150 FP64 and 160 matrix instructions per
// wavefront of 128 nodes).  It runs p = 1 and, below the size where the tiles of
// dgx_line_state.hpp fill the chip, p = 3.  Per RK4 stage, 64^3 p = 3 cube: 1266 us
// against 1698 us (traffic 5.1 against 7.5 GB); 64^3 p = 1 cube: 267 us against
// 369 us (one-row record kernel: 442); 61x37x43 p = 1 curved channel 137 us
// against 188 us one-row.
// Included by dgx_stage.hpp inside namespace dgx, after dgx_tile.hpp.
#pragma once

template <int I>
struct Const
{
  static constexpr int value = I;
};

// Fills the face table as tile_face_table does; whether a face of the tile's E
// elements lies on a characteristic boundary (uniform), whose state the next
// stage reads instead of forming it (wall_state) at the face point.
template <int E>
__device__ __forceinline__ bool state_face_table(const MeshArgs& mesh, int e0, int (*sNb)[6],
                                                 int (*sBt)[6])
{
  static_assert(E * 6 <= 64, "one face per lane");
  tile_face_table<E>(mesh, e0, sNb, sBt);
  const int x = threadIdx.x;  // each lane reads back the face it wrote
  return __any(x < E * 6 && characteristic_bc(sBt[x / 6][x % 6]));
}

// The lane index, opaque to common subexpressions: each face subpass derives
// its indices again (a few integer operations) instead of holding those of
// all subpasses in registers.
__device__ __forceinline__ void phase_fence()
{
  __syncthreads();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// Ends the live ranges of one step of a face subpass before the next begins:
// what follows (a later such tie, or a read of x or y) comes after v[0..2]
// exist.  Without these ties the two sides' traces, tractions and the face
// physics are interleaved into one block that needs over 240 registers.
__device__ __forceinline__ void order_after(double* v)
{
  asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]));
}
__device__ __forceinline__ void order_after(double* v, double& x, double& y)
{
  asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(x), "+v"(y));
}

__device__ __forceinline__ int opaque_tid()
{
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

// ---- p = 3: FP64 contractions on the matrix cores --------------------------
// v_mfma_f64_4x4x4_4b multiplies four 4x4 blocks: lane j + 4b + 16k holds
// A[b][j][k], B[b][k][j] and D[b][k][j] (measured with an in-bounds probe), so
// with 64 values laid out by three 2-bit lane fields (lo, mid, hi), mid is the
// block and one instruction contracts hi with a 4x4 table:
//   A = table, B = x:  (lo, mid, hi) -> (lo, mid, hi')
//   A = x, B = table:  (lo, mid, hi) -> (hi', mid, lo)
// (t(lane) = M[lane & 3][lane >> 4] is the operand of out[i] = sum_k M[i][k] x[k]
// in both), and lo is contracted by the second form applied twice, first
// with the identity.  The instruction takes the FP64 pipe for the 16 cycles
// of the four FMAs it replaces; what it saves is their LDS reads (4 per value
// and 8 for the table rows, each 4 cycles of a pipe that four SIMDs share) and
// the exchange through LDS with its barriers.
struct MfTabs
{
  double one, dg, dgt, ndgt;  // identity, Dg, Dg^T, -Dg^T
};

__device__ __forceinline__ MfTabs mf_tabs(const PTab& pt)
{
  const int i = threadIdx.x & 3, k = threadIdx.x >> 4;
  MfTabs t;
  t.one  = (i == k) ? 1.0 : 0.0;
  t.dg   = pt.Dg[i][k];
  t.dgt  = pt.Dg[k][i];
  t.ndgt = -t.dgt;
  return t;
}

// c + (table t along hi) x
__device__ __forceinline__ double mf_hi(double t, double x, double c)
{
  return __builtin_amdgcn_mfma_f64_4x4x4f64(t, x, c, 0, 0, 0);
}

// c + (table t along lo) x
__device__ __forceinline__ double mf_lo(double one, double t, double x, double c)
{
  return __builtin_amdgcn_mfma_f64_4x4x4f64(
      __builtin_amdgcn_mfma_f64_4x4x4f64(x, one, 0.0, 0, 0, 0), t, c, 0, 0, 0);
}

// The line of nodes behind face point (a, b) of a face normal to D: x[r][m] of
// the element's Gauss-nodal state V ([5][NB], in LDS or global memory).
template <int P, int D>
__device__ __forceinline__ void line_load(const double* V, int a, int b, double (&x)[5][P + 1])
{
  constexpr int N = P + 1, NB = N * N * N;
  int id[3];
  id[Tang<D>::T1] = a;
  id[Tang<D>::T2] = b;
#pragma unroll
  for (int r = 0; r < 5; ++r)
#pragma unroll
    for (int m = 0; m < N; ++m)
    {
      id[D]   = m;
      x[r][m] = V[r * NB + (id[2] * N + id[1]) * N + id[0]];
    }
}

// Trace U (5) and normal derivative dn (density and momentum) from the line's
// values and the end's table rows.
template <int N>
__device__ __forceinline__ void line_traces(const double (&x)[5][N], const double* L,
                                            const double* Ld, double* U, double* dn)
{
#pragma unroll
  for (int r = 0; r < 5; ++r)
  {
    double v = 0.0, dv = 0.0;
#pragma unroll
    for (int m = 0; m < N; ++m)
    {
      v += L[m] * x[r][m];
      if (r < 4)
        dv += Ld[m] * x[r][m];
    }
    U[r] = v;
    if (r < 4)
      dn[r] = dv;
  }
}

// Gradient traction tau(grad u).n of one side of a face point normal to D: its
// trace U with velocity u and reciprocal density ir, normal derivative dn,
// tangential derivatives tan(c, r) of variable r along direction c, inverse
// Jacobian Ji with mc[c] = Ji[c] . n (Ji[D] = mc[D] n is not read).  The sums of
// grad_traction, scaled by mu/rho once, one reference direction after the other,
// so that four derivatives are live at a time instead of twelve.
template <int D, typename Tan>
__device__ __forceinline__ void face_traction(Tan tan, const double* U, const double* u, double ir,
                                              const double* dn, const double Ji[3][3],
                                              const double* n, const double* mc, double mu,
                                              double* vg)
{
  double A[3] = {0.0, 0.0, 0.0}, tr = 0.0;
#pragma unroll
  for (int c = 0; c < 3; ++c)
  {
    double g[4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
      g[r] = (c == D) ? dn[r] : tan(c, r);
    // rho d u / d xi_c
    const double dv[3] = {g[1] - g[0] * u[0], g[2] - g[0] * u[1], g[3] - g[0] * u[2]};
    const double kc = dv[0] * n[0] + dv[1] * n[1] + dv[2] * n[2];
    if (c == D)
    {
      const double k = mc[c] * kc;
#pragma unroll
      for (int i = 0; i < 3; ++i)
        A[i] += dv[i] * mc[c] + k * n[i];
      tr += k;
    }
    else
    {
#pragma unroll
      for (int i = 0; i < 3; ++i)
      {
        A[i] += dv[i] * mc[c] + Ji[c][i] * kc;
        tr += dv[i] * Ji[c][i];
      }
    }
    order_after(A);
  }
  const double k = mu * ir, t = (2.0 / 3.0) * tr;
#pragma unroll
  for (int i = 0; i < 3; ++i)
    vg[i] = k * (A[i] - t * n[i]);
}

// The two tangential rows of J^-1 and mc[c] = Ji[c] . n (see face_traction) at a
// face point normal to D, from the normal column of J, the tangential ones t1
// and t2 (t1, t2 = columns D+1 and D+2, cyclic), the normal n and sg = +-1 / |t1 x t2|:
// det J = (J_D . n) / sg, so that Ji[D] = n / (J_D . n).
template <int D>
__device__ __forceinline__ void face_inverse(const double* jd, const double* t1, const double* t2,
                                             const double* n, double sg, double Ji[3][3],
                                             double* mc)
{
  constexpr int c1 = (D + 1) % 3, c2 = (D + 2) % 3;
  mc[D] = rcp(jd[0] * n[0] + jd[1] * n[1] + jd[2] * n[2]);
  const double id = mc[D] * sg;
  const double b[3] = {id * jd[0], id * jd[1], id * jd[2]};
#pragma unroll
  for (int i = 0; i < 3; ++i)
  {
    const int j = (i + 1) % 3, k = (i + 2) % 3;
    Ji[c1][i] = t2[j] * b[k] - t2[k] * b[j];
    Ji[c2][i] = b[j] * t1[k] - b[k] * t1[j];
  }
  mc[c1] = Ji[c1][0] * n[0] + Ji[c1][1] * n[1] + Ji[c1][2] * n[2];
  mc[c2] = Ji[c2][0] * n[0] + Ji[c2][1] * n[1] + Ji[c2][2] * n[2];
}

// Geometry a tile keeps per element face about the element across it: on
// affine meshes the neighbour's J^-1 (9), else the four edge vectors of the
// neighbour along the face direction (12), from which the normal column of
// its Jacobian follows at every face point; its tangential columns are the
// own side's, the face being shared up to a translation (MeshArgs::matched).
template <bool AFF>
struct NbrGeo
{
  static constexpr int n = AFF ? 9 : 12;
};

// value k of that record for face f of tile element l
template <bool AFF>
__device__ __forceinline__ double nbr_geo_load(const MeshArgs& mesh, int en, int f, int k)
{
  if constexpr (AFF)
    return mesh.arec[(size_t)en * GREC + 10 + k];
  const int c = k / 3, d = k % 3, nd = f >> 1;  // corner pair c, component d
  const int t1 = (nd == 0) ? 2 : 1, t2 = (nd == 2) ? 2 : 4, hi = 1 << nd;  // node strides
  const int lo = (c & 1) * t1 + (c >> 1) * t2;
  const double* X = mesh.nodes + (size_t)en * 24;
  return X[3 * (lo + hi) + d] - X[3 * lo + d];
}

// The columns of J = d x / d xi at point (a, b) of face (D, hi) of a trilinear
// element with nodes X (x fastest): j[c], with ga and gb the point's coordinates
// along the face, and the bilinear weights w4 of the face's corners.  The face's
// columns follow from its own four nodes and the normal one from the four
// edges that leave it: 52 operations, half of the sums over 8 nodes of the
// general form (jac_at).  With face_inverse and LineGeo, per stage: 48x24x24 p = 3
// channel 157 -> 138 us (TVD-RK3), 61x37x43 p = 1 139 -> 133, 30x24x28 p = 2 88 -> 83 (RK4).
template <int D>
__device__ __forceinline__ void trilinear_face(const double* X, int hi, double ga, double gb,
                                               double (&w4)[4], double j[3][3])
{
  constexpr int T1 = Tang<D>::T1, T2 = Tang<D>::T2, s1 = 3 << T1, s2 = 3 << T2, sn = 3 << D;
  const double fa = 1.0 - ga, fb = 1.0 - gb;
  w4[0] = fa * fb;
  w4[1] = ga * fb;
  w4[2] = fa * gb;
  w4[3] = ga * gb;
  const double* F = X + hi * sn;
#pragma unroll
  for (int i = 0; i < 3; ++i)
  {
    const double a0 = F[s1 + i] - F[i], a1 = F[s1 + s2 + i] - F[s2 + i];
    const double b0 = F[s2 + i] - F[i], b1 = F[s1 + s2 + i] - F[s1 + i];
    j[T1][i] = fb * a0 + gb * a1;
    j[T2][i] = fa * b0 + ga * b1;
    j[D][i]  = w4[0] * (X[sn + i] - X[i]) + w4[1] * (X[sn + s1 + i] - X[s1 + i]) +
              w4[2] * (X[sn + s2 + i] - X[s2 + i]) +
              w4[3] * (X[sn + s1 + s2 + i] - X[s1 + s2 + i]);
  }
}

// Physics of one face point from both sides' traces (UL, Ub) and normal
// derivatives (dL, dR) with tangential derivatives tanL, tanR: the flux G and
// the test-function fluxes hc, as face_point_fp64.  X, g, h: geometry of the
// own element (nodes or record) and of the neighbour (NbrGeo); en, bt: neighbour
// and boundary code; w: the point's quadrature weight.  next() starts the loads
// that follow, when the registers of the tractions are free.
template <int P, int Q, int D, bool AFF, typename TanL, typename TanR, typename Next>
__device__ __forceinline__ void face_states(const MeshArgs& mesh, const Phys& ph, const QTab& qt,
                                            const double* __restrict__ Tin, const double* X,
                                            const double* g, const double* h, int en, int bt,
                                            int hi, int a, int b, double w, double* UL,
                                            const double* dL, double* Ub, const double* dR,
                                            double lamL, double lamR, TanL tanL, TanR tanR,
                                            Next next, double* G, double (&hc)[3][4])
{
  constexpr int N = P + 1, NF = N * N;
  double j[3][3], w4[4];                // curved: columns of the own J, corner weights
  double JiL[3][3], nv[3], mcL[3], fJ, sg = 0.0;
  if constexpr (AFF)
  {
    fJ = face_geometry<Q, AFF>(qt, X, g, D, hi, 0, 0, 0, JiL, nv);
#pragma unroll
    for (int i = 0; i < 3; ++i)
      mcL[i] = JiL[i][0] * nv[0] + JiL[i][1] * nv[1] + JiL[i][2] * nv[2];
  }
  else
  {
    trilinear_face<D>(X, hi, qt.Bq[a][1], qt.Bq[b][1], w4, j);
    const double *t1 = j[(D + 1) % 3], *t2 = j[(D + 2) % 3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
      nv[i] = t1[(i + 1) % 3] * t2[(i + 2) % 3] - t1[(i + 2) % 3] * t2[(i + 1) % 3];
    const double n2 = nv[0] * nv[0] + nv[1] * nv[1] + nv[2] * nv[2], r = rsq(n2);
    fJ = n2 * r;
    sg = hi ? r : -r;
#pragma unroll
    for (int i = 0; i < 3; ++i)
      nv[i] *= sg;
    face_inverse<D>(j[D], t1, t2, nv, sg, JiL, mcL);
  }
  double uL[3], uR[3], vgL[3], vgR[3];
  const double irL = rcp(UL[0]), irR = rcp(Ub[0]);
#pragma unroll
  for (int i = 0; i < 3; ++i)
  {
    uL[i] = UL[1 + i] * irL;
    uR[i] = Ub[1 + i] * irR;
  }
  face_traction<D>(tanL, UL, uL, irL, dL, JiL, nv, mcL, ph.mu, vgL);
  order_after(vgL);
  {
    double JiR[3][3], mcR[3];
    if constexpr (AFF)
    {
#pragma unroll
      for (int c = 0; c < 3; ++c)
      {
#pragma unroll
        for (int i = 0; i < 3; ++i)
          JiR[c][i] = h[3 * c + i];
        mcR[c] = JiR[c][0] * nv[0] + JiR[c][1] * nv[1] + JiR[c][2] * nv[2];
      }
    }
    else
    {
      double jd[3] = {0.0, 0.0, 0.0};
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int i = 0; i < 3; ++i)
          jd[i] += w4[c] * h[3 * c + i];
      face_inverse<D>(jd, j[(D + 1) % 3], j[(D + 2) % 3], nv, sg, JiR, mcR);
    }
    face_traction<D>(tanR, Ub, uR, irR, dR, JiR, nv, mcR, ph.mu, vgR);
  }
  order_after(vgR, UL[0], Ub[0]);
  next();
  double irB = irR;
  if (en < 0)
  {
    if (characteristic_bc(bt))
    {
      // written with Vin
      const double* B =
          Tin + (size_t)mesh.nelem * 6 * 8 * NF + (size_t)(-1 - en) * 5 * NF + a + N * b;
#pragma unroll
      for (int r = 0; r < 5; ++r)
        Ub[r] = B[r * NF];
    }
    else
      wall_state(bt, UL, nv, ph, Ub);
    irB = rcp(Ub[0]);
#pragma unroll
    for (int i = 0; i < 3; ++i)
    {
      uR[i]  = Ub[1 + i] * irB;
      vgR[i] = 0.0;
    }
  }
  face_point_fp64<D>(en >= 0, UL, uL, irL, Ub, uR, irB, vgL, vgR, nv, JiL, mcL, lamL, lamR, fJ * w,
                  ph, G, hc);
}

// This lane's face point in subpass D of a tile, the tile's 2 E faces normal to
// direction D: face point (a, b) of local face f of tile element l, whose
// element is e.  Every lane has one (p = 1 and 3: 64 face points a subpass);
// faces of elements past the end of the mesh give values that no node gathers.
template <int P, int R, int D>
struct FaceLane
{
  using TD = TileDims<P, R>;
  static_assert(2 * TD::E * TD::NF == 64, "one face point of the subpass per lane");
  int tid, slot, a, b, l, hi, f, e;
  __device__ __forceinline__ FaceLane(const MeshArgs& mesh, int e0)
  {
    tid  = opaque_tid();
    slot = (P == 3) ? (tid >> 2) & 3 : tid / TD::NF;  // element slot / 2, side slot % 2
    const int t = tid % TD::NF;
    a  = (P == 3) ? tid & 3 : t % TD::N;
    b  = (P == 3) ? tid >> 4 : t / TD::N;
    l  = slot >> 1;
    hi = slot & 1;
    f  = 2 * D + hi;
    e  = min(e0 + l, mesh.nelem - 1);
  }
};

// What a face point reads from global memory about the element across its
// face: the line of nodes behind the point and both lifting coefficients.
// Loaded one subpass ahead (before the volume terms for the first subpass),
// so that the loads are in flight during the face physics.
template <int P>
struct FaceData
{
  double x[5][P + 1];
  double lamL, lamR;
};

template <int P, int R, int D, bool AFF>
__device__ __forceinline__ void face_load(const MeshArgs& mesh, const double* __restrict__ Vin,
                                          const double* __restrict__ lam, const int (*sNb)[6],
                                          int e0, FaceData<P>& fd)
{
  constexpr int NB = TileDims<P, R>::NB, NF = TileDims<P, R>::NF;
  const FaceLane<P, R, D> fl(mesh, e0);
  // (a boundary face reads its own element here; those values are not used)
  const int nb = sNb[fl.l][fl.f], en = nb >= 0 ? nb : fl.e;
  line_load<P, D>(Vin + (size_t)en * 5 * NB, fl.a, fl.b, fd.x);
  // affine meshes: the face's constant coefficient (48 B per element instead
  // of 6 (p+1)^2 doubles, read for the own and the neighbour side)
  const size_t iL = (size_t)fl.e * 6 + fl.f, iR = (size_t)en * 6 + (fl.f ^ 1);
  const int fpt = fl.a + (P + 1) * fl.b;
  fd.lamL = AFF ? mesh.lamf[iL] : lam[iL * NF + fpt];
  fd.lamR = AFF ? mesh.lamf[iR] : lam[iR * NF + fpt];
}

// Subpass D: both sides' traces and gradient tractions from the states (own
// from LDS, neighbour in fd), face point physics of the faces normal to
// direction D, the tangential (T) phase and the gather into the nodes'
// accumulators.  next() starts the loads that follow.
template <int P, int Q, int R, int D, bool AFF, typename Next>
__device__ __forceinline__ void state_face_subpass(
    const MeshArgs& mesh, const Phys& ph, const PTab& pt, const QTab& qt,
    const double* __restrict__ Tin, const double (*sV)[5][TileDims<P, R>::NB],
    const double (*sX)[(Q + 1) * (Q + 1) * (Q + 1) * 3], const double (*sG)[GREC],
    const double (*sH)[NbrGeo<AFF>::n], const int (*sNb)[6], const int (*sBt)[6], double* sR,
    const MfTabs& mf, int e0, double (&acc)[R][5], FaceData<P>& fd, Next next)
{
  using TD = TileDims<P, R>;
  constexpr int N = TD::N, NB = TD::NB, NF = TD::NF, EPR = TD::EPR;
  constexpr int T1 = Tang<D>::T1, T2 = Tang<D>::T2;
  const FaceLane<P, R, D> fl(mesh, e0);
  const int tid = fl.tid, a = fl.a, b = fl.b, l = fl.l, hi = fl.hi, f = fl.f;
  const int fbase = fl.slot * NF;

  double UL[5], dL[4], Ub[5], dR[4];
  const int en = sNb[l][f];
  {
    double xL[5][N];
    line_load<P, D>(&sV[l][0][0], a, b, xL);
    line_traces<N>(xL, pt.L[hi], pt.Ld[hi], UL, dL);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
    asm volatile("" : "+v"(UL[r]), "+v"(dL[r]), "+v"(fd.x[r][0]));
  line_traces<N>(fd.x, pt.L[1 - hi], pt.Ld[1 - hi], Ub, dR);
  const double lamL = fd.lamL, lamR = fd.lamR;
  if constexpr (P != 3)
  {
#pragma unroll
    for (int r = 0; r < 4; ++r)
    {
      sR[r * 64 + tid]       = UL[r];
      sR[(4 + r) * 64 + tid] = Ub[r];
    }
    phase_fence();
  }
  double G[5], hn[4], hc[3][4];
  {
    auto tan = [&](const double* U, const double* s, int c, int r) __attribute__((always_inline)) {
      if constexpr (P == 3)
        return (c == T1) ? mf_lo(mf.one, mf.dg, U[r], 0.0) : mf_hi(mf.dg, U[r], 0.0);
      double d = 0.0;
#pragma unroll
      for (int m = 0; m < N; ++m)
        d += (c == T1) ? pt.Dg[a][m] * s[r * 64 + fbase + m + N * b]
                       : pt.Dg[b][m] * s[r * 64 + fbase + a + N * m];
      return d;
    };
    face_states<P, Q, D, AFF>(
        mesh, ph, qt, Tin, sX[l], sG[l], sH[6 * l + f], en, sBt[l][f], hi, a, b,
        pt.w[a] * pt.w[b], UL, dL, Ub, dR, lamL, lamR,
        [&](int c, int r) __attribute__((always_inline)) { return tan(UL, sR, c, r); },
        [&](int c, int r) __attribute__((always_inline)) { return tan(Ub, sR + 4 * 64, c, r); },
        next, G, hc);
  }
  // T = G - Dg^T(t1) h_t1 - Dg^T(t2) h_t2 (the mass row has no viscous part)
#pragma unroll
  for (int r = 0; r < 4; ++r)
    hn[r] = hc[D][r];
  if constexpr (P == 3)
  {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      G[1 + r] = mf_hi(mf.ndgt, hc[T2][r], mf_lo(mf.one, mf.ndgt, hc[T1][r], G[1 + r]));
  }
  else
  {
    phase_fence();
#pragma unroll
    for (int r = 0; r < 4; ++r)
    {
      sR[r * 64 + tid]       = hc[T1][r];
      sR[(4 + r) * 64 + tid] = hc[T2][r];
    }
    phase_fence();
#pragma unroll
    for (int r = 1; r < 5; ++r)
    {
      double t = G[r];
#pragma unroll
      for (int m = 0; m < N; ++m)
      {
        t -= pt.Dg[m][a] * sR[(r - 1) * 64 + fbase + m + N * b];
        t -= pt.Dg[m][b] * sR[(3 + r) * 64 + fbase + a + N * m];
      }
      G[r] = t;
    }
  }
  phase_fence();
#pragma unroll
  for (int r = 0; r < 5; ++r)
    sR[r * 64 + tid] = G[r];
#pragma unroll
  for (int r = 0; r < 4; ++r)
    sR[(5 + r) * 64 + tid] = hn[r];
  phase_fence();
  // gather: each node takes its element's low and high face of direction D
#pragma unroll
  for (int rr = 0; rr < R; ++rr)
  {
    const int le = rr * EPR + tid / NB;
    const int nd0 = tid % NB;
    if (tid < EPR * NB && e0 + le < mesh.nelem)
    {
      const int idx[3] = {nd0 % N, (nd0 / N) % N, nd0 / (N * N)};
      const int m = idx[D];
#pragma unroll
      for (int h = 0; h < 2; ++h)
      {
        const int gg = 2 * le + h;
        const int fp = (P == 3) ? idx[T1] + 4 * gg + 16 * idx[T2]
                                : gg * NF + idx[T2] * N + idx[T1];
        acc[rr][0] += pt.L[h][m] * sR[fp];
#pragma unroll
        for (int r = 1; r < 5; ++r)
          acc[rr][r] += pt.L[h][m] * sR[r * 64 + fp] - pt.Ld[h][m] * sR[(4 + r) * 64 + fp];
      }
    }
  }
  phase_fence();
}

// Of the tile's new states in sV: the boundary states of its characteristic
// boundary faces (what the next tiled stage reads), or with records != 0 the trace
// records of every face too (see produce_traces, whose layout they have).  One
// loop over passes of whole faces, the face direction a per-lane value: run
// by tiles at the domain boundary and by the adjoint's forward sweep only, so
// one compact copy of the code.  Every lane calls.
template <int P, int Q, int R, bool AFF>
__device__ __forceinline__ void state_traces(const MeshArgs& mesh, const Phys& ph, const PTab& pt,
                                            const QTab& qt,
                                            const double (*sV)[5][TileDims<P, R>::NB],
                                            const double (*sX)[(Q + 1) * (Q + 1) * (Q + 1) * 3],
                                            const double (*sG)[GREC], const int (*sNb)[6],
                                            const int (*sBt)[6], double* sR, int e0, int records,
                                            double* __restrict__ Tout, bool& ok)
{
  using TD = TileDims<P, R>;
  constexpr int N = TD::N, NF = TD::NF, FPS = TD::FPS, NFACE = 6 * TD::E;
  double* Tb = Tout + (size_t)mesh.nelem * 6 * 8 * NF;
  const int tid = threadIdx.x, slot = tid / NF, fpt = tid % NF;
  const int a = fpt % N, b = fpt / N, fbase = slot * NF;
#pragma unroll 1
  for (int g0 = 0; g0 < NFACE; g0 += FPS)
  {
    const int g = g0 + slot, l = g / 6, f = g % 6, ee = e0 + l;
    const bool fact = (slot < FPS) && (g < NFACE) && (ee < mesh.nelem);
    const int nb = fact && (records || characteristic_bc(sBt[l][f])) ? sNb[l][f] : 0;
    if (!records && !__any(nb < 0))
      continue;
    const int nd = f >> 1, hi = f & 1;
    double U[5], dn[4];
    if (fact)
    {
#pragma unroll
      for (int r = 0; r < 5; ++r)
      {
        double v = 0.0, dv = 0.0;
#pragma unroll
        for (int m = 0; m < N; ++m)
        {
          const double x = sV[l][r][line_node<N>(nd, m, a, b)];
          v += pt.L[hi][m] * x;
          if (r < 4)
            dv += pt.Ld[hi][m] * x;
        }
        U[r] = v;
        if (r < 4)
        {
          dn[r]            = dv;
          sR[r * 64 + tid] = v;
        }
      }
    }
    __syncthreads();
    if (fact && (records || nb < 0))
    {
      const int gi0 = (nd == 0) ? 0 : a;
      const int gi1 = (nd == 1) ? 0 : ((nd == 0) ? a : b);
      const int gi2 = (nd == 2) ? 0 : b;
      double Ji[3][3], nv[3];
      face_geometry<Q, AFF, true>(qt, sX[l], sG[l], nd, hi, gi0, gi1, gi2, Ji, nv);
      if (records)
      {
        double gr[3][4];
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
          double d1 = 0.0, d2 = 0.0;
#pragma unroll
          for (int m = 0; m < N; ++m)
          {
            d1 += pt.Dg[a][m] * sR[r * 64 + fbase + m + N * b];
            d2 += pt.Dg[b][m] * sR[r * 64 + fbase + a + N * m];
          }
          gr[0][r] = pick3(nd, dn[r], d1, d1);
          gr[1][r] = pick3(nd, d1, dn[r], d2);
          gr[2][r] = pick3(nd, d2, d2, dn[r]);
        }
        double vg[3];
        grad_traction(gr, U, Ji, nv, ph.mu, vg);
        double* T = Tout + ((size_t)ee * 6 + f) * 8 * NF + fpt;
#pragma unroll
        for (int r = 0; r < 5; ++r)
          T[r * NF] = U[r];
#pragma unroll
        for (int i = 0; i < 3; ++i)
          T[(5 + i) * NF] = vg[i];
      }
      if (nb < 0)
      {
        double Ub[5];
        ok = boundary_state(sBt[l][f], U, nv, ph, Ub) && ok;
        double* B = Tb + (size_t)(-1 - nb) * 5 * NF + fpt;
#pragma unroll
        for (int r = 0; r < 5; ++r)
          B[r * NF] = Ub[r];
      }
    }
    __syncthreads();
  }
}

// LDS of one tile, carved from a byte buffer (see StageLds).
template <int P, int Q, int R, bool AFF>
struct StateLds
{
  using TD = TileDims<P, R>;
  static constexpr int E = TD::E, NB = TD::NB, NG = (Q + 1) * (Q + 1) * (Q + 1);
  static constexpr size_t oV  = 0;
  static constexpr size_t oX  = oV + sizeof(double) * E * 5 * NB;  // nodes, or affine records
  static constexpr size_t oH  = oX + sizeof(double) * E * (AFF ? GREC : NG * 3);
  static constexpr size_t oR  = oH + sizeof(double) * E * 6 * NbrGeo<AFF>::n;
  static constexpr size_t oPT = oR + sizeof(double) * TD::SR;
  static constexpr size_t oQT = oPT + sizeof(PTab);
  static constexpr size_t oNb = oQT + sizeof(QTab);
  static constexpr size_t oBt = oNb + sizeof(int) * E * 6;
  static constexpr size_t bytes = oBt + sizeof(int) * E * 6;
};

// The tiled stage: f_g of the tile's E elements (tile number `block`)
// fused with the RK stage of StageArgs, then of the new state the boundary
// states of characteristic faces or, with sa.records, every face's trace record
// (see stage_body_lds for the meaning of every argument; the arithmetic per
// point is the same up to rounding), in the LDS region lds
// (StateLds<P, Q, R, AFF>::bytes, 16-byte aligned).  NORM: the instance that also
// writes the tile's sum of R^2 to sa.normp (the first stage of a step with its
// residual norm); kept apart so that the other stages run code without it.
template <int P, int Q, int R, bool AFF, bool NORM>
__device__ __forceinline__ void state_body(const MeshArgs& mesh, const Phys& ph,
                                              const StageArgs& sa,
                                              const double* __restrict__ lam, int* status,
                                              int block, unsigned char* lds)
{
  using TD = TileDims<P, R>;
  using TL = StateLds<P, Q, R, AFF>;
  constexpr int N = TD::N, NB = TD::NB, EPR = TD::EPR, E = TD::E;
  constexpr int NG = (Q + 1) * (Q + 1) * (Q + 1);

  auto sV  = reinterpret_cast<double(*)[5][NB]>(lds + TL::oV);
  auto sX  = reinterpret_cast<double(*)[NG * 3]>(lds + TL::oX);  // curved meshes
  auto sG  = reinterpret_cast<double(*)[GREC]>(lds + TL::oX);    // affine meshes
  auto sH  = reinterpret_cast<double(*)[NbrGeo<AFF>::n]>(lds + TL::oH);
  double* sR = reinterpret_cast<double*>(lds + TL::oR);
  PTab& sPT = *reinterpret_cast<PTab*>(lds + TL::oPT);
  QTab& sQT = *reinterpret_cast<QTab*>(lds + TL::oQT);
  auto sNb = reinterpret_cast<int(*)[6]>(lds + TL::oNb);
  auto sBt = reinterpret_cast<int(*)[6]>(lds + TL::oBt);
  stage_tables<P, Q>(&sPT, &sQT);
  const PTab& pt = sPT;
  const QTab& qt = sQT;

  const int tid = threadIdx.x;
  const int e0  = block * E;
  const int nd0 = tid % NB;
  const double* __restrict__ Tin = sa.Tin;
  const bool wall = state_face_table<E>(mesh, e0, sNb, sBt);

  // ---- load the tile's states and element geometry ----
#pragma unroll
  for (int rr = 0; rr < R; ++rr)
  {
    const int le = rr * EPR + tid / NB;
    if (tid < EPR * NB && e0 + le < mesh.nelem)
    {
#pragma unroll
      for (int r = 0; r < 5; ++r)
        sV[le][r][nd0] = sa.Vin[((size_t)(e0 + le) * 5 + r) * NB + nd0];
    }
  }
  {
    constexpr int NX = AFF ? GREC : NG * 3;
    const double* src = (AFF ? mesh.arec : mesh.nodes) + (size_t)e0 * NX;
    double* dst       = reinterpret_cast<double*>(lds + TL::oX);
    const int left    = min(mesh.nelem - e0, E) * NX;
    for (int x = tid; x < E * NX; x += 64)
      dst[x] = (x < left) ? src[x] : 0.0;
  }
  __syncthreads();
  const MfTabs mf = (P == 3) ? mf_tabs(pt) : MfTabs{};
  // geometry of the elements across the tile's faces (read in the face phase)
  constexpr int NH = (E * 6 * NbrGeo<AFF>::n + 63) / 64;
  double hg[NH];
#pragma unroll
  for (int k = 0; k < NH; ++k)
  {
    const int x = tid + 64 * k, fc = x / NbrGeo<AFF>::n;
    const int en = (fc < E * 6) ? sNb[fc / 6][fc % 6] : -1;
    hg[k] = (en >= 0) ? nbr_geo_load<AFF>(mesh, en, fc % 6, x % NbrGeo<AFF>::n) : 0.0;
  }

  FaceData<P> fd;
  face_load<P, R, 0, AFF>(mesh, sa.Vin, lam, sNb, e0, fd);

  const int idx[3] = {nd0 % N, (nd0 / N) % N, nd0 / (N * N)};
  double acc[R][5];
  double wJ[R];

  // ---- volume, one row at a time: velocity gradient, flux, divergence ----
#pragma unroll
  for (int rr = 0; rr < R; ++rr)
  {
    const int le = rr * EPR + tid / NB;
    const bool vact = (tid < EPR * NB) && (e0 + le < mesh.nelem);
#pragma unroll
    for (int r = 0; r < 5; ++r)
      acc[rr][r] = 0.0;
    wJ[rr] = 1.0;
    double F[3][5];
    if (P == 3 || vact)
    {
      NodeGeo ng;
      const double w = pt.w[idx[0]] * pt.w[idx[1]] * pt.w[idx[2]];
      if constexpr (AFF)
        ng.inverse(sG[le] + 10, w * sG[le][9], ph.mu);
      else
      {
        double J[3][3];
        jac_at<Q, true>(qt, sX[le], -1, 0, idx[0], idx[1], idx[2], J);
        ng.curved(J, w, ph.mu);
      }
      wJ[rr] = ng.wJ;
      double Vq[5], gr[3][4];
#pragma unroll
      for (int r = 0; r < 5; ++r)
        Vq[r] = sV[le][r][nd0];
#pragma unroll
      for (int r = 0; r < 4; ++r)
      {
        double g0 = 0.0, g1 = 0.0, g2 = 0.0;
#pragma unroll
        for (int m = 0; m < N; ++m)
        {
          g1 += pt.Dg[idx[1]][m] * sV[le][r][nid<N>(idx[0], m, idx[2])];
          if constexpr (P != 3)
          {
            g0 += pt.Dg[idx[0]][m] * sV[le][r][nid<N>(m, idx[1], idx[2])];
            g2 += pt.Dg[idx[2]][m] * sV[le][r][nid<N>(idx[0], idx[1], m)];
          }
        }
        if constexpr (P == 3)  // the node index is the lane: x is lo, z is hi
        {
          g0 = mf_lo(mf.one, mf.dg, Vq[r], 0.0);
          g2 = mf_hi(mf.dg, Vq[r], 0.0);
        }
        gr[0][r] = g0;
        gr[1][r] = g1;
        gr[2][r] = g2;
      }
      volume_flux_fp64(Vq, gr, ng.B, ng.kv, ng.A, ph.gamma, F);
    }
#pragma unroll
    for (int c = 0; c < 3; ++c)
    {
      if (P == 3 && c != 1)
      {
#pragma unroll
        for (int r = 0; r < 5; ++r)
          acc[rr][r] = (c == 0) ? mf_lo(mf.one, mf.dgt, F[c][r], acc[rr][r])
                                : mf_hi(mf.dgt, F[c][r], acc[rr][r]);
        continue;
      }
      if (P == 3 || vact)
      {
#pragma unroll
        for (int r = 0; r < 5; ++r)
          sR[r * 64 + tid] = F[c][r];
      }
      phase_fence();
      if (P == 3 || vact)
      {
        const int base = (tid / NB) * NB;
#pragma unroll
        for (int r = 0; r < 5; ++r)
        {
          double s = 0.0;
#pragma unroll
          for (int m = 0; m < N; ++m)
          {
            int id2[3] = {idx[0], idx[1], idx[2]};
            id2[c] = m;
            s += pt.Dg[m][idx[c]] * sR[r * 64 + base + nid<N>(id2[0], id2[1], id2[2])];
          }
          acc[rr][r] += s;
        }
      }
      phase_fence();
    }
  }

#pragma unroll
  for (int k = 0; k < NH; ++k)
    if (tid + 64 * k < E * 6 * NbrGeo<AFF>::n)
      (&sH[0][0])[tid + 64 * k] = hg[k];
  if constexpr (P == 3)  // at p = 1 the first subpass has a fence before it reads sH
    phase_fence();

  // ---- faces, one reference direction at a time ----
  bool ok = true;
  double pbase[R][5], pacc[R][5];  // base state and accumulator, loaded ahead
  auto subpass = [&](auto sc) __attribute__((always_inline)) {
    constexpr int D = decltype(sc)::value;
    state_face_subpass<P, Q, R, D, AFF>(
        mesh, ph, pt, qt, Tin, sV, sX, sG, sH, sNb, sBt, sR, mf, e0, acc, fd,
        [&]() __attribute__((always_inline)) {
          if constexpr (D < 2)
            face_load<P, R, D + 1, AFF>(mesh, sa.Vin, lam, sNb, e0, fd);
          else
          {
#pragma unroll
            for (int rr = 0; rr < R; ++rr)
            {
              const int le = rr * EPR + tid / NB;
              if (tid < EPR * NB && e0 + le < mesh.nelem)
              {
                const size_t base = (size_t)(e0 + le) * 5 * NB + nd0;
                if (sa.Vout && sa.ca != 0.0)  // Vbase may be null without Vout
#pragma unroll
                  for (int r = 0; r < 5; ++r)
                    pbase[rr][r] = __builtin_nontemporal_load(sa.Vbase + base + (size_t)r * NB);
                if (sa.accmode >= 2)
#pragma unroll
                  for (int r = 0; r < 5; ++r)
                    pacc[rr][r] = __builtin_nontemporal_load(sa.acc + base + (size_t)r * NB);
              }
            }
          }
        });
  };
  subpass(Const<0>{});
  subpass(Const<1>{});
  subpass(Const<2>{});

  // ---- form f_g and the RK epilogue, one row at a time; with NORM, each
  // row's R = -B3^T W f_g in sR (three passes) and the lane's running sum of
  // R^2 in sR[5 * 64 + lane] ----
#pragma unroll
  for (int rr = 0; rr < R; ++rr)
  {
    const int le = rr * EPR + tid / NB;
    const int e  = e0 + le;
    const bool act = tid < EPR * NB && e < mesh.nelem;
    if (act)
    {
      const double iwJ = rcp(wJ[rr]);
      const size_t base = (size_t)e * 5 * NB + nd0;
#pragma unroll
      for (int r = 0; r < 5; ++r)
      {
        const size_t ix = base + (size_t)r * NB;
        const double fv = ph.source[r] - acc[rr][r] * iwJ;
        if (NORM)
          sR[r * 64 + tid] = -wJ[rr] * fv;
        if (sa.fout)
          sa.fout[ix] = fv;
        double ft = fv;
        if (sa.accmode == 1)
          __builtin_nontemporal_store(fv, sa.acc + ix);
        else if (sa.accmode == 2)
          __builtin_nontemporal_store(pacc[rr][r] + 2.0 * fv, sa.acc + ix);
        else if (sa.accmode == 3)
          ft = (pacc[rr][r] + fv) * (1.0 / 6.0);
        if (sa.Vout)
        {
          double o = sa.cf * ft;
          if (sa.ca != 0.0)
            o += sa.ca * pbase[rr][r];
          if (sa.cb != 0.0)
            o += sa.cb * sV[le][r][nd0];
          __builtin_nontemporal_store(o, sa.Vout + ix);
          sV[le][r][nd0] = o;  // only this lane reads this node from here on
        }
      }
    }
    if constexpr (NORM)
    {
      // the modal residual whose RMS the step reports, one direction per
      // pass; only this lane reads and writes its running-sum slot
#pragma unroll
      for (int c = 0; c < 3; ++c)
        tile_modal_pass<N, NB>(sR, pt.B, c, idx, act);
      double s2 = 0.0;
      if (act)
#pragma unroll
        for (int r = 0; r < 5; ++r)
          s2 += sR[r * 64 + tid] * sR[r * 64 + tid];
      sR[5 * 64 + tid] = (rr == 0) ? s2 : sR[5 * 64 + tid] + s2;
      __syncthreads();
    }
  }
  if constexpr (NORM)
  {
    // the tile's sum of R^2: a butterfly over the wavefront (fixed order:
    // deterministic)
    double sq = sR[5 * 64 + tid];
#pragma unroll
    for (int w = 32; w > 0; w >>= 1)
      sq += __shfl_xor(sq, w, 64);
    if (tid == 0)
      sa.normp[block] = sq;
  }

  // ---- of the new state: the states of characteristic boundary faces for the
  // next stage, or (sa.records) the trace records of every face ----
  if (sa.Tout && (sa.records || wall))
  {
    __syncthreads();
    state_traces<P, Q, R, AFF>(mesh, ph, pt, qt, sV, sX, sG, sNb, sBt, sR, e0, sa.records,
                                  sa.Tout, ok);
  }
  if (!ok)
    atomicOr(status, 1);
}

