// dgx_line_state.hpp -- the FP64 tiled stage of p = 2 and 3 with one line of
// nodes per lane: the method and the per-point arithmetic of
// dgx_tile_state.hpp, from the states and without trace records, but a tile is
// 64 / (p+1)^2 elements (7 at p = 2, 4 at p = 3) and lane (element, a, b) has
// the element's nodes (a, b, 0..p), whose accumulators and z contractions stay
// in its registers, and point (a, b) of each of its faces, one face of every
// element per subpass.
//   * Every lane works: 63 of 64 at p = 2, where whole elements per row of 64
//     nodes leave 54 (volume) and 54 (faces).
//   * A lane's indices (a, b) are the same in every phase, so its table rows
//     are loaded once; the side of a face is uniform, so the rows at the
//     element's ends and the z derivative come through the scalar cache.
//   * LDS is read for the other points of a line only, a third less per node;
//     faces normal to z need no gather.
// What bounds it is FP64 issue at p = 3 (3900 FP64 and 324 matrix instructions
// per wavefront of 256 nodes at 2 wavefronts per SIMD) together with the traffic
// of the state arrays (64^3 cube: 4.09 GB per launch, 78 % of the rate of a large
// copy), and at p = 2 issue and LDS in equal parts.  Per RK4 stage against the
// 2-element tile of dgx_tile_state.hpp, 64^3 p = 3 cube: 1083 against 1266 us (1083
// to 1140 from card to card), 48x24x24 p = 3 curved channel (TVD-RK3) 132 against
// 162 (both with the longer geometry 149 against 162); against the one-row kernel, 32^3 p = 2 cube 107
// against 136 us, 30x24x28 p = 2 curved channel 81 against 106.  One wavefront
// takes 20 us against 11 (p = 3) and 12 us (p = 2) of the others, so small meshes
// keep those (line_tiled, apply_defaults).  At
// p = 1 the same layout measured 4 % slower (16 elements of 6 faces take 18 KB
// of LDS).
// Included by dgx_stage.hpp inside namespace dgx, after dgx_tile_state.hpp.
#pragma once

constexpr bool line_order(int p)
{
  return p == 2 || p == 3;
}

// Whether tile 1 in FP64 runs this kernel: always at p = 2; at p = 3 from three
// wavefronts per SIMD (1024 SIMDs, 4 elements each), where it was the quicker one
// before its epilogue's loads ran ahead.  With them, per RK4 stage, 2-element against
// 4-element tile: 5202 elements 35.8 against 38.0 us, 8000 47.5 / 45.2, 11132 62.4 /
// 60.9, 13824 74.4 / 72.9, 32768 163 / 143; curved (TVD-RK3) 5202 40.2 / 42.0, 8000
// 52.8 / 48.0, 11132 71.9 / 67.2, 27648 154 / 135: from 8000 on it is 2 to 9 %
// quicker below the line too.
constexpr bool line_tiled(int p, int nelem)
{
  return p == 2 || (p == 3 && nelem >= 12288);
}

template <int P>
struct LineDims
{
  static_assert(line_order(P), "orders of this kernel");
  static constexpr int N  = P + 1;
  static constexpr int NF = N * N;
  static constexpr int NB = N * N * N;
  static constexpr int E  = 64 / NF;            // elements per tile
  static constexpr int JS = (P == 3) ? 16 : N;  // lane stride of the second face index
  // states: [variable][z][lane]; stride of a z row: at p = 2 the lines along x
  // behind the points of a face normal to x lie in all three rows
  static constexpr int RS = (P == 2) ? 65 : 64;
  static constexpr int SV = 5 * N * RS;
  // exchange region: a face subpass (9 per lane), the volume fluxes along x and
  // y (10, not at p = 3)
  static constexpr int SR = (P == 3 ? 9 : 10) * 64;
  // lane of point (a, b) of element l: at p = 3 the element is the middle
  // 2-bit field, the block of the 4x4x4 matrix instruction
  static __device__ __forceinline__ int lane(int l, int a, int b)
  {
    return (P == 3) ? a + 4 * l + 16 * b : l * NF + b * N + a;
  }
};

// This lane's element and point (a, b): nodes (a, b, 0..p) of the element and
// face point (a, b) of each of its faces.  Lanes beyond the E elements repeat
// the last element's first point, elements past the end of the mesh the last one;
// neither stores anything.
template <int P>
struct LineLane
{
  using LD = LineDims<P>;
  int tid, a, b, l, e;
  bool act;
  __device__ __forceinline__ LineLane(const MeshArgs& mesh, int e0)
  {
    tid = opaque_tid();
    if constexpr (P == 3)
    {
      a = tid & 3;
      l = (tid >> 2) & 3;
      b = tid >> 4;
      act = e0 + l < mesh.nelem;
    }
    else
    {
      const bool in = tid < LD::E * LD::NF;
      const int t = in ? tid : (LD::E - 1) * LD::NF;
      l = t / LD::NF;
      a = t % LD::N;
      b = (t / LD::N) % LD::N;
      act = in && e0 + l < mesh.nelem;
    }
    e = min(e0 + l, mesh.nelem - 1);
  }
};

// What the lane's point of face S (local face number; subpass S) needs of the
// element across it (see FaceData), loaded one subpass ahead.
template <int P, int S, bool AFF>
__device__ __forceinline__ void line_face_load(const MeshArgs& mesh, const double* __restrict__ Vin,
                                        const double* __restrict__ lam, const int (*sNb)[6],
                                        int e0, FaceData<P>& fd)
{
  using LD = LineDims<P>;
  constexpr int D = S >> 1, f = S;
  const LineLane<P> ln(mesh, e0);
  const int nb = sNb[ln.l][f], en = nb >= 0 ? nb : ln.e;
  line_load<P, D>(Vin + (size_t)en * 5 * LD::NB, ln.a, ln.b, fd.x);
  const size_t iL = (size_t)ln.e * 6 + f, iR = (size_t)en * 6 + (f ^ 1);
  const int fpt = ln.a + LD::N * ln.b;
  fd.lamL = AFF ? mesh.lamf[iL] : lam[iL * LD::NF + fpt];
  fd.lamR = AFF ? mesh.lamf[iR] : lam[iR * LD::NF + fpt];
}

// The neighbour geometry (NbrGeo) of the tile's faces normal to one direction,
// in registers between its loads and its copy into LDS.
template <int P, bool AFF>
struct NbrLoad
{
  static constexpr int M = LineDims<P>::E * 2 * NbrGeo<AFF>::n, NH = (M + 63) / 64;
  double h[NH];
  __device__ __forceinline__ void load(const MeshArgs& mesh, const int (*sNb)[6], int d)
  {
    const int tid = opaque_tid();
#pragma unroll
    for (int k = 0; k < NH; ++k)
    {
      const int x = min(tid + 64 * k, M - 1), fc = x / NbrGeo<AFF>::n, f = 2 * d + (fc & 1);
      const int en = sNb[fc >> 1][f];
      h[k] = (en >= 0) ? nbr_geo_load<AFF>(mesh, en, f, x % NbrGeo<AFF>::n) : 0.0;
    }
  }
  __device__ __forceinline__ void store(double* sH) const
  {
    const int tid = opaque_tid();
#pragma unroll
    for (int k = 0; k < NH; ++k)
      if (tid + 64 * k < M)
        sH[tid + 64 * k] = h[k];
  }
};

// The 1D tables of a lane's two indices a and b and where the other points of
// its lines along them are exchanged: entry m belongs to index (a + m) mod N, so
// that entry 0 meets the lane's own value, which stays in a register.
template <int P>
struct LineTabs
{
  static constexpr int N = P + 1;
  double da[N], db[N], ta[N], tb[N];  // Dg[a][.], Dg[b][.], Dg[.][a], Dg[.][b]
  int na[N], nb[N];                   // lanes of the points along a and b
  __device__ __forceinline__ void load(const PTab& pt, int l, int a, int b)
  {
#pragma unroll
    for (int m = 0; m < N; ++m)
    {
      const int am = a + m < N ? a + m : a + m - N, bm = b + m < N ? b + m : b + m - N;
      da[m] = pt.Dg[a][am];
      db[m] = pt.Dg[b][bm];
      ta[m] = pt.Dg[am][a];
      tb[m] = pt.Dg[bm][b];
      na[m] = LineDims<P>::lane(l, am, b);
      nb[m] = LineDims<P>::lane(l, a, bm);
    }
  }
};

// c + sum over a line: t[0] x of the lane's own value x, t[m] s[n[m]] of the others
template <int N>
__device__ __forceinline__ double row_sum(const double (&t)[N], const int (&n)[N], const double* s,
                                          double x, double c)
{
  c += t[0] * x;
#pragma unroll
  for (int m = 1; m < N; ++m)
    c += t[m] * s[n[m]];
  return c;
}

// Forms the accumulators here: their sums are used in the epilogue's branch
// only, and would be sunk there with all their operands kept (in scratch)
// until then.
template <int N>
__device__ __forceinline__ void form_now(double (&acc)[N][5])
{
#pragma unroll
  for (int k = 0; k < N; ++k)
#pragma unroll
    for (int r = 0; r < 5; ++r)
      asm volatile("" : "+v"(acc[k][r]));
}

// J = d x / d xi along the lane's line of nodes of a trilinear element: the z
// column is constant on it and the others are linear in z.
struct LineGeo
{
  double x0[3], dx[3], y0[3], dy[3], z[3];
  __device__ __forceinline__ LineGeo(const double* X, double ga, double gb)
  {
    const double fa = 1.0 - ga, fb = 1.0 - gb;
#pragma unroll
    for (int i = 0; i < 3; ++i)
    {
      double n[8];
#pragma unroll
      for (int c = 0; c < 8; ++c)
        n[c] = X[3 * c + i];
      x0[i] = fb * (n[1] - n[0]) + gb * (n[3] - n[2]);
      y0[i] = fa * (n[2] - n[0]) + ga * (n[3] - n[1]);
      dx[i] = fb * (n[5] - n[4]) + gb * (n[7] - n[6]) - x0[i];
      dy[i] = fa * (n[6] - n[4]) + ga * (n[7] - n[5]) - y0[i];
      z[i]  = fb * (fa * (n[4] - n[0]) + ga * (n[5] - n[1])) +
             gb * (fa * (n[6] - n[2]) + ga * (n[7] - n[3]));
    }
  }
  __device__ __forceinline__ void at(double g, double J[3][3]) const
  {
#pragma unroll
    for (int i = 0; i < 3; ++i)
    {
      J[i][0] = x0[i] + g * dx[i];
      J[i][1] = y0[i] + g * dy[i];
      J[i][2] = z[i];
    }
  }
};

struct AffineLine
{
  __device__ __forceinline__ AffineLine(const double*, double, double) {}
};

// Subpass S: local face S of every element of the tile: both sides' traces and
// gradient tractions from the states (own from LDS, neighbour in fd), the face
// point physics, the tangential (T) phase and the gather into the nodes'
// accumulators.  next() starts the loads that follow.  ct: the tables at
// uniform indices (scalar loads).
template <int P, int S, bool AFF, typename Next>
__device__ __forceinline__ void line_face_subpass(
    const MeshArgs& mesh, const Phys& ph, const PTab& pt, const PTab& ct, const QTab& qt,
    const double* __restrict__ Tin, const double* sV, const double (*sX)[24],
    const double (*sG)[GREC], const double (*sH)[NbrGeo<AFF>::n], const int (*sNb)[6],
    const int (*sBt)[6], double* sR, const MfTabs& mf, const LineTabs<P>& lt, double wab, int e0,
    double (&acc)[P + 1][5], FaceData<P>& fd, Next next)
{
  using LD = LineDims<P>;
  constexpr int N = LD::N, JS = LD::JS, D = S >> 1, hi = S & 1, f = S;
  constexpr int T1 = Tang<D>::T1, T2 = Tang<D>::T2;
  const LineLane<P> ln(mesh, e0);
  const int tid = ln.tid, a = ln.a, b = ln.b, l = ln.l;
  const int bb = LD::lane(l, a, 0);

  double UL[5], dL[4], Ub[5], dR[4];
  const int en = sNb[l][f];
  {
    // nodes (m, a, b), (a, m, b) or (a, b, m)
    double xL[5][N];
    const int n0 = (D == 0) ? b * LD::RS + LD::lane(l, 0, a) : ((D == 1) ? b * LD::RS + bb : tid);
    constexpr int ns = (D == 0) ? 1 : ((D == 1) ? JS : LD::RS);
#pragma unroll
    for (int r = 0; r < 5; ++r)
#pragma unroll
      for (int m = 0; m < N; ++m)
        xL[r][m] = sV[r * N * LD::RS + n0 + m * ns];
    line_traces<N>(xL, ct.L[hi], ct.Ld[hi], UL, dL);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
    asm volatile("" : "+v"(UL[r]), "+v"(dL[r]), "+v"(fd.x[r][0]));
  line_traces<N>(fd.x, ct.L[1 - hi], ct.Ld[1 - hi], Ub, dR);
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
      return (c == T1) ? row_sum(lt.da, lt.na, s + r * 64, U[r], 0.0)
                       : row_sum(lt.db, lt.nb, s + r * 64, U[r], 0.0);
    };
    face_states<P, 1, D, AFF>(
        mesh, ph, qt, Tin, sX[l], sG[l], sH[2 * l + hi], en, sBt[l][f], hi, a, b, wab, UL, dL, Ub,
        dR, lamL, lamR,
        [&](int c, int r) __attribute__((always_inline)) { return tan(UL, sR, c, r); },
        [&](int c, int r) __attribute__((always_inline)) { return tan(Ub, sR + 4 * 64, c, r); },
        next, G, hc);
  }
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
      G[r] -= row_sum(lt.tb, lt.nb, sR + (3 + r) * 64, hc[T2][r - 1],
                      row_sum(lt.ta, lt.na, sR + (r - 1) * 64, hc[T1][r - 1], 0.0));
  }
  if constexpr (D == 2)
  {
    // the lane's face point is the end of its own line of nodes
#pragma unroll
    for (int k = 0; k < N; ++k)
    {
      acc[k][0] += ct.L[hi][k] * G[0];
#pragma unroll
      for (int r = 1; r < 5; ++r)
        acc[k][r] += ct.L[hi][k] * G[r] - ct.Ld[hi][k] * hn[r - 1];
    }
    form_now<N>(acc);
    phase_fence();
    return;
  }
  phase_fence();
#pragma unroll
  for (int r = 0; r < 5; ++r)
    sR[r * 64 + tid] = G[r];
#pragma unroll
  for (int r = 0; r < 4; ++r)
    sR[(5 + r) * 64 + tid] = hn[r];
  phase_fence();
  {
    // node (i, j, k) of the lane's line lies behind point (j, k) of the faces
    // normal to x and (i, k) of those normal to y
    const int m = (D == 0) ? a : b, p0 = LD::lane(l, (D == 0) ? b : a, 0);
    const double Lh = pt.L[hi][m], Ldh = pt.Ld[hi][m];
#pragma unroll
    for (int k = 0; k < N; ++k)
    {
      const double* s = sR + p0 + k * JS;
      acc[k][0] += Lh * s[0];
#pragma unroll
      for (int r = 1; r < 5; ++r)
        acc[k][r] += Lh * s[r * 64] - Ldh * s[(4 + r) * 64];
    }
  }
  form_now<N>(acc);
  phase_fence();
}

// Of the tile's new states in sV: the boundary states of its characteristic
// boundary faces, or with records != 0 every face's trace records (state_traces).
template <int P, bool AFF>
__device__ __forceinline__ void line_state_traces(const MeshArgs& mesh, const Phys& ph, const PTab& pt,
                                          const PTab& ct, const QTab& qt, const double* sV,
                                          const double (*sX)[24], const double (*sG)[GREC],
                                          const int (*sNb)[6], const int (*sBt)[6], double* sR,
                                          int e0, int records, double* __restrict__ Tout, bool& ok)
{
  using LD = LineDims<P>;
  constexpr int N = LD::N, NF = LD::NF, JS = LD::JS;
  double* Tb = Tout + (size_t)mesh.nelem * 6 * 8 * NF;
  const LineLane<P> ln(mesh, e0);
  const int tid = ln.tid, a = ln.a, b = ln.b, l = ln.l, fpt = a + N * b;
  const int ba = LD::lane(l, 0, b), bb = LD::lane(l, a, 0);
#pragma unroll 1
  for (int f = 0; f < 6; ++f)
  {
    const int nd = f >> 1, hi = f & 1;
    const int nb = ln.act && (records || characteristic_bc(sBt[l][f])) ? sNb[l][f] : 0;
    if (!records && !__any(nb < 0))
      continue;
    const int n0 = (nd == 0) ? b * LD::RS + LD::lane(l, 0, a) : ((nd == 1) ? b * LD::RS + bb : tid);
    const int ns = (nd == 0) ? 1 : ((nd == 1) ? JS : LD::RS);
    double U[5], dn[4];
#pragma unroll
    for (int r = 0; r < 5; ++r)
    {
      double v = 0.0, dv = 0.0;
#pragma unroll
      for (int m = 0; m < N; ++m)
      {
        const double x = sV[r * N * LD::RS + n0 + m * ns];
        v += ct.L[hi][m] * x;
        if (r < 4)
          dv += ct.Ld[hi][m] * x;
      }
      U[r] = v;
      if (r < 4)
      {
        dn[r]            = dv;
        sR[r * 64 + tid] = v;
      }
    }
    __syncthreads();
    if (ln.act && (records || nb < 0))
    {
      const int gi0 = (nd == 0) ? 0 : a;
      const int gi1 = (nd == 1) ? 0 : ((nd == 0) ? a : b);
      const int gi2 = (nd == 2) ? 0 : b;
      double Ji[3][3], nv[3];
      face_geometry<1, AFF, true>(qt, sX[l], sG[l], nd, hi, gi0, gi1, gi2, Ji, nv);
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
            d1 += pt.Dg[a][m] * sR[r * 64 + ba + m];
            d2 += pt.Dg[b][m] * sR[r * 64 + bb + m * JS];
          }
          gr[0][r] = pick3(nd, dn[r], d1, d1);
          gr[1][r] = pick3(nd, d1, dn[r], d2);
          gr[2][r] = pick3(nd, d2, d2, dn[r]);
        }
        double vg[3];
        grad_traction(gr, U, Ji, nv, ph.mu, vg);
        double* T = Tout + ((size_t)ln.e * 6 + f) * 8 * NF + fpt;
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
template <int P, bool AFF>
struct LineLds
{
  using LD = LineDims<P>;
  static constexpr int E = LD::E;
  static constexpr size_t oV  = 0;
  static constexpr size_t oX  = oV + sizeof(double) * LD::SV;  // nodes, or affine records
  static constexpr size_t oH  = oX + sizeof(double) * E * (AFF ? GREC : 24);
  static constexpr size_t oR  = oH + sizeof(double) * E * 2 * NbrGeo<AFF>::n;
  static constexpr size_t oPT = oR + sizeof(double) * LD::SR;
  static constexpr size_t oQT = oPT + sizeof(PTab);
  static constexpr size_t oNb = oQT + sizeof(QTab);
  static constexpr size_t oBt = oNb + sizeof(int) * E * 6;
  static constexpr size_t bytes = oBt + sizeof(int) * E * 6;
};

// The stage of tile `block` (arguments as state_body).
template <int P, bool AFF, bool NORM>
__device__ __forceinline__ void line_body(const MeshArgs& mesh, const Phys& ph, const StageArgs& sa,
                                          const double* __restrict__ lam, int* status, int block,
                                          unsigned char* lds)
{
  using LD = LineDims<P>;
  using TL = LineLds<P, AFF>;
  constexpr int N = LD::N, NB = LD::NB, NF = LD::NF, E = LD::E, JS = LD::JS;
  // z rows of the base state and accumulator loaded during the last subpass: all
  // at p = 2; at p = 3 the registers of three are there (four spill).  Against
  // none at p = 3: 64^3 cube 1104 -> 1083 us per RK4 stage, 32^3 144 -> 137,
  // 48x24x24 channel 132.4 -> 131.6
  constexpr int KP = P == 3 ? 3 : N;

  double* sV = reinterpret_cast<double*>(lds + TL::oV);
  auto sX  = reinterpret_cast<double(*)[24]>(lds + TL::oX);    // curved meshes
  auto sG  = reinterpret_cast<double(*)[GREC]>(lds + TL::oX);  // affine meshes
  auto sH  = reinterpret_cast<double(*)[NbrGeo<AFF>::n]>(lds + TL::oH);
  double* sR = reinterpret_cast<double*>(lds + TL::oR);
  PTab& sPT = *reinterpret_cast<PTab*>(lds + TL::oPT);
  QTab& sQT = *reinterpret_cast<QTab*>(lds + TL::oQT);
  auto sNb = reinterpret_cast<int(*)[6]>(lds + TL::oNb);
  auto sBt = reinterpret_cast<int(*)[6]>(lds + TL::oBt);
  stage_tables<P, 1>(&sPT, &sQT);
  const PTab& pt = sPT;
  const PTab& ct = c_ptab[P - 1];
  const QTab& qt = sQT;

  const int e0 = block * E;
  const double* __restrict__ Tin = sa.Tin;
  const LineLane<P> ln(mesh, e0);
  const int tid = ln.tid, a = ln.a, b = ln.b, l = ln.l;
  const size_t gbase = (size_t)ln.e * 5 * NB + a + N * b;  // node (a, b, 0)
  tile_face_table<E>(mesh, e0, sNb, sBt);

  double v[N][5];
#pragma unroll
  for (int r = 0; r < 5; ++r)
#pragma unroll
    for (int k = 0; k < N; ++k)
      v[k][r] = sa.Vin[gbase + r * NB + k * NF];
  {
    constexpr int NX = AFF ? GREC : 24;
    const double* src = (AFF ? mesh.arec : mesh.nodes) + (size_t)e0 * NX;
    double* dst       = reinterpret_cast<double*>(lds + TL::oX);
    // elements past the end: the last element's, as their states
    const int left = min(mesh.nelem - e0, E) * NX;
    for (int x = tid; x < E * NX; x += 64)
      dst[x] = src[x < left ? x : left - NX + x % NX];
  }
#pragma unroll
  for (int r = 0; r < 5; ++r)
#pragma unroll
    for (int k = 0; k < N; ++k)
      sV[(r * N + k) * LD::RS + tid] = v[k][r];
  __syncthreads();
  bool wall = false;
#pragma unroll
  for (int x0 = 0; x0 < E * 6; x0 += 64)
  {
    const int x = min(x0 + tid, E * 6 - 1);
    wall = wall || characteristic_bc(sBt[x / 6][x % 6]);
  }
  wall = __any(wall);
  const MfTabs mf = (P == 3) ? mf_tabs(pt) : MfTabs{};
  LineTabs<P> lt;
  if constexpr (P != 3)
    lt.load(pt, l, a, b);
  const double wab = pt.w[a] * pt.w[b];
  double acc[N][5];
  double wJ[N];
#pragma unroll
  for (int k = 0; k < N; ++k)
#pragma unroll
    for (int r = 0; r < 5; ++r)
      acc[k][r] = 0.0;
  std::conditional_t<AFF, AffineLine, LineGeo> geo(sX[l], qt.Bq[a][1], qt.Bq[b][1]);
  const QTab& cq = c_qtab[P - 1][0];
  // volume, one z row at a time: velocity gradient, flux, divergence
#pragma unroll
  for (int k = 0; k < N; ++k)
  {
    double F[3][5], gr[3][4];
    NodeGeo ng;
    if constexpr (AFF)
      ng.inverse(sG[l] + 10, wab * ct.w[k] * sG[l][9], ph.mu);
    else
    {
      double J[3][3];
      geo.at(cq.Bq[k][1], J);
      ng.curved(J, wab * ct.w[k], ph.mu);
    }
    wJ[k] = ng.wJ;
#pragma unroll
    for (int r = 0; r < 4; ++r)
    {
      if constexpr (P == 3)
      {
        gr[0][r] = mf_lo(mf.one, mf.dg, v[k][r], 0.0);
        gr[1][r] = mf_hi(mf.dg, v[k][r], 0.0);
      }
      else
      {
        gr[0][r] = row_sum(lt.da, lt.na, sV + (r * N + k) * LD::RS, v[k][r], 0.0);
        gr[1][r] = row_sum(lt.db, lt.nb, sV + (r * N + k) * LD::RS, v[k][r], 0.0);
      }
      double g2 = 0.0;
#pragma unroll
      for (int m = 0; m < N; ++m)
        g2 += ct.Dg[k][m] * v[m][r];
      gr[2][r] = g2;
    }
    volume_flux_fp64(v[k], gr, ng.B, ng.kv, ng.A, ph.gamma, F);
#pragma unroll
    for (int r = 0; r < 5; ++r)
    {
      if constexpr (P == 3)
        acc[k][r] = mf_hi(mf.dgt, F[1][r], mf_lo(mf.one, mf.dgt, F[0][r], acc[k][r]));
      else
      {
        sR[r * 64 + tid]       = F[0][r];
        sR[(5 + r) * 64 + tid] = F[1][r];
      }
#pragma unroll
      for (int m = 0; m < N; ++m)
        acc[m][r] += ct.Dg[k][m] * F[2][r];
    }
    if constexpr (P != 3)
    {
      phase_fence();
#pragma unroll
      for (int r = 0; r < 5; ++r)
        acc[k][r] = row_sum(lt.tb, lt.nb, sR + (5 + r) * 64, F[1][r],
                            row_sum(lt.ta, lt.na, sR + r * 64, F[0][r], acc[k][r]));
    }
    form_now<N>(acc);
    phase_fence();
  }

  NbrLoad<P, AFF> hg;
  hg.load(mesh, sNb, 0);
  FaceData<P> fd;
  line_face_load<P, 0, AFF>(mesh, sa.Vin, lam, sNb, e0, fd);

  hg.store(&sH[0][0]);
  phase_fence();

  bool ok = true;
  double pbase[N][5], pacc[N][5];
  auto subpass = [&](auto sc) __attribute__((always_inline)) {
    constexpr int S = decltype(sc)::value;
    line_face_subpass<P, S, AFF>(
        mesh, ph, pt, ct, qt, Tin, sV, sX, sG, sH, sNb, sBt, sR, mf, lt, wab, e0, acc, fd,
        [&]() __attribute__((always_inline)) {
          if constexpr (S + 1 < 6)
          {
            line_face_load<P, S + 1, AFF>(mesh, sa.Vin, lam, sNb, e0, fd);
            if constexpr (S & 1)
              hg.load(mesh, sNb, (S + 1) / 2);
          }
          else if (ln.act)
          {
#pragma unroll
            for (int k = 0; k < KP; ++k)
            {
              if (sa.Vout && sa.ca != 0.0)  // Vbase may be null without Vout
#pragma unroll
                for (int r = 0; r < 5; ++r)
                  pbase[k][r] = __builtin_nontemporal_load(sa.Vbase + gbase + r * NB + k * NF);
              if (sa.accmode >= 2)
#pragma unroll
                for (int r = 0; r < 5; ++r)
                  pacc[k][r] = __builtin_nontemporal_load(sa.acc + gbase + r * NB + k * NF);
            }
          }
        });
    if constexpr ((S & 1) && S < 5)
    {
      hg.store(&sH[0][0]);
      phase_fence();
    }
  };
  subpass(Const<0>{});
  subpass(Const<1>{});
  subpass(Const<2>{});
  subpass(Const<3>{});
  subpass(Const<4>{});
  subpass(Const<5>{});

  double q[NORM ? N : 1][5];
  if (KP < N && ln.act)
  {
#pragma unroll
    for (int k = KP; k < N; ++k)
    {
      if (sa.Vout && sa.ca != 0.0)  // Vbase may be null without Vout
#pragma unroll
        for (int r = 0; r < 5; ++r)
          pbase[k][r] = __builtin_nontemporal_load(sa.Vbase + gbase + r * NB + k * NF);
      if (sa.accmode >= 2)
#pragma unroll
        for (int r = 0; r < 5; ++r)
          pacc[k][r] = __builtin_nontemporal_load(sa.acc + gbase + r * NB + k * NF);
    }
  }
#pragma unroll
  for (int k = 0; k < N; ++k)
  {
    const double iwJ = rcp(wJ[k]);
#pragma unroll
    for (int r = 0; r < 5; ++r)
    {
      const size_t ix = gbase + r * NB + k * NF;
      const double fv = ph.source[r] - acc[k][r] * iwJ;
      if (NORM)
        q[NORM ? k : 0][r] = -wJ[k] * fv;
      if (ln.act)
      {
        if (sa.fout)
          sa.fout[ix] = fv;
        double ft = fv;
        if (sa.accmode == 1)
          __builtin_nontemporal_store(fv, sa.acc + ix);
        else if (sa.accmode == 2)
          __builtin_nontemporal_store(pacc[k][r] + 2.0 * fv, sa.acc + ix);
        else if (sa.accmode == 3)
          ft = (pacc[k][r] + fv) * (1.0 / 6.0);
        if (sa.Vout)
        {
          double o = sa.cf * ft;
          if (sa.ca != 0.0)
            o += sa.ca * pbase[k][r];
          if (sa.cb != 0.0)
            o += sa.cb * sV[(r * N + k) * LD::RS + tid];
          __builtin_nontemporal_store(o, sa.Vout + ix);
          sV[(r * N + k) * LD::RS + tid] = o;  // only this lane reads this node from here on
        }
      }
    }
  }
  if constexpr (NORM)
  {
    // R = -B3^T W f_g: along z within the lane, then along x and y
    const int ba = LD::lane(l, 0, b), bb = LD::lane(l, a, 0);
    double sq = 0.0;
#pragma unroll
    for (int k = 0; k < N; ++k)
    {
      phase_fence();
#pragma unroll
      for (int r = 0; r < 5; ++r)
      {
        double z = 0.0;
#pragma unroll
        for (int m = 0; m < N; ++m)
          z += ct.B[m][k] * q[m][r];
        sR[r * 64 + tid] = z;
      }
      phase_fence();
      double o[5];
#pragma unroll
      for (int r = 0; r < 5; ++r)
      {
        o[r] = 0.0;
#pragma unroll
        for (int m = 0; m < N; ++m)
          o[r] += pt.B[m][a] * sR[r * 64 + ba + m];
      }
      phase_fence();
#pragma unroll
      for (int r = 0; r < 5; ++r)
        sR[r * 64 + tid] = o[r];
      phase_fence();
#pragma unroll
      for (int r = 0; r < 5; ++r)
      {
        double y = 0.0;
#pragma unroll
        for (int m = 0; m < N; ++m)
          y += pt.B[m][b] * sR[r * 64 + bb + m * JS];
        sq += y * y;
      }
    }
    if (!ln.act)
      sq = 0.0;
#pragma unroll
    for (int w = 32; w > 0; w >>= 1)
      sq += __shfl_xor(sq, w, 64);
    if (tid == 0)
      sa.normp[block] = sq;
  }

  if (sa.Tout && (sa.records || wall))
  {
    __syncthreads();
    line_state_traces<P, AFF>(mesh, ph, pt, ct, qt, sV, sX, sG, sNb, sBt, sR, e0, sa.records, sa.Tout, ok);
  }
  if (!ok)
    atomicOr(status, 1);
}
