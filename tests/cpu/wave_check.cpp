// The FP64 state-reading stage bodies, lane by lane on the CPU: the same results
// whether a lane's LDS writes reach the others at once, in either order of the
// lanes, or at the next barrier only (tests/cpu/wave/hip/hip_runtime.h), and no
// two lanes write different values to one word between barriers.  Affine and
// curved elements, partly filled tiles, walls, inflow and outflow, with the fused
// norm and with every face's trace records.
#include <hip/hip_runtime.h>

#include <random>
#include <string>

#include "dgx_stage.hpp"

using namespace dgx;

namespace dgx
{
namespace host
{
void build_tables(PTab* pt, QTab* qt);
}
}  // namespace dgx

static std::mt19937_64 rng(11);
static double U1() { return std::uniform_real_distribution<double>(-1.0, 1.0)(rng); }

template <int P, bool AFF, bool NORM, bool LINE>
static int check()
{
  constexpr int N = P + 1, NB = N * N * N, NF = N * N, R = tile_rows(P);
  const int n[3] = {3, 1, 3}, ne = 9;
  std::vector<double> X(ne * 24), V(ne * 5 * NB), base, lam(ne * 6 * NF), lamf(ne * 6);
  std::vector<double> arec(ne * GREC);
  for (int e = 0; e < ne; ++e)
    for (int c = 0; c < 8; ++c)
      for (int d = 0; d < 3; ++d)
      {
        const int i[3] = {e % 3, 0, e / 3};
        X[e * 24 + c * 3 + d] = 0.5 * (i[d] + ((c >> d) & 1)) * (1.0 + 0.2 * d) +
                                (AFF ? 0.0 : 0.03 * U1());
      }
  for (int e = 0; e < ne; ++e)
    affine_record(X.data(), e, ne, &arec[e * GREC]);
  for (int e = 0; e < ne; ++e)
    for (int k = 0; k < NB; ++k)
    {
      double* u = &V[(e * 5) * NB + k];
      u[0] = 1.0 + 0.05 * U1();
      for (int r = 1; r < 4; ++r)
        u[r * NB] = 0.2 * (r == 1) + 0.05 * U1();
      u[4 * NB] = 1.8 + 0.05 * U1();
    }
  base = V;
  for (double& x : lam)
    x = 10.0 + U1();
  for (double& x : lamf)
    x = 10.0 + U1();
  MeshArgs m{};
  m.nodes = X.data();
  m.nelem = ne;
  m.nx    = n[0];
  m.ny    = n[1];
  m.nz    = n[2];
  const int bounds[6] = {-5, -6, -7, -4, -2, -2};
  std::memcpy(m.bounds, bounds, sizeof(bounds));
  m.affine = AFF;
  m.lamf   = lamf.data();
  m.arec   = arec.data();
  Phys ph{};
  ph.gamma = 1.4;
  ph.mu    = 1e-2;
  ph.eta   = 6.0;
  ph.Rgas  = 287.0;
  ph.P     = 0.714;
  ph.Pt    = 0.735;
  ph.Tt    = 0.00251;
  ph.Ufr[0] = 1.0;
  ph.Ufr[1] = 0.2;
  ph.Ufr[4] = 1.8;
  const size_t nt = (size_t)ne * 6 * 8 * NF + boundary_faces(3, 1, 3) * 5 * NF;
  std::vector<double> Tin(nt);
  for (size_t i = 0; i < nt; ++i)
  {
    const int r = (int)((i - (size_t)ne * 6 * 8 * NF) / NF % 5);
    Tin[i] = r == 0 ? 1.0 : (r == 4 ? 1.8 : 0.1);
  }
  constexpr int E = LINE ? LineDims<LINE ? P : 3>::E : TileDims<P, R>::E;
  const int blocks = (ne + E - 1) / E;
  size_t lds;
  if constexpr (LINE)
    lds = LineLds<P, AFF>::bytes;
  else
    lds = StateLds<P, 1, R, AFF>::bytes;
  std::vector<double> out[3];
  static Wave w;
  w.conflicts = 0;
  for (int mode = 0; mode < 3; ++mode)
  {
    std::vector<double> f(V.size(), -1.0), Vo(V.size(), -1.0), acc(V.size(), 0.5), T(nt, -1.0);
    std::vector<double> np(blocks, -1.0);
    int status = 0;
    for (int b = 0; b < blocks; ++b)
    {
      StageArgs sa{};
      sa.Vin     = V.data();
      sa.Tin     = Tin.data();
      sa.Vbase   = base.data();
      sa.acc     = acc.data();
      sa.Vout    = Vo.data();
      sa.Tout    = T.data();
      sa.fout    = f.data();
      sa.ca      = 0.75;
      sa.cb      = 0.25;
      sa.cf      = 1e-3;
      sa.accmode = 2;
      sa.normp   = np.data();
      sa.records = 1;
      w.run((Wave::Mode)mode, lds, [&](unsigned char* l) {
        if constexpr (LINE)
          line_body<P, AFF, NORM>(m, ph, sa, lam.data(), &status, b, l);
        else
          state_body<P, 1, R, AFF, NORM>(m, ph, sa, lam.data(), &status, b, l);
      });
    }
    for (auto* v : {&f, &Vo, &acc, &T, &np})
      out[mode].insert(out[mode].end(), v->begin(), v->end());
    out[mode].push_back(status);
  }
  size_t bad = 0, nan = 0;
  for (size_t i = 0; i < out[0].size(); ++i)
  {
    nan += !(out[0][i] == out[0][i]);
    bad += std::memcmp(&out[0][i], &out[1][i], 8) != 0 || std::memcmp(&out[0][i], &out[2][i], 8) != 0;
  }
  std::printf("p %d %s %s%s: %zu of %zu values differ, %zu NaN, %d conflicting writes\n", P,
              LINE ? "line" : "state", AFF ? "affine" : "curved", NORM ? " norm" : "", bad,
              out[0].size(), nan, w.conflicts);
  return bad || nan || w.conflicts;
}

template <int P, bool LINE>
static int order()
{
  return check<P, true, false, LINE>() + check<P, true, true, LINE>() +
         check<P, false, false, LINE>() + check<P, false, true, LINE>();
}

int main()
{
  static PTab pt[3];
  static QTab qt[9];
  host::build_tables(pt, qt);
  std::memcpy(c_ptab, pt, sizeof(pt));
  std::memcpy(c_qtab, qt, sizeof(qt));
  return order<1, false>() + order<3, false>() + order<2, true>() + order<3, true>() ? 1 : 0;
}
