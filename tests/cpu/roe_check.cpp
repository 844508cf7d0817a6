// roe_flux_fp64 against roe_flux: the same flux on admissible states, and no
// finite flux where roe_flux gives none (a density, pressure or sound speed
// without a real root on one side or on both, zeros, infinities, NaN).  Prints
// the worst relative error and the number of states answered where roe_flux
// refuses.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <limits>
#include <random>

#include "dgx_device.hpp"

using namespace dgx;

static std::mt19937_64 rng(7);
static double U1() { return std::uniform_real_distribution<double>(-1.0, 1.0)(rng); }

int main()
{
  double worst = 0.0;
  int lost = 0, refused = 0;
  const double odd[] = {0.0, -0.0, std::numeric_limits<double>::infinity(),
                        -std::numeric_limits<double>::infinity(),
                        std::numeric_limits<double>::quiet_NaN()};
  for (int it = 0; it < 40000; ++it)
  {
    double U[2][5], n[3], len = 0.0;
    for (int k = 0; k < 3; ++k)
    {
      n[k] = U1();
      len += n[k] * n[k];
    }
    for (int k = 0; k < 3; ++k)
      n[k] /= std::sqrt(len);
    for (auto& W : U)
    {
      W[0] = 1.0 + 0.5 * U1();
      for (int k = 0; k < 3; ++k)
        W[1 + k] = W[0] * U1();
      W[4] = 2.5 * (1.0 + 0.5 * U1()) +
             0.5 * (W[1] * W[1] + W[2] * W[2] + W[3] * W[3]) / W[0];
    }
    const int kind = it % 8;  // 0..2 admissible
    if (kind == 3 || kind == 4)
      for (int s = 0; s < 2; ++s)  // both sides, or one, negated
        for (int r = 0; r < 5; ++r)
          U[s][r] *= (kind == 3 || s == (it / 8) % 2) ? -1.0 : 1.0;
    if (kind == 5)  // any signs
      for (auto& W : U)
        for (int r = 0; r < 5; ++r)
          W[r] *= U1() < 0.0 ? -1.0 : 1.0;
    if (kind == 6)  // no real sound speed
      for (auto& W : U)
        W[4] *= -1.0;
    if (kind == 7)
      U[(it / 8) % 2][(it / 16) % 5] = odd[(it / 80) % 5];
    double a[5], b[5], scale = 0.0;
    roe_flux(U[0], U[1], n, 1.4, a);
    roe_flux_fp64(U[0], U[1], n, 1.4, b);
    bool fa = true, fb = true;
    for (int r = 0; r < 5; ++r)
    {
      fa = fa && std::isfinite(a[r]);
      fb = fb && std::isfinite(b[r]);
      scale = std::fmax(scale, std::fabs(a[r]));
    }
    refused += !fa;
    lost += fb && !fa;
    lost += fa && !fb;
    if (kind < 3)
      for (int r = 0; r < 5; ++r)
        worst = std::fmax(worst, std::fabs(a[r] - b[r]) / scale);
  }
  std::printf("worst %.3e different %d of %d refused\n", worst, lost, refused);
  // a hundred operations, each side's rounding
  return worst < 200 * 1.1102230246251565e-16 && lost == 0 && refused > 10000 ? 0 : 1;
}
