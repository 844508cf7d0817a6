// dgx_api.cpp on a stand-in for the HIP runtime with little memory: a context
// that fits without what another one keeps to be faster is created, and the
// other goes on; what a captured launch reads stays.  The kernels are stubs that
// note the mesh they were given.
#include <cstdio>
#include <vector>

#include <hip/hip_runtime.h>

#include "../../include/dgx.h"
#include "dgx_pool.hpp"

using namespace dgx;

static MeshArgs g_mesh;  // of the last stage

namespace dgx
{
hipError_t rhs_dispatch(int, int, const MeshArgs& m, const Phys&, const StageArgs&, const double*,
                        int*, int, hipStream_t, int)
{
  g_mesh = m;
  return hipSuccess;
}
hipError_t affine_record_dispatch(const double*, int, double*, hipStream_t) { return hipSuccess; }
size_t affine_record_doubles(int n) { return (size_t)n * 31; }
hipError_t basis_dispatch(int, const double*, double*, int, int, hipStream_t, bool)
{
  return hipSuccess;
}
hipError_t boundary_dispatch(int, const MeshArgs&, const Phys&, const double*, double*, int*,
                             hipStream_t)
{
  return hipSuccess;
}
hipError_t copy_dispatch(const void*, void*, size_t, hipStream_t) { return hipSuccess; }
hipError_t geometry_dispatch(int, int, const MeshArgs&, double*, double*, hipStream_t)
{
  return hipSuccess;
}
hipError_t lift_coef_dispatch(int, int, const MeshArgs&, double*, hipStream_t) { return hipSuccess; }
hipError_t lift_face_dispatch(int, const double*, int, double*, hipStream_t) { return hipSuccess; }
hipError_t matched_dispatch(const MeshArgs&, int*, hipStream_t) { return hipSuccess; }
hipError_t mean_dispatch(const double*, double*, size_t, double, double, hipStream_t)
{
  return hipSuccess;
}
int norm_blocks(int, int, int) { return 1; }
hipError_t norm_dispatch(const double*, int, double, double*, hipStream_t) { return hipSuccess; }
hipError_t norm_partials_dispatch(int, int, const MeshArgs&, const double*, double*, hipStream_t)
{
  return hipSuccess;
}
int resid_out_blocks(int, int, int) { return 1; }
hipError_t resid_out_dispatch(int, int, const MeshArgs&, const double*, double*, double*, double*,
                              hipStream_t)
{
  return hipSuccess;
}
hipError_t sample_dispatch(int, const double*, int, int, int, double, double*, hipStream_t)
{
  return hipSuccess;
}
hipError_t sum_dispatch(const double*, int, double*, hipStream_t) { return hipSuccess; }
size_t sum_scratch(int) { return 0; }
int tile_blocks(int, int, bool) { return 1; }
bool tile_valid(int, int, int tile, int waves) { return tile != 1 || waves > 1; }
hipError_t trace_dispatch(int, int, const MeshArgs&, const Phys&, const double*, double*, int*,
                          hipStream_t, bool)
{
  return hipSuccess;
}
size_t trace_doubles(int p, int nx, int ny, int nz)
{
  return (size_t)nx * ny * nz * 6 * 8 * (p + 1) * (p + 1);
}
hipError_t upload_gen_tables(const GenTab*) { return hipSuccess; }
hipError_t upload_tables(const PTab*, const QTab*) { return hipSuccess; }
hipError_t upload_tables_ensemble(const PTab*, const QTab*) { return hipSuccess; }
hipError_t upload_tables_tile(const PTab*, const QTab*) { return hipSuccess; }
}  // namespace dgx

static int g_failed = 0;
#define CHECK(x)                                               \
  do                                                           \
    if (!(x))                                                  \
    {                                                          \
      ++g_failed;                                              \
      std::printf("line %d: %s\n", __LINE__, #x);              \
    }                                                          \
  while (0)

struct Case
{
  dgx_mesh mesh{};
  dgx_params prm{};
  std::vector<double> nodes;
  Case(int p, int q, int n)
  {
    const int nq = q + 1;
    for (int e = 0; e < n * n * n; ++e)
      for (int c = 0; c < nq * nq * nq; ++c)
      {
        nodes.push_back(e % n + (c % nq) / (double)q);
        nodes.push_back(e / n % n + (c / nq % nq) / (double)q);
        nodes.push_back(e / (n * n) + (c / (nq * nq)) / (double)q);
      }
    mesh.p  = p;
    mesh.q  = q;
    mesh.nx = mesh.ny = mesh.nz = n;
    for (auto& b : mesh.bounds)
      b = DGX_BT_PERIODIC;
    mesh.nodes = nodes.data();
    dgx_make_reference_state(1.4, 287.0, 1e-3, 1.0, 1.0, 0.2, 0.0, 0.0, 6.0, nullptr, &prm);
  }
  dgx_status create(dgx_ctx** c) { return dgx_create(&mesh, &prm, c); }
};

static bool steps(dgx_ctx* c) { return dgx_step_async(c, DGX_RK4, 1e-3, 1) == DGX_OK; }

int main()
{
  const size_t huge = (size_t)1 << 34;
  // what each part takes
  Case curved(2, 2, 6), affine(0, 1, 8);
  g_hip.capacity[0] = huge;
  dgx_ctx *a = nullptr, *b = nullptr;
  CHECK(curved.create(&a) == DGX_OK);
  const size_t with = g_hip.used[0], store = a->geo_bytes, need = with - store;
  CHECK(store == 216 * 8 * (10 * 27 + 6 * 13 * 9) && steps(a) && g_mesh.geov && g_mesh.geof);
  uint64_t sz[4];
  CHECK(dgx_get_sizes(a, sz) == DGX_OK && sz[3] >= store);

  // one byte short of both contexts without either's store: refused, nothing lost
  g_hip.capacity[0] = 2 * need - 1;
  CHECK(curved.create(&b) == DGX_ERR_HIP && !b && g_hip.used[0] == need);
  CHECK(steps(a) && !g_mesh.geov && !g_mesh.geof);

  // room for both without a store: the earlier context's goes
  g_hip.capacity[0] = huge;
  CHECK(dgx_set_stored_geometry(a, 1) == DGX_OK && steps(a) && g_mesh.geov);
  g_hip.capacity[0] = 2 * need;
  CHECK(curved.create(&b) == DGX_OK);
  int on = 1;
  CHECK(dgx_get_stored_geometry(a, &on) == DGX_OK && !on);
  CHECK(steps(a) && !g_mesh.geov && steps(b) && !g_mesh.geov);
  CHECK(dgx_destroy(b) == DGX_OK);
  b = nullptr;

  // not while a captured launch reads it
  g_hip.capacity[0] = huge;
  CHECK(dgx_set_stored_geometry(a, 1) == DGX_OK);
  g_capturing = true;
  CHECK(steps(a) && g_mesh.geov);
  g_capturing = false;
  CHECK(dgx_set_stored_geometry(a, 0) == DGX_ERR_INVALID);
  g_hip.capacity[0] = 2 * need;
  CHECK(curved.create(&b) == DGX_ERR_HIP && !b && steps(a) && g_mesh.geov);
  CHECK(dgx_destroy(a) == DGX_OK);
  CHECK(g_hip.used[0] == 0);

  // an affine mesh without the room for its elements' records
  g_hip.capacity[0] = huge;
  CHECK(affine.create(&a) == DGX_OK && steps(a) && g_mesh.affine && g_mesh.arec && g_mesh.lamf);
  const size_t full = g_hip.used[0], records = 512 * 31 * 8;
  CHECK(dgx_destroy(a) == DGX_OK);
  g_hip.capacity[0] = full - 1;
  CHECK(affine.create(&a) == DGX_OK && g_hip.used[0] < full - records);
  CHECK(steps(a) && !g_mesh.affine && !g_mesh.arec && !g_mesh.lamf);
  CHECK(dgx_destroy(a) == DGX_OK);
  CHECK(g_hip.blocks.empty());
  return g_failed ? 1 : 0;
}
