// dgx_ctx.hpp -- the device context behind the dgx_ctx handle, shared by
// the C ABI translation units of libdgx (single cases and ensembles).
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>

#include "../../include/dgx.h"
#include "dgx_launch.hpp"

struct dgx_ctx
{
  int device;
  int p, q;
  int nx, ny, nz, nelem, nbf;
  int bounds[6];
  size_t nstate;  // nelem*5*nbf
  dgx_params params;
  dgx::Phys phys;
  hipStream_t stream;
  double* nodes;    // [e][(q+1)^3][3]
  double* U;        // state, Gauss-nodal basis
  double* Ua;       // stage buffer / staging
  double* Ub;       // stage buffer
  double* acc;      // RK4 accumulator
  double* fs;       // f_g scratch
  double* partial;  // per-block sums of R^2
  double* sum;      // reduced sum
  double* lam;      // BR2 lifting coefficients [e][6][(p+1)^2]
  double* lamf;     // affine meshes: one coefficient per element face [e][6]
  double* arec;     // affine meshes: each element's constant geometry
  double* geo;      // stored geometry (geov, then geof), or null
  size_t geo_bytes;
  int geo_users;    // launches and graphs that read geo; -1: none is to be read
  double* TU;       // face trace records of U, Ua, Ub [e][6][8][(p+1)^2]
  double* TUa;
  double* TUb;
  bool tu_valid;    // TU holds the traces of the current U
  bool tb_valid;    // TU holds its boundary states (all the tiled kernel reads)
  int stage_waves;  // occupancy target of the stage kernel (1..3)
  int stage_tile;   // 0: one-row stage kernel, 1: tiled stage kernel
  bool tile_chosen, waves_chosen;  // by the caller (else the defaults)
  int prec;         // DGX_PREC_* (float trace records in the mixed forms)
  int affine;       // q = 1 and every element a parallelepiped
  int matched;      // both elements at a face have the same face up to a translation (q = 1)
  double* mean;     // running mean (Gauss-nodal), allocated on first use
  double* adj_store;       // stored stages of the last dgx_adjoint_rk4 (kept:
  size_t adj_store_bytes;  // freeing tens of GB can take seconds)
  size_t adj_store_limit;  // most bytes that store may take (0: no limit)
  double* adj_ws;          // workspace of the adjoint calls, kept likewise
  size_t adj_ws_bytes;
  int adj_busy;            // the workspace is in use (see dgx_pool.hpp)
  int* status;      // kernel-side error flags
  int npartial;
  size_t bytes;
  char err[512];
};

namespace dgx
{
// MeshArgs of the context's mesh
// trace records of U, recomputed when U was set from outside
hipError_t ensure_traces(dgx_ctx* c);
// what a stage of the context's kernel reads besides U: the boundary states
// (tiled kernel) or the trace records
hipError_t ensure_stage_inputs(dgx_ctx* c);
hipError_t ensure_boundary(dgx_ctx* c);
// whether the context's stages read states instead of trace records
inline bool reads_states(const dgx_ctx* c)
{
  return c->stage_tile == 1 && c->prec == DGX_PREC_FP64 && c->matched;
}
// the last stage of a step has written U and what the next stage reads
inline void stage_outputs_valid(dgx_ctx* c)
{
  c->tb_valid = true;
  c->tu_valid = !reads_states(c);  // such stages write no records
}
// U was set or changed from outside: nothing stored belongs to it
inline void drop_traces(dgx_ctx* c)
{
  c->tu_valid = c->tb_valid = false;
}
// StageArgs of the stages of one step without a norm (returns the number of
// stages: 4 for RK4, 3 for TVD-RK3); the last stage writes U and its traces
int stage_plan(const dgx_ctx* c, int scheme, double dt, StageArgs sa[4]);
int default_stage_waves(int p, int q);
}  // namespace dgx
