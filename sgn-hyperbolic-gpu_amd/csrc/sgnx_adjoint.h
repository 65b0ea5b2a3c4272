// =============================================================================
// sgnx_adjoint.h -- device side of the discrete adjoint: the arguments of the
// RHS vector-Jacobian product and the launchers of sgnx_adjoint.hip.
// =============================================================================
#ifndef SGNX_ADJOINT_H
#define SGNX_ADJOINT_H

#include <hip/hip_runtime.h>

#include "../../include/sgnx.h"
#include "sgnx_internal.h"

namespace sgnx {

// W = ca*A (+ cb*B when B is given); out = (dR/dU (U))^T W, or, when acc is
// given (with B), ((A + acc) + B) + that; thetaBar += (dR/dtheta)^T W (when not
// null; set to 0 + that where `fresh`, which takes A only). 5*Nd arrays; out is
// none of the inputs (a workgroup reads its neighbours' A and B).
struct VjpArgs {
  const double* U;
  const double* A;
  double ca;
  const double* B;
  double cb;
  const double* acc;
  double* out;
  double* thetaBar;
  bool fresh = false;
};

// One product with its geometry and decomposition: a launch's arguments, or
// one member of a batched launch (tiles packed behind a per-member offset
// table as in the batched RHS)
struct VjpMember {
  VjpArgs va;
  Geometry g;
  Phys ph;
  GhostTime gt;
  int nStrips, nTiles;
};
VjpMember vjp_member(const Geometry& g, const Phys& ph, const VjpArgs& va, GhostTime gt);
// ... and one gauge log row's cotangents per member (Gb null: none)
struct GaugeMember {
  const double* Gb;
  const long long* nodes;
  int n;
  double* lam;
  double* thetaBar;
};
long long vjp_row_tiles(const Geometry& g);   // strips times element rows
// element rows per workgroup for the grids of one launch (Geometry::vrows[third])
int vjp_rows(const Geometry* const* g, int n, int cus, bool third);
// about what a reversed step's three products of these grids take, packed, at the
// heights rows[0] (the first two) and rows[1], in us
double vjp_step_cost(const Geometry* const* g, int n, int cus, const int* rows);
// nop: 1 = A only, 2 = A and B, 3 = with acc too, for all members
hipError_t launch_rhs_vjp_batch(const VjpMember* mem, const long long* tileStart, int nMem,
                                long long totalTiles, int nop, hipStream_t st);
hipError_t launch_gauge_bar_batch(const GaugeMember* gm, int nMem, hipStream_t st);

hipError_t launch_rhs_vjp(const Geometry& g, const Phys& ph, const VjpArgs& va, GhostTime gt,
                          hipStream_t st);
// HfX, HfY from the nodal still depth theta: the mean of the two edge values
// meeting at a line node (the wrapped pair on a periodic axis), the one
// interior edge value on a non-periodic side.
hipError_t launch_face_depth(const Geometry& g, const double* theta, double* HfX, double* HfY,
                             hipStream_t st);
// lam[nodes[k]] += Gb[k]; thetaBar[nodes[k]] -= Gb[k] (thetaBar may be null)
hipError_t launch_gauge_bar(const double* Gb, const long long* nodes, int n, double* lam,
                            double* thetaBar, hipStream_t st);

}  // namespace sgnx

#endif  // SGNX_ADJOINT_H
