// =============================================================================
// sgnx_adjoint.hip -- kernels of the discrete adjoint: the vector-Jacobian
// product of the FR/SGN right-hand side, the still depth set from one nodal
// field theta, and the gauge cotangent scatter. No counterpart in the
// reference, which has no adjoint.
//
// R is the composition of the five phases of src/solver/sgn2d.cpp:125-290
// (with the wall / inflow sides): nodal fluxes, sources and non-conservative
// products, a Rusanov flux on every interface line, the FR lift of the jumps.
// For a cotangent W of dU/dt the product returns
//   Ubar      = (dR/dU)^T W
//   thetaBar += (dR/dtheta)^T W,  theta the nodal still depth, with
//               Hx, Hy = (D theta)/J per element line (sgn2d.cpp:54-71) and the
//               face depth of an interface line node the mean of the two edge
//               values meeting there (the one interior value on a non-periodic
//               side); sgnx_set_depth builds that still depth.
// One launch (vjp_tile): the transposed lift gives each face node the cotangents
// of its line's face jumps, Lambda = -(g' . W)/J, and of the central face depths
// of the non-conservative products, lambda = (g' . W_hp c^2 u)/J; each interface
// line's Rusanov adjoint takes them, the derivative of max(sL, sR) on the side
// that attains it, walls mirrored back onto the interior state, the inflow ghost
// constant; the volume adjoint (source, non-conservative products, nodal fluxes
// through D^T) adds each node's parts of the lines around its element.
// Every sum has one writer and a fixed order, so the results are
// deterministic. The products are the derivatives of R away from its
// non-smooth points (a zero normal velocity, sL = sR off a wall, a clamped
// wave-speed argument). The Manning term is not differentiated (the entry
// points refuse nManning != 0).
// =============================================================================

#include <hip/hip_runtime.h>

#include <algorithm>

#include "sgnx_adjoint.h"
#include "sgnx_device.h"

namespace sgnx {
namespace {

constexpr int kT = 256;    // threads per block of the elementwise kernels

// --- pointwise adjoints of sgnx_phys.h (nManning = 0) --------------------------
// Every term is differentiated with the primitives u = hu/h, v, w, p as
// intermediate variables: a term adds its explicit U-derivatives to Ub and its
// primitive cotangents to a PrimBar, and prims_fin maps the summed PrimBar
// onto U once per state.

// a state with its reciprocal depth and primitives, formed once
struct St {
  double h, hu, hv, hw, hp;
  double ih, u, v, w, p;
};
__device__ __forceinline__ St make_st(const double* U) {
  St s;
  s.h = U[IH];
  s.hu = U[IHU];
  s.hv = U[IHV];
  s.hw = U[IHW];
  s.hp = U[IHP];
  s.ih = 1.0 / s.h;
  s.u = s.hu * s.ih;
  s.v = s.hv * s.ih;
  s.w = s.hw * s.ih;
  s.p = s.hp * s.ih;
  return s;
}

struct PrimBar { double u, v, w, p; };

// Ub += (d(u, v, w, p)/dU)^T q
__device__ __forceinline__ void prims_fin(const St& s, const PrimBar& q, double* Ub) {
  Ub[IHU] += q.u * s.ih;
  Ub[IHV] += q.v * s.ih;
  Ub[IHW] += q.w * s.ih;
  Ub[IHP] += q.p * s.ih;
  Ub[IH] -= (((q.u * s.u + q.v * s.v) + q.w * s.w) + q.p * s.p) * s.ih;
}

// flux along x (DIR 0, normal momentum hu) or y (DIR 1, hv) at still depth Hl,
// F = (m, m u, m v, m w, m (p + c^2)) + P e_N,  P = g/2 (h^2 - Hl^2) + h p:
// cotangent Fb; returns (dF/dHl) . Fb
template <int DIR>
__device__ __forceinline__ double flux_acc(const St& s, double Hl, const Phys& ph,
                                           const double* Fb, double* Ub, PrimBar& q) {
  constexpr int N = DIR == 0 ? IHU : IHV;
  const double m = DIR == 0 ? s.hu : s.hv;
  Ub[N] += Fb[IH] + (((Fb[IHU] * s.u + Fb[IHV] * s.v) + Fb[IHW] * s.w) + Fb[IHP] * (s.p + ph.c2));
  const double Pb = Fb[N];
  Ub[IH] += Pb * (ph.g * s.h + s.p);
  q.u += Fb[IHU] * m;
  q.v += Fb[IHV] * m;
  q.w += Fb[IHW] * m;
  q.p += Fb[IHP] * m + Pb * s.h;
  return -Pb * (ph.g * Hl);
}

// wave speed |vn| + sig, sig = sqrt(max(g h + p + c^2, 0)) given: cotangent sb
template <int DIR>
__device__ __forceinline__ void speed_acc(const St& s, double sig, const Phys& ph, double sb,
                                          double* Ub, PrimBar& q) {
  const double vn = DIR == 0 ? s.u : s.v;
  const double sg = vn > 0.0 ? sb : (vn < 0.0 ? -sb : 0.0);
  if (DIR == 0) q.u += sg;
  else q.v += sg;
  if (sig > 0.0) {
    const double ab = sb * (0.5 / sig);
    Ub[IH] += ab * ph.g;
    q.p += ab;
  }
}

// the node's own state terms: source S and the non-conservative products
// -Bx - By = c^2 (u hx + v hy) e_hp, with cotangent W; sets the still-depth
// cotangents Hlb, Hxb, Hyb
__device__ __forceinline__ void node_terms_acc(const St& s, double Hl, double Hx, double Hy,
                                               double hx, double hy, const Phys& ph,
                                               const double* W, double* Ub, PrimBar& q,
                                               double& Hlb, double& Hxb, double& Hyb) {
  const double bath = ph.g * (s.h - Hl) + ph.gamma * s.p;
  const double bathb = W[IHU] * Hx + W[IHV] * Hy;
  const double k = ph.m2c2 * W[IHP];              // S_hp = -2 c^2 (w + u Hx + v Hy)
  const double c = W[IHP] * ph.c2;                // ncp: c^2 (u hx + v hy)
  Hxb = W[IHU] * bath + k * s.u;
  Hyb = W[IHV] * bath + k * s.v;
  Hlb = -ph.g * bathb;
  Ub[IH] += ph.g * bathb;
  q.u += k * Hx + c * hx;
  q.v += k * Hy + c * hy;
  q.w += k;
  q.p += ph.gamma * W[IHW] + ph.gamma * bathb;
}

// a value that is the same on every lane, in scalar registers
__device__ __forceinline__ double uniform_value(double x) {
  return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(x)),
                          __builtin_amdgcn_readfirstlane(__double2loint(x)));
}

// ---- the product, row sweep ---------------------------------------------------
//
// A workgroup owns a strip of kEW element columns and a chunk of g.vrows
// element rows and walks up the chunk. Per row r:
//   stage  row r's nodes (one per lane; the elements left and right of the
//          strip too, whose lines' Lambda the strip's outer lines need): state,
//          cotangent W and the integrands of the depth-gradient cotangents,
//          c^2 W_hp u / Jx and c^2 W_hp v / Jy, to LDS; row r + 1's loads are
//          issued
//   faces  two lanes per interface line node, one per side: the x lines of
//          row r and the y line between rows r - 1 and r. Each lane forms its
//          own side's lift cotangents from its element's line,
//            Lambda = -(g' . W)/J (of the FR lift's face jump) and
//            lambda = g' . (c^2 W_hp vel / J) (of the central face depth),
//          the pair exchanges states and Lambda by lane permutes, and each
//          lane keeps the Rusanov adjoint of its own side. The lower row's
//          side of a y line (Lambda, lambda, edge state) was kept in LDS when
//          that row was staged. A y line is handled in the x frame: with P the
//          exchange of hu and hv, flux_y(U) = P flux_x(P U), so its adjoint is
//          P applied to the x adjoint of the exchanged states and cotangents.
//   lines  meanwhile on the wave without interface lines, a lane per element
//          line: D^T along it of W and of the depth gradients' integrand, of row
//          r - 1's Hx, Hy cotangents, and D of h, all five nodes at once, with
//          D in scalar registers
//   nodes  row r - 1 is finished (the upper y line's part of its top nodes, the
//          Hx, Hy cotangents' sums, the stores) and row r's node adjoint formed
//          from the line sums: source, non-conservative products, nodal fluxes,
//          depth gradients, its other faces' parts.
// One row below the chunk is staged for the lower side of its first y line and
// one above for the upper side of its last.
//
// The face depths drop out: an interface's flux and the two elements' own face
// fluxes take the same depth, and its cotangents, with FbL + FbR = Fsb - LamL -
// LamR = 0 in the momentum row, cancel. A periodic axis has two lines on its
// wrap, each feeding one element; the adjoint is linear in Lambda and, but for
// the face depth, the same on both, so one evaluation with both Lambda serves.
//
// What bounds it: a step's products move 160, 200 and 240 B a node, 434, 543 and
// 651 us at 1024x512 at a copy's rate; they take 560, 668 and 850 us (2.1 to 2.2
// ms for the three; per-element coefficients written to and read from memory by
// a launch of their own, each line evaluated by both of its elements: 3.8 ms).
// The rest is LDS traffic and the row's barriers, met by the four workgroups
// that 160 KB and 168 registers let a compute unit hold (three of the third
// product, whose sum of the other cotangents waits in LDS for a row). The line
// sums taken by the line lanes instead of by every node for itself, each
// reading 80 values: 615 -> 560 and 700 -> 668 us. A third product that keeps
// that sum in global memory between the rows, for four workgroups: 1028 us.
constexpr int kEW = 5;                       // element columns of a strip
constexpr int kVT = 192;                     // threads: 125 nodes, 50 halo nodes
static_assert(NPP * (kEW + 2) <= kVT && kVT % 64 == 0, "one lane per staged node");

struct VjpLds {
  static constexpr int kRec = 13;            // odd: no bank conflicts
  static constexpr int kW = 0, kU = 5, kDX = 10, kDY = 11, kDhx = 12;
  static constexpr int kF = NP * (kEW + 1), kNY = NP * kEW, kN = NPP * kEW;
  static constexpr int kCen = 2 * NV * kF;   // from an own-side cotangent to its central depth
  static constexpr int kTop = NV + 1 + NV;   // Lambda, lambda, edge state
  double rec[NPP * (kEW + 2) * kRec];        // strip nodes, left halo, right halo
  double xU[2][NV][kF], xh[kF];              // own side's cotangents, central depth
  double yU[2][NV][kF], yh[kF], yhT[kNY];    // the line below row r; central depth above
  double top[kNY][kTop];                     // the top faces of row r - 1
  // per node: D^T along x and along y of W and of the depth-gradient
  // cotangents' integrand, D h along y (along x: kDhx of its record)
  double sx[NV + 1][kN], sy[NV + 1][kN], dhy[kN];
  // per node: cotangent of Hx over Jx, of Hy over Jy; then D^T of them
  double tx[kN], ty[kN];
  double gw[2][NP];                          // gL', gR'
};

// W = ca A (+ cb B) as the host forms it: products and sum rounded apart
template <int NOP>
__device__ __forceinline__ void cotangent(const double* A, const double* B, double ca, double cb,
                                          double* W) {
#pragma unroll
  for (int c = 0; c < NV; ++c) {
    W[c] = ca * A[c];
    if (NOP > 1) W[c] = W[c] + cb * B[c];
  }
}

// the third product's workgroup also holds a row's sums of the other cotangents
template <int NOP>
struct VjpLdsOf : VjpLds {};
template <>
struct VjpLdsOf<3> : VjpLds {
  double base[2][NV][kN];                    // (A + acc) + B by row parity
};

// NOP: 1: W = ca A; 2: W = ca A + cb B; 3: that, and out = ((A + acc) + B) +
// the product. FRESH: thetaBar is set to 0 + the product and not read (a product
// by itself: 597 -> 566 us at 1024x512 against clearing it and adding; as a
// run-time switch 583, and 0.6 % of a reverse sweep for the registers it takes).
template <int NOP, bool FRESH>
__device__ __forceinline__ void vjp_tile(ConstArgs<VjpMember> M, int tile) {
  using L = VjpLds;
  constexpr int kRec = L::kRec;
  __shared__ VjpLdsOf<NOP> lds;
  const int t = threadIdx.x;
  if (t < NP) {
    lds.gw[0][t] = M->g.ops->gLp[t];
    lds.gw[1][t] = M->g.ops->gRp[t];
  }
  const double iJx = uniform_value(1.0 / M->g.Jx), iJy = uniform_value(1.0 / M->g.Jy);
  // read where it is used: kept, it would take scalar registers of the other phases
  auto phys = [&] {
    const ConstArgs<VjpMember> P = opaque(M);
    return Phys{P->ph.g, P->ph.c, P->ph.gamma, 0.0, P->ph.halfg, P->ph.c2, P->ph.mc2, P->ph.m2c2};
  };
  const int Nx = M->g.Nx, Ny = M->g.Ny, nStrips = M->nStrips, rows = M->g.vrows[NOP > 2];
  const int bcL = M->g.bc[0], bcR = M->g.bc[1];
  const bool wallB = M->g.bc[2] != SGNX_BC_PERIODIC, wallT = M->g.bc[3] != SGNX_BC_PERIODIC;
  const int chunk = __builtin_amdgcn_readfirstlane(tile / nStrips);
  const int ex0 = (tile - chunk * nStrips) * kEW, nW = min(kEW, Nx - ex0);
  const int ey0 = chunk * rows, ey1 = min(Ny, ey0 + rows);
  const size_t plane0 = (size_t)M->g.Nd * sizeof(double);
  const unsigned rowBytes = (unsigned)Nx * (NPP * 8u);
  const double ca = M->va.ca, cb = NOP > 1 ? M->va.cb : 0.0;

  // Staged node: a strip node, a halo node (its own record also where there is
  // no such element), or node 0 again.
  const bool hasL = ex0 > 0 || bcL == SGNX_BC_PERIODIC;
  const bool hasR = ex0 + nW < Nx || bcR == SGNX_BC_PERIODIC;
  const bool isNode = t < NPP * nW;
  constexpr int kHaloL = NPP * kEW, kHaloR = NPP * (kEW + 1);
  const bool inL = t >= kHaloL && t < kHaloR, inR = t >= kHaloR && t < NPP * (kEW + 2);
  const int tn = isNode ? t : 0;
  const int j = tn / NPP, loc = tn - NPP * j, b = loc / NP, a = loc - NP * b;
  const int sRecIdx = inL || inR ? t : tn;
  unsigned n8;                               // its byte offset within a row of a plane
  if (inL) n8 = (unsigned)((hasL ? (ex0 > 0 ? ex0 - 1 : Nx - 1) : ex0) * NPP + t - kHaloL) * 8u;
  else if (inR) n8 = (unsigned)((hasR ? (ex0 + nW < Nx ? ex0 + nW : 0) : ex0) * NPP + t - kHaloR) * 8u;
  else n8 = (unsigned)(ex0 * NPP + tn) * 8u;

  // Interface half-items, from the third wave (which has no node) on: two
  // lanes per line node, lane 2k + side taking side 0 (left / lower) or 1.
  const int nX = NP * (nW + 1);
  const int it = t < 128 ? t + 64 : t - 128, side = it & 1, kk = it >> 1;
  const bool isItem = kk < nX + NP * nW;
  const bool isX = kk < nX;
  const int xi = isX ? kk / NP : 0, xn = isX ? kk - NP * xi : 0;
  const int ky = !isX && isItem ? kk - nX : 0, jj = ky / NP, aa = ky - NP * jj;
  const bool outL = isX && side == 0 && xi == 0, outR = isX && side == 1 && xi == nW;
  const bool ghostX = (outL && !hasL) || (outR && !hasR);
  const bool inflow = ghostX && outL && bcL == SGNX_BC_INFLOW;
  // the other side of this lane's line is a wall's ghost
  const bool wallX = isX && ((side == 1 && xi == 0 && !hasL && bcL == SGNX_BC_WALL) ||
                             (side == 0 && xi == nW && !hasR));
  const bool lowerY = !isX && side == 0, upperY = !isX && side == 1;
  // the element line whose Lambda the lane forms (y, lower side: that of row
  // r's top, kept for the next row), its weights, and its edge node
  int rec0;
  if (isX) rec0 = outL ? kHaloL : outR ? kHaloR : NPP * (xi - 1 + side);
  else rec0 = NPP * jj;
  LdsDouble* sLine = (LdsDouble*)lds.rec + (rec0 + (isX ? NP * xn : aa)) * kRec;
  const int step = (isX ? 1 : NP) * kRec;
  LdsDouble* sEdge = sLine + (side == 0 ? NP - 1 : 0) * step;
  LdsDouble* sGw = (LdsDouble*)lds.gw[side == 0 ? 1 : 0];
  const int dOff = isX ? L::kDX : L::kDY;
  const double miJ = isX ? -iJx : -iJy;
  LdsDouble* sTop = (LdsDouble*)lds.top[ky];
  LdsDouble* sOut = isX ? (LdsDouble*)lds.xU[side][0] + kk : (LdsDouble*)lds.yU[side][0] + ky;
  unsigned h8 = (unsigned)((ex0 + jj) * NPP + aa) * 8u;   // the column's bottom face node

  // Element lines, on the second wave (which has no half-item): lanes 0-24 the
  // x lines, 25-49 the y lines, each all five nodes of its line.
  const int ln = t - 64, ll = ln < NP * kEW ? ln : ln - NP * kEW;
  const bool lineX = ln < NP * kEW, isLine = ln >= 0 && ln < 2 * NP * kEW && ll < NP * nW;
  const int le = isLine ? ll / NP : 0, lq = isLine ? ll - NP * le : 0;
  const int lNode = NPP * le + (lineX ? NP * lq : lq), lStep = lineX ? 1 : NP;

  struct Raw {
    double U[NV], A[NV], B[NOP > 1 ? NV : 1], acc[NOP > 2 ? NV : 1];
  };
  // row `to`, clamped to the grid (where it is beyond a wall nothing of it is
  // used) and wrapped on a periodic axis
  auto row_of = [&](int to) {
    to = to < 0 ? (wallB ? 0 : Ny - 1) : to;
    to = to >= Ny ? (wallT ? Ny - 1 : min(to - Ny, Ny - 1)) : to;
    return __builtin_amdgcn_readfirstlane((int)((unsigned)to * rowBytes));
  };
  auto load_row = [&](ConstArgs<VjpMember> R, int to, size_t plane, unsigned off, Raw& x) {
    const unsigned first = (unsigned)row_of(to);
    load_vars(R->va.U, first, plane, off, x.U);
    load_vars(R->va.A, first, plane, off, x.A);
    if (NOP > 1) load_vars(R->va.B, first, plane, off, x.B);
    if (NOP > 2) load_vars(R->va.acc, first, plane, off, x.acc);
  };
  auto load_h = [&](ConstArgs<VjpMember> R, int to, unsigned off) {
    return load_at(global_at(R->va.U, (unsigned)row_of(to)), off);
  };

  LdsDouble* sRec = (LdsDouble*)lds.rec + sRecIdx * kRec;
  LdsDouble* sXU = (LdsDouble*)lds.xU[0][0] + NP * j + b;
  LdsDouble* sYU = (LdsDouble*)lds.yU[0][0] + NP * j + a;
  LdsDouble* sNode = (LdsDouble*)lds.sx[0] + (t < L::kN ? t : 0);
  constexpr int kSy = (NV + 1) * L::kN, kDhy = 2 * kSy, kTx = kDhy + L::kN, kTy = kTx + L::kN;
  LdsDouble* sL = (LdsDouble*)lds.rec + lNode * kRec;
  LdsDouble* sSum = (LdsDouble*)(lineX ? lds.sx[0] : lds.sy[0]) + lNode;

  Raw raw;
  load_row(M, ey0 - 1, plane0, n8, raw);
  double hAbove = load_h(M, ey0, h8);          // of the row after the one staged next
  // row r - 1's node results: the product without its top faces' part, what it
  // is added to, its still-depth cotangent
  double pend[NV], th = 0.0;

  for (int r = ey0 - 1; r <= ey1; ++r) {
    size_t plane = plane0;
    __asm__ volatile("" : "+s"(plane));
    __asm__ volatile("" : "+v"(n8));
    __asm__ volatile("" : "+v"(h8));
    for (LdsDouble** q : {&sRec, &sXU, &sYU, &sNode, &sLine, &sEdge, &sOut, &sTop, &sL, &sSum})
      __asm__ volatile("" : "+v"(*q));
    // ---- stage ---------------------------------------------------------------
    const ConstArgs<VjpMember> R0 = opaque(M);
    double* const tbar = R0->va.thetaBar;
    // (a fresh one isn't read: every lane takes the same entry in its place)
    const double thOld =
        FRESH ? 0.0 : load_at(global_at(tbar ? tbar : R0->va.U, (unsigned)row_of(r - 1)), n8);
    const double hNext = load_h(R0, r + 2, h8);
    const unsigned rowAt = (unsigned)row_of(r);
    const double Hl = load_at(global_at(R0->g.Hnod, rowAt), n8);
    const double Hx = load_at(global_at(R0->g.Hx, rowAt), n8);
    const double Hy = load_at(global_at(R0->g.Hy, rowAt), n8);
    {
      double W[NV];
      cotangent<NOP>(raw.A, raw.B, ca, cb, W);
      const double q = W[IHP] * R0->ph.c2 / raw.U[IH];
#pragma unroll
      for (int c = 0; c < NV; ++c) {
        sRec[L::kW + c] = W[c];
        sRec[L::kU + c] = raw.U[c];
        if constexpr (NOP > 2)
          if (t < NPP * kEW) lds.base[r & 1][c][t] = (raw.A[c] + raw.acc[c]) + raw.B[c];
      }
      sRec[L::kDX] = q * raw.U[IHU] * iJx;
      sRec[L::kDY] = q * raw.U[IHV] * iJy;
    }
    __builtin_amdgcn_sched_barrier(0);
    load_row(opaque(M), r + 1, plane, n8, raw);
    row_sync();

    // ---- faces -----------------------------------------------------------------
    if (isItem && (!isX || (r >= ey0 && r < ey1))) {
      double La[NV], la, E[NV];
      {
        double w = sGw[0];
#pragma unroll
        for (int c = 0; c < NV; ++c) La[c] = w * sLine[L::kW + c];
        la = w * sLine[dOff];
#pragma unroll
        for (int k = 1; k < NP; ++k) {
          w = sGw[k];
#pragma unroll
          for (int c = 0; c < NV; ++c) La[c] = fma(w, sLine[k * step + L::kW + c], La[c]);
          la = fma(w, sLine[k * step + dOff], la);
        }
#pragma unroll
        for (int c = 0; c < NV; ++c) {
          La[c] = La[c] * miJ;
          E[c] = sEdge[L::kU + c];
        }
      }
      if (lowerY) {
        // row r's top faces for the next row; row r - 1's for this line
        const bool atWall = wallT && r + 1 == Ny;
        lds.yhT[ky] = 0.5 * (E[IH] + (atWall ? E[IH] : hAbove));
        double o[L::kTop];
#pragma unroll
        for (int c = 0; c < L::kTop; ++c) o[c] = sTop[c];
#pragma unroll
        for (int c = 0; c < NV; ++c) {
          sTop[c] = La[c];
          sTop[NV + 1 + c] = E[c];
          La[c] = o[c];
          E[c] = o[NV + 1 + c];
        }
        sTop[NV] = la;
        la = o[NV];
      }
      auto to_frame = [&](double* x) {
        const double u_ = x[IHU], v_ = x[IHV];
        x[IHU] = isX ? u_ : v_;
        x[IHV] = isX ? v_ : u_;
      };
      to_frame(E);
      to_frame(La);
      const bool lowWall = wallB && r == 0, topWall = wallT && r == Ny;
      const bool ghost = ghostX || (lowerY && lowWall) || (upperY && topWall);
      const bool wallOther = wallX || (upperY && lowWall) || (lowerY && topWall);
      if (wave_any(ghost)) {
        double o[NV];
#pragma unroll
        for (int c = 0; c < NV; ++c) o[c] = lane_swap(E[c]);
        if (ghost) {
#pragma unroll
          for (int c = 0; c < NV; ++c) {
            E[c] = c == IHU ? -o[c] : o[c];
            La[c] = 0.0;
          }
          la = 0.0;
          if (inflow) {
            const int rr = min(max(r, 0), Ny - 1);   // (rows outside the grid are not used)
            const GlobalDouble* cf =
                (const GlobalDouble*)R0->g.inflow + ((size_t)rr * NP + xn) * (NV * 3);
#pragma unroll
            for (int c = 0; c < NV; ++c)
              E[c] = (cf[3 * c] + cf[3 * c + 1] * R0->gt.s) + cf[3 * c + 2] * R0->gt.c;
          }
        }
      }
      // Fs = 0.5 (FL + FR) - 0.5 lam (UR - UL) with its cotangent LamL + LamR,
      // the sides' own face fluxes with cotangents -LamL, -LamR, the central
      // depth 0.5 (hL + hR) with cotangent lamL + lamR and the own edge depth
      // with -lam
      const Phys ph = phys();
      const St s = make_st(E);
      const double arg = ph.g * s.h + s.p + ph.c2;
      const double sig = sqrt(arg > 0.0 ? arg : 0.0);
      const double sp = fabs(s.u) + sig, so = lane_swap(sp);
      const double hl = flip_sign(0.5 * fmax(sp, so), side << 31);
      double Ub[NV], Fb[NV], dot = 0.0;
#pragma unroll
      for (int c = 0; c < NV; ++c) {
        const double Fsb = La[c] + lane_swap(La[c]);
        const double Eo = lane_swap(E[c]);
        if (c == IH && side == 0) sOut[L::kCen] = 0.5 * (E[c] + Eo);
        Ub[c] = hl * Fsb;
        Fb[c] = fma(0.5, Fsb, -La[c]);
        dot = fma(Fsb, Eo - E[c], dot);
      }
      Ub[IH] = fma(0.5, la + lane_swap(la), Ub[IH]) - la;
      PrimBar q{0.0, 0.0, 0.0, 0.0};
      const double hlb = side == 0 ? -dot : dot;
      if (side == 0 ? sp > so : !(so > sp)) speed_acc<0>(s, sig, ph, 0.5 * hlb, Ub, q);
      flux_acc<0>(s, 0.0, ph, Fb, Ub, q);
      prims_fin(s, q, Ub);
      if (wave_any(wallOther)) {
        // a wall's ghost is the own state with the normal momentum negated
#pragma unroll
        for (int c = 0; c < NV; ++c) {
          const double o = lane_swap(Ub[c]);
          if (wallOther) Ub[c] = c == IHU ? Ub[c] - o : Ub[c] + o;
        }
      }
      to_frame(Ub);
#pragma unroll
      for (int c = 0; c < NV; ++c) sOut[c * L::kF] = Ub[c];
    }
    // ---- lines -----------------------------------------------------------------
    if (isLine) {
      const auto* const T = (ConstArgs<OpTables>)opaque(M)->g.ops;
      // out[a] = sum over k of D[k][a] in[k]
      auto transposed = [&](const LdsDouble* in, int inStep, LdsDouble* out) {
        double x[NP];
#pragma unroll
        for (int k = 0; k < NP; ++k) x[k] = in[k * inStep];
#pragma unroll
        for (int q = 0; q < NP; ++q) {
          double v = T->D[q] * x[0];
#pragma unroll
          for (int k = 1; k < NP; ++k) v = fma(T->D[k * NP + q], x[k], v);
          out[q * lStep] = v;
        }
        __builtin_amdgcn_sched_barrier(0);
      };
      const int in = lStep * kRec;
#pragma unroll
      for (int c = 0; c < NV; ++c) transposed(sL + L::kW + c, in, sSum + c * L::kN);
      transposed(sL + (lineX ? L::kDX : L::kDY), in, sSum + NV * L::kN);
      LdsDouble* const sT = sSum + (lineX ? kTx : kTy - kSy);
      transposed(sT, lStep, sT);
      double h[NP];
#pragma unroll
      for (int k = 0; k < NP; ++k) h[k] = sL[k * in + L::kU];
      LdsDouble* const to = lineX ? sL + L::kDhx : sSum + (kDhy - kSy);
      const int toStep = lineX ? kRec : NP;
#pragma unroll
      for (int q = 0; q < NP; ++q) {
        double v = T->D[q * NP] * h[0];
#pragma unroll
        for (int k = 1; k < NP; ++k) v = fma(T->D[q * NP + k], h[k], v);
        to[q * toStep] = v;
      }
    }
    row_sync();

    // ---- nodes -----------------------------------------------------------------
    if (t < NPP * kEW) {
      if (r > ey0) {
        // row r - 1
        const unsigned first = (unsigned)row_of(r - 1);
        if (b == NP - 1) {
#pragma unroll
          for (int c = 0; c < NV; ++c) pend[c] += sYU[c * L::kF];
        }
        GlobalByte* p = global_at(R0->va.out, first);
#pragma unroll
        for (int c = 0; c < NV; ++c) {
          double o = pend[c];
          if constexpr (NOP > 2) o = lds.base[(r - 1) & 1][c][t] + o;
          if (isNode) store_at(p, n8, o);
          p += plane;
        }
        if (tbar) {
          // still depth: Hnod = theta, Hx = (D theta)/Jx, Hy = (D theta)/Jy per line
          th = (th + sNode[kTx]) + sNode[kTy];
          if (isNode) store_at(global_at(tbar, first), n8, thOld + th);
        }
      }
      if (r >= ey0 && r < ey1) {
        double U[NV], W[NV];
#pragma unroll
        for (int c = 0; c < NV; ++c) {
          U[c] = sRec[L::kU + c];
          W[c] = sRec[L::kW + c];
        }
        const Phys ph = phys();
        const St s = make_st(U);
        // the depth gradient: the line sums and the jumps to the central depths
        double dhx = sRec[L::kDhx], dhy = sNode[kDhy];
        {
          LdsDouble* const x0 = (LdsDouble*)lds.rec + (NPP * j + NP * b) * kRec + L::kU;
          LdsDouble* const y0 = (LdsDouble*)lds.rec + (NPP * j + a) * kRec + L::kU;
          LdsDouble* const cx = sXU + L::kCen;
          LdsDouble* const cy = sYU + L::kCen;
          dhx += (cx[0] - x0[0]) * lds.gw[0][a] + (cx[NP] - x0[(NP - 1) * kRec]) * lds.gw[1][a];
          dhy += (cy[0] - y0[0]) * lds.gw[0][b] +
                 (cy[L::kF] - y0[(NP - 1) * NP * kRec]) * lds.gw[1][b];
        }
        double Fb[NV], Gb[NV];
        double Hlb, Hxb, Hyb;
        PrimBar q{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int c = 0; c < NV; ++c) {
          pend[c] = 0.0;
          Fb[c] = -sNode[c * L::kN] * iJx;
          Gb[c] = -sNode[kSy + c * L::kN] * iJy;
        }
        node_terms_acc(s, Hl, Hx, Hy, dhx * iJx, dhy * iJy, ph, W, pend, q, Hlb, Hxb, Hyb);
        Hlb += flux_acc<0>(s, Hl, ph, Fb, pend, q);
        Hlb += flux_acc<1>(s, Hl, ph, Gb, pend, q);
        prims_fin(s, q, pend);
        pend[IH] += sNode[NV * L::kN] + sNode[kSy + NV * L::kN];
        auto face_add = [&](LdsDouble* f) {
#pragma unroll
          for (int c = 0; c < NV; ++c) pend[c] += f[c * L::kF];
        };
        if (a == 0) face_add(sXU + NV * L::kF);        // upper side of the line on the left
        if (a == NP - 1) face_add(sXU + NP);            // lower side of the one on the right
        if (b == 0) face_add(sYU + NV * L::kF);        // upper side of the line below
        th = Hlb;
        sNode[kTx] = Hxb * iJx;
        sNode[kTy] = Hyb * iJy;
      }
    }
    hAbove = hNext;
    row_sync();
  }
}

// The arguments are the kernel's only parameter, read where they lie.
template <int NOP, bool FRESH>
__global__ void __launch_bounds__(kVT, 3) k_vjp_sweep(VjpMember) {
  vjp_tile<NOP, FRESH>((ConstArgs<VjpMember>)__builtin_amdgcn_kernarg_segment_ptr(),
                     xcd_tile(blockIdx.x, gridDim.x));
}

// every member's tiles in one launch: the member of workgroup w has
// tileStart[m] <= w < tileStart[m + 1], multiples of the XCDs' number
template <int NOP>
__global__ void __launch_bounds__(kVT, 3)
k_vjp_sweep_batch(const VjpMember* __restrict__ mem, const long long* __restrict__ tileStart,
                  int nMem) {
  const long long w = blockIdx.x;
  int lo = 0, hi = nMem - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (tileStart[mid] <= w) lo = mid;
    else hi = mid - 1;
  }
  const int own = __builtin_amdgcn_readfirstlane((int)(w - tileStart[lo]));
  const ConstArgs<VjpMember> M = const_entry(mem, lo);
  if (own >= M->nTiles) return;   // (filling up)
  vjp_tile<NOP, false>(M, xcd_tile(own, M->nTiles));
}

// lam[node] += Gb[k], thetaBar[node] -= Gb[k] for the n gauges of one log row,
// by one block: the thread of a node's first gauge adds that node's gauges in
// gauge order, so every node receives the sums a sequential scan over the
// gauges forms (a node may carry several gauges), bit for bit, and distinct
// nodes proceed in parallel instead of one dependent load after another.
__device__ __forceinline__ void gauge_bar_block(const double* __restrict__ Gb,
                                                const long long* __restrict__ nodes, int n,
                                                double* __restrict__ lam,
                                                double* __restrict__ thetaBar) {
  for (int k = threadIdx.x; k < n; k += blockDim.x) {
    const long long i = nodes[k];
    bool first = true;
    for (int j = 0; j < k && first; ++j) first = nodes[j] != i;
    if (!first) continue;
    double l = lam[i];
    double th = thetaBar ? thetaBar[i] : 0.0;
    for (int j = k; j < n; ++j) {
      if (nodes[j] != i) continue;
      l += Gb[j];
      th -= Gb[j];
    }
    lam[i] = l;
    if (thetaBar) thetaBar[i] = th;
  }
}

// the gauge cotangents of one log row per member (one block per member)
__global__ void k_gauge_bar_batch(const GaugeMember* __restrict__ gm, int nMem) {
  if ((int)blockIdx.x >= nMem) return;
  const GaugeMember q = gm[blockIdx.x];
  if (!q.Gb) return;
  gauge_bar_block(q.Gb, q.nodes, q.n, q.lam, q.thetaBar);
}

// ---- still depth from theta -------------------------------------------------------
__global__ void __launch_bounds__(kT)
k_face_depth(const double* __restrict__ th, int Nx, int Ny, int perX, int perY,
             double* __restrict__ HfX, double* __restrict__ HfY) {
  const long long nfx = (long long)(Nx + 1) * Ny * NP, nfy = (long long)Nx * (Ny + 1) * NP;
  const long long gid = (long long)blockIdx.x * kT + threadIdx.x;
  if (gid < nfx) {
    const long long q = gid / NP;
    const int n = (int)(gid - q * NP);
    const int ey = (int)(q / (Nx + 1)), l = (int)(q - (long long)ey * (Nx + 1));
    const long long row = (long long)ey * Nx;
    const double lo = th[(row + (l > 0 ? l - 1 : Nx - 1)) * NPP + NP - 1 + NP * n];
    const double hi = th[(row + (l < Nx ? l : 0)) * NPP + NP * n];
    double v;
    if ((l > 0 && l < Nx) || perX) v = 0.5 * (lo + hi);
    else v = l == 0 ? hi : lo;
    HfX[gid] = v;
  } else if (gid < nfx + nfy) {
    const long long k = gid - nfx;
    const long long q = k / NP;
    const int n = (int)(k - q * NP);
    const int l = (int)(q / Nx), ex = (int)(q - (long long)l * Nx);
    const double lo = th[((long long)(l > 0 ? l - 1 : Ny - 1) * Nx + ex) * NPP + n + NP * (NP - 1)];
    const double hi = th[((long long)(l < Ny ? l : 0) * Nx + ex) * NPP + n];
    double v;
    if ((l > 0 && l < Ny) || perY) v = 0.5 * (lo + hi);
    else v = l == 0 ? hi : lo;
    HfY[k] = v;
  }
}

// the gauge cotangents of one log row (one block)
__global__ void k_gauge_bar(const double* __restrict__ Gb, const long long* __restrict__ nodes,
                            int n, double* __restrict__ lam, double* __restrict__ thetaBar) {
  if (blockIdx.x != 0) return;
  gauge_bar_block(Gb, nodes, n, lam, thetaBar);
}

}  // namespace

namespace {
int vjp_strips(const Geometry& g) { return (g.Nx + kEW - 1) / kEW; }
// which build a product takes: its operands
int vjp_nop(const VjpArgs& va) { return va.acc ? 3 : va.B ? 2 : 1; }
}  // namespace

long long vjp_row_tiles(const Geometry& g) { return (long long)vjp_strips(g) * g.Ny; }

// Per row a lone workgroup on a unit takes 2.8 us, two, three and four together
// 3.6, 4.4 and 5.2 (a unit holds four), of the third product 3.2, 4.1 and 5.0
// (three); the rows staged beside a chunk cost as much as its own.
namespace {
constexpr SweepPace kPace[2] = {{4, 2.0, 0.8, 2.0, 2.0}, {3, 2.3, 0.9, 2.0, 2.0}};

double vjp_cost(const Geometry* const* g, int n, int cus, bool third, int rows) {
  long long tiles = 0;
  for (int i = 0; i < n; ++i)
    tiles += (long long)vjp_strips(*g[i]) * (((long long)g[i]->Ny + rows - 1) / rows);
  return sweep_cost(tiles, rows, cus, kPace[third]);
}
}  // namespace

// The lowest time by sweep_cost:
//   first two products, us     rows: 2    3    4    7   10   16   32
//    128 x   64                     44   46   46   65   73
//    256 x  128                    126  115  112   99  107  130  199
//   1024 x  512                   1800 1552 1426 1306 1271 1224 1224
//   third product
//    128 x   64                     30   27   25   36   40
//    256 x  128                     81   71   70   68   62   74  111
//   1024 x  512                   1269 1121 1038  948  906  854  829
int vjp_rows(const Geometry* const* g, int n, int cus, bool third) {
  cus = std::max(cus, 1);
  return choose_rows(32, [&](int r) { return vjp_cost(g, n, cus, third, r); });
}

double vjp_step_cost(const Geometry* const* g, int n, int cus, const int* rows) {
  cus = std::max(cus, 1);
  return 2.0 * vjp_cost(g, n, cus, false, rows[0]) + vjp_cost(g, n, cus, true, rows[1]);
}

VjpMember vjp_member(const Geometry& g, const Phys& ph, const VjpArgs& va, GhostTime gt) {
  const long long rows = g.vrows[vjp_nop(va) > 2];
  const int strips = vjp_strips(g);
  return VjpMember{va, g, ph, gt, strips, (int)(strips * ((g.Ny + rows - 1) / rows))};
}

hipError_t launch_rhs_vjp(const Geometry& g, const Phys& ph, const VjpArgs& va, GhostTime gt,
                          hipStream_t st) {
  const VjpMember m = vjp_member(g, ph, va, gt);
  const int nop = vjp_nop(va);
  if ((va.fresh && nop != 1) || va.out == va.A || va.out == va.B || (va.acc && !va.B))
    return hipErrorInvalidValue;
  const dim3 grid((unsigned)m.nTiles), block(kVT);
#define SGNX_VJP(...) hipLaunchKernelGGL((k_vjp_sweep<__VA_ARGS__>), grid, block, 0, st, m)
  if (va.fresh) SGNX_VJP(1, true);
  else if (nop == 1) SGNX_VJP(1, false);
  else if (nop == 2) SGNX_VJP(2, false);
  else SGNX_VJP(3, false);
#undef SGNX_VJP
  return hipGetLastError();
}

hipError_t launch_rhs_vjp_batch(const VjpMember* mem, const long long* tileStart, int nMem,
                                long long totalTiles, int nop, hipStream_t st) {
  if (totalTiles <= 0) return hipSuccess;
  if (totalTiles > 0x7fffffffLL || nop < 1 || nop > 3) return hipErrorInvalidValue;
  const dim3 grid((unsigned)totalTiles), block(kVT);
#define SGNX_VJP(N) \
  hipLaunchKernelGGL(k_vjp_sweep_batch<N>, grid, block, 0, st, mem, tileStart, nMem)
  switch (nop) {
    case 1: SGNX_VJP(1); break;
    case 2: SGNX_VJP(2); break;
    default: SGNX_VJP(3);
  }
#undef SGNX_VJP
  return hipGetLastError();
}

hipError_t launch_gauge_bar_batch(const GaugeMember* gm, int nMem, hipStream_t st) {
  if (nMem <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_gauge_bar_batch, dim3((unsigned)nMem), dim3(64), 0, st, gm, nMem);
  return hipGetLastError();
}

hipError_t launch_face_depth(const Geometry& g, const double* theta, double* HfX, double* HfY,
                             hipStream_t st) {
  const long long n = (long long)(g.Nx + 1) * g.Ny * NP + (long long)g.Nx * (g.Ny + 1) * NP;
  hipLaunchKernelGGL(k_face_depth, dim3((unsigned)((n + kT - 1) / kT)), dim3(kT), 0, st, theta,
                     g.Nx, g.Ny, (int)(g.bc[0] == SGNX_BC_PERIODIC),
                     (int)(g.bc[2] == SGNX_BC_PERIODIC), HfX, HfY);
  return hipGetLastError();
}

hipError_t launch_gauge_bar(const double* Gb, const long long* nodes, int n, double* lam,
                            double* thetaBar, hipStream_t st) {
  hipLaunchKernelGGL(k_gauge_bar, dim3(1), dim3(64), 0, st, Gb, nodes, n, lam, thetaBar);
  return hipGetLastError();
}

}  // namespace sgnx
