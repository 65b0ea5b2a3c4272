// =============================================================================
// sgnx_kernels.hip -- gfx950 kernels of the FR/SGN right-hand side and of the
// Bogacki-Shampine 3(2) stage, update and error-norm passes.
//
// RHS (one launch, replaces the five phases of src/solver/sgn2d.cpp:125-290):
//   A workgroup owns a tile of TW consecutive elements of one element row
//   (25*TW nodes, one work-item per node; the state layout keeps each
//   variable's element blocks contiguous, so the tile is one coalesced span
//   per variable). Three phases separated by workgroup barriers:
//     0  load U, H at the node; primitives; nodal fluxes F, G -> LDS
//     1  one work-item per interface node of the tile (TW+1 x-lines, TW
//        bottom and TW top y-lines): Rusanov flux, central depth h*, and the
//        two one-sided fluxes, which are the elements' own face fluxes
//     2  one work-item per node: D.F and D.G from LDS, FR lift of the face
//        jumps, FR depth gradients, non-conservative products, source, dU
//   Face extrapolation on GLL points is the edge node itself: the reference's
//   sum 0 + 1*v0 + 0*v1 + ... equals v0 + 0.0 for finite values (the +0.0
//   turns -0 into +0 as that sum does), so it is never materialised.
//   Neighbour face nodes outside the tile are read from global memory; the
//   domain sides are periodic (wrapped index), walls (mirror ghost) or the
//   left inflow ghost.
//   Tiles are handed out XCD-contiguously: consecutive workgroup ids land on
//   different XCDs, so ids are remapped such that each XCD sweeps its own
//   contiguous band of tiles and finds the row below still in its L2.
//
// Every floating-point expression keeps the reference's evaluation order; the
// file is compiled with -ffp-contract=off.
// =============================================================================

#include <algorithm>

#include "sgnx_device.h"
#include "sgnx_internal.h"

namespace sgnx {

namespace {

constexpr int kThreads = 256;     // elementwise / reduction kernels

template <int TW>
struct Tile {
  static constexpr int NT = ((NPP * TW + 63) / 64) * 64;  // work-items (whole waves)
  static constexpr int NXI = NP * (TW + 1);               // x-interface nodes
  static constexpr int NYI = NP * TW;                     // y-interface nodes per side
};

// Node (a, b) of element (ex, ey), variable v (sgn2d.h:22-27, mesh2d.h:31).
__device__ __forceinline__ long long nidx(const Geometry& g, int ex, int ey, int a, int b) {
  return ((long long)ey * g.Nx + ex) * NPP + a + NP * b;
}

// Face state of a node: the GLL extrapolation value v + 0.0 (see header).
__device__ __forceinline__ void load_face(const double* __restrict__ U, long long Nd,
                                          long long node, double* W) {
#pragma unroll
  for (int v = 0; v < NV; ++v) W[v] = U[(long long)v * Nd + node] + 0.0;
}

// Compensated accumulation (Knuth's TwoSum): s + c carries the running sum
// with the rounding error of every addition kept in c.
__device__ __forceinline__ void acc_add(double& s, double& c, double x) {
  const double t = s + x;
  const double bp = t - s;
  const double e = (s - (t - bp)) + (x - bp);
  s = t;
  c = c + e;
}

// Fixed-order reductions of (s, c, m) triples: a compensated sum s + c and a
// max m. Within a wavefront, five butterfly levels of swizzles (lane ^ 1, 2,
// 4, 8, 16 inside each half) and lane 32's triple read into lane 0; then the
// waves' triples in wave order. Each level merges the partner's triple into
// the lane's own in the same way, so lane 0's result is one fixed tree and
// the same bits on every run.
template <int XOR>
__device__ __forceinline__ double swz_xor(double x) {
  constexpr int kPat = (XOR << 10) | 0x1F;   // bit mode: and 0x1f, or 0, xor XOR
  const int lo = __builtin_amdgcn_ds_swizzle(__double2loint(x), kPat);
  const int hi = __builtin_amdgcn_ds_swizzle(__double2hiint(x), kPat);
  return __hiloint2double(hi, lo);
}

__device__ __forceinline__ void merge3(double& s, double& c, double& m, double s2, double c2,
                                       double m2) {
  acc_add(s, c, s2);
  c = c + c2;
  m = fmax(m, m2);
}

template <int XOR>
__device__ __forceinline__ void wave_level(double& s, double& c, double& m) {
  const double s2 = swz_xor<XOR>(s), c2 = swz_xor<XOR>(c), m2 = swz_xor<XOR>(m);
  merge3(s, c, m, s2, c2, m2);
}

__device__ __forceinline__ double lane32(double x) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(x), 32);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(x), 32);
  return __hiloint2double(hi, lo);
}

// a wavefront's triples into its lane 0
__device__ __forceinline__ void wave_reduce(double& s, double& c, double& m) {
  wave_level<1>(s, c, m);
  wave_level<2>(s, c, m);
  wave_level<4>(s, c, m);
  wave_level<8>(s, c, m);
  wave_level<16>(s, c, m);
  const double s2 = lane32(s), c2 = lane32(c), m2 = lane32(m);
  merge3(s, c, m, s2, c2, m2);
}

// Every thread of the block calls it (no divergence); the result is in
// thread 0's s, c, m. ws: 3 doubles of LDS per wave.
__device__ __forceinline__ void block_reduce(double& s, double& c, double& m, double* ws) {
  wave_reduce(s, c, m);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) {
    ws[3 * w] = s;
    ws[3 * w + 1] = c;
    ws[3 * w + 2] = m;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < (int)(blockDim.x >> 6); ++k) merge3(s, c, m, ws[3 * k], ws[3 * k + 1], ws[3 * k + 2]);
  }
}

// Ghost state across a non-periodic side.
__device__ __forceinline__ void wall_ghost(const double* In, int normal, double* G) {
#pragma unroll
  for (int v = 0; v < NV; ++v) G[v] = In[v];
  G[normal] = -In[normal];
}

template <int TW>
__global__ void __launch_bounds__(Tile<TW>::NT)
k_rhs(const double* __restrict__ U, double* __restrict__ dU, Geometry g, Phys ph, GhostTime gt,
      int tilesPerRow) {
  constexpr int NT = Tile<TW>::NT, NXI = Tile<TW>::NXI, NYI = Tile<TW>::NYI;
  __shared__ double sU[NV][NT];
  __shared__ double sF[NV][NT];
  __shared__ double sG[NV][NT];
  __shared__ double xFs[NV][NXI], xFl[NV][NXI], xFr[NV][NXI];
  __shared__ double xhs[NXI], xhl[NXI], xhr[NXI];
  __shared__ double yFsB[NV][NYI], yFrB[NV][NYI], yhsB[NYI], yhrB[NYI];
  __shared__ double yFsT[NV][NYI], yFlT[NV][NYI], yhsT[NYI], yhlT[NYI];

  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int ey = tile / tilesPerRow;
  const int ex0 = (tile - ey * tilesPerRow) * TW;
  const int nW = min(TW, g.Nx - ex0);
  const int nNodes = NPP * nW;
  const int t = threadIdx.x;
  const long long Nd = g.Nd;
  const long long gbase = ((long long)ey * g.Nx + ex0) * NPP;

  // ---- phase 0: nodal state and fluxes (sgn2d.cpp:188-196) -----------------
  double Un[NV] = {0.0, 0.0, 0.0, 0.0, 0.0};
  Prim q{0.0, 0.0, 0.0, 0.0};
  double Hn = 0.0;
  if (t < nNodes) {
#pragma unroll
    for (int v = 0; v < NV; ++v) Un[v] = U[(long long)v * Nd + gbase + t];
    Hn = g.Hnod[gbase + t];
    q = prims(Un);
    double F[NV], G[NV];
    flux_x(Un, q, Hn, ph, F);
    flux_y(Un, q, Hn, ph, G);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      sU[v][t] = Un[v];
      sF[v][t] = F[v];
      sG[v][t] = G[v];
    }
  }
  __syncthreads();

  // ---- phase 1: interface fluxes (sgn2d.cpp:198-239) -----------------------
  const int nXI = NP * (nW + 1);
  if (t < nXI) {
    const int i = t / NP, b = t - NP * i;
    const int ex = ex0 + i;                   // this interface is the left edge of column ex
    double UL[NV], UR[NV];
    bool ghostL = false, ghostR = false;
    if (i < nW) {
#pragma unroll
      for (int v = 0; v < NV; ++v) UR[v] = sU[v][i * NPP + NP * b] + 0.0;
    } else if (ex < g.Nx) {
      load_face(U, Nd, nidx(g, ex, ey, 0, b), UR);
    } else if (g.bc[1] == 0) {
      load_face(U, Nd, nidx(g, 0, ey, 0, b), UR);
    } else {
      ghostR = true;
    }
    if (i > 0) {
#pragma unroll
      for (int v = 0; v < NV; ++v) UL[v] = sU[v][(i - 1) * NPP + (NP - 1) + NP * b] + 0.0;
    } else if (ex > 0) {
      load_face(U, Nd, nidx(g, ex - 1, ey, NP - 1, b), UL);
    } else if (g.bc[0] == 0) {
      load_face(U, Nd, nidx(g, g.Nx - 1, ey, NP - 1, b), UL);
    } else {
      ghostL = true;
    }
    if (ghostL) {
      if (g.bc[0] == 1) {
        wall_ghost(UR, IHU, UL);
      } else {
        const double* c = g.inflow + ((long long)ey * NP + b) * (NV * 3);
#pragma unroll
        for (int v = 0; v < NV; ++v) UL[v] = (c[3 * v] + c[3 * v + 1] * gt.s) + c[3 * v + 2] * gt.c;
      }
    }
    if (ghostR) wall_ghost(UL, IHU, UR);
    const double Hf = g.HfX[((long long)ey * (g.Nx + 1) + ex) * NP + b];
    double Fs[NV], FL[NV], FR[NV];
    interface_flux<0>(UL, UR, Hf, ph, Fs, FL, FR);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      xFs[v][t] = Fs[v];
      xFl[v][t] = FL[v];
      xFr[v][t] = FR[v];
    }
    xhs[t] = 0.5 * (UL[IH] + UR[IH]);
    xhl[t] = UL[IH];
    xhr[t] = UR[IH];
  } else if (t < nXI + 2 * NP * nW) {
    const int r2 = t - nXI;
    const int side = r2 / (NP * nW);          // 0 bottom edge, 1 top edge
    const int r = r2 - side * NP * nW;
    const int j = r / NP, a = r - NP * j;
    const int ex = ex0 + j;
    double UL[NV], UR[NV];
    if (side == 0) {
#pragma unroll
      for (int v = 0; v < NV; ++v) UR[v] = sU[v][j * NPP + a] + 0.0;
      if (ey > 0) load_face(U, Nd, nidx(g, ex, ey - 1, a, NP - 1), UL);
      else if (g.bc[2] == 0) load_face(U, Nd, nidx(g, ex, g.Ny - 1, a, NP - 1), UL);
      else wall_ghost(UR, IHV, UL);
      const double Hf = g.HfY[((long long)ey * g.Nx + ex) * NP + a];
      double Fs[NV], FL[NV], FR[NV];
      interface_flux<1>(UL, UR, Hf, ph, Fs, FL, FR);
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        yFsB[v][r] = Fs[v];
        yFrB[v][r] = FR[v];
      }
      yhsB[r] = 0.5 * (UL[IH] + UR[IH]);
      yhrB[r] = UR[IH];
    } else {
#pragma unroll
      for (int v = 0; v < NV; ++v) UL[v] = sU[v][j * NPP + a + NP * (NP - 1)] + 0.0;
      if (ey + 1 < g.Ny) load_face(U, Nd, nidx(g, ex, ey + 1, a, 0), UR);
      else if (g.bc[3] == 0) load_face(U, Nd, nidx(g, ex, 0, a, 0), UR);
      else wall_ghost(UL, IHV, UR);
      const double Hf = g.HfY[((long long)(ey + 1) * g.Nx + ex) * NP + a];
      double Fs[NV], FL[NV], FR[NV];
      interface_flux<1>(UL, UR, Hf, ph, Fs, FL, FR);
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        yFsT[v][r] = Fs[v];
        yFlT[v][r] = FL[v];
      }
      yhsT[r] = 0.5 * (UL[IH] + UR[IH]);
      yhlT[r] = UL[IH];
    }
  }
  __syncthreads();

  // ---- phase 2: FR lift and assembly (sgn2d.cpp:241-288) -------------------
  if (t < nNodes) {
    const int j = t / NPP, loc = t - NPP * j;
    const int b = loc / NP, a = loc - NP * b;
    const OpTables* T = g.ops;
    double Da[NP], Db[NP];
#pragma unroll
    for (int k = 0; k < NP; ++k) { Da[k] = T->D[a * NP + k]; Db[k] = T->D[b * NP + k]; }
    const double gLa = T->gLp[a], gRa = T->gRp[a], gLb = T->gLp[b], gRb = T->gRp[b];
    const int ixL = j * NP + b, ixR = (j + 1) * NP + b, iy = j * NP + a;
    const int rowx = j * NPP + NP * b, coly = j * NPP + a;
    double out[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      double dfx = 0.0, dgy = 0.0;
#pragma unroll
      for (int k = 0; k < NP; ++k) {
        dfx = dfx + Da[k] * sF[v][rowx + k];
        dgy = dgy + Db[k] * sG[v][coly + NP * k];
      }
      const double cx = (xFs[v][ixL] - xFr[v][ixL]) * gLa + (xFs[v][ixR] - xFl[v][ixR]) * gRa;
      const double cy = (yFsB[v][iy] - yFrB[v][iy]) * gLb + (yFsT[v][iy] - yFlT[v][iy]) * gRb;
      const double dF = (dfx + cx) / g.Jx;
      const double dG = (dgy + cy) / g.Jy;
      out[v] = -dF - dG;
    }
    double dhx = 0.0, dhy = 0.0;
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      dhx = dhx + Da[k] * sU[IH][rowx + k];
      dhy = dhy + Db[k] * sU[IH][coly + NP * k];
    }
    dhx = dhx + ((xhs[ixL] - xhr[ixL]) * gLa + (xhs[ixR] - xhl[ixR]) * gRa);
    dhy = dhy + ((yhsB[iy] - yhrB[iy]) * gLb + (yhsT[iy] - yhlT[iy]) * gRb);
    const double hx = dhx / g.Jx, hy = dhy / g.Jy;
    // ncpX / ncpY (sgn_flux2d.h:150-161): only the hp entry is non-zero, and
    // subtracting the zero entries leaves the other sums unchanged
    const double Bx = ph.mc2 * q.u * hx;
    const double By = ph.mc2 * q.v * hy;
    double S[NV];
    source(Un, q, Hn, g.Hx[gbase + t], g.Hy[gbase + t], ph, S);
    out[IHP] = out[IHP] - Bx - By;
#pragma unroll
    for (int v = 0; v < NV; ++v) dU[(long long)v * Nd + gbase + t] = out[v] + S[v];
  }
}

// ---- RHS, row sweep ---------------------------------------------------------
//
// A workgroup owns a strip of TW element columns and a chunk of `rows`
// element rows and walks up the chunk one element row r per iteration:
//   A  the row's nodes: stage input, primitives, nodal F and G, source -> LDS
//      / registers. Node operands are loaded two rows ahead: row r + 1 has
//      landed, and its bottom faces go to LDS too (with the halo nodes of the
//      strip's outer x lines); row r + 2's loads are issued here.
//   B  interface items: the TW+1 x-interface lines of row r, and the
//      y-interface line r+1 on top of the row (the line at its bottom was
//      done in the previous iteration, or before the loop). A y-interface is
//      the x-interface arithmetic applied to the states with hu and hv
//      exchanged (fluxY(U) is fluxX of the exchanged state with the hu and hv
//      components exchanged back, and |v| is the exchanged |u|), so all items
//      follow one code path. Each interface stores the flux jumps
//      F* - F(left/lower state) and F* - F(right/upper state) and the depth
//      jumps h* - h, which are the jumps the reference forms for each of the
//      two elements (sgn2d.cpp:251-257, :268-275); y lines are double-buffered.
//   C  nodes: the complete RHS of row r (and, in the candidate stage, its
//      scaled embedded error).
// Every y-interface is evaluated once; the stage input is read once per chunk,
// plus the faces of the rows below and above the chunk and the x-halo nodes.
//
// What bounds it: the stage launches, their traffic (at 1024x512 stage 2 moves
// 2.3 GB, stage 3 3.3, k4 2.6, all at 5.1 to 5.25 TB/s; a large copy reaches
// 4.8); the plain launch, vector and LDS instructions (each 70 % busy: 640 and 80
// per wave and row, three waves per SIMD); small grids, a workgroup's pace (2.7
// to 3.2 us a row alone on its compute unit, 6 us around them). Hence no branch
// around a global access, no face loaded twice, quotients without a branch each,
// and no vector instruction spent on an address. On 1024x512, per launch, before
// and after these (one MI355X, both builds in turn): plain 0.409 -> 0.348 ms,
// stage 2 0.549 -> 0.436, stage 3 0.725 -> 0.640, k4 0.628 -> 0.505; with what
// is noted further down 0.340, 0.435, 0.631 and 0.496.
template <int TW>
struct Sweep {
  static constexpr int NT = ((NPP * TW + 63) / 64) * 64;
  static constexpr int NXI = NP * (TW + 1);   // x-interface nodes per row
  static constexpr int NYI = NP * TW;         // y-interface nodes per line
  static_assert(2 * (NXI + NYI) <= NT, "two lanes per interface node");
};

// kCand of a step that takes no error norm: without the embedded sum (a build of
// its own: a test of zOut in kCand costs the adaptive step's launch 0.5 %)
constexpr int kCandOnly = 4;
constexpr bool is_cand(int mode) { return mode == kCand || mode == kCandOnly; }

// Operands of the stage input at one node (5 variables each): u, and the
// increment k of u + a*k in the modes that have one.
template <int MODE>
struct StageRaw {
  static constexpr bool kHasK = MODE == kAxpy || is_cand(MODE);
  double u[NV], k[kHasK ? NV : 1];
};
// Per-node operands beyond the stage input: kCand: x0 = kc; kErr: x0 = u0,
// x1 = z. Faces and halos never need them.
template <int MODE>
struct NodeExtra {
  double x0[(is_cand(MODE) || MODE == kErr) ? NV : 1], x1[MODE == kErr ? NV : 1];
};

// The launch's arguments: its kernel's own, or one entry of a batch's table.
typedef ConstArgs<BatchMember> SweepArgs;

template <int MODE>
__device__ __forceinline__ void stage_load(SweepArgs A, size_t first, size_t plane, unsigned off,
                                           StageRaw<MODE>& R) {
  load_vars(A->sa.u, first, plane, off, R.u);
  if (StageRaw<MODE>::kHasK) load_vars(A->sa.k1, first, plane, off, R.k);
}

template <int MODE>
__device__ __forceinline__ void extra_load(SweepArgs A, size_t first, size_t plane, unsigned off,
                                           NodeExtra<MODE>& E) {
  if (is_cand(MODE) || MODE == kErr) load_vars(is_cand(MODE) ? A->sa.kc : A->sa.u0, first, plane, off, E.x0);
  if (MODE == kErr) load_vars(A->sa.z, first, plane, off, E.x1);
}

// rk.cpp:100, :102: the stage input u + (c dt) k from its operands (a = c dt)
template <int MODE>
__device__ __forceinline__ void stage_combine(const StageRaw<MODE>& R, double a, double* W) {
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    if (StageRaw<MODE>::kHasK) W[v] = R.u[v] + a * R.k[v];
    else W[v] = R.u[v];
  }
}

// a face's state: the stage input + 0.0
template <int MODE>
__device__ __forceinline__ void stage_combine_face(const StageRaw<MODE>& R, double a, double* W) {
  stage_combine<MODE>(R, a, W);
#pragma unroll
  for (int v = 0; v < NV; ++v) W[v] = W[v] + 0.0;
}

// The primitives of prims() by one refined reciprocal of h for the four
// quotients where h and the four dividends are in the range of DivBy; else, on
// some lane of the wave, by IEEE division for the wave. Same bits.
__device__ __forceinline__ Prim prims_shared(const double* U) {
  const DivBy d = make_div_by(U[IH], __builtin_amdgcn_rcp(U[IH]));
  Prim q;
  q.u = d.quotient(U[IHU]);
  q.v = d.quotient(U[IHV]);
  q.w = d.quotient(U[IHW]);
  q.p = d.quotient(U[IHP]);
  const double big = fmax(fmax(fabs(U[IHU]), fabs(U[IHV])), fmax(fabs(U[IHW]), fabs(U[IHP])));
  const int bad = (int)!div_by_ok(U[IH]) | (int)!(big <= 0x1p+800) |
                  (int)div_needs_exact(U[IHU]) | (int)div_needs_exact(U[IHV]) |
                  (int)div_needs_exact(U[IHW]) | (int)div_needs_exact(U[IHP]);
  if (__builtin_expect(wave_any(bad), 0)) q = prims(U);
  return q;
}

// LDS of one workgroup. A node's record holds h, hu, hv, hw, hp, the fluxes
// F[1..4] and G[1..4] (F[0] is hu and G[0] is hv) and, with HXR, the still
// depth; every operand of phase C is then an immediate offset from the lane's
// row, its column or its own record. 13 and 15 doubles are odd multiples of a
// bank pair, so neither the records' writes nor the row and column reads
// conflict. Interface jumps: F* - F(side) and, as a sixth entry, h* - h(side)
// (side 0 = left / lower, 1 = right / upper), for the x lines of the row and
// the y lines below and above it (by line parity).
template <int TW, bool HXR>
struct SweepLds {
  static constexpr int kRec = HXR ? 15 : 13;
  static constexpr int kF = 4, kG = 8, kH = 13;      // record offsets: F[v] at kF + v, v >= 1
  static constexpr int kJ = NP * (TW + 1);           // interface nodes of one jump plane
  static constexpr int kJSide = (NV + 1) * kJ, kJLine = 2 * kJSide;
  double node[NPP * TW * kRec];
  double jump[3 * kJLine];                           // x lines, even y line, odd y line
  double face[(NP * TW + 2 * NP) * NV];              // bottom faces of the row above, halo nodes
  double tab[NP][NP + 2];                            // per node index a: D[a][.], gL'[a], gR'[a]
  static __device__ __forceinline__ constexpr int offF(int v) { return v == IH ? IHU : kF + v; }
  static __device__ __forceinline__ constexpr int offG(int v) { return v == IH ? IHV : kG + v; }
};

// One workgroup's strip x chunk `tile` of one grid (the body of the plain and
// the batched launches).
template <int TW, int MODE, int WAVES, bool KEEP = false, bool HXR = false>
__device__ __forceinline__ void sweep_tile(SweepArgs A, int tile, int rows, int base) {
  using L = SweepLds<TW, HXR>;
  constexpr int kRec = L::kRec, kJ = L::kJ, kJSide = L::kJSide, kJLine = L::kJLine;
  // the row sweep runs without the Manning friction term (the launchers
  // refuse it; solvers with friction use the element-row tiles), so its
  // branch is compiled out
  Phys ph{A->ph.g, A->ph.c, A->ph.gamma, 0.0, A->ph.halfg, A->ph.c2, A->ph.mc2, A->ph.m2c2};
  const ConstDiv divX{A->g.dx.b, A->g.dx.rh, A->g.dx.rl, 1}, divY{A->g.dy.b, A->g.dy.rh, A->g.dy.rl, 1};
  const double stA = A->sa.a, stDt = A->sa.dt, atol = A->sa.atol, rtol = A->sa.rtol;
  const int bcL = A->g.bc[0], bcR = A->g.bc[1], bcB = A->g.bc[2], bcT = A->g.bc[3];
  const int nStrips = A->nStrips, Nx = A->g.Nx, Ny = A->g.Ny;
  __shared__ L lds;

  // The lane's rows of D and weights are kept in registers by the plain launch,
  // which LDS reads bound (2000x1000 1302 -> 1256 us, 1024x512 350 -> 343); the
  // stage launches wait for memory and gain nothing from that, but from fetching
  // their first rows before anything else: the latency is then behind the rest of
  // the preparation (387x191 stage 3 103.9 -> 102.5 us, 1024x512 635 -> 631). The
  // plain launch, which waits for its tables, loses by it (8x6 6.14 -> 6.25 us).
  constexpr bool kTabRegs = MODE == kPlain;
  if (kTabRegs && threadIdx.x < NP) {
    const OpTables* const T = A->g.ops;
    double* const to = lds.tab[threadIdx.x];
#pragma unroll
    for (int k = 0; k < NP; ++k) to[k] = T->D[threadIdx.x * NP + k];
    to[NP] = T->gLp[threadIdx.x];
    to[NP + 1] = T->gRp[threadIdx.x];
  }

  const int chunk = __builtin_amdgcn_readfirstlane(tile / nStrips);
  const int strip = tile - chunk * nStrips, ex0 = strip * TW;
  const int nW = min(TW, Nx - ex0);
  const int ey0 = base + chunk * rows;
  const int ey1 = min(Ny, ey0 + rows);
  const int nNodes = NPP * nW;
  const int t = threadIdx.x;
  const size_t plane0 = (size_t)A->g.Nd * sizeof(double);
  const unsigned rowBytes = (unsigned)Nx * (NPP * 8u);   // a plane has at most 2^31 bytes

  // Every lane has an item in every phase, so that no branch stands around a
  // global access: the compiler then knows how many accesses are in flight at
  // each wait and waits for the oldest only. Lanes beyond the strip's items
  // repeat item 0, with the same values at the same addresses.
  //
  // node work item: node (a, b) of element j of the strip
  const bool isNode = t < nNodes;
  const int tn = isNode ? t : 0;
  const int j = tn / NPP, loc = tn - NPP * j;
  const int b = loc / NP, a = loc - NP * b;
  unsigned t8 = (unsigned)tn * 8u;                       // the node
  unsigned f8 = (unsigned)(j * NPP + a) * 8u;            // the bottom face of its column
  const bool wallTop = bcT != 0;
  // The nodes' operands, two rows ahead: while row r is worked on, row r + 1
  // has landed (its bottom faces are the upper side of the y line between the
  // two, so no lane loads a face a second time) and row r + 2 is in flight.
  // Above the chunk only the bottom faces are needed (from the first row
  // across a periodic top side), so every lane takes its column's; with
  // nothing to load, row r's first nodes stand in.
  struct Node {
    StageRaw<MODE> s;
    double H, Hx, Hy;
    __device__ __forceinline__ void take(const Node& o) {
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        move_to(s.u[v], o.s.u[v]);
        if (StageRaw<MODE>::kHasK) move_to(s.k[v], o.s.k[v]);
      }
      move_to(H, o.H);
      if (!HXR) {
        move_to(Hx, o.Hx);
        move_to(Hy, o.Hy);
      }
    }
  };
  Node cur, nxt;
  const unsigned row0 = (unsigned)ex0 * (NPP * 8u);
  unsigned rowOff = row0 + (unsigned)ey0 * rowBytes;     // row r's first node (bytes)
  auto node_load = [&](SweepArgs R, int r, int ahead, size_t plane, Node& n) {
    int to = r + ahead;
    const bool full = to < ey1;
    to = to > ey1 ? r : to;
    to = to == Ny ? (wallTop ? r : 0) : to;
    const unsigned first =
        __builtin_amdgcn_readfirstlane((int)(row0 + (unsigned)to * rowBytes));
    const unsigned off = full ? t8 : f8;
    stage_load<MODE>(R, first, plane, off, n.s);
    n.H = load_at(global_at(R->g.Hnod, first), off);
    if (!HXR) {
      n.Hx = load_at(global_at(R->g.Hx, first), off);
      n.Hy = load_at(global_at(R->g.Hy, first), off);
    }
  };
  static_assert(offsetof(OpTables, gLp) == NPP * 8 && offsetof(OpTables, gRp) == (NPP + NP) * 8, "");
  const int te = threadIdx.x < NPP + 2 * NP ? threadIdx.x : 0;   // a table entry per lane
  double tabEntry = 0.0;
  if (!kTabRegs) {
    node_load(A, ey0, 0, plane0, cur);
    node_load(A, ey0, 1, plane0, nxt);
    tabEntry = ((const GlobalDouble*)A->g.ops)[te];
  }
  // Interface half-items: two lanes per interface node, lane 2k + side
  // taking one side (0 = left / lower, 1 = right / upper) of interface k.
  // Items 0 .. nX - 1 are the x-interface nodes of the row (k = i NP + bb:
  // line i on the left edge of strip column i, node bb); the next NP nW items
  // the y-interface nodes of the line above the row (k = nX + jj NP + aa).
  // Each lane evaluates its own side (primitives, one-sided flux, wave speed)
  // and the pair exchanges them with lane permutes, so the interface work is
  // spread over every wave of the workgroup.
  const int nX = NP * (nW + 1);
  const int side = t & 1, kk = (t >> 1) < nX + NP * nW ? t >> 1 : 0;
  const bool isX = kk < nX, isY = !isX;
  const int xi = isX ? kk / NP : 0, xb = isX ? kk - NP * xi : 0;
  const int ky = isY ? kk - nX : 0;
  const int jj = ky / NP, aa = ky - NP * jj;
  // The side's state: a node of the row in LDS, the bottom face of the row
  // above for the upper side of a y line (gY, in LDS too), or the halo node of
  // the strip's outer x lines (gX, a global node). At a wall it is the other
  // side's node, mirrored. The inflow side's ghost is data.
  const bool outer = isX && (side == 0 ? xi == 0 : xi == nW);
  const bool gX = outer && (side == 0 ? ex0 > 0 || bcL == 0 : ex0 + nW < Nx || bcR == 0);
  const bool gY = isY && side == 1;
  const bool inflow = outer && side == 0 && ex0 == 0 && bcL == 2;
  int src;
  if (isX) {
    const int col = outer ? (side == 0 ? 0 : nW - 1) : (side == 0 ? xi - 1 : xi);
    const bool high = outer ? side == 1 : side == 0;
    src = col * NPP + (high ? NP - 1 : 0) + NP * xb;
  } else {
    src = jj * NPP + aa + NP * (NP - 1);
  }
  int mirror = outer && !gX ? (int)0x80000000 : 0;
  LdsDouble* sSrc = (LdsDouble*)lds.node + src * kRec;
  LdsDouble* sHalo = (LdsDouble*)lds.face + (NP * TW + NP * side + xb) * NV;
  LdsDouble* sFrom = gX ? sHalo : gY ? (LdsDouble*)lds.face + ky * NV : sSrc;
  // the global node of the gX lanes (byte offset), for the row whose
  // interfaces are next (the others: the strip's first node); it moves up one
  // element row with r
  unsigned fOff = node_of(Nx, ex0, ey0, 0, 0) * 8u;
  if (gX) {
    const int col = side == 0 ? (ex0 > 0 ? ex0 - 1 : Nx - 1) : (ex0 + nW < Nx ? ex0 + nW : 0);
    fOff = node_of(Nx, col, ey0, side == 0 ? NP - 1 : 0, xb) * 8u;
  }
  // face depth of the lane's line of row r, and its step to the next row
  const GlobalDouble* pHf =
      isX ? (const GlobalDouble*)A->g.HfX + ((size_t)ey0 * (Nx + 1) + ex0 + xi) * NP + xb
          : (const GlobalDouble*)A->g.HfY + ((size_t)(ey0 + 1) * Nx + ex0 + jj) * NP + aa;
  const unsigned hfStep = (unsigned)(Nx + (isX ? 1 : 0)) * NP;
  LdsDouble* sJ = (LdsDouble*)lds.jump + (isX ? 0 : kJLine) + side * kJSide + (isX ? kk : ky);

  // One interface node evaluated by a lane pair. W is this lane's side's
  // state in the interface frame (a y interface has hu and hv exchanged:
  // fluxY(U) is fluxX of the exchanged state with hu and hv of the result
  // exchanged back, and |v| is the exchanged |u|). Stores this side's flux
  // jump F* - F(W) and depth jump h* - h(W), with the Rusanov flux of
  // sgn_flux2d.h:169-179: F* = 0.5 (FL + FR) - 0.5 max(sL, sR) (UR - UL).
  // Both lanes take the other's values by one swap: UR - UL is other - own on
  // the lower side and its negative on the upper one, which the sign of hl
  // carries (where the difference is zero, F* - F is the same +0 either way).
  auto half_iface = [&](const double* W, double Hf, LdsDouble* to) {
    const Prim q = prims_shared(W);
    double F[NV];
    flux_x(W, q, Hf, ph, F);
    const double so = fabs(q.u) + signal_speed(W[IH], q, ph);
    const double lam = fmax(so, lane_swap(so));
    const double hl = flip_sign(0.5 * lam, side << 31);
    double jf[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const double o = lane_swap(W[v]);
      // FL + FR in either lane order (addition commutes exactly)
      const double Fs = 0.5 * (F[v] + lane_swap(F[v])) - hl * (o - W[v]);
      jf[v] = Fs - F[v];
      if (v == IH) to[NV * kJ] = 0.5 * (W[IH] + o) - W[IH];
    }
    to[IH * kJ] = jf[IH];
    to[IHU * kJ] = isY ? jf[IHV] : jf[IHU];
    to[IHV * kJ] = isY ? jf[IHU] : jf[IHV];
    to[IHW * kJ] = jf[IHW];
    to[IHP * kJ] = jf[IHP];
  };
  auto to_frame = [&](double* W) {             // exchange hu, hv on y lanes
    const double u_ = W[IHU], v_ = W[IHV];
    W[IHU] = isY ? v_ : u_;
    W[IHV] = isY ? u_ : v_;
  };

  // The interface lanes' global operands: the halo nodes and the face depths.
  // Those of row r + 1 are issued at the start of phase C of row r, so phase C
  // and the next phase A cover their latency.
  StageRaw<MODE> fR;
  double fH;
  auto face_load = [&](SweepArgs R, size_t plane) {
    stage_load<MODE>(R, 0, plane, fOff, fR);
    fH = *pHf;
  };

  if (kTabRegs) {
    node_load(A, ey0, 0, plane0, cur);
    node_load(A, ey0, 1, plane0, nxt);
  }
  face_load(A, plane0);
  if (!kTabRegs)
    (&lds.tab[0][0])[te < NPP ? te / NP * (NP + 2) + te % NP
                              : (te - NPP) % NP * (NP + 2) + NP + (te - NPP) / NP] = tabEntry;
  // the y line at the bottom of the chunk, both sides from global memory (the
  // bottom wall's ghost mirrors the upper side)
  if (isY) {
    const bool below = ey0 > 0 || bcB == 0;
    const bool lower = side == 0 && below;
    const unsigned n = lower ? node_of(Nx, ex0 + jj, ey0 > 0 ? ey0 - 1 : Ny - 1, aa, NP - 1)
                             : node_of(Nx, ex0 + jj, ey0, aa, 0);
    StageRaw<MODE> R;
    stage_load<MODE>(A, 0, plane0, n * 8u, R);
    double W[NV];
    stage_combine_face<MODE>(R, stA, W);
    to_frame(W);
    if (side == 0 && !below) W[IHU] = -W[IHU];
    half_iface(W, ((const GlobalDouble*)A->g.HfY)[((size_t)ey0 * Nx + ex0 + jj) * NP + aa],
               sJ + (ey0 & 1) * kJLine);
  }
  // a Jacobian outside the branch-free quotient's range: always IEEE division
  const bool never_fast = !A->g.dx.fast || !A->g.dy.fast;
  // scaled embedded error of this work-item's nodes (kErr)
  double eS = 0.0, eC = 0.0, eM = 0.0;

  LdsDouble* sOwn = (LdsDouble*)lds.node + tn * kRec;
  LdsDouble* sRow = (LdsDouble*)lds.node + (j * NPP + NP * b) * kRec;
  LdsDouble* sCol = (LdsDouble*)lds.node + (j * NPP + a) * kRec;
  LdsDouble* sBot = (LdsDouble*)lds.face + (j * NP + a) * NV;
  LdsDouble* sJx = (LdsDouble*)lds.jump + j * NP + b;   // the line on the element's left
  LdsDouble* sJy = (LdsDouble*)lds.jump + kJLine + j * NP + a;
  LdsDouble* sTa = (LdsDouble*)lds.tab[a];
  LdsDouble* sTb = (LdsDouble*)lds.tab[b];

  // the lane's rows of D and weights
  double Da[NP], Db[NP], gLa, gRa, gLb, gRb;
  auto load_tab = [&](auto* ta, auto* tb) {
#pragma unroll
    for (int k = 0; k < NP; ++k) { Da[k] = ta[k]; Db[k] = tb[k]; }
    gLa = ta[NP], gRa = ta[NP + 1], gLb = tb[NP], gRb = tb[NP + 1];
  };
  if (kTabRegs) {
    __syncthreads();
    load_tab(sTa, sTb);
  }

  auto row = [&](int r) {
    // opaque in every row: the planes of all operands kept across rows would
    // exceed the scalar registers, and a lane offset folded into them would
    // make the addresses vectors
    size_t plane = plane0;
    __asm__ volatile("" : "+s"(plane));
    __asm__ volatile("" : "+v"(t8));
    __asm__ volatile("" : "+v"(f8));
    // likewise the lane's places in LDS, whose offset forms the rows would
    // otherwise share through registers of their own
    for (LdsDouble** q : {&sOwn, &sRow, &sCol, &sBot, &sJx, &sJy, &sTa, &sTb, &sFrom, &sHalo, &sJ})
      __asm__ volatile("" : "+v"(*q));
    // ---- A ---------------------------------------------------------------------
    double S[NV], qu, qv, qw;
    SrcPart sp;
    // row r's operands that phase C needs again: the stage operands and those
    // of the candidate and the error, which nothing needs before phase C
    NodeExtra<MODE> ext;
    extra_load<MODE>(opaque(A), rowOff, plane, t8, ext);
    const StageRaw<MODE> own = cur.s;
    {
      double Un[NV];
      stage_combine<MODE>(own, stA, Un);
      double* const yOut = KEEP ? opaque(A)->sa.yOut : nullptr;
      if (KEEP && yOut) {
        // the stage input, kept for a later reverse sweep
        GlobalByte* p = global_at(yOut, rowOff);
#pragma unroll
        for (int v = 0; v < NV; ++v) {
          store_at(p, t8, Un[v]);
          p += plane;
        }
      }
      const double Hn = cur.H;
      const Prim q = prims_shared(Un);
      qu = q.u;
      qv = q.v;
      if (HXR) {
        // the gradient terms wait for phase C
        sp = source_part(Un, q, Hn, ph);
        qw = q.w;
        sOwn[L::kH] = Hn;
      } else {
        source(Un, q, Hn, cur.Hx, cur.Hy, ph, S);
      }
      double F[NV], G[NV];
      flux_x(Un, q, Hn, ph, F);
      flux_y(Un, q, Hn, ph, G);
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        sOwn[v] = Un[v];
        if (v > IH) {
          sOwn[L::offF(v)] = F[v];
          sOwn[L::offG(v)] = G[v];
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (b == 0) {
      // the bottom faces of row r + 1
      double W[NV];
      stage_combine_face<MODE>(nxt.s, stA, W);
#pragma unroll
      for (int v = 0; v < NV; ++v) sBot[v] = W[v];
    }
    if (gX) {
      double W[NV];
      stage_combine_face<MODE>(fR, stA, W);
#pragma unroll
      for (int v = 0; v < NV; ++v) sHalo[v] = W[v];
    }
    // Row r + 1's operands into row r's registers, row r + 2's loads into
    // theirs. The moves are written out: left to itself the compiler moves at
    // the end of the row, and there waits for the loads in flight.
    __builtin_amdgcn_sched_barrier(0);
    cur.take(nxt);
    node_load(opaque(A), r, 2, plane, nxt);
    row_sync();

    // ---- B ---------------------------------------------------------------------
    {
      if (wallTop && r + 1 == Ny && gY) {
        sFrom = sSrc;                            // the top wall mirrors the row's own nodes
        mirror = (int)0x80000000;
      }
      double W[NV];
#pragma unroll
      for (int v = 0; v < NV; ++v) W[v] = sFrom[v] + 0.0;
      to_frame(W);
      W[IHU] = flip_sign(W[IHU], mirror);
      if (inflow) {
        const SweepArgs R = opaque(A);
        const GlobalDouble* c = (const GlobalDouble*)R->g.inflow + ((size_t)r * NP + xb) * (NV * 3);
#pragma unroll
        for (int v = 0; v < NV; ++v)
          W[v] = (c[3 * v] + c[3 * v + 1] * R->gt.s) + c[3 * v + 2] * R->gt.c;
      }
      half_iface(W, fH, isX ? sJ : sJ + ((r + 1) & 1) * kJLine);
    }
    row_sync();

    // ---- C: dU of row r ---------------------------------------------------------
    if (r + 1 < ey1) {
      fOff += rowBytes;
      pHf += hfStep;
    }
    face_load(opaque(A), plane);
    __builtin_amdgcn_sched_barrier(0);
    {
      if (!kTabRegs) load_tab(sTa, sTb);
      LdsDouble* const jB = sJy + (r & 1) * kJLine;         // the line below the row
      LdsDouble* const jT = sJy + ((r + 1) & 1) * kJLine;   // and the one above it
      // The dividends of one pair of quotients, along x and along y: D . f of
      // the records' entry `fx` / `fy` plus the lift of the jump plane v. The
      // reference's sums start from 0.0; here they start from the first
      // product, which differs only in a zero's sign, and div_unchecked takes
      // both zeros to +0.
      auto sums = [&](int fx, int fy, int v, double& ax, double& ay) {
        double dx = Da[0] * sRow[fx], dy = Db[0] * sCol[fy];
#pragma unroll
        for (int k = 1; k < NP; ++k) {
          dx = dx + Da[k] * sRow[k * kRec + fx];
          dy = dy + Db[k] * sCol[NP * k * kRec + fy];
        }
        if (v < 0) { ax = dx; ay = dy; return; }
        ax = dx + (sJx[kJSide + v * kJ] * gLa + sJx[v * kJ + NP] * gRa);
        ay = dy + (jB[kJSide + v * kJ] * gLb + jT[v * kJ] * gRb);
      };
      double hx, hy;
      const SweepArgs R = opaque(A);
      auto finish = [&](int v, double k4, size_t pl) {
        auto put = [&](double* base, double x) { store_at(global_at(base, pl), t8, x); };
        if (is_cand(MODE)) {
          // rk.cpp:106-108 and the first three terms of :119-120 (k4 is k3 here)
          const double k1 = ext.x0[v], k2 = own.k[v];
          put(R->sa.uNew, own.u[v] + stDt * (2.0 / 9.0 * k1 + 1.0 / 3.0 * k2 + 4.0 / 9.0 * k4));
          if (MODE == kCand) put(R->sa.zOut, 7.0 / 24.0 * k1 + 0.25 * k2 + 1.0 / 3.0 * k4);
        } else if (!(MODE == kAxpy && KEEP) || R->dU) {
          put(R->dU, k4);
        }
        if (MODE == kAxpy && KEEP && R->sa.y3Out) {
          // the stage-3 input u + (3/4 dt) k2 of a recomputed step
          // (rk.cpp:104), formed as the elementwise combination forms it
          put(R->sa.y3Out, own.u[v] + R->sa.a3 * k4);
        }
        if (MODE == kErr) {
          // rk.cpp:119-129 for this entry
          const double u0 = ext.x0[v], un = sOwn[v];
          const double uEmb = u0 + stDt * (ext.x1[v] + 0.125 * k4);
          const double e = un - uEmb;
          const double au = fabs(u0), an = fabs(un);
          const double r_ = e / (atol + rtol * ((au < an) ? an : au));
          acc_add(eS, eC, r_ * r_);
          const double ar = fabs(r_);
          eM = (eM < ar) ? ar : eM;
        }
      };
      // A scheduling group: the quotients of the entries [e0, e1), -2 the
      // still-depth gradient (HXR), -1 the depth gradient, v >= 0 variable v,
      // by the branch-free sequence; then, where a lane of the wave has one
      // outside its range or not finite, by IEEE division (+ 0.0: the
      // reference's sums are never -0); then the variables' results.
      auto group = [&](auto e0_, auto e1_) {
        constexpr int e0 = decltype(e0_)::value, e1 = decltype(e1_)::value, n = e1 - e0;
        double ax[n], ay[n], qx[n], qy[n];
        int bad = never_fast;
#pragma unroll
        for (int i = 0; i < n; ++i) {
          const int v = e0 + i;
          if (v == -2) sums(L::kH, L::kH, -1, ax[i], ay[i]);
          else if (v == -1) sums(IH, IH, NV, ax[i], ay[i]);
          else sums(L::offF(v), L::offG(v), v, ax[i], ay[i]);
          qx[i] = div_unchecked(ax[i], divX);
          qy[i] = div_unchecked(ay[i], divY);
          bad |= (int)div_needs_exact(ax[i]) | (int)div_needs_exact(ay[i]) |
                 (int)!(fabs(qx[i] + qy[i]) < HUGE_VAL);
        }
        if (__builtin_expect(wave_any(bad), 0)) {
#pragma unroll
          for (int i = 0; i < n; ++i) {
            qx[i] = (ax[i] + 0.0) / divX.b;
            qy[i] = (ay[i] + 0.0) / divY.b;
          }
        }
#pragma unroll
        for (int i = 0; i < n; ++i) {
          const int v = e0 + i;
          if (v == -2) {
            // sgn2d.cpp:54-71: Hx, Hy = (D H) / J along the node's x and y lines
            source_rest(sp, qu, qv, qw, qx[i], qy[i], ph, S);
          } else if (v == -1) {
            hx = qx[i];
            hy = qy[i];
          } else {
            // the non-conservative products enter hp only (the others' are
            // zero, and subtracting zero changes no sum)
            double o = -qx[i] - qy[i];
            if (v == IHP) o = o - ph.mc2 * qu * hx - ph.mc2 * qv * hy;
            finish(v, o + S[v], rowOff + (size_t)v * plane);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      };
      // One entry per group: with two or more, the compiler hoists the LDS
      // operands of the later ones over the first and needs 30 to 70 registers
      // more, which costs a wave per SIMD.
      if (HXR) group(IntC<-2>{}, IntC<-1>{});
      group(IntC<-1>{}, IntC<0>{});
      group(IntC<0>{}, IntC<1>{});
      group(IntC<1>{}, IntC<2>{});
      group(IntC<2>{}, IntC<3>{});
      group(IntC<3>{}, IntC<4>{});
      group(IntC<4>{}, IntC<5>{});
    }
    row_sync();
    rowOff += rowBytes;
  };
  if (MODE != kErr) {
    for (int r = ey0; r < ey1; ++r) row(r);
    return;
  }
  // the norm's partials: one for every g.rows rows
  int done = ey0;
  for (long long at = (long long)(ey0 / A->g.rows) * nStrips + strip; done < ey1; at += nStrips) {
    const int to = min(ey1, done + A->g.rows);
    for (; done < to; ++done) row(done);
    if (!isNode) eS = eC = eM = 0.0;                     // node 0 counts once
    // fixed-order reduction over the workgroup (LDS of the last row reused)
    block_reduce(eS, eC, eM, lds.node);
    if (t == 0) {
      double* const part = A->sa.part + 3 * at;
      part[0] = eS;
      part[1] = eC;
      part[2] = eM;
    }
    eS = eC = eM = 0.0;
    row_sync();
  }
}

// The arguments are the kernel's only parameter, read where they lie.
template <int TW, int MODE, int WAVES, bool KEEP = false, bool HXR = false>
__global__ void __launch_bounds__(Sweep<TW>::NT, WAVES) k_rhs_sweep(BatchMember) {
  const SweepArgs A = (SweepArgs)__builtin_amdgcn_kernarg_segment_ptr();
  const int b = blockIdx.x, low = b - A->tallBlocks;
  int tile = xcd_tile(low, A->lowTiles), rows = A->rows, base = A->lowFrom;
  if (low < 0) {
    if (b >= A->tallTiles) return;           // (filling up)
    tile = xcd_tile(b, A->tallTiles);
    rows = A->tall;
    base = 0;
  }
  sweep_tile<TW, MODE, WAVES, KEEP, HXR>(A, tile, rows, base);
}

// Many grids in one launch: the workgroups of every member's tiles, one member
// after the other (tileStart[m] = first workgroup of member m, ascending, a
// multiple of the XCDs' number); each member keeps its own tile decomposition, so its error partials, and
// everything else, equal its own launch's.
template <int TW, int MODE, int WAVES, bool KEEP = false, bool HXR = false>
__global__ void __launch_bounds__(Sweep<TW>::NT, WAVES)
k_rhs_sweep_batch(const BatchMember* __restrict__ mem, const long long* __restrict__ tileStart,
                  int nMem) {
  const long long w = blockIdx.x;
  int lo = 0, hi = nMem - 1;                  // last member with tileStart <= w
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (tileStart[mid] <= w) lo = mid; else hi = mid - 1;
  }
  const SweepArgs M = const_entry(mem, lo);
  const int own = __builtin_amdgcn_readfirstlane((int)(w - tileStart[lo]));
  if (own >= M->nTiles) return;               // (filling up)
  sweep_tile<TW, MODE, WAVES, KEEP, HXR>(M, xcd_tile(own, M->nTiles), M->rows, 0);
}

// Hx, Hy at every node (sgn2d.cpp:54-71).
__global__ void __launch_bounds__(kThreads)
k_bathy_grad(const double* __restrict__ H, double* __restrict__ Hx, double* __restrict__ Hy,
             const OpTables* __restrict__ T, long long Nd, double Jx, double Jy) {
  const long long gn = (long long)blockIdx.x * kThreads + threadIdx.x;
  if (gn >= Nd) return;
  const long long e = gn / NPP;
  const int loc = (int)(gn - e * NPP);
  const int b = loc / NP, a = loc - NP * b;
  const double* He = H + e * NPP;
  double dHx = 0.0, dHy = 0.0;
#pragma unroll
  for (int k = 0; k < NP; ++k) {
    dHx = dHx + T->D[a * NP + k] * He[k + NP * b];
    dHy = dHy + T->D[b * NP + k] * He[a + NP * k];
  }
  Hx[gn] = dHx / Jx;
  Hy[gn] = dHy / Jy;
}

// Whether Hx, Hy hold (D Hnod) / J (sgn2d.cpp:54-71, the arithmetic of
// k_bathy_grad) bit for bit at every node: any difference sets *bad.
__global__ void __launch_bounds__(kThreads)
k_bathy_check(const double* __restrict__ H, const double* __restrict__ Hx,
              const double* __restrict__ Hy, const OpTables* __restrict__ T, long long Nd,
              double Jx, double Jy, int* bad) {
  const long long gn = (long long)blockIdx.x * kThreads + threadIdx.x;
  if (gn >= Nd) return;
  const long long e = gn / NPP;
  const int loc = (int)(gn - e * NPP);
  const int b = loc / NP, a = loc - NP * b;
  const double* He = H + e * NPP;
  double dHx = 0.0, dHy = 0.0;
#pragma unroll
  for (int k = 0; k < NP; ++k) {
    dHx = dHx + T->D[a * NP + k] * He[k + NP * b];
    dHy = dHy + T->D[b * NP + k] * He[a + NP * k];
  }
  if (__double_as_longlong(dHx / Jx) != __double_as_longlong(Hx[gn]) ||
      __double_as_longlong(dHy / Jy) != __double_as_longlong(Hy[gn]))
    atomicOr(bad, 1);
}

// ---- RK stage arithmetic (src/solver/rk.cpp) ----------------------------------

__global__ void __launch_bounds__(kThreads)
k_comb1(double* __restrict__ out, const double* __restrict__ u, double a1,
        const double* __restrict__ k1, size_t n) {
  const size_t stride = (size_t)gridDim.x * kThreads;
  for (size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += stride)
    out[i] = u[i] + a1 * k1[i];
}

__global__ void __launch_bounds__(kThreads)
k_bs3_update(double* __restrict__ out, const double* __restrict__ u, double dt,
             const double* __restrict__ k1, const double* __restrict__ k2,
             const double* __restrict__ k3, size_t n) {
  const size_t stride = (size_t)gridDim.x * kThreads;
  for (size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += stride)
    out[i] = u[i] + dt * (2.0 / 9.0 * k1[i] + 1.0 / 3.0 * k2[i] + 4.0 / 9.0 * k3[i]);
}

__global__ void __launch_bounds__(kThreads)
k_rk4_update(double* __restrict__ u, double dt, const double* __restrict__ k1,
             const double* __restrict__ k2, const double* __restrict__ k3,
             const double* __restrict__ k4, size_t n) {
  const size_t stride = (size_t)gridDim.x * kThreads;
  const double d6 = dt / 6.0;
  for (size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += stride)
    u[i] += d6 * (k1[i] + 2.0 * k2[i] + 2.0 * k3[i] + k4[i]);
}

// rk.cpp:118-131: r = (uNew - uEmb) / (atol + rtol*max(|u|, |uNew|)).
__global__ void __launch_bounds__(kThreads)
k_err_norm(const double* __restrict__ u, const double* __restrict__ uNew,
           const double* __restrict__ k1, const double* __restrict__ k2,
           const double* __restrict__ k3, const double* __restrict__ k4, double dt, double atol,
           double rtol, size_t n, double* __restrict__ part) {
  __shared__ double ws[3 * kThreads / 64];
  double s = 0.0, c = 0.0, m = 0.0;
  const size_t stride = (size_t)gridDim.x * kThreads;
  for (size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += stride) {
    const double uEmb =
        u[i] + dt * (7.0 / 24.0 * k1[i] + 0.25 * k2[i] + 1.0 / 3.0 * k3[i] + 0.125 * k4[i]);
    const double e = uNew[i] - uEmb;
    const double au = fabs(u[i]), an = fabs(uNew[i]);
    const double sc_ = atol + rtol * ((au < an) ? an : au);   // std::max(|u|, |uNew|)
    const double r = e / sc_;
    acc_add(s, c, r * r);
    const double ar = fabs(r);
    m = (m < ar) ? ar : m;                                     // std::max(errMax, |r|)
  }
  block_reduce(s, c, m, ws);
  if (threadIdx.x == 0) {
    part[3 * blockIdx.x] = s;
    part[3 * blockIdx.x + 1] = c;
    part[3 * blockIdx.x + 2] = m;
  }
}

// Second level: one block folds the nb partial triples in a fixed order.
// out[0] = sum, out[1] = max. Its time is that of its loads, one after the
// other where each waits for the last: eight triples a thread are on their way
// at once (13120 triples, of 1024x512: 25.3 -> 9.5 us; 832: 3.8 either way; twice
// the threads: 9.4, but 2 % of a 128x64 step).
constexpr int kFinish = 512;
__device__ __forceinline__ void finish_block(const double* __restrict__ part, int nb,
                                             double* __restrict__ out) {
  static_assert(kFinish == 8 * 64, "a tree of 8 waves");
  __shared__ double ws[kFinish / 64][3];
  constexpr int kAhead = 8;
  double s = 0.0, c = 0.0, m = 0.0;
  for (int i0 = threadIdx.x; i0 < nb; i0 += kAhead * kFinish) {
    double x[kAhead][3];
#pragma unroll
    for (int q = 0; q < kAhead; ++q) {
      const size_t i = (size_t)min(i0 + q * kFinish, nb - 1);
#pragma unroll
      for (int k = 0; k < 3; ++k) x[q][k] = part[3 * i + k];
    }
#pragma unroll
    for (int q = 0; q < kAhead; ++q) {
      if (i0 + q * kFinish < nb) {
        acc_add(s, c, x[q][0]);
        c = c + x[q][1];
        m = fmax(m, x[q][2]);
      }
    }
  }
  wave_reduce(s, c, m);
  if ((threadIdx.x & 63) == 0) {
    ws[threadIdx.x >> 6][0] = s;
    ws[threadIdx.x >> 6][1] = c;
    ws[threadIdx.x >> 6][2] = m;
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    // the waves' triples by a tree of their own (each half of the wave alike)
    const int w = threadIdx.x & (kFinish / 64 - 1);
    s = ws[w][0];
    c = ws[w][1];
    m = ws[w][2];
    wave_level<1>(s, c, m);
    wave_level<2>(s, c, m);
    wave_level<4>(s, c, m);
    if (threadIdx.x == 0) {
      out[0] = s + c;
      out[1] = m;
    }
  }
}

__global__ void __launch_bounds__(kFinish)
k_finish(const double* __restrict__ part, int nb, double* __restrict__ out) {
  finish_block(part, nb, out);
}

// k_finish writing straight into host memory mapped for the device: the
// (sum, max) pair, then, after a system-scope fence, the attempt's sequence
// number, for which the host polls.
__global__ void __launch_bounds__(kFinish)
k_finish_post(const double* __restrict__ part, int nb, double* __restrict__ host,
              unsigned long long seq) {
  __shared__ double pair[2];
  finish_block(part, nb, pair);
  if (threadIdx.x == 0) {
    host[0] = pair[0];
    host[1] = pair[1];
    __threadfence_system();
    reinterpret_cast<volatile unsigned long long*>(host)[2] = seq;
  }
}

// k_finish_post for every member, a block each: member m's pair and the
// attempt's sequence number into host[3m], host[3m + 1], host[3m + 2]
__global__ void __launch_bounds__(kFinish)
k_finish_batch(const BatchMember* __restrict__ mem, int nMem, double* __restrict__ host,
               const unsigned long long* __restrict__ seq) {
  const BatchMember& M = mem[blockIdx.x];
  double* const out = host + 3 * (size_t)blockIdx.x;
  __shared__ double pair[2];
  finish_block(M.sa.part, M.parts, pair);
  if (threadIdx.x == 0) {
    out[0] = pair[0];
    out[1] = pair[1];
    __threadfence_system();
    reinterpret_cast<volatile unsigned long long*>(out)[2] = *seq;
  }
}

// Max of eta = h - H over the nodes inside the open window (x0, x1) x (y0, y1)
// and the lowest node index attaining it (the result of a sequential scan with
// a strict ">", apps/shoal_focus_mpi.cu:199-204): per block, (value, index)
// partials in part[2 b], part[2 b + 1]; empty: (-1e300, -1). Node coordinates
// are formed as the host forms them, ex hx + xo[a] with xo[a] = 0.5 hx (xi_a + 1).
__global__ void __launch_bounds__(kThreads)
k_eta_max(const double* __restrict__ U, const double* __restrict__ Hn, Geometry g, double hx,
          double hy, EtaWindow w, double* __restrict__ part) {
  __shared__ double sv[kThreads];
  __shared__ long long si[kThreads];
  double best = -1e300;
  long long bi = -1;
  const long long Nd = g.Nd;
  const long long stride = (long long)gridDim.x * kThreads;
  for (long long i = (long long)blockIdx.x * kThreads + threadIdx.x; i < Nd; i += stride) {
    const long long e = i / NPP;
    const int loc = (int)(i - e * NPP);
    const int b = loc / NP, a = loc - NP * b;
    const int ey = (int)(e / g.Nx), ex = (int)(e - (long long)ey * g.Nx);
    const double x = ex * hx + w.xo[a];
    const double y = ey * hy + w.yo[b];
    if (!(x > w.x0 && x < w.x1 && y > w.y0 && y < w.y1)) continue;
    const double eta = U[i] - Hn[i];
    if (eta > best) { best = eta; bi = i; }
  }
  sv[threadIdx.x] = best;
  si[threadIdx.x] = bi;
  __syncthreads();
  for (int off = kThreads / 2; off > 0; off >>= 1) {
    if (threadIdx.x < off) {
      const double v2 = sv[threadIdx.x + off];
      const long long i2 = si[threadIdx.x + off];
      const double v1 = sv[threadIdx.x];
      const long long i1 = si[threadIdx.x];
      if (v2 > v1 || (v2 == v1 && i2 >= 0 && (i1 < 0 || i2 < i1))) {
        sv[threadIdx.x] = v2;
        si[threadIdx.x] = i2;
      }
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = sv[0];
    part[2 * blockIdx.x + 1] = (double)si[0];
  }
}

// eta = h - H at n given nodes
__global__ void __launch_bounds__(kThreads)
k_gather_eta(const double* __restrict__ U, const double* __restrict__ Hn,
             const long long* __restrict__ nodes, int n, double* __restrict__ out) {
  const int k = blockIdx.x * kThreads + threadIdx.x;
  if (k < n) out[k] = U[nodes[k]] - Hn[nodes[k]];
}

// Element means of eta, u, v, p, H (src/io/vtk2d.h:39-44, :67-81): for each
// field, 0.25 * sum over b, a of qw[a] qw[b] f at the element's nodes, in that
// order; out[f * Ne + e].
__global__ void __launch_bounds__(kThreads)
k_elem_means(const double* __restrict__ U, const double* __restrict__ Hn,
             const OpTables* __restrict__ T, long long Nd, long long Ne,
             double* __restrict__ out) {
  const long long e = (long long)blockIdx.x * kThreads + threadIdx.x;
  if (e >= Ne) return;
  double m[5];
#pragma unroll
  for (int f = 0; f < 5; ++f) {
    double s = 0.0;
    for (int b = 0; b < NP; ++b)
      for (int a = 0; a < NP; ++a) {
        const long long i = e * NPP + a + NP * b;
        const double h = U[i];
        double v;
        if (f == 0) v = h - Hn[i];
        else if (f == 1) v = U[(long long)IHU * Nd + i] / h;
        else if (f == 2) v = U[(long long)IHV * Nd + i] / h;
        else if (f == 3) v = U[(long long)IHP * Nd + i] / h;
        else v = Hn[i];
        s += T->qw[a] * T->qw[b] * v;
      }
    m[f] = 0.25 * s;
  }
#pragma unroll
  for (int f = 0; f < 5; ++f) out[f * Ne + e] = m[f];
}

// Diagnostics over nodes: 0 = max wave speed (sgn2d.cpp:295-304), 1 = mass
// integrand qw_a qw_b h (:319-332), 2 = energy integrand (:334-350).
__global__ void __launch_bounds__(kThreads)
k_diag(const double* __restrict__ U, Geometry g, Phys ph, int which, double* __restrict__ part) {
  __shared__ double ws[3 * kThreads / 64];
  double s = 0.0, c = 0.0, m = 0.0;
  const long long Nd = g.Nd;
  const size_t stride = (size_t)gridDim.x * kThreads;
  for (size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x; i < (size_t)Nd; i += stride) {
    double Un[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) Un[v] = U[(long long)v * Nd + i];
    if (which == 0) {
      const Prim q = prims(Un);
      const double ce = signal_speed(Un[IH], q, ph);
      const double s0 = fabs(q.u) + ce, s1 = fabs(q.v) + ce;
      m = fmax(m, fmax(s0, s1));
    } else {
      const int loc = (int)(i % NPP);
      const int b = loc / NP, a = loc - NP * b;
      const double wq = g.ops->qw[a] * g.ops->qw[b];
      double val;
      if (which == 1) {
        val = wq * Un[IH];
      } else {
        const double h = Un[IH];
        const double u = Un[IHU] / h, v = Un[IHV] / h, w = Un[IHW] / h;
        const double ed = 0.5 * h *
                          (u * u + v * v + (1.0 / ph.gamma) * w * w + ph.g * (h - 2.0 * g.Hnod[i]));
        val = wq * ed;
      }
      acc_add(s, c, val);
    }
  }
  block_reduce(s, c, m, ws);
  if (threadIdx.x == 0) {
    part[3 * blockIdx.x] = s;
    part[3 * blockIdx.x + 1] = c;
    part[3 * blockIdx.x + 2] = m;
  }
}

inline unsigned elementwise_blocks(size_t n) {
  const size_t want = (n + kThreads - 1) / kThreads;
  return (unsigned)(want < 16384 ? (want ? want : 1) : 16384);
}

constexpr int kTileW = kStripW;   // elements per RHS tile / sweep strip

}  // namespace

long long sweep_tiles(const Geometry& g) {
  const long long strips = (g.Nx + kTileW - 1) / kTileW;
  const long long chunks = ((long long)g.Ny + g.rows - 1) / g.rows;   // (rows up to 2^31 - 1)
  return strips * chunks;
}

namespace {

// one row-sweep launch of a (mode, waves, keep) build, with the still-depth
// gradients read (hxr false) or formed from Hnod (hxr true)
template <int M, int W, bool K>
void sweep_launch(bool hxr, dim3 grid, dim3 block, hipStream_t st, const BatchMember& a) {
  if (hxr) hipLaunchKernelGGL((k_rhs_sweep<kTileW, M, W, K, true>), grid, block, 0, st, a);
  else hipLaunchKernelGGL((k_rhs_sweep<kTileW, M, W, K, false>), grid, block, 0, st, a);
}

template <int M, int W, bool K>
void sweep_launch_batch(bool hxr, dim3 grid, dim3 block, hipStream_t st, const BatchMember* mem,
                        const long long* tileStart, int nMem) {
  if (hxr)
    hipLaunchKernelGGL((k_rhs_sweep_batch<kTileW, M, W, K, true>), grid, block, 0, st, mem,
                       tileStart, nMem);
  else
    hipLaunchKernelGGL((k_rhs_sweep_batch<kTileW, M, W, K, false>), grid, block, 0, st, mem,
                       tileStart, nMem);
}

}  // namespace

// A launch of a grid by itself takes its rows in tall tiles first and the last
// kLowTiles or so in low ones (g.rows high): tall tiles start and load their
// borders less often, low ones even out the end. Tall and low heights against
// one height, us:
//   387 x 191   9, 3 against 5    plain 59.6 -> 58.2   76.0 -> 72.6   100.8 -> 96.5   86.4 -> 80.4
//   603 x 301  12, 4 against 8         135.0 -> 129.0 170.4 -> 166.6  228.7 -> 226.9 192.1 -> 193.4
//  1024 x 512  12, 4 against 8         341.9 -> 330.0 440.0 -> 426.2  635.6 -> 628.6 498.7 -> 493.7
//  2000 x 1000 16, 4 against 18         1239 -> 1221   1607 -> 1588    2396 -> 2376   1887 -> 1858
// (1024 x 512 at 16, 4: 333, 427, 630, 502; 2000 x 1000 at 12, 4: 1234, 1620, 2391,
// 1871.) 16, 4 against 12, 4, by the sets of four workgroups per compute unit that
// 16 rows make (the place of the arrays moves stage 3 by more than that):
//   6.4  1024 x 512   plain 377, 369   443, 451   k4 504, 514
//   8.8  1200 x 600         503, 513   600, 600      696, 689
//  10.4  1300 x 650         588, 589   699, 709      810, 814
//  13.0  1448 x 724         731, 737   868, 880     1004, 1002
//  15.6  1600 x 800         886, 894  1051, 1059    1206, 1210
// 6, 2 against one height, plain and the step's three together, at 1.6 to 2.4 sets
// of 6 rows: 303 x 161 50.6 185 -> 43.9 172, 256 x 210 50.5 198 -> 47.5 189, 370 x 185
// 60.7 247 -> 57.0 236, but 320 x 160 46.6 170 -> 44.3 176, 330 x 165 52.0 191 -> 51.7
// 203, where the one height makes just one set, which stage 3 takes in one go; in the
// mean of 16 sizes 1 % faster, the plain launch 5 %.
// A grid that has not 1.6 sets of four workgroups per compute unit at 6
// rows takes one height (sweep_rows), and so does a flat one: the rows that a
// strip has left beside its tall tiles all go into low ones, which costs more than
// their even end gives where there is no tall tile, or, with two sets of strips or
// more, not four of them. The plain launch and a step's three, one height against
// tall and low:
//    8201 x 16   104  435, 12, 4: 105  434      14800 x 13   147  600,  9, 3: 160  662
//   20000 x 11   164  673,  6, 2: 188  774      61440 x 11   488 1987,  6, 2: 548 2424
constexpr int kLowTiles = 1280;

// chunks of `tall` rows, which leave the rest of the rows to the low tiles
static int tall_chunks(const Geometry& g, int strips, int tall, int rows) {
  const int lowChunks = (kLowTiles + strips - 1) / strips;
  return std::max(0, (g.Ny - lowChunks * rows) / tall);
}

int sweep_tall(const Geometry& g, int cus, int* rows) {
  const long long strips = (g.Nx + kTileW - 1) / kTileW, unit = 4LL * std::max(cus, 1);
  constexpr struct { int tall, rows; double sets; } kHeights[] = {
      {16, 4, 12.0}, {12, 4, 1.6}, {9, 3, 1.6}, {6, 2, 1.6}};
  for (const auto& h : kHeights) {
    if (strips * ((g.Ny + h.tall - 1) / h.tall) < h.sets * unit) continue;
    if (tall_chunks(g, (int)strips, h.tall, h.rows) < (strips < 2 * unit ? 1 : 4)) break;
    *rows = h.rows;
    return h.tall / h.rows;
  }
  return 1;
}

hipError_t launch_rhs_stage(const Geometry& g, const Phys& ph, int mode, const Stage& sa,
                            double* dU, GhostTime gt, hipStream_t st) {
  if (sweep_tiles(g) > 0x7fffffffLL || g.rows < 1) return hipErrorInvalidValue;
  BatchMember args = sweep_member(g, ph, sa.u, dU, gt, sa);
  args.lowTiles = args.nTiles;
  if (g.tall > 1) {
    const int strips = args.nStrips;
    args.tall = g.tall * g.rows;
    const int tallChunks = tall_chunks(g, strips, args.tall, g.rows);
    args.lowFrom = tallChunks * args.tall;
    args.tallTiles = tallChunks * strips;
    args.tallBlocks = (int)packed_tiles(args.tallTiles);
    args.lowTiles = strips * ((g.Ny - args.lowFrom + g.rows - 1) / g.rows);
    args.nTiles = args.tallTiles + args.lowTiles;
  }
  const dim3 grid((unsigned)(args.tallBlocks + args.lowTiles)), block(Sweep<kTileW>::NT);
  // waves per SIMD the register allocation targets, per stage mode (bit m of
  // g.waves3 set: 3 waves, else 2)
  const bool w3 = (g.waves3 >> mode) & 1;
  if (mode < kPlain || mode > kErr || ph.nManning != 0.0) return hipErrorInvalidValue;
  const bool hxr = g.hxr != 0;   // Hx, Hy formed from Hnod
#define SGNX_SWEEP(M, W, K) sweep_launch<M, W, K>(hxr, grid, block, st, args)
  const bool keep = sa.yOut != nullptr;
  if (mode == kCand && keep && !sa.zOut) return hipErrorInvalidValue;
  if (mode == kPlain) { if (w3) SGNX_SWEEP(kPlain, 3, false); else SGNX_SWEEP(kPlain, 2, false); }
  else if (mode == kAxpy) {
    if (keep) { if (w3) SGNX_SWEEP(kAxpy, 3, true); else SGNX_SWEEP(kAxpy, 2, true); }
    else { if (w3) SGNX_SWEEP(kAxpy, 3, false); else SGNX_SWEEP(kAxpy, 2, false); }
  } else if (mode == kCand) {
    if (keep) { if (w3) SGNX_SWEEP(kCand, 3, true); else SGNX_SWEEP(kCand, 2, true); }
    else if (!sa.zOut) { if (w3) SGNX_SWEEP(kCandOnly, 3, false); else SGNX_SWEEP(kCandOnly, 2, false); }
    else { if (w3) SGNX_SWEEP(kCand, 3, false); else SGNX_SWEEP(kCand, 2, false); }
  } else { if (w3) SGNX_SWEEP(kErr, 3, false); else SGNX_SWEEP(kErr, 2, false); }
#undef SGNX_SWEEP
  return hipGetLastError();
}

BatchMember sweep_member(const Geometry& g, const Phys& ph, const double* U, double* dU,
                         GhostTime gt, const Stage& sa, int times) {
  BatchMember m{U, dU, g, ph, gt, sa, times * g.rows, (g.Nx + kTileW - 1) / kTileW, 0, 0, 0, 0, 0, 0, 0};
  m.nTiles = (int)(m.nStrips * (((long long)g.Ny + m.rows - 1) / m.rows));
  m.parts = (int)sweep_tiles(g);
  return m;
}

// The lowest time of a step by sweep_cost, in us: six workgroups fit on a compute
// unit, four of stage 3 (kStripW). The last stage fits six times too, yet the rule
// counts it with stage 3: counted with the others it picks 1 row for 103 x 77 (62.6
// us a step, 57.6 at the 2 rows taken), 3 for 156 x 117 (94.1, 90.5 at 4), 4 for 197 x
// 147 (127.6, 120.0 at 6), 3 for 333 x 133 (175.3, 165.5 at 9). Measured (plain, stage
// 2, stage 3, last):
//   rows            1            2            5            7            8           12           16
//   128 x  64  16 20 22 20  15 18 19 19  24 28 28 30  31 34 36 37  29 31 33 34  40 43 46 47  51 54 58 60
//   256 x 128  38 47 58 49  34 41 50 43  33 40 55 42  35 40 43 43  38 43 46 47  50 55 58 61  63 68 72 76
//   387 x 191 73 104 145 109 63 87 118 92 60 77 105 88 66 82 108 89 72 86 100 96 65 78 109 88 71 85 100 96
//   603 x 301 (all four) 1033  833  734  728  735  786  770;  1024 x 512  -  -  -  -  1932 1943 1951
// It takes 2, 7, 5, 8 and 8 rows there (launches by themselves: sweep_tall).
int sweep_rows(const Geometry* const* g, int n, int cus) {
  constexpr SweepPace six{6, 2.5, 0.5, 0.5, 1.8}, four{4, 2.6, 0.65, 0.5, 1.6};
  cus = std::max(cus, 1);
  return choose_rows(24, [&](int r) {
    long long tiles = 0;
    for (int i = 0; i < n; ++i)
      tiles += (long long)((g[i]->Nx + kTileW - 1) / kTileW) * ((g[i]->Ny + r - 1) / r);
    return sweep_cost(tiles, r, cus, six) + sweep_cost(tiles, r, cus, four);
  });
}

hipError_t launch_rhs_stage_batch(const BatchMember* mem, const long long* tileStart, int nMem,
                                  long long totalTiles, int mode, bool waves3, hipStream_t st,
                                  bool keep, bool hxr) {
  if (nMem < 1 || totalTiles < 1 || totalTiles > 0x7fffffffLL) return hipErrorInvalidValue;
  if (mode < kPlain || mode > kErr) return hipErrorInvalidValue;
  const dim3 grid((unsigned)totalTiles), block(Sweep<kTileW>::NT);
#define SGNX_SWEEPB(M, W, K) sweep_launch_batch<M, W, K>(hxr, grid, block, st, mem, tileStart, nMem)
  if (mode == kPlain) { if (waves3) SGNX_SWEEPB(kPlain, 3, false); else SGNX_SWEEPB(kPlain, 2, false); }
  else if (mode == kAxpy && keep) { if (waves3) SGNX_SWEEPB(kAxpy, 3, true); else SGNX_SWEEPB(kAxpy, 2, true); }
  else if (mode == kAxpy) { if (waves3) SGNX_SWEEPB(kAxpy, 3, false); else SGNX_SWEEPB(kAxpy, 2, false); }
  else if (mode == kCand && keep) { if (waves3) SGNX_SWEEPB(kCand, 3, true); else SGNX_SWEEPB(kCand, 2, true); }
  else if (mode == kCand) { if (waves3) SGNX_SWEEPB(kCand, 3, false); else SGNX_SWEEPB(kCand, 2, false); }
  else { if (waves3) SGNX_SWEEPB(kErr, 3, false); else SGNX_SWEEPB(kErr, 2, false); }
#undef SGNX_SWEEPB
  return hipGetLastError();
}

hipError_t launch_finish_batch(const BatchMember* mem, int nMem, double* host,
                               const long long* seq, hipStream_t st) {
  if (nMem < 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_finish_batch, dim3((unsigned)nMem), dim3(kFinish), 0, st, mem, nMem, host,
                     reinterpret_cast<const unsigned long long*>(seq));
  return hipGetLastError();
}

hipError_t launch_finish_post(const double* part, long long nb, double* host,
                              unsigned long long seq, hipStream_t st) {
  hipLaunchKernelGGL(k_finish_post, dim3(1), dim3(kFinish), 0, st, part, (int)nb, host, seq);
  return hipGetLastError();
}

hipError_t launch_finish(const double* part, long long nb, double* out, hipStream_t st) {
  hipLaunchKernelGGL(k_finish, dim3(1), dim3(kFinish), 0, st, part, (int)nb, out);
  return hipGetLastError();
}

hipError_t launch_rhs(const Geometry& g, const Phys& ph, const double* U, double* dU,
                      GhostTime gt, hipStream_t st) {
  if (g.variant == 1) {
    Stage sa{};
    sa.u = U;
    return launch_rhs_stage(g, ph, kPlain, sa, dU, gt, st);
  }
  const int tpr = (g.Nx + kTileW - 1) / kTileW;
  const long long tiles = (long long)tpr * g.Ny;
  if (tiles > 0x7fffffffLL) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_rhs<kTileW>, dim3((unsigned)tiles), dim3(Tile<kTileW>::NT), 0, st, U, dU,
                     g, ph, gt, tpr);
  return hipGetLastError();
}

hipError_t launch_bathy_check(const Geometry& g, const double* Hnod, const double* Hx,
                              const double* Hy, int* bad, hipStream_t st) {
  const long long nb = (g.Nd + kThreads - 1) / kThreads;
  hipLaunchKernelGGL(k_bathy_check, dim3((unsigned)nb), dim3(kThreads), 0, st, Hnod, Hx, Hy,
                     g.ops, g.Nd, g.Jx, g.Jy, bad);
  return hipGetLastError();
}

hipError_t launch_bathy_grad(const Geometry& g, const double* Hnod, double* Hx, double* Hy,
                             hipStream_t st) {
  const long long nb = (g.Nd + kThreads - 1) / kThreads;
  hipLaunchKernelGGL(k_bathy_grad, dim3((unsigned)nb), dim3(kThreads), 0, st, Hnod, Hx, Hy,
                     g.ops, g.Nd, g.Jx, g.Jy);
  return hipGetLastError();
}

hipError_t launch_comb1(double* out, const double* u, double a1, const double* k1, size_t n,
                        hipStream_t st) {
  hipLaunchKernelGGL(k_comb1, dim3(elementwise_blocks(n)), dim3(kThreads), 0, st, out, u, a1, k1,
                     n);
  return hipGetLastError();
}

hipError_t launch_bs3_update(double* out, const double* u, double dt, const double* k1,
                             const double* k2, const double* k3, size_t n, hipStream_t st) {
  hipLaunchKernelGGL(k_bs3_update, dim3(elementwise_blocks(n)), dim3(kThreads), 0, st, out, u,
                     dt, k1, k2, k3, n);
  return hipGetLastError();
}

hipError_t launch_rk4_update(double* u, double dt, const double* k1, const double* k2,
                             const double* k3, const double* k4, size_t n, hipStream_t st) {
  hipLaunchKernelGGL(k_rk4_update, dim3(elementwise_blocks(n)), dim3(kThreads), 0, st, u, dt, k1,
                     k2, k3, k4, n);
  return hipGetLastError();
}

hipError_t launch_err_norm(const double* u, const double* uNew, const double* k1,
                           const double* k2, const double* k3, const double* k4, double dt,
                           double atol, double rtol, size_t n, double* part, double* out,
                           hipStream_t st) {
  hipLaunchKernelGGL(k_err_norm, dim3(kReduceBlocks), dim3(kThreads), 0, st, u, uNew, k1, k2, k3,
                     k4, dt, atol, rtol, n, part);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_finish, dim3(1), dim3(kFinish), 0, st, part, kReduceBlocks, out);
  return hipGetLastError();
}

hipError_t launch_eta_max(const Geometry& g, const double* U, double hx, double hy,
                          const EtaWindow& w, double* part, hipStream_t st) {
  hipLaunchKernelGGL(k_eta_max, dim3(kReduceBlocks), dim3(kThreads), 0, st, U, g.Hnod, g, hx, hy,
                     w, part);
  return hipGetLastError();
}

hipError_t launch_gather_eta(const Geometry& g, const double* U, const long long* nodes, int n,
                             double* out, hipStream_t st) {
  if (n < 1) return hipSuccess;
  hipLaunchKernelGGL(k_gather_eta, dim3((n + kThreads - 1) / kThreads), dim3(kThreads), 0, st, U,
                     g.Hnod, nodes, n, out);
  return hipGetLastError();
}

hipError_t launch_elem_means(const Geometry& g, const double* U, double* out, hipStream_t st) {
  const long long Ne = (long long)g.Nx * g.Ny;
  hipLaunchKernelGGL(k_elem_means, dim3((unsigned)((Ne + kThreads - 1) / kThreads)),
                     dim3(kThreads), 0, st, U, g.Hnod, g.ops, g.Nd, Ne, out);
  return hipGetLastError();
}

hipError_t launch_diag(const Geometry& g, const Phys& ph, const double* U, int which,
                       double* part, double* out, hipStream_t st) {
  hipLaunchKernelGGL(k_diag, dim3(kReduceBlocks), dim3(kThreads), 0, st, U, g, ph, which, part);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_finish, dim3(1), dim3(kFinish), 0, st, part, kReduceBlocks, out);
  return hipGetLastError();
}

}  // namespace sgnx
