// =============================================================================
// sgnx_device.h -- what the row-sweep kernels (sgnx_kernels.hip) and the
// adjoint's product kernel (sgnx_adjoint.hip) share on the device: addressing
// by scalar bases, lane permutes, per-row barriers.
// =============================================================================
#ifndef SGNX_DEVICE_H
#define SGNX_DEVICE_H

#include <hip/hip_runtime.h>

#include "sgnx_internal.h"

namespace sgnx {

// Global operands are addressed as a wave-uniform base (scalar registers and
// scalar adds) plus a 32-bit byte offset of the lane, so that no vector
// instruction forms an address. Variable v of an operand lies v planes of
// `plane` bytes above its base; the planes are stepped to one after another,
// which needs one scalar pair per operand instead of five.
typedef __attribute__((address_space(1))) char GlobalByte;
typedef __attribute__((address_space(1))) double GlobalDouble;
typedef __attribute__((address_space(3))) double LdsDouble;
__device__ __forceinline__ GlobalByte* global_at(const double* base, size_t first) {
  GlobalByte* p = (GlobalByte*)base + first;
  __asm__ volatile("" : "+s"(p));   // formed by scalar instructions, before the lane's part
  return p;
}
__device__ __forceinline__ double load_at(const GlobalByte* base, unsigned off) {
  return *(const GlobalDouble*)(base + off);
}
__device__ __forceinline__ void store_at(GlobalByte* base, unsigned off, double x) {
  *(GlobalDouble*)(base + off) = x;
}
__device__ __forceinline__ void load_vars(const double* base, size_t first, size_t plane,
                                          unsigned off, double* W) {
  const GlobalByte* p = global_at(base, first);
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    W[v] = load_at(p, off);
    p += plane;
  }
}

// A launch's arguments in constant memory (kernel arguments, or one entry of a
// batch's table) are read by scalar loads. What a phase needs once per row is
// read there again, through a pointer made opaque in that row: all of it kept
// across rows exceeds the scalar registers, and the excess would travel
// through vector lanes.
template <class T>
using ConstArgs = const T __attribute__((address_space(4))) *;
template <class P>
__device__ __forceinline__ P opaque(P A) {
  __asm__ volatile("" : "+s"(A));
  return A;
}
// entry i of a table in global memory, i the same on every lane
template <class T>
__device__ __forceinline__ ConstArgs<T> const_entry(const T* table, int i) {
  const size_t at = reinterpret_cast<size_t>(table + __builtin_amdgcn_readfirstlane(i));
  return reinterpret_cast<ConstArgs<T>>(
      (size_t)(unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)at) |
      (size_t)(unsigned)__builtin_amdgcn_readfirstlane((int)(at >> 32)) << 32);
}

// The other lane's value within each pair of lanes (DPP quad_perm [1,0,3,2]).
__device__ __forceinline__ double lane_swap(double x) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), 0xB1, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), 0xB1, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}

// barrier that instructions of the two phases do not cross in either direction
// (arithmetic hoisted over it only lengthens registers' lives)
__device__ __forceinline__ void row_sync() {
  __builtin_amdgcn_sched_barrier(0);
  __syncthreads();
  __builtin_amdgcn_sched_barrier(0);
}

// whether the condition holds on some active lane of the wave
__device__ __forceinline__ bool wave_any(int c) { return __builtin_amdgcn_ballot_w64(c != 0) != 0; }

// y = x as a move at this place
__device__ __forceinline__ void move_to(double& y, double x) {
  __asm__ volatile("v_mov_b64 %0, %1" : "=v"(y) : "v"(x));
}

// x with its sign bit changed where mask = 0x80000000 (0: unchanged)
__device__ __forceinline__ double flip_sign(double x, int mask) {
  return __hiloint2double(__double2hiint(x) ^ mask, __double2loint(x));
}

// Node (a, b) of element (ex, ey) within a variable (at most 2^28 of them).
__device__ __forceinline__ unsigned node_of(int Nx, int ex, int ey, int a, int b) {
  return ((unsigned)ey * (unsigned)Nx + (unsigned)ex) * NPP + a + NP * b;
}

template <int V>
struct IntC { static constexpr int value = V; };

}  // namespace sgnx

#endif  // SGNX_DEVICE_H
