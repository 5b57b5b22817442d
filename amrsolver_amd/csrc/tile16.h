// Workgroups of 16x16 cells that march in z with a halo of two cells: the
// plane's layout in LDS, the ring of cells around the tile and the lane shifts
// of the forward and the reverse stage kernel.
#pragma once

#include <hip/hip_runtime.h>

namespace amr {
namespace tile16 {

constexpr int TX = 16, TY = 16, NT = 256, HX = 2, RX = TX + 2 * HX, RY = TY + 2 * HX, PL = RX * RY;
constexpr int NRING = 64, RB = NT - NRING;  // ring threads: the last wave
constexpr int NOUT = PL - NT - NRING;       // halo cells that are not ring cells

// Ring cell r (0..63): left, right, bottom, top; (a, b) its tile coordinates.
__device__ __forceinline__ void ring_cell(int r, bool& isx, int& a, int& b) {
  isx = r < 2 * TY;
  const int s = r & 15, hi = (r >> 4) & 1;
  a = isx ? (hi ? TX : -1) : s;
  b = isx ? s : (hi ? TY : -1);
}

// LDS cell of a thread's halo load: ring threads load their ring cell, threads
// OB .. OB+NOUT-1 the other halo cells (rows 0 and RY-1, columns 0
// and RX-1, then the ring's four corners); -1 for threads with none.
template <int OB>
__device__ __forceinline__ int halo_cell(int tid) {
  static_assert(OB >= 0 && OB + NOUT <= RB, "halo cells fit the first three waves");
  if (tid >= RB) {
    bool isx;
    int a, b;
    ring_cell(tid - RB, isx, a, b);
    return (b + HX) * RX + (a + HX);
  }
  if (tid < OB || tid >= OB + NOUT) return -1;
  const int o = tid - OB;
  int i, j;
  if (o < RX) { i = o; j = 0; }
  else if (o < 2 * RX) { i = o - RX; j = RY - 1; }
  else if (o < 2 * RX + RY - 2) { i = 0; j = o - 2 * RX + 1; }
  else if (o < 2 * RX + 2 * (RY - 2)) { i = RX - 1; j = o - 2 * RX - (RY - 2) + 1; }
  else {
    const int q = o - 2 * RX - 2 * (RY - 2);
    i = (q & 1) ? RX - 2 : 1;
    j = (q & 2) ? RY - 2 : 1;
  }
  return j * RX + i;
}

// The value of the lane to the left (SHR) or right (SHL) in the 16-lane row;
// the row's first (last) lane gets `edge`.
template <int CTRL>
__device__ __forceinline__ double dpp_row(double edge, double v) {
  const int lo = __builtin_amdgcn_update_dpp(__double2loint(edge), __double2loint(v), CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(__double2hiint(edge), __double2hiint(v), CTRL, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}
constexpr int ROW_SHL1 = 0x101, ROW_SHR1 = 0x111;

// A wave-uniform value held in scalar registers.
__device__ __forceinline__ double uniform(double v) {
  return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                          __builtin_amdgcn_readfirstlane(__double2loint(v)));
}

// Ends a section: nothing is scheduled across, and LDS values are read again
// rather than held in registers (with them held the kernel spilled).
__device__ __forceinline__ void section() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_sched_barrier(0);
}

}  // namespace tile16
}  // namespace amr
