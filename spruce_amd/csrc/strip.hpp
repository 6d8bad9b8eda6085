// Building blocks of the wavefront-strip stencil kernels (mhd2.hip, the ideal_2F strip kernel in
// twofluid.hip): one 64-lane wavefront owns 64 columns (y, contiguous in memory) and marches down
// the rows (x) of a strip; y-neighbours come from neighbouring lanes through DPP shifts, x-neighbours
// from a rotating register window.  Face arithmetic follows derivs.cpp:10-73 and 477-499 operation
// for operation.
#pragma once
#include <hip/hip_runtime.h>

#include "arith.hpp"
#include "mhd.hpp"
#include "range.hpp"

namespace spruce {
namespace strip {

constexpr int OUT_COLS = 60;   // lanes 2..61 produce outputs; 0, 1, 62, 63 supply the y-halo

// lane l receives the value of lane l-1 (wave_shr:1) / lane l+1 (wave_shl:1); 0 at the ends
__device__ __forceinline__ double shr1(double x) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), 0x138, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), 0x138, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double shl1(double x) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), 0x130, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), 0x130, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}

__device__ __forceinline__ int wrapn(int k, int n) {
  k %= n;
  return k < 0 ? k + n : k;
}
__device__ __forceinline__ int clampn(int k, int n) { return k < 0 ? 0 : (k >= n ? n - 1 : k); }

// k brought into [0, n) when it is at most n away from it
__device__ __forceinline__ int wrap_near(int k, int n) { return k < 0 ? k + n : (k >= n ? k - n : k); }

// Element jb bytes into row `row` (an offset in elements, the same in every lane).  The row's address
// is formed in scalar registers (the empty asm keeps the compiler from adding the lane's part to the
// array's address first and holding one 64-bit sum per array in vector registers), and the lane
// supplies one 32-bit offset for every array and row.  p and row are the same in every lane.
using gdouble = __attribute__((address_space(1))) double;
using gchar = __attribute__((address_space(1))) char;
__device__ __forceinline__ gdouble* row_at(const double* p, size_t row, uint32_t jb) {
  uint64_t base = reinterpret_cast<uint64_t>(p + row);
  asm("" : "+s"(base));
  return reinterpret_cast<gdouble*>(reinterpret_cast<gchar*>(base) + jb);
}
// The lane's offset as a value of its own in the block that uses it: carried in from another block
// it would arrive widened to 64 bits, and each access would add it in vector registers.
__device__ __forceinline__ void lane_offset(uint32_t& jb) { asm("" : "+v"(jb)); }
__device__ __forceinline__ double ld_row(const double* p, size_t row, uint32_t jb) { return *row_at(p, row, jb); }
__device__ __forceinline__ void st_row(double* p, size_t row, uint32_t jb, double v) { *row_at(p, row, jb) = v; }

// the face between cells c-1 and c of an axis, -1 <= c <= n+1 (wrapped on periodic axes, clamped otherwise)
__device__ __forceinline__ FaceGeom face_geom(const Axis& ax, int c) {
  return ax.face[ax.per ? wrap_near(c, ax.n) : clampn(c, ax.n)];
}

// The same face for an index that is the same in every lane, through the scalar cache: the table never
// changes, so its address space is the constant one.  As vector loads these would be waited for in
// order with the rows being fetched.
__device__ __forceinline__ FaceGeom face_geom_row(const Axis& ax, int c) {
  using cdouble = const __attribute__((address_space(4))) double;
  cdouble* p = reinterpret_cast<cdouble*>(reinterpret_cast<uint64_t>(ax.face + (ax.per ? wrap_near(c, ax.n) : clampn(c, ax.n))));
  return FaceGeom{p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], p[8], p[9], p[10], p[11], p[12], p[13]};
}

// boundaryInterpolate(a at the lower cell, b at the upper cell) (derivs.cpp:477-487); IN: the
// operands are in range (range.hpp)
template <bool IN = false>
__device__ __forceinline__ double interp(const FaceGeom& g, double a, double b) {
  return qdiv_t<IN>(a * g.hup + b * g.hlo, g.den, g.rden);
}

// Upwind side of a face from its velocity (derivs.cpp:47-68).
struct FaceDir {
  double vf, ge, de, rde;
  bool pos, moving;
};
__device__ __forceinline__ FaceDir face_dir(double vf, const FaceGeom& g) {
  FaceDir d;
  d.vf = vf;
  d.pos = vf > 0.0;
  d.moving = d.pos || vf < 0.0;
  d.ge = d.pos ? g.gup : g.gdn;
  d.de = d.pos ? g.denm : g.denp;
  d.rde = d.pos ? g.rdenm : g.rdenp;
  return d;
}

// surf * face velocity * (Barton-limited upwind value) of one transported quantity, from the four
// cells c-2, c-1 (lo), c (up), c+1 along the face's axis; d2 = the plain interpolation.
template <bool IN = false>
__device__ __forceinline__ double face_flux(double q0, double q1, double q2, double q3, const FaceGeom& g,
                                            const FaceDir& fd, double& d2) {
  d2 = interp<IN>(g, q1, q2);
  const double ea = fd.pos ? q0 : q3, eb = fd.pos ? q1 : q2;
  const double d1 = ea + qdiv_t<IN>((eb - ea) * fd.ge, fd.de, fd.rde);
  const bool le = q2 <= q1;
  const bool outer_min = fd.pos == le;
  if (IN) {
    // finite values: both orders by min and max, then one choice; a face at rest (vf = 0) carries
    // lim * 0 = 0, as d2 * 0
    const double lo = hw_min(eb, hw_max(d1, d2)), up = hw_max(eb, hw_min(d1, d2));
    return (outer_min ? lo : up) * fd.vf;
  }
  const double inner = outer_min ? smax(d1, d2) : smin(d1, d2);
  const double lim = outer_min ? smin(eb, inner) : smax(eb, inner);
  return (fd.moving ? lim : d2) * fd.vf;
}

// Workgroups go to the 8 XCDs round-robin by launch index (index % 8), and each XCD has its own
// L2: launch index L (of `total`) is mapped to the logical tile t so that XCD x takes the x-th
// eighth of the tiles in order, and tiles that run together on one XCD are neighbours.
__device__ __forceinline__ int xcd_tile(int L, int total) {
  const int xcd = L & 7, k = L >> 3;
  const int q = total >> 3, rem = total & 7;
  return xcd * q + (xcd < rem ? xcd : rem) + k;
}

}  // namespace strip
}  // namespace spruce
