// Building blocks of the wavefront-strip form of the conduction update (k_tc_strip, solar.hip) and
// of its reverse (k_adj_tc_strip, adj_modules.hip): one 64-lane wavefront owns consecutive columns
// (y) and marches down the rows (x) of a strip; the face values the energy derivative takes are
// formed once and shared by the two cells of the face, along y through DPP lane shifts, along x
// by keeping the previous row's faces in registers.  Each value is the same sequence of IEEE
// operations as tc_core's (tc_cell.hpp).
#pragma once
#include <hip/hip_runtime.h>

#include "arith.hpp"
#include "range.hpp"
#include "solar.hpp"
#include "strip.hpp"

namespace spruce {
namespace tcs {

// temp = max((gamma-1) te / (2 K_B n), temp_min) (thermalconduction.cpp:109; idealmhd.cpp:254)
__device__ __forceinline__ double temp_of(double te, double n, const MhdConst& K) {
  return smax(te * K.gm1 / (n * (2.0 * K_B)), K.tmin);
}

// How the geometric divisions are taken: as products with the prepared reciprocal (within an ulp; the
// adjoint's recompute of the values its partial derivatives take), IEEE divisions (qdiv), or the same
// without the operand test, for rows in range (range.hpp).
enum Div { DIV_PRODUCT, DIV_TESTED, DIV_IN };
template <int D>
__device__ __forceinline__ double qd(double a, double b, double rb) {
  return D == DIV_PRODUCT ? a * rb : (D == DIV_IN ? qdiv_in(a, b, rb) : qdiv(a, b, rb));
}

// one row of the strip at this lane: cell values and the quantities that need only y-neighbours
struct Row {
  double T, te, gy, s1, bx, by, dbxy, dbyy;
  int i;                     // wrapped row index (clamped into [0, nx) when the row lies outside)
  bool val, inx;             // row exists; row inside the interior bounds
};
struct Raw { double te, n, bx, by, rho; };   // rho: flux saturation only
struct XFaces { double T, gy, bx, by; };

struct Lane {
  int j;                     // wrapped column (clamped into [0, ny) when it lies outside)
  bool val, iny, out;        // column exists; inside the interior bounds; writes an output
  double hc, hn, fd, rfd;    // upper y-face: weight of this lane's value, of the next lane's, denominator
  double dy, rdy, hsq, rhsq;
};

// k (at most n away from the grid) wrapped on a periodic axis, else clamped; val: whether it exists
__device__ __forceinline__ int row_index(int k, int n, int per, bool& val) {
  if (per) { val = true; return strip::wrap_near(k, n); }
  val = k >= 0 && k < n;
  return strip::clampn(k, n);
}

// column jc of the mesh as this lane's (out is left to the caller)
__device__ __forceinline__ Lane lane_at(const Mesh& M, int jc) {
  Lane L;
  bool vp;
  L.j = row_index(M.y.per ? strip::wrapn(jc, M.ny) : jc, M.ny, M.y.per, L.val);
  L.iny = L.val && L.j >= M.y.lo && L.j <= M.y.hi;
  const int jp = row_index(L.j + 1, M.ny, M.y.per, vp);
  L.hc = M.y.h[jp];
  L.hn = M.y.h[L.j];
  L.fd = M.y.fden[jp];
  L.rfd = M.y.rfden[jp];
  L.dy = M.y.d[L.j];
  L.rdy = M.y.rd[L.j];
  L.hsq = M.y.hsq[L.j];
  L.rhsq = M.y.rhsq[L.j];
  L.out = false;
  return L;
}

// boundaryInterpolate across this lane's upper y-face (derivs.cpp:477-487), from its own value and
// the next lane's
template <int D>
__device__ __forceinline__ double yface(const Lane& L, double q) {
  const double up = strip::shl1(q);
  return qd<D>(q * L.hc + up * L.hn, L.fd, L.rfd);
}
// derivative1D along y at this lane from the upper faces of this lane and of the previous one
template <int D>
__device__ __forceinline__ double yderiv(const Lane& L, double fup) {
  return qd<D>(fup - strip::shr1(fup), L.dy, L.rdy);
}

// Rows and columns outside a closed side are read from the nearest cell: what they hold reaches only
// values that are masked.
template <bool SAT>
__device__ __forceinline__ Raw load_raw(const TcStepArgs& a, const Lane& L, int k) {
  bool v;
  const size_t row = (size_t)row_index(k, a.mesh.nx, a.mesh.x.per, v) * a.mesh.ny;
  uint32_t jb = 8u * (uint32_t)L.j;
  strip::lane_offset(jb);
  Raw r;
  r.te = strip::ld_row(a.te_src, row, jb);
  r.n = strip::ld_row(a.n, row, jb);
  r.bx = strip::ld_row(a.bhx, row, jb);
  r.by = strip::ld_row(a.bhy, row, jb);
  r.rho = SAT ? strip::ld_row(a.rho, row, jb) : 0.0;
  return r;
}

template <int D>
__device__ __forceinline__ Row make_row(const TcStepArgs& a, const Lane& L, int k, const Raw& r) {
  const Mesh& M = a.mesh;
  Row w;
  w.i = row_index(k, M.nx, M.x.per, w.val);
  w.inx = w.val && w.i >= M.x.lo && w.i <= M.x.hi;
  w.te = r.te;
  const double den = r.n * (2.0 * K_B);
  w.T = D == DIV_IN ? smax(qdiv_in(r.te * a.k.gm1, den, recip_in(den)), a.k.tmin) : temp_of(r.te, r.n, a.k);
  w.bx = r.bx;
  w.by = r.by;
  const double fT = yface<D>(L, w.T);
  const double fTlo = strip::shr1(fT);
  // dtemp_dy is zero outside the interior (derivs.cpp:229-233)
  w.gy = (w.inx && L.iny) ? qd<D>(fT - fTlo, L.dy, L.rdy) : 0.0;
  w.s1 = qd<D>(fT - 2.0 * w.T + fTlo, L.hsq, L.rhsq);      // secondDerivative1D (derivs.cpp:450)
  w.dbxy = yderiv<D>(L, yface<D>(L, w.bx));
  w.dbyy = yderiv<D>(L, yface<D>(L, w.by));
  return w;
}

// whether a row's values at this lane are outside the range of the untested divisions and powers
template <bool SAT>
__device__ __forceinline__ bool row_out(const Row& w, const Raw& r) {
  RangeTest t;
  t.add(w.bx);
  t.add(w.by);
  if (SAT) t.density(r.rho);
  return t.out() || !(w.T >= 0x1p-100 && w.T <= 0x1p+100) || !(r.n >= 0x1p-100 && r.n <= 0x1p+150);
}

// boundaryInterpolate across the x-face between rows A (lower) and B (upper), whose geometry is g
template <int D>
__device__ __forceinline__ XFaces xfaces(const FaceGeom& g, const Row& A, const Row& B) {
  XFaces f;
  f.T = qd<D>(A.T * g.hup + B.T * g.hlo, g.den, g.rden);
  f.gy = qd<D>(A.gy * g.hup + B.gy * g.hlo, g.den, g.rden);
  f.bx = qd<D>(A.bx * g.hup + B.bx * g.hlo, g.den, g.rden);
  f.by = qd<D>(A.by * g.hup + B.by * g.hlo, g.den, g.rden);
  return f;
}

}  // namespace tcs
}  // namespace spruce
