// IdealMHD stage kernel, wavefront-strip form (the production path of launch_mhd_stage).
//
// A block of two 64-lane wavefronts owns a strip of 64 columns (y, contiguous in memory) and marches
// down R rows (x).  Lanes 2..61 produce outputs; lanes 0, 1, 62, 63 only supply the y-halo.  Along x
// the four rows a face needs (c-2 .. c+1) stay in a rotating register window, so every x-face is
// computed once and reused by the two cells that share it; along y the neighbouring columns are
// read from the neighbouring lanes with DPP wave shifts, so every y-face is computed once too.
// One wavefront transports the fluid (rho, mom, thermal energy), the other the field (bi, be); each
// forms the velocities it needs once per row, and the field hands its terms of the momentum
// equations over in LDS.  The arithmetic of each value is the reference's (derivs.cpp,
// idealmhd.cpp), operation for operation.
//
// What bounds it: FP64 instruction issue and the latency of a row's chain.  Each row is one
// straight run of about 550 VALU instructions per wavefront, because the divisions' range tests are
// made once per loaded value (range.hpp) instead of at each of the ~90 divisions per cell, where
// they cost twice the instructions and ended a basic block each.  One wavefront for all eleven
// quantities needs more than 256 registers once the code is straight, and a spilled value's reload
// also waits for the rows being fetched; the split leaves room (231 to 240 vector registers, none spilled, two
// wavefronts per SIMD) to fetch a row two rows ahead.  Measured on 2048x2048 (RK2, periodic): 536 us
// a stage with tested divisions and one wavefront per strip, 404 us with untested ones, 350 us with
// the split, 281 us with the longer fetch distance, the geometry gathered and read through the scalar
// cache, and the static rows; 0.81 GB of HBM traffic a launch, VALU 46% busy.  512x1024: 110 -> 41 us;
// 64x48: 17 (8x8 tiles) -> 9 us.
#include <cfloat>
#include <type_traits>

#include "arith.hpp"
#include "mhd.hpp"
#include "strip.hpp"

namespace spruce {
namespace {


using namespace strip;

// The eleven transported quantities (idealmhd.cpp:52-86) are split between the two wavefronts of a
// block: the fluid's and the field's (bi and be, component by component).
enum Role { FLUID = 0, FIELD = 1 };
enum { Q_RHO = 0, Q_MX, Q_MY, Q_MZ, Q_TE };                  // FLUID
enum { Q_BIX = 0, Q_BEX, Q_BIY, Q_BEY, Q_BIZ, Q_BEZ };       // FIELD

// qdiv for a data-dependent divisor: the reciprocal is exact-rounded only if it is a normal number.
__device__ __forceinline__ double qdiv_d(double a, double b, double rb) {
  const double ab = __builtin_fabs(b);
  if (__builtin_expect(ab > 0x1p-900 && ab < 0x1p+900, 1)) return qdiv(a, b, rb);
  return a / b;
}

// What a block shares.  The geometry of every column's lower y-face and its cell size are read from
// here once per row (24 registers otherwise, or a chain of an address and a load at the head of
// every row); force holds the field's terms of the momentum equations for the row being finished,
// in two slots so that one barrier per row orders the wavefronts; out_of_range says whether a
// wavefront found a value outside the range of the untested divisions in a row it loaded.
enum { F_EXT0 = 0, F_EXT1, F_IN0, F_IN1, F_INZ0, F_INZ1, F_EXTZ0, F_EXTZ1, F_ZEXT, F_ZIN, NF };
struct Shared {
  double2 geom[6][64];
  double force[2][NF][64];
  double b2[2][64];          // |b|^2 after the update, for the step size
  int out_of_range[2][2];
};
__device__ __forceinline__ void put_ygeom(Shared& s, const Axis& ax, int j, int l) {
  const FaceGeom g = face_geom(ax, j);
  s.geom[0][l] = double2{g.hlo, g.hup};
  s.geom[1][l] = double2{g.den, g.rden};
  s.geom[2][l] = double2{g.gup, g.denm};
  s.geom[3][l] = double2{g.rdenm, g.gdn};
  s.geom[4][l] = double2{g.denp, g.rdenp};
  s.geom[5][l] = double2{g.d, g.rd};
}
__device__ __forceinline__ FaceGeom get_ygeom(const Shared& s, int l) {
  const double2 a = s.geom[0][l], b = s.geom[1][l], c = s.geom[2][l], d = s.geom[3][l], e = s.geom[4][l],
                f = s.geom[5][l];
  return FaceGeom{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y, e.x, e.y, f.x, f.y, 0.0, 0.0};
}
// LDS written before is seen by both wavefronts after; loads from memory stay in flight
__device__ __forceinline__ void block_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// This lane's column in a strip.
struct Column {
  int j;                     // wrapped (periodic) or clamped
  bool interior, out;        // inside the interior bounds; this lane writes it
};

// Strip of a workgroup: launch index L mapped XCD-aware (xcd_tile) onto the strips in column-major
// order, so strips that run together on one XCD are x-neighbours and share their halo rows in L2.
__device__ __forceinline__ void strip_of(int L, int nstrips, int total, int& col, int& strip) {
  const int t = xcd_tile(L, total);
  col = t / nstrips;
  strip = t - col * nstrips;
}

// One wavefront's row: its transported quantities, and for the field the fluid values v needs.
template <int ROLE> struct Row;
template <> struct Row<FLUID> {
  double q[5];
  __device__ __forceinline__ bool out_of_range() const {
    RangeTest t;
    t.density(q[Q_RHO]);
#pragma unroll
    for (int k = Q_MX; k <= Q_TE; ++k) t.add(q[k]);
    return t.out();
  }
};
template <> struct Row<FIELD> {
  double q[6];
  double rho, m[3];
  __device__ __forceinline__ bool out_of_range() const {   // be is checked at set-up, the fluid by the other wavefront
    RangeTest t;
    t.add(q[Q_BIX]);
    t.add(q[Q_BIY]);
    t.add(q[Q_BIZ]);
    return t.out();
  }
};

// Rows and columns beyond a closed side are clamped to the grid: their values reach only the faces
// of ghost cells, whose derivatives are masked.
template <int ROLE>
__device__ __forceinline__ void load_row(const StageArgs& a, int i, uint32_t jb, Row<ROLE>& r) {
  const size_t row = (size_t)i * a.mesh.ny;
  lane_offset(jb);
  if constexpr (ROLE == FLUID) {
    r.q[Q_RHO] = ld_row(a.S.rho, row, jb);
    r.q[Q_MX] = ld_row(a.S.mx, row, jb);
    r.q[Q_MY] = ld_row(a.S.my, row, jb);
    r.q[Q_MZ] = ld_row(a.S.mz, row, jb);
    r.q[Q_TE] = ld_row(a.S.te, row, jb);
  } else {
    r.rho = ld_row(a.S.rho, row, jb);
    r.m[0] = ld_row(a.S.mx, row, jb);
    r.m[1] = ld_row(a.S.my, row, jb);
    r.m[2] = ld_row(a.S.mz, row, jb);
    r.q[Q_BIX] = ld_row(a.S.bx, row, jb);
    r.q[Q_BEX] = ld_row(a.st.bex, row & a.row_mask[ST_BEX], jb);
    r.q[Q_BIY] = ld_row(a.S.by, row, jb);
    r.q[Q_BEY] = ld_row(a.st.bey, row & a.row_mask[ST_BEY], jb);
    r.q[Q_BIZ] = ld_row(a.S.bz, row, jb);
    r.q[Q_BEZ] = ld_row(a.st.bez, row & a.row_mask[ST_BEZ], jb);
  }
}

// v = mom/rho (idealmhd.cpp:248-250), N components (the fluid's wavefront never needs v_z)
template <bool IN, int N>
__device__ __forceinline__ void velocities(double rho, const double* m, double* v) {
  const double rr = IN ? recip_in(rho) : 1.0 / rho;
#pragma unroll
  for (int k = 0; k < N; ++k) v[k] = IN ? qdiv_in(m[k], rho, rr) : qdiv_d(m[k], rho, rr);
}

// The inverse of IdealMHD::recomputeDT at one cell (idealmhd.cpp:279-304).  IN: rho, te, mom, b2, the mesh
// and gamma are in range and te is positive.  There |v| stands for sqrt(v*v), which equals it, and the slow speed,
// never above the fast one (or NaN with it), is left out of the maximum.
template <bool IN>
__device__ __forceinline__ double dt_inverse(double rho, double te, double mx, double my, double b2, const MhdConst& K,
                                             double dx, double rdx, double dy, double rdy) {
  const double press = te * K.gm1;
  if constexpr (IN) {
    const double rr = recip_in(rho);
    const double vx = qdiv_in(mx, rho, rr), vy = qdiv_in(my, rho, rr);
    const double bmag = b2 == 0.0 ? 0.0 : sqrt_in(b2);
    const double cs = sqrt_in(qdiv_in(press * K.gamma, rho, rr));
    const double cs2 = cs * cs;
    const double den = sqrt_in(rho * (4.0 * PI));
    const double va = qdiv_in(bmag, den, recip_in(den));
    const double va2 = va * va;
    const double sum = cs2 + va2, sum2 = sum * sum;
    const double delta = sqrt(1.0 - qdiv_in(cs2 * 4.0 * va2, sum2, recip_in(sum2)));
    const double vfast = sqrt_in(sum * 0.5 * (1.0 + delta));
    const double cmax = smax(smax(cs, va), vfast);
    return qdiv_in(__builtin_fabs(vx) + cmax, dx, rdx) + qdiv_in(__builtin_fabs(vy) + cmax, dy, rdy);
  } else {
    const double bmag = sqrt(b2);
    const double vx = mx / rho, vy = my / rho;
    const double cs = sqrt(press * K.gamma / rho);
    const double cs2 = cs * cs;
    const double va = bmag / sqrt(rho * (4.0 * PI));
    const double va2 = va * va;
    const double sum = cs2 + va2;
    const double delta = sqrt(1.0 - cs2 * 4.0 * va2 / (sum * sum));
    const double vfast = sqrt(sum * 0.5 * (1.0 + delta));
    const double vslow = sqrt(sum * 0.5 * (1.0 - delta));
    const double vmx = sqrt(vx * vx), vmy = sqrt(vy * vy);
    const double cmax = smax(smax(smax(cs, va), vfast), vslow);
    return qdiv(vmx + cmax, dx, rdx) + qdiv(vmy + cmax, dy, rdy);
  }
}
// What the fluid's wavefront keeps of an updated row until the field's |b|^2 of it is there, and the
// largest inverse step size so far (1/x falls as x grows, so the smallest step size is 1 over the
// largest inverse; a NaN never replaces it, as std::min drops it).  The mesh and gamma are in range: without
// that the host has the step size formed by a kernel of its own.
struct DtState {
  double rho, te, mx, my, dx, rdx;
  bool cell = false;           // this lane's cell takes part
  bool pending = false;
  double worst = 0.0;
  __device__ __forceinline__ void finish(double b2, const MhdConst& K, double dy, double rdy) {
    RangeTest t;
    t.density(rho);
    t.add(te);
    t.add(mx);
    t.add(my);
    t.add(b2);
    const bool out = t.out() || !(te > 0.0);
    double s;
    if (__any(cell && out)) s = dt_inverse<false>(rho, te, mx, my, b2, K, dx, rdx, dy, rdy);
    else s = dt_inverse<true>(rho, te, mx, my, b2, K, dx, rdx, dy, rdy);
    worst = (cell && s > worst) ? s : worst;
    pending = false;
  }
};

// Rows rs .. rend-1 of a strip for one of the block's two wavefronts.  IN: the untested divisions;
// every row is tested as it is loaded, and both wavefronts stop before the first row whose stencil
// holds a value out of range.  Returns the row they stopped at (rend when done).  SAME: the update's
// base is the set the derivatives are evaluated on.  DT: the final stage of a step that nothing but a
// ghost fill follows: the fluid's wavefront also forms the step size of each updated row, one row
// later, when the field's wavefront has put its |b|^2 into LDS.
template <int ROLE, int MODE, bool IN, bool SAME, bool DT>
__device__ __forceinline__ int march(const StageArgs& a, const Column& col, Shared& sh, double stepv, int rs, int rend,
                                     DtState& dt) {
  constexpr int NQ = ROLE == FLUID ? 5 : 6;     // transported quantities
  constexpr int NV = ROLE == FLUID ? 2 : 3;     // velocity components held per row
  constexpr int NO = ROLE == FLUID ? 5 : 3;     // evolved variables
  constexpr int O0 = ROLE == FLUID ? 0 : 5;     // the first of them in evolved order
  const Mesh& M = a.mesh;
  const MhdConst& K = a.k;
  const int nx = M.nx, ny = M.ny, lane = threadIdx.x;
  const size_t N = (size_t)nx * ny;
  const uint32_t jcol = 8u * (uint32_t)col.j;
  auto row_of = [&](int r) -> int { return M.x.per ? wrap_near(r, nx) : clampn(r, nx); };
  // whether either wavefront saw a value out of range, after the next barrier
  auto post_test = [&](bool bad, int slot) {
    const bool any = __any(bad);
    if (lane == 0) sh.out_of_range[slot][ROLE] = any ? 1 : 0;
  };
  auto tested_out = [&](int slot) -> bool {
    return __builtin_amdgcn_readfirstlane(sh.out_of_range[slot][0] | sh.out_of_range[slot][1]) != 0;
  };

  Row<ROLE> w[4], next;       // rotating window of rows r-1 .. r+2, and row r+3 arriving
  double v[2][NV], p[2];      // velocities and (fluid) pressure of rows r and r+1
  double Px[NQ];              // flux through row r's lower x-face
  double gdx, grdx;           // size of row r's cells
  double xiv[NV], xip = 0.0, xib0 = 0.0, xib1 = 0.0;   // interpolated values of that face
  auto derive = [&](const Row<ROLE>& r, double* vv, double& pp) {
    if constexpr (ROLE == FLUID) {
      velocities<IN, NV>(r.q[Q_RHO], r.q + Q_MX, vv);
      pp = r.q[Q_TE] * K.gm1;                          // press = (gamma-1) te (idealmhd.cpp:253)
    } else {
      velocities<IN, NV>(r.rho, r.m, vv);
      pp = 0.0;
    }
  };

  {  // prologue: rows rs-2 .. rs+1 and the lower x-face of row rs
    load_row<ROLE>(a, row_of(rs - 2), jcol, w[3]);
    load_row<ROLE>(a, row_of(rs - 1), jcol, w[0]);
    load_row<ROLE>(a, row_of(rs), jcol, w[1]);
    load_row<ROLE>(a, row_of(rs + 1), jcol, w[2]);
    load_row<ROLE>(a, row_of(rs + 2), jcol, next);
    if (IN) {
      post_test(w[3].out_of_range() || w[0].out_of_range() || w[1].out_of_range() || w[2].out_of_range(), (rs + 1) & 1);
      block_barrier();
      if (tested_out((rs + 1) & 1)) return rs;
    }
    double vt[NV], pt;
    derive(w[0], vt, pt);
    derive(w[1], v[0], p[0]);
    const FaceGeom gx = face_geom_row(M.x, rs);
    gdx = gx.d;
    grdx = gx.rd;
#pragma unroll
    for (int k = 0; k < NV; ++k)
      if (ROLE == FIELD || k == 0) xiv[k] = interp<IN>(gx, vt[k], v[0][k]);
    if (ROLE == FLUID) xip = interp<IN>(gx, pt, p[0]);
    const FaceDir fd = face_dir(xiv[0], gx);
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
      double d2;
      Px[k] = face_flux<IN>(w[3].q[k], w[0].q[k], w[1].q[k], w[2].q[k], gx, fd, d2);
      if (ROLE == FIELD && k == Q_BIY) xib0 = d2;
      if (ROLE == FIELD && k == Q_BIZ) xib1 = d2;
    }
  }

  // one row; false when the march ends before it
  auto step = [&](auto BC, int r) -> bool {
    constexpr int B = decltype(BC)::value;
    constexpr int SM = B % 4, S0 = (B + 1) % 4, S1 = (B + 2) % 4, S2 = (B + 3) % 4;
    constexpr int D0 = B % 2, D1 = (B + 1) % 2;
    if (r >= rend) return false;
    const int slot = r & 1;
    // row r+2 was asked for a row ago; row r+3, the update's base and gravity are on their way while
    // row r is computed
    w[S2] = next;
    load_row<ROLE>(a, row_of(r + 3), jcol, next);
    const size_t row = (size_t)r * ny;
    uint32_t jb = jcol;
    lane_offset(jb);
    double b[NO], grx = 0.0, gry = 0.0;
    if constexpr (ROLE == FLUID) {
      if (!SAME) {
        b[0] = ld_row(a.B.rho, row, jb); b[1] = ld_row(a.B.mx, row, jb); b[2] = ld_row(a.B.my, row, jb);
        b[3] = ld_row(a.B.mz, row, jb); b[4] = ld_row(a.B.te, row, jb);
      }
      grx = ld_row(a.st.gx, row & a.row_mask[ST_GX], jb);
      gry = ld_row(a.st.gy, row & a.row_mask[ST_GY], jb);
    } else if (!SAME) {
      b[0] = ld_row(a.B.bx, row, jb); b[1] = ld_row(a.B.by, row, jb); b[2] = ld_row(a.B.bz, row, jb);
    }
    const FaceGeom gx = face_geom_row(M.x, r + 1);
    const double dx = gdx, rdx = grdx;   // cell r's size came with its lower face
    gdx = gx.d;
    grdx = gx.rd;
    // lower y-face of this lane's column in row r (cells j-2, j-1, j, j+1 from neighbouring lanes):
    // the upper y-face of the column is the next lane's lower one
    const FaceGeom gy = get_ygeom(sh, lane);
    auto ddx = [&](double up, double lo) { return qdiv_t<IN>(up - lo, dx, rdx); };
    auto ddy = [&](double lo) { return qdiv_t<IN>(shl1(lo) - lo, gy.d, gy.rd); };
    const double fvy = interp<IN>(gy, shr1(v[D0][1]), v[D0][1]);
    const FaceDir fdy = face_dir(fvy, gy);
    // derivative1D along y (derivs.cpp:259)
    const double dvy_y = ddy(fvy);
    double dpy = 0.0, dvx_y = 0.0, dvz_y = 0.0, dbix_y = 0.0, dbiz_y = 0.0;
    if constexpr (ROLE == FLUID) {
      dpy = ddy(interp<IN>(gy, shr1(p[D0]), p[D0]));
    } else {
      dvx_y = ddy(interp<IN>(gy, shr1(v[D0][0]), v[D0][0]));
      dvz_y = ddy(interp<IN>(gy, shr1(v[D0][2]), v[D0][2]));
    }
    double tdiv[NQ];       // y part first; the x part is added when the upper x-face is known
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
      const double qc = w[S0].q[k];
      const double qm1 = shr1(qc);
      const double qm2 = shr1(qm1);
      const double qp1 = shl1(qc);
      double d2;
      const double Pl = face_flux<IN>(qm2, qm1, qc, qp1, gy, fdy, d2);
      if (ROLE == FIELD && k == Q_BIX) dbix_y = ddy(d2);
      if (ROLE == FIELD && k == Q_BIZ) dbiz_y = ddy(d2);
      tdiv[k] = ddy(Pl);
    }
    // row r+2: its values are the only ones of row r's stencil not tested yet
    if (IN) post_test(w[S2].out_of_range(), slot);
    // upper x-face of row r from rows r-1 .. r+2; divergence term (up - lo)/dx + y term
    derive(w[S1], v[D1], p[D1]);
    double dpx = 0.0, dvx_x = 0.0, dvy_x = 0.0, dvz_x = 0.0, dbiy_x = 0.0, dbiz_x = 0.0;
    {
      double niv[NV];
#pragma unroll
      for (int k = 0; k < NV; ++k)
        if (ROLE == FIELD || k == 0) niv[k] = interp<IN>(gx, v[D0][k], v[D1][k]);
      const FaceDir fd = face_dir(niv[0], gx);
      dvx_x = ddx(niv[0], xiv[0]);
      xiv[0] = niv[0];
      if constexpr (ROLE == FLUID) {
        const double nip = interp<IN>(gx, p[D0], p[D1]);
        dpx = ddx(nip, xip);
        xip = nip;
      } else {
        dvy_x = ddx(niv[1], xiv[1]);
        dvz_x = ddx(niv[2], xiv[2]);
        xiv[1] = niv[1];
        xiv[2] = niv[2];
      }
#pragma unroll
      for (int k = 0; k < NQ; ++k) {
        double d2;
        const double Pn = face_flux<IN>(w[SM].q[k], w[S0].q[k], w[S1].q[k], w[S2].q[k], gx, fd, d2);
        if (ROLE == FIELD && k == Q_BIY) { dbiy_x = ddx(d2, xib0); xib0 = d2; }
        if (ROLE == FIELD && k == Q_BIZ) { dbiz_x = ddx(d2, xib1); xib1 = d2; }
        const double tx = ddx(Pn, Px[k]);
        tdiv[k] = tx + tdiv[k];
        Px[k] = Pn;
      }
    }
    const double* qc = w[S0].q;
    if constexpr (ROLE == FIELD) {
      // the momentum equations' field terms (idealmhd.cpp:54-60), in the order they are summed
      const double bix = qc[Q_BIX], biy = qc[Q_BIY], biz = qc[Q_BIZ];
      const double bex = qc[Q_BEX], bey = qc[Q_BEY], bez = qc[Q_BEZ];
      const double curl_db = qdiv_t<IN>(dbiy_x - dbix_y, 4.0 * PI, K.r4pi);
      const double cz0 = dbiz_y, cz1 = -dbiz_x;
      const double bzi = qdiv_t<IN>(biz, 4.0 * PI, K.r4pi), bze = qdiv_t<IN>(bez, 4.0 * PI, K.r4pi);
      double(*f)[64] = sh.force[slot];
      f[F_EXT0][lane] = (-curl_db) * bey;
      f[F_EXT1][lane] = curl_db * bex;
      f[F_IN0][lane] = (-curl_db) * biy;
      f[F_IN1][lane] = curl_db * bix;
      f[F_INZ0][lane] = bzi * cz1;
      f[F_INZ1][lane] = (-bzi) * cz0;
      f[F_EXTZ0][lane] = bze * cz1;
      f[F_EXTZ1][lane] = (-bze) * cz0;
      f[F_ZEXT][lane] = qdiv_t<IN>(cz0 * bey - cz1 * bex, 4.0 * PI, K.r4pi);
      f[F_ZIN][lane] = qdiv_t<IN>(cz0 * biy - cz1 * bix, 4.0 * PI, K.r4pi);
    }
    block_barrier();
    if (DT && ROLE == FLUID && dt.pending) dt.finish(sh.b2[slot ^ 1][lane], K, gy.d, gy.rd);
    if (IN && tested_out(slot)) return false;
    if (!DT && !col.out) return true;
    double o_rho = 1.0, o_te = 1.0, o_mx = 0.0, o_my = 0.0, o_b2 = 0.0;   // what the step size reads
    if (!DT || col.out) {
    double k8[NO];
    if (r >= M.x.lo && r <= M.x.hi && col.interior) {
      if constexpr (ROLE == FLUID) {
        const double rho = qc[Q_RHO], vx = v[D0][0], vy = v[D0][1];
        const double(*f)[64] = sh.force[slot];
        k8[0] = -tdiv[Q_RHO] + 0.0;
        k8[1] = (-tdiv[Q_MX] - dpx + rho * grx + f[F_EXT0][lane] + f[F_IN0][lane] + f[F_INZ0][lane] + f[F_EXTZ0][lane]) +
                (IN ? 0.0 : rho * 0.0 + vx * 0.0);
        k8[2] = (-tdiv[Q_MY] - dpy + rho * gry + f[F_EXT1][lane] + f[F_IN1][lane] + f[F_INZ1][lane] + f[F_EXTZ1][lane]) +
                (IN ? 0.0 : rho * 0.0 + vy * 0.0);
        // v_z enters only through v_z * 0 (NaN or a zero's sign)
        k8[3] = (-tdiv[Q_MZ] + f[F_ZEXT][lane] + f[F_ZIN][lane]) +
                (IN ? 0.0 : rho * 0.0 + (qc[Q_MZ] / rho) * 0.0);
        k8[4] = (-tdiv[Q_TE] - p[D0] * (dvx_x + dvy_y)) + 0.0;
      } else {
        const double btx = qc[Q_BIX] + qc[Q_BEX], bty = qc[Q_BIY] + qc[Q_BEY];
        k8[0] = (-tdiv[Q_BIX] - tdiv[Q_BEX] + btx * dvx_x + bty * dvx_y) + 0.0;
        k8[1] = (-tdiv[Q_BIY] - tdiv[Q_BEY] + btx * dvy_x + bty * dvy_y) + 0.0;
        k8[2] = (-tdiv[Q_BIZ] - tdiv[Q_BEZ] + btx * dvz_x + bty * dvz_y) + 0.0;
      }
    } else if (a.moc) {  // open_moc ghost cells: masked RHS (0) + characteristic terms (idealmhd.cpp:99-103)
#pragma unroll
      for (int o = 0; o < NO; ++o) k8[o] = 0.0 + ld_row(a.moc, (O0 + o) * N + row, jb);
    } else {
#pragma unroll
      for (int o = 0; o < NO; ++o) k8[o] = 0.0;
    }
    for (int e = 0; e < a.n_extra; ++e) {
#pragma unroll
      for (int o = 0; o < NO; ++o)
        if (O0 + o == a.extra_var[e]) k8[o] = k8[o] + ld_row(a.extra[e], row, jb);
    }
    if (MODE == STAGE_STORE_K) {
#pragma unroll
      for (int o = 0; o < NO; ++o) st_row(a.kbuf, (O0 + o) * N + row, jb, k8[o]);
    } else if (MODE == STAGE_RK4_FINAL) {
#pragma unroll
      for (int o = 0; o < NO; ++o) {
        const double k1 = ld_row(a.kbuf, (O0 + o) * N + row, jb), k2 = ld_row(a.k2buf, (O0 + o) * N + row, jb),
                     k3 = ld_row(a.k3buf, (O0 + o) * N + row, jb);
        k8[o] = qdiv(k1 + k8[o], 6.0, K.r6) + qdiv(k2 + k3, 3.0, K.r3);
      }
      if (a.kf_out) {
#pragma unroll
        for (int o = 0; o < NO; ++o) st_row(a.kf_out, (O0 + o) * N + row, jb, k8[o]);
      }
    }
    if (SAME) {
#pragma unroll
      for (int o = 0; o < NO; ++o) b[o] = ROLE == FLUID ? qc[o] : qc[2 * o];
    }
    if constexpr (ROLE == FLUID) {
      const double rho_new = b[0] + k8[0] * stepv;
      const double rho1 = smax(qdiv(rho_new, K.m, K.rm), K.nmin) * K.m;
      const double te1 = smax(b[4] + k8[4] * stepv, K.temin);
      const double n = smax(qdiv(rho1, K.m, K.rm), K.nmin);
      o_rho = n * K.m;
      o_mx = b[1] + k8[1] * stepv;
      o_my = b[2] + k8[2] * stepv;
      o_te = smax(te1, K.temin);
      st_row(a.T.rho, row, jb, o_rho);
      if (a.write_n) st_row(a.T.n, row, jb, n);
      if (a.write_pre) st_row(a.T.rho_pre, row, jb, rho1);
      st_row(a.T.mx, row, jb, o_mx);
      st_row(a.T.my, row, jb, o_my);
      st_row(a.T.mz, row, jb, b[3] + k8[3] * stepv);
      st_row(a.T.te, row, jb, o_te);
    } else {
      const double nbx = b[0] + k8[0] * stepv, nby = b[1] + k8[1] * stepv, nbz = b[2] + k8[2] * stepv;
      st_row(a.T.bx, row, jb, nbx);
      st_row(a.T.by, row, jb, nby);
      st_row(a.T.bz, row, jb, nbz);
      if (DT) {
        const double bx = qc[Q_BEX] + nbx, by = qc[Q_BEY] + nby, bz = qc[Q_BEZ] + nbz;
        o_b2 = bx * bx + by * by + bz * bz;
      }
    }
    }
    if (DT && ROLE == FIELD) sh.b2[slot][lane] = o_b2;
    if (DT && ROLE == FLUID) {
      // a fixed or reflecting side's ghost fill zeroes the momenta of the interior row next to it
      const bool still = (r == M.x.lo && (a.dt_still & 1)) || (r == M.x.hi && (a.dt_still & 2)) ||
                         (col.j == M.y.lo && (a.dt_still & 4)) || (col.j == M.y.hi && (a.dt_still & 8));
      dt.rho = o_rho;
      dt.te = o_te;
      dt.mx = still ? 0.0 : o_mx;
      dt.my = still ? 0.0 : o_my;
      dt.dx = dx;
      dt.rdx = rdx;
      dt.cell = col.out && col.interior && r >= M.x.lo && r <= M.x.hi;
      dt.pending = true;
    }
    return true;
  };

  for (int r = rs; r < rend; r += 4) {
    if (!step(std::integral_constant<int, 0>{}, r)) return r;
    if (!step(std::integral_constant<int, 1>{}, r + 1)) return r + 1;
    if (!step(std::integral_constant<int, 2>{}, r + 2)) return r + 2;
    if (!step(std::integral_constant<int, 3>{}, r + 3)) return r + 3;
  }
  return rend;
}

template <int ROLE, int MODE, bool SAME, bool DT>
__device__ __forceinline__ void strip_rows(const StageArgs& a, const Column& col, Shared& sh, double stepv, int r,
                                           int rend) {
  DtState dt;
  if (a.in_range) r = march<ROLE, MODE, true, SAME, DT>(a, col, sh, stepv, r, rend, dt);
  if (r < rend) (void)march<ROLE, MODE, false, SAME, DT>(a, col, sh, stepv, r, rend, dt);
  if constexpr (DT) {
    block_barrier();
    if constexpr (ROLE == FLUID) {
      const double2 d = sh.geom[5][threadIdx.x];
      if (dt.pending) dt.finish(sh.b2[(rend - 1) & 1][threadIdx.x], a.k, d.x, d.y);
      double m = dt.worst;
      for (int off = 32; off > 0; off >>= 1) {
        const double o = __shfl_xor(m, off, 64);
        m = m < o ? o : m;
      }
      if (threadIdx.x == 0) a.dt_partial[blockIdx.x] = m > 0.0 ? 1.0 / m : DBL_MAX;
    }
  }
}

template <int MODE, bool SAME, bool DT>
__global__ void __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(2)))
k_mhd_stage_strip(StageArgs a, int R, int nstrips) {
  const Mesh& M = a.mesh;
  __shared__ Shared sh;
  const int lane = threadIdx.x;
  int tile, strip;
  strip_of(blockIdx.x, nstrips, gridDim.x, tile, strip);
  const int jraw = tile * OUT_COLS + lane - 2;
  Column col;
  bool valid = true;
  if (M.y.per) col.j = wrapn(jraw, M.ny);
  else { valid = jraw >= 0 && jraw < M.ny; col.j = clampn(jraw, M.ny); }
  col.out = lane >= 2 && lane < 62 && jraw >= 0 && jraw < M.ny;
  col.interior = valid && col.j >= M.y.lo && col.j <= M.y.hi;
  const double stepv = a.step_mult * (*a.step);
  const int r0 = strip * R, rend = min(r0 + R, M.nx);
  put_ygeom(sh, M.y, col.j, lane);   // both wavefronts write, and each reads, the same values
  if (__builtin_amdgcn_readfirstlane(threadIdx.y) == 0) strip_rows<FLUID, MODE, SAME, DT>(a, col, sh, stepv, r0, rend);
  else strip_rows<FIELD, MODE, SAME, DT>(a, col, sh, stepv, r0, rend);
}

}  // namespace

int mhd_strip_rows_default(int nx, int ny) {
  // 1024 blocks (2 wavefronts per SIMD) run at once and a strip costs its rows plus about three (four
  // halo rows read, one face and the start of the pipeline): the height with the least rounds x cost,
  // the taller one of equals, which reads fewer halo rows
  const long tiles = (ny + OUT_COLS - 1) / OUT_COLS;
  int best = 1;
  long least = 0;
  for (int R = 1; R <= 96; ++R) {
    const long rounds = (tiles * ((nx + R - 1) / R) + 1023) / 1024;
    const long cost = rounds * (R + 3);
    if (R == 1 || cost <= least) { best = R; least = cost; }
  }
  return best;
}

int mhd_strip_blocks(const Mesh& m, int R) {
  return ((m.ny + OUT_COLS - 1) / OUT_COLS) * ((m.nx + R - 1) / R);
}

void launch_mhd_stage_strip(const StageArgs& a, int R, hipStream_t s) {
  const int nstrips = (a.mesh.nx + R - 1) / R;
  const dim3 grid(mhd_strip_blocks(a.mesh, R));
  const bool same = a.B.rho == a.S.rho;
  auto go = [&](auto mode, auto is_same, auto dt) {
    hipLaunchKernelGGL((k_mhd_stage_strip<decltype(mode)::value, decltype(is_same)::value, decltype(dt)::value>), grid,
                       dim3(64, 2), 0, s, a, R, nstrips);
  };
  using Y = std::true_type;
  using No = std::false_type;
  const std::integral_constant<int, STAGE_PLAIN> plain{};
  const std::integral_constant<int, STAGE_STORE_K> store{};
  const std::integral_constant<int, STAGE_RK4_FINAL> final4{};
  if (a.mode == STAGE_STORE_K) same ? go(store, Y{}, No{}) : go(store, No{}, No{});
  else if (a.mode == STAGE_RK4_FINAL) a.dt_partial ? go(final4, No{}, Y{}) : go(final4, No{}, No{});
  else if (a.dt_partial) same ? go(plain, Y{}, Y{}) : go(plain, No{}, Y{});
  else same ? go(plain, Y{}, No{}) : go(plain, No{}, No{});
}

}  // namespace spruce
