// Thermal conduction and radiative-loss kernels for gfx950 (reference:
// source/modules/solar/thermalconduction.cpp, radiativelosses.cpp).  Operation order and rounding
// follow the reference whole-grid expressions; powers are correctly rounded (crpow.hpp).
#include <cfloat>

#include "arith.hpp"
#include "crpow.hpp"
#include "solar.hpp"
#include "strip.hpp"
#include "tc_cell.hpp"
#include "tc_strip.hpp"

namespace spruce {
namespace {

__device__ __forceinline__ int wrp(int k, int n, int per) {
  if (per) {
    if (k < 0) k += n;
    else if (k >= n) k -= n;
  }
  return k;
}
__device__ __forceinline__ bool inside(const Mesh& M, int i, int j) {
  return i >= M.x.lo && i <= M.x.hi && j >= M.y.lo && j <= M.y.hi;
}
// temp = max((gamma-1) te / (2 K_B n), temp_min) (thermalconduction.cpp:109; idealmhd.cpp:254)
__device__ __forceinline__ double temp_of(double te, double n, const MhdConst& K) {
  return smax(te * K.gm1 / (n * (2.0 * K_B)), K.tmin);
}
// boundaryInterpolate across the face whose upper cell is c on axis ax (derivs.cpp:477-487)
__device__ __forceinline__ double fint(const Axis& ax, int c, int cm1, double qlo, double qup) {
  return qdiv(qlo * ax.h[c] + qup * ax.h[cm1], ax.fden[c], ax.rfden[c]);
}

__device__ __forceinline__ double block_reduce(double v, bool is_min) {
  for (int off = 32; off > 0; off >>= 1) {
    const double o = __shfl_xor(v, off, 64);
    v = is_min ? ((o < v) ? o : v) : ((v < o) ? o : v);
  }
  __shared__ double part[16];
  const int lane = threadIdx.x + threadIdx.y * blockDim.x;
  __syncthreads();
  if ((lane & 63) == 0) part[lane >> 6] = v;
  __syncthreads();
  if (lane == 0) {
    const int nw = (blockDim.x * blockDim.y + 63) >> 6;
    double m = part[0];
    for (int k = 1; k < nw; ++k) m = is_min ? ((part[k] < m) ? part[k] : m) : ((m < part[k]) ? part[k] : m);
    v = m;
  }
  return v;
}

__device__ __forceinline__ void bhat_at(const MhdSet& L, const MhdStatic& st, size_t c, double& hx, double& hy) {
  const double bx = st.bex[c] + L.bx[c], by = st.bey[c] + L.by[c], bz = st.bez[c] + L.bz[c];
  const double bm = sqrt(bx * bx + by * by + bz * bz);
  hx = bm == 0.0 ? 0.0 : bx / bm;
  hy = bm == 0.0 ? 0.0 : by / bm;
}

__global__ void __launch_bounds__(256) k_bhat(MhdSet L, MhdStatic st, Mesh M, double* bhx, double* bhy) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x, i = blockIdx.y * blockDim.y + threadIdx.y;
  if (i >= M.nx || j >= M.ny) return;
  const size_t c = (size_t)i * M.ny + j;
  double hx, hy;
  bhat_at(L, st, c, hx, hy);
  bhx[c] = hx;
  bhy[c] = hy;
}

__global__ void __launch_bounds__(256) k_bhat_derivs(const double* bhx, const double* bhy, Mesh M, double* dbxx,
                                                     double* dbxy, double* dbyx, double* dbyy) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x, i = blockIdx.y * blockDim.y + threadIdx.y;
  if (i >= M.nx || j >= M.ny) return;
  const size_t c = (size_t)i * M.ny + j;
  double r[4] = {0.0, 0.0, 0.0, 0.0};
  if (inside(M, i, j)) {
    const int ny = M.ny;
    const int im = wrp(i - 1, M.nx, M.x.per), ip = wrp(i + 1, M.nx, M.x.per);
    const int jm = wrp(j - 1, M.ny, M.y.per), jp = wrp(j + 1, M.ny, M.y.per);
    const size_t cxm = (size_t)im * ny + j, cxp = (size_t)ip * ny + j, cym = (size_t)i * ny + jm, cyp = (size_t)i * ny + jp;
    const double dx = M.x.d[i], rdx = M.x.rd[i], dy = M.y.d[j], rdy = M.y.rd[j];
    const double bx = bhx[c], by = bhy[c];
    r[0] = qdiv(fint(M.x, ip, i, bx, bhx[cxp]) - fint(M.x, i, im, bhx[cxm], bx), dx, rdx);
    r[1] = qdiv(fint(M.y, jp, j, bx, bhx[cyp]) - fint(M.y, j, jm, bhx[cym], bx), dy, rdy);
    r[2] = qdiv(fint(M.x, ip, i, by, bhy[cxp]) - fint(M.x, i, im, bhy[cxm], by), dx, rdx);
    r[3] = qdiv(fint(M.y, jp, j, by, bhy[cyp]) - fint(M.y, j, jm, bhy[cym], by), dy, rdy);
  }
  dbxx[c] = r[0]; dbxy[c] = r[1]; dbyx[c] = r[2]; dbyy[c] = r[3];
}

// Field-aligned conductive flux at an interior cell and its saturated magnitude
// (thermalconduction.cpp:198-232).
// IN: T and rho in range (range.hpp), so that T^2.5 and (T K_B)^1.5 need no operand tests.
struct SatFlux { double fx, fy, fm, sfm; };
template <bool IN = false>
__device__ __forceinline__ SatFlux sat_flux(double T, double gx, double gy, double rho, double bx, double by,
                                            double dx, double dy, const TcParams& p, const MhdConst& K) {
  const double kmax = qdiv(dx * dy * K_B * qdiv(rho, K.m, K.rm), p.dsm, 1.0 / p.dsm);
  double t15 = 0.0, t25, k15, k25 = 0.0;
  if (IN) {
    pow_1p5_2p5_in(T, t15, t25);
    pow_1p5_2p5_in(T * K_B, k15, k25);
  } else {
    t25 = pow_2p5(T);
    k15 = pow_1p5(T * K_B);
  }
  const double kap = smin(t25 * p.k0, kmax);
  const double cfx = (-kap) * gx, cfy = (-kap) * gy;
  const double fmag = cfx * bx + cfy * by;
  SatFlux s;
  s.fx = fmag * bx;
  s.fy = fmag * by;
  const double sat = qdiv(rho, K.m, K.rm) * p.c_sat * k15 / p.sqrt_me;
  s.fm = sqrt(s.fx * s.fx + s.fy * s.fy);
  const double scale = sat / sqrt(sat * sat + s.fm * s.fm);
  const double sx = s.fx * scale, sy = s.fy * scale;
  s.sfm = sqrt(sx * sx + sy * sy);
  return s;
}

// Central gradient of T at (i,j) from the temperatures of its four neighbours.
__device__ __forceinline__ void grad_at(const Mesh& M, int i, int j, double Tc, double Txm, double Txp, double Tym,
                                        double Typ, double& gx, double& gy) {
  const int ip = wrp(i + 1, M.nx, M.x.per), jp = wrp(j + 1, M.ny, M.y.per);
  const int im = wrp(i - 1, M.nx, M.x.per), jm = wrp(j - 1, M.ny, M.y.per);
  gx = qdiv(fint(M.x, ip, i, Tc, Txp) - fint(M.x, i, im, Txm, Tc), M.x.d[i], M.x.rd[i]);
  gy = qdiv(fint(M.y, jp, j, Tc, Typ) - fint(M.y, j, jm, Tym, Tc), M.y.d[j], M.y.rd[j]);
}

// The conduction time scale at an interior cell and, with saturation, |b_hat . grad T|
// (thermalconduction.cpp:179-193).
__device__ __forceinline__ void tc_timescale(const MhdSet& L, double bx, double by, const TcParams& p, const MhdConst& K,
                                             const Mesh& M, int i, int j, double& dts, double& ft) {
  auto T = [&](int a, int b) {
    const size_t q = (size_t)wrp(a, M.nx, M.x.per) * M.ny + wrp(b, M.ny, M.y.per);
    return temp_of(L.te[q], L.n[q], K);
  };
  const double Tc = T(i, j);
  const double rho = L.rho[(size_t)i * M.ny + j];
  if (!p.saturation) {
    // K_B/(w kappa_0) * (rho/m) * d_x * d_y / T^2.5 (thermalconduction.cpp:183)
    dts = qdiv(rho, K.m, K.rm) * p.c1 * M.x.d[i] * M.y.d[j] / pow_2p5(Tc);
  } else {
    double gx, gy;
    grad_at(M, i, j, Tc, T(i - 1, j), T(i + 1, j), T(i, j - 1), T(i, j + 1), gx, gy);
    const double ftg = gx * bx + gy * by;
    ft = fabs(ftg);
    const SatFlux s = sat_flux(Tc, gx, gy, rho, bx, by, M.x.d[i], M.y.d[j], p, K);
    const double kap = fabs(s.sfm / ftg);                  // saturatedKappa (:236-248)
    dts = K_B / kap * qdiv(rho, K.m, K.rm) * M.x.d[i] * M.y.d[j];
  }
}

// Block k: module k's minimum and maximum over the blocks of k_step_pre, straight to the host's copy;
// the first block also copies the step size and the error flag.  Each block then stores the ticket in its
// place behind them, which the host polls: it has the values when it sees the store, where a stream
// synchronisation also waits for the launch to retire and for a marker behind it.
__global__ void __launch_bounds__(1024) k_finish_scalars(const double* partial, int nblocks, int njobs, const double* step,
                                                         const int* err, double* host_out, uint64_t ticket) {
  if ((int)blockIdx.x < njobs) {
    const double* pmin = partial + (size_t)2 * nblocks * blockIdx.x;
    const double* pmax = pmin + nblocks;
    double a = DBL_MAX, b = -DBL_MAX;
    for (int k = threadIdx.x; k < nblocks; k += blockDim.x) {
      a = (pmin[k] < a) ? pmin[k] : a;
      b = (b < pmax[k]) ? pmax[k] : b;
    }
    a = block_reduce(a, true);
    b = block_reduce(b, false);
    if (threadIdx.x == 0) { host_out[2 * blockIdx.x] = a; host_out[2 * blockIdx.x + 1] = b; }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    host_out[2 * njobs] = *step;
    host_out[2 * njobs + 1] = (double)*err;
  }
  if (threadIdx.x == 0)
    __hip_atomic_store(reinterpret_cast<uint64_t*>(host_out) + 2 * njobs + 2 + blockIdx.x, ticket, __ATOMIC_RELEASE,
                       __HIP_MEMORY_SCOPE_SYSTEM);
}

__global__ void __launch_bounds__(256) k_tc_sat(const double* te, const double* n, const double* rho, const double* bhx,
                                                const double* bhy, TcParams p, MhdConst K, Mesh M, double* rx,
                                                double* ry, double* coef) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x, i = blockIdx.y * blockDim.y + threadIdx.y;
  if (i >= M.nx || j >= M.ny) return;
  const size_t c = (size_t)i * M.ny + j;
  if (!inside(M, i, j)) { rx[c] = 0.0; ry[c] = 0.0; coef[c] = 1.0; return; }
  auto T = [&](int a, int b) {
    const size_t q = (size_t)wrp(a, M.nx, M.x.per) * M.ny + wrp(b, M.ny, M.y.per);
    return temp_of(te[q], n[q], K);
  };
  const double Tc = T(i, j);
  double gx, gy;
  grad_at(M, i, j, Tc, T(i - 1, j), T(i + 1, j), T(i, j - 1), T(i, j + 1), gx, gy);
  const SatFlux s = sat_flux(Tc, gx, gy, rho[c], bhx[c], bhy[c], M.x.d[i], M.y.d[j], p, K);
  rx[c] = s.fx;
  ry[c] = s.fy;
  coef[c] = s.fm != 0.0 ? s.sfm / s.fm : 1.0;                  // thermalconduction.cpp:264-268
}

// ThermalConduction::thermalEnergyDerivative at an interior cell (thermalconduction.cpp:158-176),
// from the temperatures of its 3x3 neighbourhood: the unsaturated part (tc_cell.hpp), then the
// saturation factor and correction.
__device__ double tc_energy_derivative(const TcStepArgs& a, int i, int j, const double T[3][3]) {
  const Mesh& M = a.mesh;
  const int ny = M.ny;
  const int im = wrp(i - 1, M.nx, M.x.per), ip = wrp(i + 1, M.nx, M.x.per);
  const int jm = wrp(j - 1, M.ny, M.y.per), jp = wrp(j + 1, M.ny, M.y.per);
  const double dx = M.x.d[i], rdx = M.x.rd[i], dy = M.y.d[j], rdy = M.y.rd[j];
  // b_hat and its derivatives (frozen for the step, computed once by k_bhat_derivs)
  const size_t c = (size_t)i * ny + j;
  const size_t cxm = (size_t)im * ny + j, cxp = (size_t)ip * ny + j, cym = (size_t)i * ny + jm, cyp = (size_t)i * ny + jp;
  double result = tcc::tc_core<double>(M, i, j, T, a.bhx[c], a.bhy[c], a.dbxx[c], a.dbxy[c], a.dbyx[c], a.dbyy[c],
                                       a.p.k0);
  if (a.p.saturation) {                                         // thermalconduction.cpp:171-174, 255-271
    const double cc = a.coef[c];
    const double dcx = qdiv(fint(M.x, ip, i, cc, a.coef[cxp]) - fint(M.x, i, im, a.coef[cxm], cc), dx, rdx);
    const double dcy = qdiv(fint(M.y, jp, j, cc, a.coef[cyp]) - fint(M.y, j, jm, a.coef[cym], cc), dy, rdy);
    const double add = -1.0 * (dcx * a.rx[c] + dcy * a.ry[c]);
    result = cc * result + add;
  }
  return result;
}

// One conduction update.  The block's temperatures and a one-cell halo are computed once into LDS
// (each temperature is a division), then every cell reads its 3x3 neighbourhood from there.
__global__ void __launch_bounds__(256) k_tc_step(TcStepArgs a) {
  constexpr int BX = 64, BY = 4;
  __shared__ double Ts[BY + 2][BX + 2];
  const Mesh& M = a.mesh;
  const int j0 = blockIdx.x * BX, i0 = blockIdx.y * BY;
  for (int t = threadIdx.y * BX + threadIdx.x; t < (BY + 2) * (BX + 2); t += BX * BY) {
    const int r = t / (BX + 2), q = t - r * (BX + 2);
    const int ii = wrp(i0 - 1 + r, M.nx, M.x.per), jj = wrp(j0 - 1 + q, M.ny, M.y.per);
    double v = 0.0;
    if (ii >= 0 && ii < M.nx && jj >= 0 && jj < M.ny) {
      const size_t cc = (size_t)ii * M.ny + jj;
      v = temp_of(a.te_src[cc], a.n[cc], a.k);
    }
    Ts[r][q] = v;
  }
  __syncthreads();
  const int j = j0 + threadIdx.x, i = i0 + threadIdx.y;
  if (i >= M.nx || j >= M.ny) return;
  const size_t c = (size_t)i * M.ny + j;
  const double base = a.te_base[c];
  if (!inside(M, i, j)) {
    // mask = 0: te + 0*dE; every derivative is zero there, so dE = 0
    a.te_out[c] = smax(base + 0.0, a.k.temin);
    if (a.mode == TC_STORE_K) a.k_out[c] = 0.0;
    return;
  }
  double T[3][3];
#pragma unroll
  for (int a1 = 0; a1 < 3; ++a1)
#pragma unroll
    for (int b1 = 0; b1 < 3; ++b1) T[a1][b1] = Ts[threadIdx.y + a1][threadIdx.x + b1];
  double dE = tc_energy_derivative(a, i, j, T);
  double v;
  if (a.mode == TC_RK4_FINAL) {
    const double sum = a.k1[c] + 2.0 * a.k2[c] + 2.0 * a.k3[c] + dE;
    v = base + qdiv(1.0 * a.h * sum, 6.0, a.k.r6);
  } else {
    if (a.mode == TC_STORE_K) a.k_out[c] = dE;
    v = base + 1.0 * (a.mult * a.h) * dE;
  }
  a.te_out[c] = smax(v, a.k.temin);
}

// Strip form of one conduction update (the production path of launch_tc_step).  One 64-lane
// wavefront owns 64 consecutive columns (y) and marches down R rows (x): lane l holds column
// 62*tile + l - 1, lanes 1..62 write outputs and lanes 0, 63 are the y-halo.  Every face value the
// energy derivative takes -- the interpolants of T, of dT/dx along y, of dT/dy along x and of b_hat
// along both axes -- is computed once and shared by the two cells of the face: along y through DPP
// lane shifts, along x by keeping the previous row's faces in registers.  The derivatives of the
// frozen b_hat are formed here from b_hat, so a subcycle reads te, n, b_hat_x, b_hat_y and writes
// te.  Each value is the same sequence of IEEE operations as tc_core's (tc_cell.hpp), so the result
// is bit-identical to the one-thread-per-cell form.
//
// What bounds it: HBM and the latency of a row's chain.  A 2048x2048 subcycle moves at least 168 MB
// (40 B per cell), 34 us at the 4.9 TB/s a large copy reaches here; a 23-row strip's halo rows and
// lanes make it 210 MB, at 4.7 TB/s.  The divisions' range tests are made once per row (range.hpp) instead of at
// each of ~20 divisions and both powers share one square root, so a row is about 250 VALU
// instructions in one run instead of 400 in twenty pieces (1.78e7 against 2.79e7 a launch), and the
// row's geometry comes through the scalar cache, so that nothing waits for the row being fetched but
// its use.  Measured per subcycle: 2048x2048 79.5 -> 47 to 52 us, 512x1024 17.5 (one thread per cell) ->
// 11 to 12.3 us, 133x197 7.7 -> 5.0 us.  157 to 161 VGPRs, three wavefronts per SIMD: at four (128) the two register
// sets of a pair of rows spill.
//
// With flux saturation the march also forms the saturated flux and coefficient of each row, from the
// temperature gradient it has there, and writes a row once the next row's coefficient is known: its cells
// reach two rows and two lanes to each side, so lane l holds column 60*tile + l - 2 and lanes 2..61 write.
// As a kernel of its own, which formed temperatures and gradients again, the coefficient took 24.5 us
// per update at 700x1301 beside the update's 19.3; together they take 28.5.  VALU-bound; 207 to 213 VGPRs, two
// wavefronts per SIMD (three spill).
//
// Rows rs .. rend-1.  D = DIV_IN: the geometric divisions and the powers without their operand tests;
// every row is tested once it is formed, and the march stops before the first row whose stencil holds
// a value out of range.  Returns the row it stopped at (rend when done).
struct SatRow { double te, dE, fx, fy, coef, clo; };   // a row waiting for the next; clo: its lower x-face's coefficient

template <int MODE, bool SAT, bool SEP, int D>
__device__ __forceinline__ int tc_march(const TcStepArgs& a, const tcs::Lane& L, int rs, int rend) {
  using namespace tcs;
  const Mesh& M = a.mesh;
  constexpr bool IN = D == DIV_IN;
  constexpr int LAG = SAT ? 1 : 0;          // rows between the one formed and the one written
  const int lane = threadIdx.x;
  const int first = rs - LAG, last = rend + LAG;
  Row cur;
  FaceGeom g = strip::face_geom_row(M.x, first);
  XFaces lo;
  {
    const Raw rp = load_raw<SAT>(a, L, first - 1), rc = load_raw<SAT>(a, L, first);
    const Row prev = make_row<D>(a, L, first - 1, rp);
    cur = make_row<D>(a, L, first, rc);
    if (IN && __any(row_out<SAT>(prev, rp) || row_out<SAT>(cur, rc))) return rs;
    lo = xfaces<D>(g, prev, cur);
  }
  // writes row r from its energy derivative
  auto write = [&](int r, double te, double dE) {
    const size_t row = (size_t)r * M.ny;
    uint32_t jb = 8u * (uint32_t)L.j;
    strip::lane_offset(jb);
    const double base = SEP ? strip::ld_row(a.te_base, row, jb) : te;
    const bool in = r >= M.x.lo && r <= M.x.hi && L.iny;
    dE = in ? dE : 0.0;   // every derivative is zero outside the interior
    double v;
    if (MODE == TC_RK4_FINAL) {
      const double sum = strip::ld_row(a.k1, row, jb) + 2.0 * strip::ld_row(a.k2, row, jb) +
                         2.0 * strip::ld_row(a.k3, row, jb) + dE;
      v = base + qdiv(1.0 * a.h * sum, 6.0, a.k.r6);
    } else {
      v = base + 1.0 * (a.mult * a.h) * dE;
    }
    // mask = 0 there: te + 0*dE
    const double out = smax(in ? v : base + 0.0, a.k.temin);
    if (L.out) {
      if (MODE == TC_STORE_K) strip::st_row(a.k_out, row, jb, dE);
      strip::st_row(a.te_out, row, jb, out);
    }
  };
  // Row r from row r+1's values (raw), with row r+2 asked for first; false when the march ends before
  // it.  What row r leaves for the next is written to the second of each pair, so that two rows in
  // turn swap the pairs and nothing is copied.
  auto step = [&](int r, const Raw& rc, const Raw& raw, Raw& ahead, const Row& cur, Row& nxt, const XFaces& lo,
                  XFaces& hi, const FaceGeom& g, FaceGeom& gn, const SatRow& sp, SatRow& sn, double dx_p,
                  double rdx_p) -> bool {
    ahead = load_raw<SAT>(a, L, r + 2);
    gn = strip::face_geom_row(M.x, r + 1);
    nxt = make_row<D>(a, L, r + 1, raw);
    if (IN && __any(row_out<SAT>(nxt, raw))) return false;
    hi = xfaces<D>(gn, cur, nxt);
    // cell values at row r along x
    const double dx = g.d, rdx = g.rd;
    const bool in = cur.inx && L.iny;
    const double gx = qd<D>(hi.T - lo.T, dx, rdx);
    // dtemp_dx is zero outside the interior; its y-derivative takes the neighbouring lanes' values
    const double dgx_y = yderiv<D>(L, yface<D>(L, in ? gx : 0.0));
    const double s0 = qd<D>(hi.T - 2.0 * cur.T + lo.T, g.hsq, g.rhsq);
    const double dgy_x = qd<D>(hi.gy - lo.gy, dx, rdx);
    const double dbxx = qd<D>(hi.bx - lo.bx, dx, rdx);
    const double dbyx = qd<D>(hi.by - lo.by, dx, rdx);
    const double dE = tcc::tc_combine<double, IN>(cur.T, gx, cur.gy, s0, cur.s1, dgx_y, dgy_x, cur.bx, cur.by, dbxx,
                                                  cur.dbxy, dbyx, cur.dbyy, a.p.k0);
    if (!SAT) {
      write(r, cur.te, dE);
      return true;
    }
    const SatFlux f = sat_flux<IN>(cur.T, gx, cur.gy, rc.rho, cur.bx, cur.by, dx, L.dy, a.p, a.k);
    sn.te = cur.te;
    sn.dE = dE;
    sn.fx = f.fx;
    sn.fy = f.fy;
    sn.coef = in && f.fm != 0.0 ? f.sfm / f.fm : 1.0;           // thermalconduction.cpp:264-268
    if (IN) {
      RangeTest t;
      t.add(sn.coef);
      if (__any(t.out() && lane >= 1 && lane <= 62)) return false;
    }
    // row r-1, whose upper x-face the coefficient now has (thermalconduction.cpp:171-174, 255-271)
    sn.clo = qd<D>(sp.coef * g.hup + sn.coef * g.hlo, g.den, g.rden);
    if (r <= rs) return true;
    const double dcx = qd<D>(sn.clo - sp.clo, dx_p, rdx_p);
    const double dcy = yderiv<D>(L, yface<D>(L, sp.coef));
    const double add = -1.0 * (dcx * sp.fx + dcy * sp.fy);
    write(r - 1, sp.te, sp.coef * sp.dE + add);
    return true;
  };
  Raw raw[2], rowraw = {};
  Row rows[2];
  XFaces faces[2];
  FaceGeom geom[2];
  SatRow sat[2] = {};
  raw[0] = load_raw<SAT>(a, L, first + 1);
  if (SAT) raw[1] = load_raw<SAT>(a, L, first);     // its density is the first row's
  rows[0] = cur;
  faces[0] = lo;
  geom[0] = g;
  geom[1] = g;
  for (int r = first; r < last; r += 2) {
    rowraw.rho = raw[1].rho;
    double d = geom[1].d, rd = geom[1].rd;
    if (!step(r, rowraw, raw[0], raw[1], rows[0], rows[1], faces[0], faces[1], geom[0], geom[1], sat[0], sat[1], d, rd))
      return max(r - LAG, rs);
    if (r + 1 >= last) break;
    rowraw.rho = raw[0].rho;
    d = geom[0].d, rd = geom[0].rd;
    if (!step(r + 1, rowraw, raw[1], raw[0], rows[1], rows[0], faces[1], faces[0], geom[1], geom[0], sat[1], sat[0], d, rd))
      return max(r + 1 - LAG, rs);
  }
  return rend;
}

template <int MODE, bool SAT, bool SEP>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(SAT ? 2 : 3)))
k_tc_strip(TcStepArgs a, int R, int nstrips, int total) {
  const Mesh& M = a.mesh;
  const int t = strip::xcd_tile(blockIdx.x, total);
  const int tile = t / nstrips, sidx = t - tile * nstrips;
  constexpr int HALO = SAT ? 2 : 1;
  const int lane = threadIdx.x, jc = tile * (64 - 2 * HALO) + lane - HALO;
  tcs::Lane L = tcs::lane_at(M, jc);
  L.out = lane >= HALO && lane < 64 - HALO && jc < M.ny;
  const int r0 = sidx * R, r1 = min(r0 + R, M.nx);
  int r = r0;
  if (a.in_range) r = tc_march<MODE, SAT, SEP, tcs::DIV_IN>(a, L, r, r1);
  if (r < r1) (void)tc_march<MODE, SAT, SEP, tcs::DIV_TESTED>(a, L, r, r1);
}

// RadiativeLosses::computeLosses at one interior cell (radiativelosses.cpp:149-197).
__device__ __forceinline__ double rl_loss(double t, double n, double te_live, double dt_live, const RlParams& p) {
  if (t < p.cut) return 0.0;
  // log10(t) <= 4.97 etc. as the host's log10 decides it (p.tb)
  double chi, pw;
  if (t <= p.tb[0]) { chi = 1.09e-31; pw = t * t; }
  else if (t <= p.tb[1]) { chi = 8.87e-17; pw = 1.0 / t; }
  else if (t <= p.tb[2]) { chi = 1.90e-22; pw = 1.0; }
  else if (t <= p.tb[3]) { chi = 3.53e-13; pw = pow_m1p5(t); }
  else if (t <= p.tb[4]) { chi = 3.46e-25; pw = pow_third(t); }
  else if (t <= p.tb[5]) { chi = 5.49e-16; pw = 1.0 / t; }
  else { chi = 1.96e-27; pw = sqrt(t); }
  double v = n * n * chi * pw;
  if (t < p.cut_plus_ramp) {
    const double ramp = (t - p.cut) / p.ramp;
    v *= ramp;
  }
  if (p.prevent) {
    if (0.1 * p.eps * (te_live / v) < p.pd_eps * (dt_live)) v = 0.1 * p.eps * (te_live) / (p.pd_eps * (dt_live));
  }
  return v;
}

// What the modules need before their subcycles, one pass over the live grids: b_hat, and per block the
// least and greatest values of the conduction and the radiation reductions.  Launch-bound on small grids:
// as one kernel for each and one more to finish each reduction they were six launches of 1 to 4.5 us with
// 4 us between two, 48 us of the 137 us a step of a 133x197 arcade took; this pass and k_finish_scalars
// take 7 and 5.5 us there.
__global__ void __launch_bounds__(256) k_step_pre(StepPreArgs a) {
  const Mesh& M = a.mesh;
  const int j = blockIdx.x * blockDim.x + threadIdx.x, i = blockIdx.y * blockDim.y + threadIdx.y;
  double tmin = DBL_MAX, tmax = -DBL_MAX, rmin = DBL_MAX, rmax = -DBL_MAX;
  if (i < M.nx && j < M.ny) {
    const size_t c = (size_t)i * M.ny + j;
    double hx = 0.0, hy = 0.0;
    if (a.bhx) {
      bhat_at(a.L, a.st, c, hx, hy);
      a.bhx[c] = hx;
      a.bhy[c] = hy;
    }
    if (!inside(M, i, j)) {
      tmax = 0.0;   // |b_hat . grad T| and the losses are zero outside the interior
      rmax = 0.0;
    } else {
      if (a.tc_partial) {
        double dts;
        tc_timescale(a.L, hx, hy, a.tc, a.k, M, i, j, dts, tmax);
        tmin = (dts < tmin) ? dts : tmin;
      }
      if (a.rl_partial) {
        const double te = a.L.te[c], n = a.L.n[c];
        const double l = rl_loss(temp_of(te, n, a.k), n, te, a.rl.prevent ? a.dt_grid[c] : 0.0, a.rl);
        rmax = l;
        const double r = fabs(te / l);
        rmin = (r < rmin) ? r : rmin;
      }
    }
  }
  const int blk = blockIdx.y * gridDim.x + blockIdx.x, nblk = gridDim.x * gridDim.y;
  const bool first = threadIdx.x == 0 && threadIdx.y == 0;
  if (a.tc_partial) {
    const double lo = block_reduce(tmin, true), hi = block_reduce(tmax, false);
    if (first) { a.tc_partial[blk] = lo; a.tc_partial[nblk + blk] = hi; }
  }
  if (a.rl_partial) {
    const double lo = block_reduce(rmin, true), hi = block_reduce(rmax, false);
    if (first) { a.rl_partial[blk] = lo; a.rl_partial[nblk + blk] = hi; }
  }
}

// enforceMinimums then recomputeDerivedVarsFromEvolvedVars at one cell (idealmhd.cpp:234-252)
__device__ __forceinline__ void propagate_cell(const MhdSet& L, const MhdConst& K, size_t c, double te, double* te_out,
                                               int write_pre) {
  const double rho1 = smax(qdiv(L.rho[c], K.m, K.rm), K.nmin) * K.m;
  const double te1 = smax(te, K.temin);
  const double n = smax(qdiv(rho1, K.m, K.rm), K.nmin);
  if (write_pre) L.rho_pre[c] = rho1;
  L.n[c] = n;
  L.rho[c] = n * K.m;
  te_out[c] = smax(te1, K.temin);
}

// propagate: te_out is the live thermal energy from here on and the cell is propagated too, which as a pass
// of its own costs a small grid 3 us and a launch's gap of 4.
__global__ void __launch_bounds__(256) k_rl_iterate(MhdSet L, const double* dtg, RlParams p, MhdConst K, Mesh M,
                                                    int nsub, double h, int integ, double* te_out, int propagate,
                                                    int write_pre) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x, i = blockIdx.y * blockDim.y + threadIdx.y;
  if (i >= M.nx || j >= M.ny) return;
  const size_t c = (size_t)i * M.ny + j;
  const double te_live = L.te[c];
  if (!inside(M, i, j)) {
    if (propagate) propagate_cell(L, K, c, te_live, te_out, write_pre);
    else te_out[c] = te_live;
    return;
  }
  const double n = L.n[c];
  const double dtl = p.prevent ? dtg[c] : 0.0;
  auto loss = [&](double te) { return rl_loss(temp_of(te, n, K), n, te_live, dtl, p); };
  double te = te_live;
  const double hh = 1.0 * h, half = 1.0 * (0.5 * h);
  for (int s = 0; s < nsub; ++s) {
    if (integ == 0) {                                             // radiativelosses.cpp:92-96
      te = smax(te - hh * loss(te), K.temin);
    } else if (integ == 1) {                                      // :97-108
      const double hs = smax(te - half * loss(te), K.temin);
      te = smax(te - hh * loss(hs), K.temin);
    } else {                                                      // :109-130
      const double k1 = -loss(te);
      double im = smax(te + half * k1, K.temin);
      const double k2 = -loss(im);
      im = smax(te + half * k2, K.temin);
      const double k3 = -loss(im);
      im = smax(te + hh * k3, K.temin);
      const double k4 = -loss(im);
      te = smax(te + qdiv(hh * (k1 + 2.0 * k2 + 2.0 * k3 + k4), 6.0, K.r6), K.temin);
    }
  }
  if (propagate) propagate_cell(L, K, c, te, te_out, write_pre);
  else te_out[c] = te;
}

__global__ void __launch_bounds__(256) k_propagate_live(MhdSet L, MhdConst K, size_t N, int write_pre) {
  const size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c < N) propagate_cell(L, K, c, L.te[c], L.te, write_pre);
}

inline dim3 g2(const Mesh& m, dim3 b) { return dim3((m.ny + b.x - 1) / b.x, (m.nx + b.y - 1) / b.y); }

}  // namespace

int solar_blocks(const Mesh& m) {
  dim3 g = g2(m, dim3(64, 4));
  return (int)(g.x * g.y);
}

void launch_bhat(MhdSet L, MhdStatic st, Mesh mesh, double* bhx, double* bhy, hipStream_t s) {
  hipLaunchKernelGGL(k_bhat, g2(mesh, dim3(64, 4)), dim3(64, 4), 0, s, L, st, mesh, bhx, bhy);
}

void launch_bhat_derivs(const double* bhx, const double* bhy, Mesh mesh, double* dbxx, double* dbxy, double* dbyx,
                        double* dbyy, hipStream_t s) {
  hipLaunchKernelGGL(k_bhat_derivs, g2(mesh, dim3(64, 4)), dim3(64, 4), 0, s, bhx, bhy, mesh, dbxx, dbxy, dbyx, dbyy);
}

void launch_step_pre(const StepPreArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(k_step_pre, g2(a.mesh, dim3(64, 4)), dim3(64, 4), 0, s, a);
}

void launch_finish_scalars(const double* partial, int nblocks, int njobs, const double* step, const int* err,
                           double* host_out, uint64_t ticket, hipStream_t s) {
  hipLaunchKernelGGL(k_finish_scalars, dim3(njobs > 0 ? njobs : 1), dim3(1024), 0, s, partial, nblocks, njobs, step, err,
                     host_out, ticket);
}

void launch_tc_sat(const double* te_src, const double* n, const double* rho, const double* bhx, const double* bhy,
                   TcParams p, MhdConst k, Mesh mesh, double* rx, double* ry, double* coef, hipStream_t s) {
  hipLaunchKernelGGL(k_tc_sat, g2(mesh, dim3(64, 4)), dim3(64, 4), 0, s, te_src, n, rho, bhx, bhy, p, k, mesh, rx, ry,
                     coef);
}

int tc_strip_rows_default(int nx, int ny, bool saturation) {
  // 3072 wavefronts (3 per SIMD, 2 with saturation) run at once and a strip costs its rows plus about five
  // (three rows to start with, the launch; two rows more with saturation): the height with the least
  // rounds x cost, the taller one of equals
  const int cols = saturation ? 60 : 62, waves = saturation ? 2048 : 3072, extra = saturation ? 7 : 5;
  const long tiles = (ny + cols - 1) / cols;
  int best = 1;
  long least = 0;
  for (int R = 1; R <= 96; ++R) {
    const long cost = (tiles * ((nx + R - 1) / R) + waves - 1) / waves * (R + extra);
    if (R == 1 || cost <= least) { best = R; least = cost; }
  }
  return best;
}

template <int MODE, bool SAT>
static void launch_tc_strip_m(const TcStepArgs& a, int R, hipStream_t s) {
  constexpr int COLS = SAT ? 60 : 62;
  const int tiles = (a.mesh.ny + COLS - 1) / COLS, nstrips = (a.mesh.nx + R - 1) / R, total = tiles * nstrips;
  if (a.te_base != a.te_src)
    hipLaunchKernelGGL((k_tc_strip<MODE, SAT, true>), dim3(total), dim3(64), 0, s, a, R, nstrips, total);
  else
    hipLaunchKernelGGL((k_tc_strip<MODE, SAT, false>), dim3(total), dim3(64), 0, s, a, R, nstrips, total);
}

void launch_tc_step(const TcStepArgs& a, hipStream_t s) {
  if (a.rows <= 0) {
    hipLaunchKernelGGL(k_tc_step, g2(a.mesh, dim3(64, 4)), dim3(64, 4), 0, s, a);
    return;
  }
  if (a.p.saturation) {
    if (a.mode == TC_STORE_K) launch_tc_strip_m<TC_STORE_K, true>(a, a.rows, s);
    else if (a.mode == TC_RK4_FINAL) launch_tc_strip_m<TC_RK4_FINAL, true>(a, a.rows, s);
    else launch_tc_strip_m<TC_UPDATE, true>(a, a.rows, s);
  } else {
    if (a.mode == TC_STORE_K) launch_tc_strip_m<TC_STORE_K, false>(a, a.rows, s);
    else if (a.mode == TC_RK4_FINAL) launch_tc_strip_m<TC_RK4_FINAL, false>(a, a.rows, s);
    else launch_tc_strip_m<TC_UPDATE, false>(a, a.rows, s);
  }
}

void launch_rl_iterate(MhdSet L, const double* dt_grid, RlParams p, MhdConst k, Mesh mesh, int nsub, double h,
                       int integrator, double* te_out, int propagate, int write_pre, hipStream_t s) {
  hipLaunchKernelGGL(k_rl_iterate, g2(mesh, dim3(64, 4)), dim3(64, 4), 0, s, L, dt_grid, p, k, mesh, nsub, h,
                     integrator, te_out, propagate, write_pre);
}

void launch_propagate_live(MhdSet L, MhdConst k, int nx, int ny, int write_pre, hipStream_t s) {
  const size_t N = (size_t)nx * ny;
  hipLaunchKernelGGL(k_propagate_live, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, s, L, k, N, write_pre);
}

}  // namespace spruce
