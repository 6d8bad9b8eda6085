// Discrete-adjoint kernels of the IdealMHD time step for gfx950 (reverse of mhd.hip's stage, dt and
// populate kernels).  The per-cell algebra is adj_cell.hpp; these kernels sequence it over the
// grid.  Face contributions land on four cells each and are accumulated with FP64 atomics, so the
// gradient is reproducible to rounding, not bit for bit.
#include <cfloat>

#include "adj_cell.hpp"
#include "adjoint.hpp"
#include "arith.hpp"
#include "strip.hpp"

namespace spruce {
namespace {

__device__ __forceinline__ bool interior_cell(const Mesh& M, int i, int j) {
  return i >= M.x.lo && i <= M.x.hi && j >= M.y.lo && j <= M.y.hi;
}

__device__ __forceinline__ double block_sum(double v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  __shared__ double part[16];
  const int lane = threadIdx.x + threadIdx.y * blockDim.x;
  if ((lane & 63) == 0) part[lane >> 6] = v;
  __syncthreads();
  if (lane == 0) {
    const int nw = (blockDim.x * blockDim.y + 63) >> 6;
    double m = 0.0;
    for (int k = 0; k < nw; ++k) m += part[k];
    v = m;
  }
  return v;
}

// Reverse of one stage for one cell: T = minimums/derived(B + mult*h*kv) reversed (lam_B gets mu,
// lamk = mult*h*mu, the block's partial of mult*mu.kv), then the cell's own part of the transposed
// time derivative at S applied to lamk (its face coefficients to cx, cy; its own part to lam_S).
// assign_B / assign_S: this launch is the first writer of lam_B / lam_S in the step (no clear).
__global__ void __launch_bounds__(256) k_adj_stage_cells(MhdSet B, const double* kv, const double* step, double mult,
                                                         MhdSet S, MhdStatic st, MhdConst K, Mesh M,
                                                         const double* lam_T, double* lam_B, int assign_B,
                                                         double* lam_S, int assign_S, double* cx, double* cy,
                                                         double* partial) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x, i = blockIdx.y * blockDim.y + threadIdx.y;
  double dot = 0.0;
  if (i < M.nx && j < M.ny) {
    const size_t N = (size_t)M.nx * M.ny, c = (size_t)i * M.ny + j;
    const double h = mult * (*step);
    // derivative of the minimums/derived maps (idealmhd.cpp:237-238, 246-252): rho passes when
    // neither floor is active, te when its floor is not
    const double rho_new = B.rho[c] + kv[c] * h;
    const double x = rho_new / K.m;
    const double rho1 = smax(x, K.nmin) * K.m;
    const double drho = (x < K.nmin || rho1 / K.m < K.nmin) ? 0.0 : 1.0;
    const double te_new = B.te[c] + kv[4 * N + c] * h;
    const double dte = te_new < K.temin ? 0.0 : 1.0;
    double lamk[8];
    for (int v = 0; v < 8; ++v) {
      const double d = v == 0 ? drho : (v == 4 ? dte : 1.0);
      const double mu = lam_T[v * N + c] * d;
      lam_B[v * N + c] = assign_B ? mu : lam_B[v * N + c] + mu;
      lamk[v] = h * mu;
      dot += mu * kv[v * N + c];
    }
    dot *= mult;
    double fx[ADJ_NCOEF], fy[ADJ_NCOEF];
    if (interior_cell(M, i, j)) {
      double own[8];
      adj_cell_coeffs(S, st, K, M, i, j, lamk, own, fx, fy);
      for (int v = 0; v < 8; ++v) lam_S[v * N + c] = assign_S ? own[v] : lam_S[v * N + c] + own[v];
    } else {
      for (int q = 0; q < ADJ_NCOEF; ++q) { fx[q] = 0.0; fy[q] = 0.0; }
      if (assign_S) for (int v = 0; v < 8; ++v) lam_S[v * N + c] = 0.0;
    }
    for (int q = 0; q < ADJ_NCOEF; ++q) { cx[q * N + c] = fx[q]; cy[q * N + c] = fy[q]; }
  }
  dot = block_sum(dot);
  if (threadIdx.x == 0 && threadIdx.y == 0) partial[blockIdx.y * gridDim.x + blockIdx.x] = dot;
}

// Reverse of the pointwise part of one stage, T = minimums/derived(B + mult*h*kv), alone:
// lam_B (+)= mu = dT/dpre^T lam_T, lamk = mult*h*mu (written), partial: block sums of mult*mu.kv.
__global__ void __launch_bounds__(256) k_adj_update(MhdSet B, const double* kv, const double* step, double mult,
                                                    MhdConst K, Mesh M, const double* lam_T, double* lam_B,
                                                    int assign_B, double* lamk, double* partial) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x, i = blockIdx.y * blockDim.y + threadIdx.y;
  double dot = 0.0;
  if (i < M.nx && j < M.ny) {
    const size_t N = (size_t)M.nx * M.ny, c = (size_t)i * M.ny + j;
    const double h = mult * (*step);
    const double rho_new = B.rho[c] + kv[c] * h;
    const double x = rho_new / K.m;
    const double rho1 = smax(x, K.nmin) * K.m;
    const double drho = (x < K.nmin || rho1 / K.m < K.nmin) ? 0.0 : 1.0;
    const double te_new = B.te[c] + kv[4 * N + c] * h;
    const double dte = te_new < K.temin ? 0.0 : 1.0;
    for (int v = 0; v < 8; ++v) {
      const double d = v == 0 ? drho : (v == 4 ? dte : 1.0);
      const double mu = lam_T[v * N + c] * d;
      lam_B[v * N + c] = assign_B ? mu : lam_B[v * N + c] + mu;
      lamk[v * N + c] = h * mu;
      dot += mu * kv[v * N + c];
    }
    dot *= mult;
  }
  dot = block_sum(dot);
  if (threadIdx.x == 0 && threadIdx.y == 0) partial[blockIdx.y * gridDim.x + blockIdx.x] = dot;
}

// The per-cell part of the transposed time derivative at S applied to lamk = sa*ka + kb (kb may be
// null): its own part to lam_S, its face coefficients to cx, cy (then k_adj_faces).
__global__ void __launch_bounds__(256) k_adj_rhs_cells(MhdSet S, MhdStatic st, MhdConst K, Mesh M, const double* ka,
                                                       double sa, const double* kb, double* lam_S, int assign_S,
                                                       double* cx, double* cy) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x, i = blockIdx.y * blockDim.y + threadIdx.y;
  if (i >= M.nx || j >= M.ny) return;
  const size_t N = (size_t)M.nx * M.ny, c = (size_t)i * M.ny + j;
  double fx[ADJ_NCOEF], fy[ADJ_NCOEF];
  if (interior_cell(M, i, j)) {
    double lamk[8], own[8];
    for (int v = 0; v < 8; ++v) lamk[v] = kb ? sa * ka[v * N + c] + kb[v * N + c] : sa * ka[v * N + c];
    adj_cell_coeffs(S, st, K, M, i, j, lamk, own, fx, fy);
    for (int v = 0; v < 8; ++v) lam_S[v * N + c] = assign_S ? own[v] : lam_S[v * N + c] + own[v];
  } else {
    for (int q = 0; q < ADJ_NCOEF; ++q) { fx[q] = 0.0; fy[q] = 0.0; }
    if (assign_S) for (int v = 0; v < 8; ++v) lam_S[v * N + c] = 0.0;
  }
  for (int q = 0; q < ADJ_NCOEF; ++q) { cx[q * N + c] = fx[q]; cy[q * N + c] = fy[q]; }
}

// The face scatter, x and y faces in one launch of one-wavefront blocks: the first x_blocks blocks take
// the x faces, the others the y faces.
//
// x faces: one thread per column takes `rows` consecutive faces; a face adds to the rows f-2 .. f+1 of its
// column, so the thread keeps those four rows' adjoint in registers and adds a row once no later face of
// its own can reach it.  y faces: a wavefront takes 64 consecutive faces of a row, one per lane; a cell's
// four faces lie in neighbouring lanes, whose contributions are exchanged by lane shifts, so that lanes
// 1 .. 61 hold complete sums of 61 cells and neighbouring wavefronts share no cell.  What bounds both is the
// latency of one wavefront's chain of loads and divisions; at 2048x2048 the two read and write 3.0 GB at
// 2.6 TB/s.
__device__ __forceinline__ void adj_faces_x(const MhdSet& S, const MhdStatic& st, const MhdConst& K, const Mesh& M,
                                            const double* cx, double* lam_S, int block, int rows) {
  const int cols = (M.ny + 63) / 64, strip = block / cols;
  const int j = (block - strip * cols) * 64 + threadIdx.x;
  if (j >= M.ny) return;
  const Axis& ax = M.x;
  const size_t N = (size_t)M.nx * M.ny;
  const int fs = strip * rows, fe = min(fs + rows, M.nx);
  double acc[4][8];
  for (int a = 0; a < 4; ++a)
    for (int v = 0; v < 8; ++v) acc[a][v] = 0.0;
  auto flush = [&](int row, const double* a8) {
    if (!ax.per && (row < 0 || row >= ax.n)) return;
    const size_t c = (size_t)wrapi(row, ax.n, ax.per) * M.ny + j;
    for (int v = 0; v < 8; ++v)
      if (a8[v] != 0.0) atomicAdd(&lam_S[v * N + c], a8[v]);
  };
  for (int f = fs; f < fe; ++f) {
    if (ax.per || (f >= ax.lo && f <= ax.hi + 1)) {     // faces of interior cells only
      const int fl = wrapi(f - 1, ax.n, ax.per);
      const size_t cu = (size_t)f * M.ny + j, cl = (size_t)fl * M.ny + j;
      double fa[ADJ_NCOEF];
      bool any = false;
      for (int q = 0; q < ADJ_NCOEF; ++q) {
        fa[q] = cx[q * N + cl] - cx[q * N + cu];
        any = any || fa[q] != 0.0;
      }
      if (any) adj_face_slots<0>(S, st, K, M, f, j, fa, [&](int slot, int v, double val) { acc[slot][v] += val; });
    }
    flush(f - 2, acc[0]);   // complete as far as this strip goes: its later faces reach rows f-1 and above
    for (int a = 0; a < 3; ++a)
      for (int v = 0; v < 8; ++v) acc[a][v] = acc[a + 1][v];
    for (int v = 0; v < 8; ++v) acc[3][v] = 0.0;
  }
  for (int a = 0; a < 3; ++a) flush(fe - 2 + a, acc[a]);
}

constexpr int FY_CELLS = 61;   // cells a wavefront of 64 y faces completes

template <bool SHARED>
__device__ __forceinline__ void adj_faces_y(const MhdSet& S, const MhdStatic& st, const MhdConst& K, const Mesh& M,
                                            const double* cy, double* lam_S, int block) {
  const Axis& ax = M.y;
  const size_t N = (size_t)M.nx * M.ny;
  const int tiles = (M.ny + FY_CELLS - 1) / FY_CELLS;
  const int i = block / tiles, lane = threadIdx.x, base = (block - i * tiles) * FY_CELLS;
  const int ncell = min(FY_CELLS, M.ny - base);
  const bool own = lane >= 1 && lane <= ncell;
  const size_t co = (size_t)i * M.ny + (own ? base + lane - 1 : base);
  double lam[8], acc[4][8];
  if (!SHARED)
    for (int v = 0; v < 8; ++v) lam[v] = lam_S[v * N + co];
  for (int a = 0; a < 4; ++a)
    for (int v = 0; v < 8; ++v) acc[a][v] = 0.0;
  const int j = wrapi(base - 1 + lane, ax.n, ax.per);     // the lane's face: between cells j-1 and j
  if (lane < ncell + 3 && (ax.per || (j >= ax.lo && j <= ax.hi + 1))) {
    const int fl = wrapi(j - 1, ax.n, ax.per);
    const size_t cu = (size_t)i * M.ny + j, cl = (size_t)i * M.ny + fl;
    double fa[ADJ_NCOEF];
    bool any = false;
    for (int q = 0; q < ADJ_NCOEF; ++q) {
      fa[q] = cy[q * N + cl] - cy[q * N + cu];
      any = any || fa[q] != 0.0;
    }
    if (any) adj_face_slots<1>(S, st, K, M, i, j, fa, [&](int slot, int v, double val) { acc[slot][v] += val; });
  }
  // cell j: slot 2 of its own face, slot 1 of face j+1, slot 0 of face j+2, slot 3 of face j-1
  for (int v = 0; v < 8; ++v) {
    const double t = acc[2][v] + strip::shl1(acc[1][v]) + strip::shl1(strip::shl1(acc[0][v])) + strip::shr1(acc[3][v]);
    if (!own) continue;
    if (SHARED) atomicAdd(&lam_S[v * N + co], t);
    else lam_S[v * N + co] = lam[v] + t;
  }
}

__global__ void __launch_bounds__(64) k_adj_faces(MhdSet S, MhdStatic st, MhdConst K, Mesh M, const double* cx,
                                                  const double* cy, double* lam_S, int x_blocks, int rows) {
  const int b = blockIdx.x;
  if (b < x_blocks) adj_faces_x(S, st, K, M, cx, lam_S, b, rows);
  else adj_faces_y<true>(S, st, K, M, cy, lam_S, b - x_blocks);
}

__global__ void __launch_bounds__(64) k_adj_faces_x(MhdSet S, MhdStatic st, MhdConst K, Mesh M, const double* cx,
                                                    double* lam_S, int rows) {
  adj_faces_x(S, st, K, M, cx, lam_S, blockIdx.x, rows);
}

__global__ void __launch_bounds__(64) k_adj_faces_y(MhdSet S, MhdStatic st, MhdConst K, Mesh M, const double* cy,
                                                    double* lam_S) {
  adj_faces_y<false>(S, st, K, M, cy, lam_S, blockIdx.x);
}

// per-block (min dt, index) over the interior, std::min semantics (NaN never selected)
__global__ void __launch_bounds__(256) k_adj_dt_blocks(MhdSet L, MhdStatic st, MhdConst K, Mesh M, double* pmin,
                                                       int* pidx) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x, i = blockIdx.y * blockDim.y + threadIdx.y;
  double v = DBL_MAX;
  int idx = -1;
  if (i < M.nx && j < M.ny && interior_cell(M, i, j)) {
    const double dt = dt_cell_dual(L, st, K, M, i, j).v;
    if (dt < v) { v = dt; idx = i * M.ny + j; }
  }
  for (int off = 32; off > 0; off >>= 1) {
    const double ov = __shfl_xor(v, off, 64);
    const int oi = __shfl_xor(idx, off, 64);
    if (ov < v || (ov == v && oi >= 0 && (idx < 0 || oi < idx))) { v = ov; idx = oi; }
  }
  __shared__ double pv[16];
  __shared__ int pi[16];
  const int lane = threadIdx.x + threadIdx.y * blockDim.x;
  if ((lane & 63) == 0) { pv[lane >> 6] = v; pi[lane >> 6] = idx; }
  __syncthreads();
  if (lane == 0) {
    const int nw = (blockDim.x * blockDim.y + 63) >> 6;
    for (int k = 1; k < nw; ++k)
      if (pv[k] < v || (pv[k] == v && pi[k] >= 0 && (idx < 0 || pi[k] < idx))) { v = pv[k]; idx = pi[k]; }
    pmin[blockIdx.y * gridDim.x + blockIdx.x] = v;
    pidx[blockIdx.y * gridDim.x + blockIdx.x] = idx;
  }
}

__global__ void __launch_bounds__(1024) k_adj_dt_apply(MhdSet L, MhdStatic st, MhdConst K, Mesh M, double eps,
                                                       const double* p1, const double* p2, const double* gh,
                                                       const double* pmin, const int* pidx, int nb, double* lam_L) {
  // the adjoint of the step size: the sum of the stage kernels' block partials, plus the modules';
  // and the (min, lowest index) over the block results, a rule independent of the visiting order.
  // Sixteen wavefronts, each reduced by shuffles, then combined by the first thread.
  __shared__ double sg[16], sv[16];
  __shared__ int si[16];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  double g = 0.0, v = DBL_MAX;
  int idx = -1;
  for (int k = t; k < nb; k += 1024) {
    g += (p1 ? p1[k] : 0.0) + (p2 ? p2[k] : 0.0);
    if (pmin[k] < v || (pmin[k] == v && pidx[k] >= 0 && (idx < 0 || pidx[k] < idx))) { v = pmin[k]; idx = pidx[k]; }
  }
  for (int off = 32; off > 0; off >>= 1) {
    g += __shfl_xor(g, off, 64);
    const double ov = __shfl_xor(v, off, 64);
    const int oi = __shfl_xor(idx, off, 64);
    if (ov < v || (ov == v && oi >= 0 && (idx < 0 || oi < idx))) { v = ov; idx = oi; }
  }
  if (lane == 0) { sg[w] = g; sv[w] = v; si[w] = idx; }
  __syncthreads();
  if (t != 0) return;
  g = 0.0;
  v = DBL_MAX;
  idx = -1;
  for (int q = 0; q < 16; ++q) {
    g += sg[q];
    if (sv[q] < v || (sv[q] == v && si[q] >= 0 && (idx < 0 || si[q] < idx))) { v = sv[q]; idx = si[q]; }
  }
  if (gh) g += gh[0];
  if (idx < 0) return;
  const int i = idx / M.ny, j = idx - i * M.ny;
  const Dual8 dt = dt_cell_dual(L, st, K, M, i, j);
  const size_t N = (size_t)M.nx * M.ny;
  const double s = eps * g;
  for (int v8 = 0; v8 < 8; ++v8) lam_L[v8 * N + idx] += s * dt.d[v8];
}

// populateVariablesFromState (equationset.cpp:96-104; idealmhd.cpp:226-252) reversed
__global__ void __launch_bounds__(256) k_adj_populate(const double* rho_s, const double* temp_s, const double* lam,
                                                      MhdConst K, size_t N, double* g) {
  const size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= N) return;
  const double rho = rho_s[c], T = temp_s[c];
  const double x = rho / K.m;
  const double n0 = smax(x, K.nmin);
  const double Tm = smax(T, K.tmin);
  const double te = n0 * 2.0 * K_B * Tm / K.gm1;
  const double dte = te < K.temin ? 0.0 : 1.0;
  const double rho1 = n0 * K.m;
  const double drho = (x < K.nmin || rho1 / K.m < K.nmin) ? 0.0 : 1.0;
  const double l_rho = lam[c], l_te = lam[4 * N + c];
  g[0 * N + c] = l_rho * drho + l_te * dte * (2.0 * K_B * Tm / K.gm1) * (x < K.nmin ? 0.0 : 1.0 / K.m);
  g[1 * N + c] = l_te * dte * (n0 * 2.0 * K_B / K.gm1) * (T < K.tmin ? 0.0 : 1.0);
  g[2 * N + c] = lam[1 * N + c];
  g[3 * N + c] = lam[2 * N + c];
  g[4 * N + c] = lam[3 * N + c];
  g[5 * N + c] = lam[5 * N + c];
  g[6 * N + c] = lam[6 * N + c];
  g[7 * N + c] = lam[7 * N + c];
}

__global__ void __launch_bounds__(256) k_fill(double* p, double v, size_t n) {
  const size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c < n) p[c] = v;
}

inline dim3 g2(const Mesh& m, dim3 b) { return dim3((m.ny + b.x - 1) / b.x, (m.nx + b.y - 1) / b.y); }

}  // namespace

int adj_blocks(const Mesh& m) {
  const dim3 g = g2(m, dim3(64, 4));
  return (int)(g.x * g.y);
}

void launch_adj_stage_cells(MhdSet B, const double* kv, const double* step, double mult, MhdSet S, MhdStatic st,
                            MhdConst k, Mesh mesh, const double* lam_T, double* lam_B, int assign_B, double* lam_S,
                            int assign_S, double* cx, double* cy, double* partial, hipStream_t s) {
  const dim3 b(64, 4);
  hipLaunchKernelGGL(k_adj_stage_cells, g2(mesh, b), b, 0, s, B, kv, step, mult, S, st, k, mesh, lam_T, lam_B,
                     assign_B, lam_S, assign_S, cx, cy, partial);
}

void launch_adj_faces(MhdSet S, MhdStatic st, MhdConst k, Mesh mesh, const double* cx, const double* cy,
                      double* lam_S, hipStream_t s) {
  // A wavefront needs 5 us for one face per lane and 300 registers, so one fits on a SIMD.  Small grids: x
  // and y together fill the 1024 SIMDs better than two launches that each leave most of them idle, and the
  // strips are as short as one residency allows (measured, both axes, us: 128x128 12.5, 192x192 22.5,
  // 256x256 25.4, 320x320 39 in one launch against 30, 33, 36, 43 in two).  Large grids: two launches, where
  // the y faces need no atomics (512x512 89 against 96, 2048x2048 1157 against 1477).  Strips of 16 rows, as
  // many as a quarter of a residency at 256x256, took 142 us there for the x faces alone.
  const int cols = (mesh.ny + 63) / 64, tiles = (mesh.ny + FY_CELLS - 1) / FY_CELLS;
  const int y_blocks = tiles * mesh.nx;
  const auto x_blocks = [&](int rows) { return cols * ((mesh.nx + rows - 1) / rows); };
  if (y_blocks <= 2048) {
    const int rows = x_blocks(1) + y_blocks <= 1024 ? 1 : 3;
    hipLaunchKernelGGL(k_adj_faces, dim3((unsigned)(x_blocks(rows) + y_blocks)), dim3(64), 0, s, S, st, k, mesh, cx, cy,
                       lam_S, x_blocks(rows), rows);
  } else {
    const int rows = 2;
    hipLaunchKernelGGL(k_adj_faces_x, dim3((unsigned)x_blocks(rows)), dim3(64), 0, s, S, st, k, mesh, cx, lam_S, rows);
    hipLaunchKernelGGL(k_adj_faces_y, dim3((unsigned)y_blocks), dim3(64), 0, s, S, st, k, mesh, cy, lam_S);
  }
}

void launch_adj_dt(MhdSet L, MhdStatic st, MhdConst k, Mesh mesh, double eps, const double* p1, const double* p2,
                   const double* gh, double* pmin, int* pidx, double* lam_L, hipStream_t s) {
  const dim3 b(64, 4), g = g2(mesh, b);
  hipLaunchKernelGGL(k_adj_dt_blocks, g, b, 0, s, L, st, k, mesh, pmin, pidx);
  hipLaunchKernelGGL(k_adj_dt_apply, dim3(1), dim3(1024), 0, s, L, st, k, mesh, eps, p1, p2, gh, (const double*)pmin,
                     (const int*)pidx, (int)(g.x * g.y), lam_L);
}

void launch_adj_populate(const double* rho_s, const double* temp_s, const double* lam, MhdConst k, size_t N,
                         double* g_state, hipStream_t s) {
  hipLaunchKernelGGL(k_adj_populate, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, s, rho_s, temp_s, lam, k, N,
                     g_state);
}

void launch_fill(double* p, double v, size_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_fill, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, v, n);
}


void launch_adj_update(MhdSet B, const double* kv, const double* step, double mult, MhdConst k, Mesh mesh,
                       const double* lam_T, double* lam_B, int assign_B, double* lamk, double* partial,
                       hipStream_t s) {
  const dim3 b(64, 4);
  hipLaunchKernelGGL(k_adj_update, g2(mesh, b), b, 0, s, B, kv, step, mult, k, mesh, lam_T, lam_B, assign_B, lamk, partial);
}

void launch_adj_rhs_cells(MhdSet S, MhdStatic st, MhdConst k, Mesh mesh, const double* ka, double sa,
                          const double* kb, double* lam_S, int assign_S, double* cx, double* cy, hipStream_t s) {
  const dim3 b(64, 4);
  hipLaunchKernelGGL(k_adj_rhs_cells, g2(mesh, b), b, 0, s, S, st, k, mesh, ka, sa, kb, lam_S, assign_S, cx, cy);
}

}  // namespace spruce
