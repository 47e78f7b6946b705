// cv_sweep.h -- one y-line smoothing sweep of a small level in one launch
// (the residual and the line solves of stencil_tile and yline_reg_tile).
// Included by cv_poisson.hip.
#pragma once

namespace {

// As two launches a sweep of such a level takes 9-10 us, most of it launch,
// memory round trips and the passage of the residual from one to the other.
// Here a work-group takes XC columns of one k plane over their whole height: x
// with a halo of one column goes to LDS, each thread forms the residual of one
// cell and leaves it, times 1/pivot, in LDS beside the line factors, and one
// thread per CS rows solves the columns.  Every
// operand is in flight before the first is used; each face flux is formed by
// both its cells, so nothing waits for a neighbour.  Bound by latency up to
// some 10^5 points; past SWEEP_MAX points the operands of the halo columns
// (twice the traffic) cost more than the second launch: the pressure solve of
// 72x61x112 cells (520,000 points) takes 7.80 ms in FP64 with its finest level as
// launches and 8.3 without, 5.9 and 6.1 with FP16 coefficients; the fused sweep
// of 1.4 M points 37 us against 28 for the two launches, of 350,000 points 14
// and 17.5, of 39,000 points 7.4 and 16.
// Pressure solves with two launches a sweep and now: 32x32x32 mixed16 2.72 and
// 2.08 ms, 128x96x96 mixed16 9.2 and 7.8, 200x117x136 mixed 28.0 and 26.5,
// 128x192x128 FP64 17.6 and 16.3.
// Every value is formed by the expressions of the two launches, so the bits are
// theirs.
#define SWEEP_MAX 400000

// XC: 8 up to 64 rows, 4 beyond (shorter passes over the rows: FP64 96x120x96
// 8.65 ms a pressure solve with 8, 8.03 with 4; 32x32x32 2.45 and 2.58)
__host__ __device__ inline int sweep_cols(int ny) { return ny <= 64 ? 8 : 4; }
// chunks of cs rows lie XC values past a multiple of the LDS banks
__host__ __device__ inline int sweep_rows(int ny, int cs, int xc) { return xc * (ny + (ny + cs - 1) / cs); }
// values in LDS: x and its halo, four per row, the carries of both recurrences;
// at most 9252 (74 KB in FP64) for the 256 rows of CS = 16
__host__ __device__ inline int sweep_lds(int ny, int cs, int xc) {
  return 3 * (xc + 2) * (ny + 2) + 4 * sweep_rows(ny, cs, xc) + 4 * xc * ((ny + cs - 1) / cs);
}
inline int sweep_patches(const CvDims &d, int xc) { return (d.mx + xc - 1) / xc * d.mz; }
// threads of a work-group, one a cell: at most 1024
inline unsigned sweep_threads(int ny, int xc) { return (unsigned)((ny * xc + 63) / 64 * 64); }
// whether a sweep of the level is one launch
inline bool sweep_fits(const CvDims &d) { return d.n <= SWEEP_MAX && d.my - 2 >= 1 && d.my - 2 <= 256; }

// the operands of one cell: the operator words and face coefficients of its
// upper faces and of those of the cells at i-1, j-1 and k-1, b, the line
// factors, and the cell's own x where the halo holds the periodic image
template <class T, bool HG>
struct SwCell {
  uint32_t w, wi, wj, wk;
  T g[9], gi[3], gj[3], gk[3], aj, b, ip, a, cp, xg;
};
template <class T>
struct SwCell<T, true> {
  cv_u4 ha;
  cv_u2 hb, hj, ai, ak;
  uint32_t bi, bk, yh;
  uint16_t yc;
  T b, xg;
};

template <class T, bool HG, int CS, int XC>
__device__ __forceinline__ void sweep_body(const OpV<T> &A, const T *__restrict__ x, const T *__restrict__ b,
                                           T *__restrict__ xo, T om, int patch, T *lds) {
  const int tid = threadIdx.x, NT = blockDim.x;
  const int mx = A.mx, my = A.my, mz = A.mz, ny = my - 2;
  const unsigned pl = (unsigned)mx * (unsigned)my, n = pl * (unsigned)mz;
  constexpr int TC = XC + 2;   // columns of the tile
  const int px = (mx + XC - 1) / XC;
  const int x0 = patch % px * XC, gk = patch / px;
  const int plane = TC * my;
  const int rows = sweep_rows(ny, CS, XC), nch = (ny + CS - 1) / CS;
  T *const X = lds, *const Y = X + 3 * plane, *const Fa = Y + rows, *const Fc = Fa + rows;
  T *const D = Fc + rows, *const SA = D + rows, *const SB = SA + 2 * XC * nch;
  const CvBuf Bx = cv_buf(x, n * sizeof(T)), Bb = cv_buf(b, n * sizeof(T));
  auto in_grid = [&](bool ok, unsigned t, unsigned sz) { return ok ? t * sz : CV_OOB; };

  // this thread's cell
  const int col = tid % XC, gi = x0 + col;
  const bool on = gi < mx;
  const bool ghost = (A.xper && (gi == 0 || gi == mx - 1)) || (A.zper && (gk == 0 || gk == mz - 1));
  const unsigned base = (unsigned)gi + pl * (unsigned)gk;
  const int j = 1 + tid / XC;
  const bool cell = on && j < my - 1;
  SwCell<T, HG> C;
  auto fetch = [&]() {
    const bool ok = cell, oi = ok && gi > 0, ok_ = ok && gk > 0;
    const unsigned t = base + (unsigned)(mx * j);
    if constexpr (HG) {
      const CvBuf a = cv_buf(A.hA, n * 16ul), h = cv_buf(A.hB, n * 8ul);
      C.ha = cv_bld<cv_u4>(a, in_grid(ok, t, 16), 0);
      C.hb = cv_bld<cv_u2>(h, in_grid(ok, t, 8), 0);
      C.ai = cv_bld<cv_u2>(a, in_grid(oi, t - 1, 16), 0);
      C.bi = cv_bld<uint32_t>(h, oi ? (t - 1) * 8u + 4u : CV_OOB, 0);
      C.hj = cv_bld<cv_u2>(h, in_grid(ok, t - mx, 8), 0);
      C.ak = cv_bld<cv_u2>(a, ok_ ? (t - pl) * 16u + 4u : CV_OOB, 0);
      C.bk = cv_bld<uint32_t>(h, ok_ ? (t - pl) * 8u + 4u : CV_OOB, 0);
      C.yh = cv_bld<uint32_t>(cv_buf(A.yh, n * 4ul), in_grid(ok, t, 4), 0);
      C.yc = A.yc[ok ? t : 0];
    } else {
      const CvBuf f = cv_buf(A.fl, n * 4ul);
      C.w = cv_bld<uint32_t>(f, in_grid(ok, t, 4), 0);
      C.wi = cv_bld<uint32_t>(f, in_grid(oi, t - 1, 4), 0);
      C.wj = cv_bld<uint32_t>(f, in_grid(ok, t - mx, 4), 0);
      C.wk = cv_bld<uint32_t>(f, in_grid(ok_, t - pl, 4), 0);
#pragma unroll
      for (int q = 0; q < 9; q++) {
        const CvBuf g = cv_buf(A.g[q], n * sizeof(T));
        C.g[q] = cv_bld<T>(g, in_grid(ok, t, sizeof(T)), 0);
        if (q < 3) C.gi[q] = cv_bld<T>(g, in_grid(oi, t - 1, sizeof(T)), 0);
        else if (q < 6) C.gj[q - 3] = cv_bld<T>(g, in_grid(ok, t - mx, sizeof(T)), 0);
        else C.gk[q - 6] = cv_bld<T>(g, in_grid(ok_, t - pl, sizeof(T)), 0);
      }
      C.aj = cv_bld<T>(cv_buf(A.aj, n * sizeof(T)), in_grid(ok, t, sizeof(T)), 0);
      C.ip = cv_bld<T>(cv_buf(A.yip, n * sizeof(T)), in_grid(ok, t, sizeof(T)), 0);
      C.a = cv_bld<T>(cv_buf(A.ylo, n * sizeof(T)), in_grid(ok, t, sizeof(T)), 0);
      C.cp = cv_bld<T>(cv_buf(A.ycp, n * sizeof(T)), in_grid(ok, t, sizeof(T)), 0);
    }
    C.b = cv_bld<T>(Bb, in_grid(ok, t, sizeof(T)), 0);
    C.xg = cv_bld<T>(Bx, in_grid(ok && ghost, t, sizeof(T)), 0);
  };

  // x of the patch and its halo (periodic images, 0 outside the grid)
  const int nx = 3 * plane;
  auto x_off = [&](int e) -> unsigned {
    const int row = e / TC, c = e - row * TC;
    const int q = (row >= my) + (row >= 2 * my), jj = row - q * my;
    const int ii = x0 - 1 + c, kk = gk - 1 + q;
    const bool ok = e < nx && ii >= 0 && ii < mx && kk >= 0 && kk < mz;
    return in_grid(ok, (unsigned)cv_wrap(ii, mx, A.xper) + (unsigned)(mx * jj) + pl * (unsigned)cv_wrap(kk, mz, A.zper),
                   sizeof(T));
  };
  constexpr int XB = 4;
  T xv[XB];
#pragma unroll
  for (int q = 0; q < XB; q++) xv[q] = cv_bld<T>(Bx, x_off(tid + q * NT), 0);
  fetch();
#pragma unroll
  for (int q = 0; q < XB; q++)
    if (tid + q * NT < nx) X[tid + q * NT] = xv[q];
  for (int e = tid + XB * NT; e < nx; e += XB * NT) {
#pragma unroll
    for (int q = 0; q < XB; q++) xv[q] = cv_bld<T>(Bx, x_off(e + q * NT), 0);
#pragma unroll
    for (int q = 0; q < XB; q++)
      if (e + q * NT < nx) X[e + q * NT] = xv[q];
  }
  // the rows this thread solves
  const int tc = tid / XC;
  const int r0 = tc * CS, nrow = on && tc < nch ? min(CS, ny - r0) : 0;

  // the residual of one cell and its line solve's terms to LDS
  const T *M = X, *P = M + plane, *Q = P + plane;
  const int c = col + 1;
  __syncthreads();
  if (cell) {
    uint32_t w, wi, wj, wk;
    T g[9], gi_[3], gj_[3], gk_[3], aj, ip, a, cp;
    if constexpr (HG) {
      w = C.hb.y >> 16; wi = C.bi >> 16; wj = C.hj.y >> 16; wk = C.bk >> 16;
      g[0] = half_lo(C.ha.x); g[1] = half_hi(C.ha.x); g[2] = half_lo(C.ha.y);
      g[3] = half_lo(C.hb.x); g[4] = half_hi(C.hb.x); g[5] = half_lo(C.hb.y);
      g[6] = half_hi(C.ha.y); g[7] = half_lo(C.ha.z); g[8] = half_hi(C.ha.z);
      gi_[0] = half_lo(C.ai.x); gi_[1] = half_hi(C.ai.x); gi_[2] = half_lo(C.ai.y);
      gj_[0] = half_lo(C.hj.x); gj_[1] = half_hi(C.hj.x); gj_[2] = half_lo(C.hj.y);
      gk_[0] = half_hi(C.ak.x); gk_[1] = half_lo(C.ak.y); gk_[2] = half_hi(C.ak.y);
      aj = __uint_as_float(C.ha.w);
      a = half_lo(C.yh); ip = half_hi(C.yh); cp = half_lo((uint32_t)C.yc);
    } else {
      w = C.w; wi = C.wi; wj = C.wj; wk = C.wk; aj = C.aj; ip = C.ip; a = C.a; cp = C.cp;
#pragma unroll
      for (int q = 0; q < 9; q++) g[q] = C.g[q];
#pragma unroll
      for (int q = 0; q < 3; q++) { gi_[q] = C.gi[q]; gj_[q] = C.gj[q]; gk_[q] = C.gk[q]; }
    }
    const T fi = tile_flux_i<T, TC>(M, P, Q, c, j, w, g[0], g[1], g[2]);
    const T fj = tile_flux_j<T, TC>(M, P, Q, c, j, w, g[3], g[4], g[5]);
    const T fk = tile_flux_k<T, TC>(P, Q, c, j, w, g[6], g[7], g[8]);
    const T fi_lo = tile_flux_i<T, TC>(M, P, Q, c - 1, j, wi, gi_[0], gi_[1], gi_[2]);
    const T fj_lo = tile_flux_j<T, TC>(M, P, Q, c, j - 1, wj, gj_[0], gj_[1], gj_[2]);
    const T fk_lo = tile_flux_k<T, TC>(M, P, c, j, wk, gk_[0], gk_[1], gk_[2]);
    const T xc = P[j * TC + c];
    T acc = 0;
    acc += fi; acc -= fi_lo;
    acc += fj; acc -= fj_lo;
    acc += fk; acc -= fk_lo;
    const T own = ghost ? C.xg : xc, rf = C.b - -aj * acc, rn = C.b - own;
    const T r = (w & 1u) ? rf : rn;
    const int row = j - 1, o = (row + row / CS) * XC + col;
    Y[o] = r * ip;
    Fa[o] = a;
    Fc[o] = cp;
    D[o] = own;
  }
  const T xe = cv_bld<T>(Bx, in_grid(nrow > 0 && tc == 0, base, sizeof(T)), 0);
  const T xt = cv_bld<T>(Bx, in_grid(nrow > 0 && tc == nch - 1, base + (unsigned)(mx * (my - 1)), sizeof(T)), 0);
  __syncthreads();

  // the columns: CS rows a thread, the recurrences as yline_reg_tile runs them
  const int o0 = (r0 + tc) * XC + col;
  T yv[CS], av[CS];
  T Aa = 1, Bb_ = 0, y = 0, e = 0;
  if (nrow > 0) {
#pragma unroll
    for (int q = 0; q < CS; q++) {
      const bool in = q < nrow;
      const int o = in ? o0 + q * XC : o0;
      const T yq = Y[o], aq = Fa[o];
      av[q] = in ? aq : (T)1;
      yv[q] = in ? yq : (T)0;
      Aa = av[q] * Aa;
      Bb_ = av[q] * Bb_ + yv[q];
    }
    SA[tid] = Aa; SB[tid] = Bb_;
  }
  __syncthreads();
  if (nrow > 0) {
#pragma unroll 4
    for (int q = 0; q < tc; q++) y = SA[q * XC + col] * y + SB[q * XC + col];
#pragma unroll
    for (int q = 0; q < CS; q++) {
      y = yv[q] + av[q] * y;
      yv[q] = y;
    }
    Aa = 1; Bb_ = 0;
#pragma unroll
    for (int q = CS - 1; q >= 0; q--) {
      const bool in = q < nrow;
      const T cq = Fc[in ? o0 + q * XC : o0];
      av[q] = in ? -cq : (T)1;
      yv[q] = in ? yv[q] : (T)0;
      Aa = av[q] * Aa;
      Bb_ = av[q] * Bb_ + yv[q];
    }
    SA[XC * nch + tid] = Aa; SB[XC * nch + tid] = Bb_;
  }
  __syncthreads();
  if (nrow > 0) {
#pragma unroll 4
    for (int q = nch - 1; q > tc; q--) e = SA[XC * (nch + q) + col] * e + SB[XC * (nch + q) + col];
#pragma unroll
    for (int q = CS - 1; q >= 0; q--) {
      e = yv[q] + av[q] * e;
      if (q < nrow) {
        xo[base + (unsigned)(mx * (1 + r0 + q))] = D[o0 + q * XC] + om * e;
      }
    }
    if (tc == 0) xo[base] = xe;
    if (tc == nch - 1) xo[base + (unsigned)(mx * (my - 1))] = xt;
  }
}

extern __shared__ double sweep_mem[];

template <class T, bool HG, int CS, int XC>
__global__ void __launch_bounds__(1024) k_sweep(OpV<T> A, const T *__restrict__ x, const T *__restrict__ b,
                                              T *__restrict__ xo, T om) {
  sweep_body<T, HG, CS, XC>(A, x, b, xo, om, cv_xcd_line(), (T *)sweep_mem);
}

}  // namespace

// f(HG, CS, XC) as compile-time constants for a precision and a number of rows
// (cs: as the line solve takes them)
template <class T, class F>
static void sweep_dispatch(bool hg, int cs, int xc, F f) {
  using std::integral_constant;
  auto by_rows = [&](auto h) {
    if (cs == 16) f(h, integral_constant<int, 16>{}, integral_constant<int, 4>{});
    else if (xc == 4) f(h, integral_constant<int, 8>{}, integral_constant<int, 4>{});
    else f(h, integral_constant<int, 8>{}, integral_constant<int, 8>{});
  };
  if constexpr (sizeof(T) == 4) {
    if (hg) { by_rows(std::true_type{}); return; }
  }
  by_rows(std::false_type{});
}
