// cv_coarse.h -- the coarsest multigrid level in one work-group: all its
// smoothing sweeps and the nullspace rule (the coarse solve of
// PoissonSolver_MG, poisson.c:1896-1910) without leaving the CU.  Included by
// cv_poisson.hip.
//
// The level holds a few thousand cells at most, so as launches every sweep
// is a residual and a line solve of 5-14 us each that wait for their own
// memory round trips.  Here x, the face fluxes and the line factors live in
// LDS and the operator of its faces in each thread's registers over all
// sweeps: a sweep forms every flux once and costs two barriers (point Jacobi)
// or five.  Bound by instruction issue on one CU.  Ten line sweeps with the
// nullspace rule on 4x32x4 cells: 98 us as launches, 36 here; 40 point Jacobi
// sweeps on 8x8x8 in FP64: 237 and 54.
// Every value is formed by the expressions of the launches (stencil_tile,
// yline_reg_tile, k_jacobi, the fluid sum's partition), so the bits are theirs.
#pragma once
#include <type_traits>

namespace {

constexpr int COARSE_NT = 1024;

// Extents and LDS plan of a level: x over the storage, the fluxes of the
// three face families at the faces of the interior cells, then (line
// smoother) the residual and the line factors of the interior cells and the
// chunk carries of the two recurrences
struct CoDims {
  int nx, ny, nz, N, n, fi, fj, fk;
  __host__ __device__ CoDims(int mx, int my, int mz)
      : nx(mx - 2), ny(my - 2), nz(mz - 2), N(nx * ny * nz), n(mx * my * mz), fi((nx + 1) * ny * nz),
        fj(nx * (ny + 1) * nz), fk(nx * ny * (nz + 1)) {}
  __host__ __device__ int faces() const { return fi + fj + fk; }
  // chunks of the line solve over all columns, cs rows each
  __host__ __device__ int chunks(int cs) const { return nx * nz * ((ny + cs - 1) / cs); }
  // values in LDS; cs = 0: point Jacobi
  __host__ __device__ int lds(int cs) const { return n + faces() + (cs ? 4 * N + 4 * chunks(cs) : 0); }
};

// makes the compiler forget what it knows of the value, so that the sweep
// loop does not hoist what it derives from it (decoded coefficients, masks,
// addresses: far more registers than the values)
template <class V>
__device__ __forceinline__ void opaque(V &v) { asm volatile("" : "+v"(v)); }

// floor(a / m) for 0 <= a < 2^16 from inv = 1 / m in FP32: (a + 1/2) / m lies at
// least 1 / 2m from an integer, far more than the product's rounding
__device__ __forceinline__ int coarse_div(int a, float inv) { return (int)(((float)a + 0.5f) * inv); }

// one face: the storage index of its lower cell and its family, the face
// bits of the operator word (open, two cross modes) and the coefficients
// (normal, first and second tangential axis)
template <class T, bool HG>
struct CoFace {
  uint32_t tw;     // storage index << 7 | family << 5 | face bits
  T g[3];
};
template <class T>
struct CoFace<T, true> {
  uint32_t tw;
  uint32_t ga, gb; // FP16: normal | first, second
};

// all sweeps of the coarsest level from a zero guess, then the nullspace
// rule, by one work-group of COARSE_NT threads.  CS: rows per thread of the
// line solve, 0 for point Jacobi; FPT: most faces a thread holds; om: the
// damping (times 2^-e for FP16 line factors), nrd and inv_nf: the partition
// and 1 / fluid rows of the nullspace sum
template <class T, bool HG, int CS, int FPT>
__device__ __forceinline__ void coarse_body(const OpV<T> &A, const T *__restrict__ b, T *__restrict__ x, T om, int nsweep,
                                            double inv_nf, int nrd, T *lds) {
  constexpr bool LINE = CS > 0;
  constexpr int CL = CS > 0 ? CS : 1;
  constexpr int CPT = (FPT + 2) / 3;   // there are at least three faces a cell
  __shared__ double shv[COARSE_NT / 64], part[64];
  const int tid = threadIdx.x;
  const int mx = A.mx, my = A.my, mz = A.mz, pl = mx * my;
  const CoDims D(mx, my, mz);
  const int nx = D.nx, ny = D.ny, nz = D.nz, N = D.N, n = D.n, NF = D.faces();
  T *const xs = lds, *const F = xs + n;
  // LINE only: carries, residual, line factors (a, ip, cp)
  const int NL = LINE ? D.chunks(CL) : 0;
  T *const SA = F + NF, *const SB = SA + 2 * NL, *const rs = SB + 2 * NL;
  T *const fa = rs + N, *const fp = fa + N, *const fc = fp + N;
  for (int t = tid; t < n; t += COARSE_NT) xs[t] = (T)0;
  const float rx = 1.0f / (float)nx, rx1 = 1.0f / (float)(nx + 1), ry = 1.0f / (float)ny, ry1 = 1.0f / (float)(ny + 1);

  // this thread's faces: tid, tid + COARSE_NT, ... of families i, j, k
  CoFace<T, HG> face[FPT];
#pragma unroll
  for (int q = 0; q < FPT; q++) {
    const int f = min(tid + q * COARSE_NT, NF - 1);
    const int d = f < D.fi ? 0 : f < D.fi + D.fj ? 1 : 2;
    const int r = f - (d == 0 ? 0 : d == 1 ? D.fi : D.fi + D.fj);
    const int ex = nx + (d == 0), ey = ny + (d == 1);
    const int jk = coarse_div(r, d == 0 ? rx1 : rx), i = r - jk * ex, k = coarse_div(jk, d == 1 ? ry1 : ry), j = jk - k * ey;
    const int t = (i + (d != 0)) + mx * ((j + (d != 1)) + my * (k + (d != 2)));
    // coefficients: normal 4d, tangential axes in order
    const int q0 = d == 0 ? 1 : d == 1 ? 3 : 6, q1 = d == 0 ? 2 : d == 1 ? 5 : 7;
    uint32_t w;
    if constexpr (HG) {
      const uint4 ha = A.hA[t];
      const uint2 hb = A.hB[t];
      w = hb.y >> 16;
      // halves: ha.x g0 g1 | ha.y g2 g6 | ha.z g7 g8; hb.x g3 g4 | hb.y g5
      face[q].ga = d == 0 ? ha.x : d == 1 ? (hb.x >> 16 | hb.x << 16) : (ha.z >> 16 | (ha.y & 0xffff0000u));
      face[q].gb = d == 0 ? ha.y & 0xffffu : d == 1 ? hb.y & 0xffffu : ha.z & 0xffffu;
    } else {
      w = A.fl[t];
      face[q].g[0] = A.g[4 * d][t];
      face[q].g[1] = A.g[q0][t];
      face[q].g[2] = A.g[q1][t];
    }
    face[q].tw = (uint32_t)t << 7 | (uint32_t)d << 5 | ((w >> (1 + 5 * d)) & 31u);
  }
  // and its cells
  // per cell its storage index << 5 | its periodic edges (i first, i last, k
  // first, k last) and fluid bit, and its lower i- and j-faces
  T bv[CPT], aj[CPT], dv[LINE ? 1 : CPT];
  uint32_t ct[CPT], cf[CPT];
#pragma unroll
  for (int q = 0; q < CPT; q++) {
    const int idx = min(tid + q * COARSE_NT, N - 1);
    const int jk = coarse_div(idx, rx), i = idx - jk * nx, k = coarse_div(jk, ry), j = jk - k * ny;
    const int t = (i + 1) + mx * ((j + 1) + my * (k + 1));
    ct[q] = (uint32_t)t << 5 | (A.fl[t] & 1u);
    if (A.xper) ct[q] |= (i == 0 ? 2u : 0u) | (i == nx - 1 ? 4u : 0u);
    if (A.zper) ct[q] |= (k == 0 ? 8u : 0u) | (k == nz - 1 ? 16u : 0u);
    cf[q] = (uint32_t)(i + (nx + 1) * (j + ny * k)) | (uint32_t)(D.fi + i + nx * (j + (ny + 1) * k)) << 16;
    bv[q] = b[t];
    if constexpr (HG) aj[q] = __uint_as_float(A.hA[t].w);
    else aj[q] = A.aj[t];
    if constexpr (!LINE) dv[q] = A.dinv[t];
    if constexpr (LINE) {
      if constexpr (HG) {
        const uint32_t h = A.yh[t];
        fa[idx] = half_lo(h); fp[idx] = half_hi(h); fc[idx] = half_lo((uint32_t)A.yc[t]);
      } else {
        fa[idx] = A.ylo[t]; fp[idx] = A.yip[t]; fc[idx] = A.ycp[t];
      }
      rs[idx] = bv[q];              // the residual of the zero guess
    }
  }
  // the fluxes of x through the thread's faces, each formed once
  auto fluxes = [&]() {
#pragma unroll
    for (int q = 0; q < FPT; q++) {
      const int f = tid + q * COARSE_NT;
      if (f >= NF) break;
      opaque(face[q].tw);
      const uint32_t tw = face[q].tw;
      const int o = (int)(tw >> 7), d = (int)(tw >> 5) & 3;
      const int sd = d == 0 ? 1 : d == 1 ? mx : pl, s0 = d == 0 ? mx : 1, s1 = d == 2 ? mx : pl, u = o + sd;
      T g[3];
      if constexpr (HG) {
        opaque(face[q].ga); opaque(face[q].gb);
        g[0] = half_lo(face[q].ga); g[1] = half_hi(face[q].ga); g[2] = half_lo(face[q].gb);
      } else {
        g[0] = face[q].g[0]; g[1] = face[q].g[1]; g[2] = face[q].g[2];
      }
      const T v = tile_flux<T>(xs[o], xs[u], g[0], tw, 1, g[1], xs[o + s0], xs[u + s0], xs[o - s0], xs[u - s0],
                               g[2], xs[o + s1], xs[u + s1], xs[o - s1], xs[u - s1]);
      F[f] = (tw & 1u) ? v : (T)0;
    }
  };
  // b - A x of the thread's cell q at storage index t
  auto resid = [&](int q, int t) -> T {
    const int ai = (int)(cf[q] & 0xffffu), bj = (int)(cf[q] >> 16), ak = D.fi + D.fj + tid + q * COARSE_NT;
    T acc = 0;
    acc += F[ai + 1]; acc -= F[ai];
    acc += F[bj + nx]; acc -= F[bj];
    acc += F[ak + nx * ny]; acc -= F[ak];
    const T rf = bv[q] - -aj[q] * acc, rn = bv[q] - xs[t];
    return (ct[q] & 1u) ? rf : rn;
  };
  // x of interior point t and its periodic images in the ghosts; e: the
  // edges it lies on, as in ct
  auto put = [&](int t, uint32_t e, T v) {
    xs[t] = v;
    if (e & 30u) {
      const int di = e & 2u ? nx : e & 4u ? -nx : 0, dk = (e & 8u ? nz : e & 16u ? -nz : 0) * pl;
      if (di) xs[t + di] = v;
      if (dk) xs[t + dk] = v;
      if (di && dk) xs[t + di + dk] = v;
    }
  };
  __syncthreads();
  if constexpr (LINE) {
    const int ncol = nx * nz, nch = (ny + CL - 1) / CL;
    const int tc = tid / ncol, col = tid - tc * ncol;
    const bool on = tc < nch;
    const int ck = col / nx, ci = col - ck * nx;
    const int nrow = on ? min(CL, ny - tc * CL) : 0;
    const uint32_t edge = (A.xper ? (ci == 0 ? 2u : 0u) | (ci == nx - 1 ? 4u : 0u) : 0u) |
                          (A.zper ? (ck == 0 ? 8u : 0u) | (ck == nz - 1 ? 16u : 0u) : 0u);
    int r0 = ci + nx * (tc * CL + ny * ck);                             // first row: interior index
    int t0 = (ci + 1) + mx * (tc * CL + 1 + my * (ck + 1));             // and storage index
    for (int s = 0; s < nsweep; s++) {
      if (s > 0) {
        fluxes();
        __syncthreads();
#pragma unroll
        for (int q = 0; q < CPT; q++) {
          if (tid + q * COARSE_NT >= N) break;
          opaque(ct[q]); opaque(cf[q]);
          rs[tid + q * COARSE_NT] = resid(q, (int)(ct[q] >> 5));
        }
        __syncthreads();
      }
      opaque(r0); opaque(t0);
      T yv[CL], av[CL];
      T Aa = 1, Bb = 0, y = 0;
      if (on) {
#pragma unroll
        for (int q = 0; q < CL; q++) {
          const bool in = q < nrow;
          const int e = in ? r0 + nx * q : 0;
          const T r = rs[e], p = fp[e], a = fa[e];
          av[q] = in ? a : (T)1;
          yv[q] = in ? r * p : (T)0;
          Aa = av[q] * Aa;
          Bb = av[q] * Bb + yv[q];
        }
        if (nch > 1) { SA[tid] = Aa; SB[tid] = Bb; }
      }
      if (nch > 1) __syncthreads();
      if (on) {
#pragma unroll 4
        for (int q = 0; q < tc; q++) y = SA[q * ncol + col] * y + SB[q * ncol + col];
#pragma unroll
        for (int q = 0; q < CL; q++) {
          y = yv[q] + av[q] * y;
          yv[q] = y;
        }
        Aa = 1; Bb = 0;
#pragma unroll
        for (int q = CL - 1; q >= 0; q--) {
          const bool in = q < nrow;
          const T c = fc[in ? r0 + nx * q : 0];
          av[q] = in ? -c : (T)1;
          yv[q] = in ? yv[q] : (T)0;
          Aa = av[q] * Aa;
          Bb = av[q] * Bb + yv[q];
        }
        if (nch > 1) { SA[NL + tid] = Aa; SB[NL + tid] = Bb; }
      }
      if (nch > 1) __syncthreads();
      if (on) {
        T e = 0;
#pragma unroll 4
        for (int q = nch - 1; q > tc; q--) e = SA[NL + q * ncol + col] * e + SB[NL + q * ncol + col];
#pragma unroll
        for (int q = CL - 1; q >= 0; q--) {
          e = yv[q] + av[q] * e;
          if (q < nrow) {
            const int t = t0 + mx * q;
            put(t, edge, xs[t] + om * e);
          }
        }
      }
      __syncthreads();
    }
  } else {
    for (int s = 0; s < nsweep; s++) {
      if (s > 0) {
        fluxes();
        __syncthreads();
      }
#pragma unroll
      for (int q = 0; q < CPT; q++) {
        if (tid + q * COARSE_NT >= N) break;
        opaque(ct[q]); opaque(cf[q]);
        const int t = (int)(ct[q] >> 5);
        const T v = s == 0 ? om * dv[q] * bv[q] : xs[t] + om * dv[q] * resid(q, t);
        put(t, ct[q], v);
      }
      __syncthreads();
    }
  }
  // the nullspace rule: the fluid sum by the partition of its launches
  // (blocks of BS threads), the final sum, the shift
  constexpr int NG = COARSE_NT / BS;
  const int grp = tid / BS, lt = tid % BS;
  for (int v0 = 0; v0 < nrd; v0 += NG) {
    const int vb = v0 + grp;
    double s = vb < nrd ? fluid_sum_thread<T>(xs, A.fl, n, vb, nrd, lt) : 0.0;
    s = cv_wave_sum(s);
    __syncthreads();
    if ((tid & 63) == 0) shv[tid >> 6] = s;
    __syncthreads();
    if (lt == 0 && vb < nrd) {
      double a = 0.0;
      for (int w = 0; w < BS / 64; w++) a += shv[grp * (BS / 64) + w];
      part[vb] = a;
    }
  }
  __syncthreads();
  {
    double s = 0.0;
    if (tid < BS)
      for (int q = tid; q < nrd; q += BS) s += part[q];
    s = cv_wave_sum(s);
    if ((tid & 63) == 0) shv[tid >> 6] = s;
    __syncthreads();
  }
  double sum = 0.0;
  for (int w = 0; w < BS / 64; w++) sum += shv[w];
  const double mean = sum * inv_nf;
  for (int t = tid; t < n; t += COARSE_NT) x[t] = (A.fl[t] & 1u) ? (T)((double)xs[t] - mean) : (T)0;
}

extern __shared__ double coarse_lds[];

template <class T, bool HG, int CS, int FPT>
__global__ void __launch_bounds__(COARSE_NT) k_coarse(OpV<T> A, const T *__restrict__ b, T *__restrict__ x, T om, int nsweep,
                                                      double inv_nf, int nrd) {
  coarse_body<T, HG, CS, FPT>(A, b, x, om, nsweep, inv_nf, nrd, (T *)coarse_lds);
}

}  // namespace

// rows per thread of the line solve, as its launches take them (0: none)
static int coarse_rows(const CvDims &d, bool line) { return !line ? 0 : d.my - 2 <= 16 * 8 ? 8 : 16; }

// whether one work-group takes a level: its LDS plan must fit, its faces the
// threads' registers, the lines' chunks one thread each, and the nullspace
// partials their array.  Past 7 faces a thread the launches are as fast (a
// sweep on 4x256x4 cells, 14 faces a thread: 17 us here, 19 as two launches)
#define COARSE_LDS (156 * 1024)
template <class T>
static bool coarse_fits(const CvDims &d, bool line) {
  if (d.mx < 5 || d.mz < 5 || d.n >= 32768 || nred(d.n) > 64) return false;
  const CoDims D(d.mx, d.my, d.mz);
  const int cs = coarse_rows(d, line);
  if (D.lds(cs) * (int)sizeof(T) > COARSE_LDS || D.faces() > 7 * COARSE_NT) return false;
  return !line || (D.ny <= 16 * 16 && D.chunks(cs) <= COARSE_NT);
}

// f(HG, CS, FPT) as compile-time constants for a precision, the rows per
// thread of the line solve (0: point Jacobi) and the level's faces
template <class T, class F>
static void coarse_dispatch(bool hg, int cs, int faces, F f) {
  using std::integral_constant;
  auto by_faces = [&](auto h, auto c) {
    if (faces <= 2 * COARSE_NT) f(h, c, integral_constant<int, 2>{});
    else if (faces <= 4 * COARSE_NT) f(h, c, integral_constant<int, 4>{});
    else f(h, c, integral_constant<int, 7>{});
  };
  auto by_rows = [&](auto h) {
    if (cs == 0) by_faces(h, integral_constant<int, 0>{});
    else if (cs == 8) by_faces(h, integral_constant<int, 8>{});
    else by_faces(h, integral_constant<int, 16>{});
  };
  if constexpr (sizeof(T) == 4) {
    if (hg) { by_rows(std::true_type{}); return; }
  }
  by_rows(std::false_type{});
}
