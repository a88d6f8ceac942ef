// Tiled kernel-vector products of the cubic co-kriging interpolant.
//
// One kernel family evaluates S(x) = sum over sources of weight * kernel(x, source)
// (+ drift) and optionally grad S, on a regular lattice regenerated in-kernel or
// on explicit points.  It serves three callers:
//   * grid / octree / custom-point evaluation (the engine's exported fields,
//     test_example_models_I.py:20-21; chunking 2-layers.approved.txt:172 is
//     unnecessary here: the lattice is never materialised),
//   * the matrix-free operator y = A x (the rows of A are the gradient of the
//     interpolant at orientation points and its increments at surface points),
//   * surface-point thresholds.
// Sources are staged through LDS in tiles of 256 and broadcast to the
// wavefront; every thread owns PPT points (a z-run on the lattice, where
// rho^2 is updated incrementally).
#include <algorithm>
#include <cmath>
#include "gk_internal.h"

namespace {

constexpr int TS = 256;   // sources per LDS tile == threads per block
// relative cost of one (point, source) pair: interface source or orientation,
// without or with the gradient
constexpr int src_cost(bool grad, bool ori) { return grad ? (ori ? 7 : 5) : (ori ? 5 : 4); }
// Explicit point sets too small to fill the GPU split their sources over
// blockIdx.y: at most SPLIT_WGS workgroups in all, at most MAX_SPLIT splits
// with the gradient and MAX_SPLIT_SCALAR without.  Measured on the
// operator product at N = 35k (scalar at 20,000 data points, gradient at
// 5,000 orientations, FP64): 288 us at 64 splits against 308 at 102 for the
// scalar, 123 us at 204 splits against 135 at 64 for the gradient.
constexpr int SPLIT_WGS = 2048, MAX_SPLIT = 256, MAX_SPLIT_SCALAR = 64;

template <typename T> struct alignas(sizeof(T) * 4) V4 { T x, y, z, w; };
template <typename T> struct alignas(sizeof(T) * 4) V8 { T x, y, z, pad0, wx, wy, wz, pad1; };

struct EvalArgs {
  int64_t n_points;
  int64_t n_runs;
  double ox, oy, oz, hx, hy, hz;
  int64_t nx, ny, nz, nzr;
  const double* xyz;
  double cx, cy, cz, inv_a;
  const void* pts;
  int64_t n_pts;
  const void* ori;
  int64_t n_ori;
  int32_t uni_degree, n_fault;
  const double* lam;          // drift then fault weights
  double gi_res;
  const double* fault_values;
  double* scalar;
  double* grad;
  int32_t* ids;
  int32_t n_thr, thr_rev;
  double thr[GK_MAX_THRESHOLDS];
  // source splitting across blockIdx.y (small point sets): partial sums go to
  // part_s [nsplit][n_points] (and part_g [nsplit][n_points][3]) and a
  // finalize kernel adds them in a fixed order.  The sources are the
  // interface sources followed by the orientations, each costing
  // src_cost(grad, orientation) units; split y takes the sources whose cost
  // interval starts in [y cost_chunk, (y + 1) cost_chunk), so every split
  // carries the same work.
  int32_t nsplit;
  int64_t cost_chunk;
  // explicit points, mask asked for: 1 for each of n_out groups of sources
  // with one outside the sphere of half the range around the centre (null:
  // not known)
  const int32_t* src_out;
  int32_t n_out;
  double* part_s;
  double* part_g;
};

__device__ __forceinline__ void drift_terms(const EvalArgs& a, double X, double Y, double Z,
                                            int64_t pidx, double& s, double* g) {
  if (a.uni_degree >= 1) {
    const double* l = a.lam;
    s += a.gi_res * (l[0] * X + l[1] * Y + l[2] * Z);
    if (g) { g[0] += a.gi_res * l[0]; g[1] += a.gi_res * l[1]; g[2] += a.gi_res * l[2]; }
    if (a.uni_degree >= 2) {
      s += a.gi_res * (l[3] * X * X + l[4] * Y * Y + l[5] * Z * Z + l[6] * X * Y + l[7] * X * Z +
                       l[8] * Y * Z);
      if (g) {
        g[0] += a.gi_res * (2 * l[3] * X + l[6] * Y + l[7] * Z);
        g[1] += a.gi_res * (2 * l[4] * Y + l[6] * X + l[8] * Z);
        g[2] += a.gi_res * (2 * l[5] * Z + l[7] * X + l[8] * Y);
      }
    }
  }
  if (a.n_fault > 0 && a.fault_values) {
    const int L = a.uni_degree == 0 ? 0 : (a.uni_degree == 1 ? 3 : 9);
    for (int f = 0; f < a.n_fault; ++f)
      s += a.gi_res * a.lam[L + f] * a.fault_values[pidx * a.n_fault + f];
  }
}

__device__ __forceinline__ int32_t segment_id(const EvalArgs& a, double s) {
  int32_t id = 1;
  if (a.thr_rev) {
    for (int k = 0; k < a.n_thr; ++k) id += (s > a.thr[k]) ? 1 : 0;
  } else {
    for (int k = 0; k < a.n_thr; ++k) id += (s < a.thr[k]) ? 1 : 0;
  }
  return id;
}

// Lattice scalar path (no gradient, no range mask), the grid evaluation:
// rho^2 never reaches 0 because a tiny positive offset rides on the
// per-source xy part (so no clamp per pair).  rho = sqrt(t) enters only as
// rho * Q(t), and one Newton step on r = t rsq(t) gives
// rho Q = r (1 + (1 - r y)/2) Q = (r Q/2) (3 - r y), so the polynomial is
// evaluated with halved coefficients and the step costs one FMA.  The source
// weight is folded into the coefficients, w C = w + t (w c0 + rho (w c1 +
// t (w c2 + w c3 t))), and the w are added once per tile.
template <typename T> struct Tiny;
template <> struct Tiny<double> { static constexpr double v = 1e-280; };
template <> struct Tiny<float> { static constexpr float v = 1e-30f; };

__device__ __forceinline__ double gk_rsq_raw(double t) { return __builtin_amdgcn_rsq(t); }
__device__ __forceinline__ float gk_rsq_raw(float t) { return __builtin_amdgcn_rsqf(t); }

// z - source z along a thread's run: points at a constant spacing, or at the
// positions of a table (interpolation nodes).
template <typename T> struct SpacedRun {
  T z0, hz;
  __device__ __forceinline__ T first(T sz) const { return z0 - sz; }
  __device__ __forceinline__ T next(int q, T e0, T) const { return fma(T(q), hz, e0); }
};
template <typename T, int PPT> struct TableRun {
  T z[PPT];
  __device__ __forceinline__ T first(T) const { return T(0); }
  __device__ __forceinline__ T next(int q, T, T sz) const { return z[q] - sz; }
};

// Sums of one LDS tile's sources over a z-run of PPT lattice points (x0, y0, zr).
// What bounds them is the issue of FP64 (FP32) vector instructions, so what
// depends on the source or the run alone is kept out of the pair, t never
// reaches 0, and the Newton step of rho = sqrt(t) rides on the polynomial (see
// above; FP32 sums with mask or gradient take the raw rsq).  The plain field
// also folds the source weight into the coefficients: 9 instructions and an
// rsq per interface pair.  With mask or gradient the coefficients stay the
// exact constants, which costs nothing there (the weight joins the last
// product) and loses nothing near the range, where C vanishes.  With a clamp
// and a full Newton step per pair instead, field and gradient of 1.2e6 points
// and 1,900 sources took 2.39 ms against 2.14 (1.78 since tiles run over the
// sources they hold), the masked field of 1.2e6 points and 6,000 sources 4.82
// against 4.28 (1.69 in blocks).
template <typename T> __device__ __forceinline__ T rho_poly(T u, T r, T h3, T c0) {
  if constexpr (sizeof(T) == 4) return fma(r, u, c0);        // u = Q
  else return fma(r * u, h3, c0);                            // u = Q / 2
}

// FOLD: the plain field's form (sums that stand in for masked ones, whose
// pairs all lie within the range, go without).
template <typename T, bool GRAD, bool MASKED, int PPT, bool FOLD = !GRAD && !MASKED, typename Run>
__device__ __forceinline__ void lattice_pts_tile(const V4<T>* s4, int nk, T x0, T y0, const Run& zr, T (&part)[PPT],
                                                 T (&gpart)[PPT][3]) {
  if constexpr (FOLD) {
    T wsum = T(0);
#pragma unroll 2
    for (int k = 0; k < nk; ++k) {
      const V4<T> s = s4[k];
      const T dx = x0 - s.x, dy = y0 - s.y;
      const T dxy = fma(dx, dx, fma(dy, dy, Tiny<T>::v));
      const T c3 = T(0.375) * s.w, c2 = T(-1.75) * s.w, c1 = T(4.375) * s.w, c0 = T(-7.0) * s.w;
      const T e0 = zr.first(s.z);
      wsum += s.w;
#pragma unroll
      for (int q = 0; q < PPT; ++q) {
        const T e = zr.next(q, e0, s.z);
        const T t = fma(e, e, dxy);
        const T y = gk_rsq_raw(t);
        const T r = t * y;
        const T h3 = fma(-r, y, T(3));
        T u = fma(c3, t, c2);
        u = fma(u, t, c1);
        const T v = fma(r * u, h3, c0);
        part[q] = fma(v, t, part[q]);
      }
    }
#pragma unroll
    for (int q = 0; q < PPT; ++q) part[q] += wsum;
  } else {
    // C: 3/4, -7/2, 35/4, -7; C'/r: 21/4, -35/2, 105/4, -14 (those of rho Q halved for the Newton step)
    constexpr T H = sizeof(T) == 4 ? T(1) : T(0.5);
    T c3 = T(0.75) * H, c2 = T(-3.5) * H, c1 = T(8.75) * H, d3 = T(5.25) * H, d2 = T(-17.5) * H, d1 = T(26.25) * H;
    asm volatile("" : "+v"(c3), "+v"(c2), "+v"(c1), "+v"(d3), "+v"(d2), "+v"(d1));
#pragma unroll 2
    for (int k = 0; k < nk; ++k) {
      const V4<T> s = s4[k];
      const T dx = x0 - s.x, dy = y0 - s.y;
      const T dxy = fma(dx, dx, fma(dy, dy, Tiny<T>::v));
      const T e0 = zr.first(s.z);
#pragma unroll
      for (int q = 0; q < PPT; ++q) {
        const T e = zr.next(q, e0, s.z);
        const T t = fma(e, e, dxy);
        const T y = gk_rsq_raw(t);
        const T r = t * y;
        const T h3 = fma(-r, y, T(3));
        T c = fma(rho_poly(fma(fma(c3, t, c2), t, c1), r, h3, T(-7)), t, T(1));
        if (MASKED) c = t < T(1) ? c : T(0);
        part[q] = fma(s.w, c, part[q]);
        if (GRAD) {
          T dp = rho_poly(fma(fma(d3, t, d2), t, d1), r, h3, T(-14));
          if (MASKED) dp = t < T(1) ? dp : T(0);
          const T wd = s.w * dp;
          gpart[q][0] = fma(wd, dx, gpart[q][0]);
          gpart[q][1] = fma(wd, dy, gpart[q][1]);
          gpart[q][2] = fma(wd, e, gpart[q][2]);
        }
      }
    }
  }
}

template <typename T, bool GRAD, bool MASKED, int PPT, bool FOLD = !GRAD && !MASKED, typename Run>
__device__ __forceinline__ void lattice_ori_tile(const V8<T>* s8, int nk, T x0, T y0, const Run& zr, T (&part)[PPT],
                                                 T (&gpart)[PPT][3]) {
  // the derivative polynomial's constants held in registers (as literals
  // the compiler would rebuild them inside the loop)
  constexpr bool NEWTON = sizeof(T) == 8 || FOLD;
  constexpr T H = NEWTON ? T(0.5) : T(1);
  T d3 = T(5.25) * H, d2 = T(-17.5) * H, d1 = T(26.25) * H, d0 = T(-14.0);
  asm volatile("" : "+v"(d3), "+v"(d2), "+v"(d1), "+v"(d0));
#pragma unroll 2
  for (int k = 0; k < nk; ++k) {
    const V8<T> s = s8[k];
    const T dx = s.x - x0, dy = s.y - y0;          // q - x
    const T dxy = fma(dx, dx, fma(dy, dy, Tiny<T>::v));
    const T base_dot = fma(s.wx, dx, s.wy * dy);
    const T e0 = zr.first(s.z);                    // x - q (z)
#pragma unroll
    for (int q = 0; q < PPT; ++q) {
      const T e = zr.next(q, e0, s.z);
      const T t = fma(e, e, dxy);
      const T y = gk_rsq_raw(t);
      const T r = t * y;
      const T h3 = fma(-r, y, T(3));
      const T u = fma(fma(d3, t, d2), t, d1);
      T p = NEWTON ? fma(r * u, h3, d0) : fma(r, u, d0);
      if (MASKED) p = t < T(1) ? p : T(0);
      const T dot = fma(-s.wz, e, base_dot);
      part[q] = fma(dot, p, part[q]);
      if (GRAD) {
        const T om = T(1) - t;
        // 26.25 (1-t)^2 / rho, 1/rho = y (3 - r y) / 2
        T dd = d1 * om * om * (NEWTON ? y * h3 : y);
        if (MASKED) dd = t < T(1) ? dd : T(0);
        const T hw = dot * dd;
        gpart[q][0] -= fma(s.wx, p, hw * dx);
        gpart[q][1] -= fma(s.wy, p, hw * dy);
        gpart[q][2] -= fma(s.wz, p, -hw * e);
      }
    }
  }
}

// Sums of one LDS tile's sources at PPT explicit points: no clamp per pair,
// Newton step folded as on the lattice.  kc: the halved constants of C (3/4,
// -7/2, 35/4) and C'/r (21/4, -35/2, 105/4), held in registers.
template <typename T, bool GRAD, bool MASKED, int PPT, bool SCALAR>
__device__ __forceinline__ void points_pts_tile(const V4<T>* s4, int nk, const T (&kc)[6], const T (&px)[PPT],
                                                const T (&py)[PPT], const T (&pz)[PPT], T (&part)[PPT],
                                                T (&gpart)[PPT][3]) {
#pragma unroll 2
  for (int k = 0; k < nk; ++k) {
    const V4<T> s = s4[k];
#pragma unroll
    for (int q = 0; q < PPT; ++q) {
      const T dx = px[q] - s.x, dy = py[q] - s.y, dz = pz[q] - s.z;
      const T t = fma(dz, dz, fma(dy, dy, fma(dx, dx, Tiny<T>::v)));
      const T y = gk_rsq_raw(t);
      const T r = t * y;
      const T h3 = fma(-r, y, T(3));
      T c = fma(fma(r * fma(fma(kc[0], t, kc[1]), t, kc[2]), h3, T(-7)), t, T(1));
      if (MASKED) c = t < T(1) ? c : T(0);
      if (SCALAR) part[q] = fma(s.w, c, part[q]);
      if (GRAD) {
        T dp = fma(r * fma(fma(kc[3], t, kc[4]), t, kc[5]), h3, T(-14));
        if (MASKED) dp = t < T(1) ? dp : T(0);
        const T wd = s.w * dp;
        gpart[q][0] = fma(wd, dx, gpart[q][0]);
        gpart[q][1] = fma(wd, dy, gpart[q][1]);
        gpart[q][2] = fma(wd, dz, gpart[q][2]);
      }
    }
  }
}

template <typename T, bool GRAD, bool MASKED, int PPT, bool SCALAR>
__device__ __forceinline__ void points_ori_tile(const V8<T>* s8, int nk, const T (&kc)[6], const T (&px)[PPT],
                                                const T (&py)[PPT], const T (&pz)[PPT], T (&part)[PPT],
                                                T (&gpart)[PPT][3]) {
#pragma unroll 2
  for (int k = 0; k < nk; ++k) {
    const V8<T> s = s8[k];
#pragma unroll
    for (int q = 0; q < PPT; ++q) {
      const T dx = s.x - px[q], dy = s.y - py[q], dz = s.z - pz[q];   // q - x
      const T t = fma(dz, dz, fma(dy, dy, fma(dx, dx, Tiny<T>::v)));
      const T y = gk_rsq_raw(t);
      const T r = t * y;
      const T h3 = fma(-r, y, T(3));
      T p = fma(r * fma(fma(kc[3], t, kc[4]), t, kc[5]), h3, T(-14));
      if (MASKED) p = t < T(1) ? p : T(0);
      const T dot = fma(s.wz, dz, fma(s.wy, dy, s.wx * dx));
      if (SCALAR) part[q] = fma(dot, p, part[q]);
      if (GRAD) {
        const T om = T(1) - t;
        T dd = T(13.125) * om * om * (y * h3);     // 26.25 (1-t)^2 / rho, 1/rho = y (3 - r y) / 2
        if (MASKED) dd = t < T(1) ? dd : T(0);
        const T hw = dot * dd;
        gpart[q][0] -= fma(s.wx, p, hw * dx);
        gpart[q][1] -= fma(s.wy, p, hw * dy);
        gpart[q][2] -= fma(s.wz, p, hw * dz);
      }
    }
  }
}

// Square of half the range (range units) less the rounding of both ends of a pair.
template <typename T> __host__ __device__ constexpr double half_range2() {
  return 0.25 * (1.0 - (sizeof(T) == 4 ? 1e-5 : 1e-9));
}

// SCALAR false (explicit points with gradient): the gradient only; the
// scalar output then holds the drift terms alone.
template <typename T, bool LATTICE, bool GRAD, bool MASKED, int PPT, bool SCALAR = true>
__global__ __launch_bounds__(TS) void eval_kernel(EvalArgs a) {
  __shared__ V8<T> s_src[TS];
  const int tid = threadIdx.x;
  const int64_t run = (int64_t)blockIdx.x * TS + tid;
  const bool run_ok = run < a.n_runs;

  // point coordinates (normalised frame) --------------------------------
  T px[PPT], py[PPT], pz[PPT];
  int64_t pidx[PPT];
  bool pok[PPT];
  T x0 = 0, y0 = 0, z0 = 0, hz = 0;
  int64_t ix = 0, iy = 0, iz0 = 0;
  if (LATTICE) {
    int64_t r = run_ok ? run : 0;
    iz0 = (r % a.nzr) * PPT;
    int64_t rest = r / a.nzr;
    iy = rest % a.ny;
    ix = rest / a.ny;
    x0 = (T)((a.ox + ix * a.hx - a.cx) * a.inv_a);
    y0 = (T)((a.oy + iy * a.hy - a.cy) * a.inv_a);
    z0 = (T)((a.oz + iz0 * a.hz - a.cz) * a.inv_a);
    hz = (T)(a.hz * a.inv_a);
#pragma unroll
    for (int q = 0; q < PPT; ++q) {
      pok[q] = run_ok && (iz0 + q) < a.nz;
      pidx[q] = (ix * a.ny + iy) * a.nz + iz0 + q;
    }
  } else {
#pragma unroll
    for (int q = 0; q < PPT; ++q) {
      int64_t p = (run_ok ? run : 0) * PPT + q;
      pok[q] = run_ok && p < a.n_points;
      pidx[q] = pok[q] ? p : 0;
      const double* X = a.xyz + 3 * pidx[q];
      px[q] = (T)((X[0] - a.cx) * a.inv_a);
      py[q] = (T)((X[1] - a.cy) * a.inv_a);
      pz[q] = (T)((X[2] - a.cz) * a.inv_a);
    }
  }

  double acc[PPT];
  double gacc[PPT][3];
  T part[PPT];
  T gpart[PPT][3];
#pragma unroll
  for (int q = 0; q < PPT; ++q) {
    acc[q] = 0.0;
    part[q] = T(0);
    gacc[q][0] = gacc[q][1] = gacc[q][2] = 0.0;
    gpart[q][0] = gpart[q][1] = gpart[q][2] = T(0);
  }

  // Explicit points come without a box.  Where every source and every point
  // of the wave lies within half the range of the centre no pair is beyond it,
  // and the same sums go without the mask: the preparing launch leaves a flag
  // per group of sources, the wave looks at its own points.  A product of
  // 25,000 data 431 us with the mask, 391 without; 100,000 points of 6,000
  // sources 390 and 351.
  bool inside = false;
  if constexpr (!LATTICE && MASKED) {
    bool out = a.src_out == nullptr;
    for (int i = tid & 63; !out && i < a.n_out; i += 64) out = a.src_out[i] != 0;
#pragma unroll
    for (int q = 0; q < PPT; ++q)
      out = out || !((double)fma(pz[q], pz[q], fma(py[q], py[q], px[q] * px[q])) <= half_range2<T>());
    inside = !__any(out);
  }

  T kc[6] = {T(0.375), T(-1.75), T(4.375), T(2.625), T(-8.75), T(13.125)};
  if constexpr (!LATTICE) asm volatile("" : "+v"(kc[0]), "+v"(kc[1]), "+v"(kc[2]), "+v"(kc[3]), "+v"(kc[4]), "+v"(kc[5]));

  // ---- interface + reference sources: weight * C(|x - p|) -----------------
  const V4<T>* pts = reinterpret_cast<const V4<T>*>(a.pts);
  V4<T>* s4 = reinterpret_cast<V4<T>*>(s_src);
  int64_t pb = 0, pe = a.n_pts, obeg = 0, oend = a.n_ori;    // the lattice is never split
  if constexpr (!LATTICE) {
    constexpr int64_t CP = src_cost(GRAD, false), CO = src_cost(GRAD, true);
    const int64_t cpts = a.n_pts * CP;
    const int64_t clo = (int64_t)blockIdx.y * a.cost_chunk, chi = clo + a.cost_chunk;
    pb = min(a.n_pts, (clo + CP - 1) / CP);
    pe = min(a.n_pts, (chi + CP - 1) / CP);
    obeg = min(a.n_ori, (max(clo - cpts, (int64_t)0) + CO - 1) / CO);
    oend = min(a.n_ori, (max(chi - cpts, (int64_t)0) + CO - 1) / CO);
  }
  for (int64_t base = pb; base < pe; base += TS) {
    // sources in this tile (always TS, padded with zero weights, cost a sketch
    // of 33 sources 512: 125,000 points 132 us of a model of 1.29 ms, 1.16 now)
    const int nk = (int)min((int64_t)TS, pe - base);
    __syncthreads();
    {
      int64_t j = base + tid;
      V4<T> v;
      if (j < pe) v = pts[j];
      else { v.x = T(0); v.y = T(0); v.z = T(0); v.w = T(0); }
      s4[tid] = v;
    }
    __syncthreads();
    if constexpr (LATTICE) {
      lattice_pts_tile<T, GRAD, MASKED, PPT>(s4, nk, x0, y0, SpacedRun<T>{z0, hz}, part, gpart);
    } else if (MASKED && !inside) {
      points_pts_tile<T, GRAD, true, PPT, SCALAR>(s4, nk, kc, px, py, pz, part, gpart);
    } else {
      points_pts_tile<T, GRAD, false, PPT, SCALAR>(s4, nk, kc, px, py, pz, part, gpart);
    }
#pragma unroll
    for (int q = 0; q < PPT; ++q) {
      acc[q] += (double)part[q];
      part[q] = T(0);
      if (GRAD) {
        for (int u = 0; u < 3; ++u) { gacc[q][u] += (double)gpart[q][u]; gpart[q][u] = T(0); }
      }
    }
  }

  // ---- orientation sources: (w . (q - x)) C'(r)/r --------------------------
  const V8<T>* ori = reinterpret_cast<const V8<T>*>(a.ori);
  for (int64_t base = obeg; base < oend; base += TS) {
    const int nk = (int)min((int64_t)TS, oend - base);
    __syncthreads();
    {
      int64_t j = base + tid;
      V8<T> v;
      if (j < oend) v = ori[j];
      else { v.x = v.y = v.z = v.pad0 = v.wx = v.wy = v.wz = v.pad1 = T(0); }
      s_src[tid] = v;
    }
    __syncthreads();
    if constexpr (LATTICE) {
      lattice_ori_tile<T, GRAD, MASKED, PPT>(s_src, nk, x0, y0, SpacedRun<T>{z0, hz}, part, gpart);
    } else if (MASKED && !inside) {
      points_ori_tile<T, GRAD, true, PPT, SCALAR>(s_src, nk, kc, px, py, pz, part, gpart);
    } else {
      points_ori_tile<T, GRAD, false, PPT, SCALAR>(s_src, nk, kc, px, py, pz, part, gpart);
    }
#pragma unroll
    for (int q = 0; q < PPT; ++q) {
      acc[q] += (double)part[q];
      part[q] = T(0);
      if (GRAD) {
        for (int u = 0; u < 3; ++u) { gacc[q][u] += (double)gpart[q][u]; gpart[q][u] = T(0); }
      }
    }
  }

  // ---- drift (FP64, raw coordinates), ids, store -----------------------------
  if (a.nsplit > 1) {
#pragma unroll
    for (int q = 0; q < PPT; ++q) {
      if (!pok[q]) continue;
      const int64_t o = (int64_t)blockIdx.y * a.n_points + pidx[q];
      a.part_s[o] = acc[q];
      if (GRAD && a.part_g) {
        a.part_g[3 * o + 0] = gacc[q][0];
        a.part_g[3 * o + 1] = gacc[q][1];
        a.part_g[3 * o + 2] = gacc[q][2];
      }
    }
    return;
  }
#pragma unroll
  for (int q = 0; q < PPT; ++q) {
    if (!pok[q]) continue;
    double X, Y, Z;
    if (LATTICE) {
      X = a.ox + ix * a.hx; Y = a.oy + iy * a.hy; Z = a.oz + (iz0 + q) * a.hz;
    } else {
      const double* P = a.xyz + 3 * pidx[q];
      X = P[0]; Y = P[1]; Z = P[2];
    }
    double s = acc[q];
    double g[3] = {gacc[q][0] * a.inv_a, gacc[q][1] * a.inv_a, gacc[q][2] * a.inv_a};
    drift_terms(a, X, Y, Z, pidx[q], s, GRAD ? g : nullptr);
    a.scalar[pidx[q]] = s;
    if (GRAD && a.grad) {
      a.grad[3 * pidx[q] + 0] = g[0];
      a.grad[3 * pidx[q] + 1] = g[1];
      a.grad[3 * pidx[q] + 2] = g[2];
    }
    if (a.ids) a.ids[pidx[q]] = segment_id(a, s);
  }
}

// ------------------------------------------------- lattice blocks, far sources
// A lattice evaluation in blocks of points.  For one block the sources fall
// into three groups:
//   beyond   no point of the block within the range: left out
//   far      well separated: their summed field is smooth over the block, so
//            it is summed at a tensor grid of N^3 Chebyshev nodes and
//            interpolated to the points
//   near     the others, summed pair by pair
// What bounds the direct sum is the issue of its pairs (85 ms for 8e6 points
// and 25,000 sources); a block of 30^3 points takes 16^3 node sums for its far
// sources instead of 27,000.
//
// Separation.  Along one axis the field of a source at lateral distance s and
// axial offset z is analytic but for the points z +- i s (C is a polynomial in
// rho^2 and rho), so the interpolation error falls with the ellipse through
// them: with the block's half width as unit, a = (|z + i s + 1| + |z + i s -
// 1|) / 2 has to reach the same bound on every axis (s taken from the nearest
// points of the block).  The bound is that of a source beside the block at a
// gap of g half widths, a = sqrt(1 + g^2).  Measured in 80-bit arithmetic for
// unit weights at half width 0.036 of the range: N = 16, g = 3: 2e-17 for C
// and 2e-15 for an orientation's term (computing one such term in FP64 rounds
// it by 4e-16 rms and up to 3.4e-15, its largest part being 14; C by 1.5e-16
// and 1.2e-15), for the worst source at that gap; four times less per 0.5 more
// of g, 15 times more per 0.5 less.  N = 8, g = 2.5: 8e-10 and
// 5e-8 (FP32 sums), 3 times more per 0.5.  The error grows with the square of
// the half width, which the gap makes up for.
// The interpolant passes rounding errors of the node sums on without growth
// (the squares of the cardinal functions of Chebyshev nodes sum to at most 1).
// Sources with a weight or position that is not finite count as near, so that
// they reach the same points as in a direct sum.
struct FarArgs {
  EvalArgs e;
  int32_t p[3], b[3];        // points of a block per axis, blocks per axis
  int32_t n;                 // nodes per axis (0: near and beyond only)
  int32_t nsplit;            // far sources of a block in this many parts
  int32_t masked;
  float amin;
  int32_t *lp, *lo;          // [block][n_pts], [block][n_ori]: near from the front, far from the back
  int32_t* cnt;              // [block][4]: near, far interface sources, near, far orientations
  int32_t* order;            // blocks by falling number of near sources
  double* nodes;             // [split][block][n^3]
  double* tab;               // [p0 + p1 + p2][n] interpolation weights per axis
};

enum { FAR_BEYOND = 0, FAR_NEAR = 1, FAR_FAR = 2 };

// Group of a source at distance d (per axis, from the block's centre) of a
// block with half widths h, in units of the range.  The margins of the range
// tests cover FP32: the near sums test each pair themselves.  slack: what the
// rounding of d, h and FP32 positions may add to the squared distance (it
// counts where the block is many ranges wide or away from the centre).
__host__ __device__ inline int far_group(const float d[3], const float h[3], bool masked, bool nodes, float amin,
                                         float slack = 0.0f) {
  float g[3], dmin = 0.0f, dmax = 0.0f;
  for (int k = 0; k < 3; ++k) {
    g[k] = d[k] > h[k] ? d[k] - h[k] : 0.0f;
    dmin += g[k] * g[k];
    dmax += (d[k] + h[k]) * (d[k] + h[k]);
  }
  if (masked && dmin >= 1.0001f + slack) return FAR_BEYOND;
  if (!nodes || (masked && !(dmax < 0.9999f))) return FAR_NEAR;
  for (int k = 0; k < 3; ++k) {
    const float s2 = dmin - g[k] * g[k], u = d[k] + h[k], v = d[k] - h[k];
    if (!(0.5f * (sqrtf(u * u + s2) + sqrtf(v * v + s2)) >= amin * h[k])) return FAR_NEAR;
  }
  return FAR_FAR;
}

template <typename T> __device__ __forceinline__ bool finite4(const V4<T>& v) {
  return isfinite(v.x) && isfinite(v.y) && isfinite(v.z) && isfinite(v.w);
}
template <typename T> __device__ __forceinline__ bool finite4(const V8<T>& v) {
  return isfinite(v.x) && isfinite(v.y) && isfinite(v.z) && isfinite(v.wx) && isfinite(v.wy) && isfinite(v.wz);
}

// Centre and half widths (signed, as the spacing) of block b in range units.
__device__ __forceinline__ void far_box(const FarArgs& f, int64_t b, double c[3], double h[3], int64_t i0[3]) {
  const int64_t ib[3] = {b / ((int64_t)f.b[1] * f.b[2]), b / f.b[2] % f.b[1], b % f.b[2]};
  const double o[3] = {f.e.ox - f.e.cx, f.e.oy - f.e.cy, f.e.oz - f.e.cz}, sp[3] = {f.e.hx, f.e.hy, f.e.hz};
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    i0[k] = ib[k] * f.p[k];
    h[k] = 0.5 * (f.p[k] - 1) * sp[k] * f.e.inv_a;
    c[k] = (o[k] + i0[k] * sp[k]) * f.e.inv_a + h[k];
  }
}

// Chebyshev nodes of the first kind on [-1, 1], ascending.
__device__ __forceinline__ double cheb_node(int k, int n) { return -cospi((2 * k + 1) / (2.0 * n)); }

// One workgroup per block sorts the sources of one kind into the block's list,
// each group in the sources' order.
template <typename T, typename V>
__device__ void far_sort(const FarArgs& f, const V* src, int64_t n, const double c[3], const float h[3], int32_t* list,
                         int32_t* cnt) {
  __shared__ int32_t w_near[16], w_far[16];
  const int t = threadIdx.x, wave = t >> 6;
  const uint64_t below = (1ull << (t & 63)) - 1;
  int32_t nnear = 0, nfar = 0;
  // 2^-24 each of d, of h (d < h + 2 where it matters) and, in FP32, of both
  // positions, on every axis, twice for the square
  const float slack = 1e-6f * (float)(fabs(c[0]) + fabs(c[1]) + fabs(c[2]) + h[0] + h[1] + h[2]);
  for (int64_t base = 0; base < n; base += 1024) {
    int g = FAR_BEYOND;
    if (base + t < n) {
      const V v = src[base + t];
      const float d[3] = {(float)fabs((double)v.x - c[0]), (float)fabs((double)v.y - c[1]),
                          (float)fabs((double)v.z - c[2])};
      g = finite4(v) ? far_group(d, h, f.masked != 0, f.n > 0, f.amin, slack) : FAR_NEAR;
    }
    const uint64_t mn = __ballot(g == FAR_NEAR), mf = __ballot(g == FAR_FAR);
    if ((t & 63) == 0) { w_near[wave] = __popcll(mn); w_far[wave] = __popcll(mf); }
    __syncthreads();
    int32_t an = nnear, af = nfar;
    for (int w = 0; w < 16; ++w) {
      if (w == wave) { an = nnear; af = nfar; }
      nnear += w_near[w];
      nfar += w_far[w];
    }
    if (g == FAR_NEAR) list[an + __popcll(mn & below)] = (int32_t)(base + t);
    if (g == FAR_FAR) list[n - 1 - (af + __popcll(mf & below))] = (int32_t)(base + t);
    __syncthreads();
  }
  if (t == 0) { cnt[0] = nnear; cnt[1] = nfar; }
}

template <typename T>
__global__ __launch_bounds__(1024) void far_sort_kernel(FarArgs f) {
  const int64_t nb = (int64_t)f.b[0] * f.b[1] * f.b[2], b = blockIdx.x;
  if (b == nb) {             // the last workgroup: interpolation weights (second barycentric form)
    const int rows = f.p[0] + f.p[1] + f.p[2];
    for (int r = threadIdx.x; r < rows; r += 1024) {
      const int k = r < f.p[0] ? 0 : (r < f.p[0] + f.p[1] ? 1 : 2);
      const int i = r - (k > 0 ? f.p[0] : 0) - (k > 1 ? f.p[1] : 0);
      const double x = (2.0 * i - (f.p[k] - 1)) / (f.p[k] - 1);
      double* o = f.tab + (int64_t)r * f.n;
      double sum = 0.0;
      int hit = -1;
      for (int m = 0; m < f.n; ++m) {
        const double dx = x - cheb_node(m, f.n);
        if (dx == 0.0) hit = m;
        const double w = ((m & 1) ? -sinpi((2 * m + 1) / (2.0 * f.n)) : sinpi((2 * m + 1) / (2.0 * f.n))) / dx;
        o[m] = w;
        sum += w;
      }
      for (int m = 0; m < f.n; ++m) o[m] = hit >= 0 ? (m == hit ? 1.0 : 0.0) : o[m] / sum;
    }
    return;
  }
  double c[3], hd[3];
  int64_t i0[3];
  far_box(f, b, c, hd, i0);
  const float h[3] = {(float)fabs(hd[0]), (float)fabs(hd[1]), (float)fabs(hd[2])};
  far_sort<T>(f, reinterpret_cast<const V4<T>*>(f.e.pts), f.e.n_pts, c, h, f.lp + b * f.e.n_pts, f.cnt + 4 * b);
  far_sort<T>(f, reinterpret_cast<const V8<T>*>(f.e.ori), f.e.n_ori, c, h, f.lo + b * f.e.n_ori, f.cnt + 4 * b + 2);
}

// Blocks by falling cost of their near sources (ties by number).  Blocks in
// the middle of the model have about twice the mean, a launch holds few more
// workgroups than fit the chip, and workgroups go round the XCDs and CUs: in
// lattice order one XCD got all the middle layers; in falling order each CU
// gets its share of heavy, middling and light ones (near part of 1.2e6 points,
// range 0.45 of the box: 4.14 ms, then 2.55 with blocks of half the size).
__global__ __launch_bounds__(256) void far_order_kernel(FarArgs f, int32_t nb) {
  constexpr int CP = src_cost(false, false), CO = src_cost(false, true);
  const int32_t b = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;    // a wave per block
  if (b >= nb) return;
  const int32_t mine = CP * f.cnt[4 * b] + CO * f.cnt[4 * b + 2];
  int32_t rank = 0;
  for (int32_t j = lane; j < nb; j += 64) {
    const int32_t c = CP * f.cnt[4 * j] + CO * f.cnt[4 * j + 2];
    rank += c > mine || (c == mine && j < b);
  }
  for (int o = 32; o > 0; o >>= 1) rank += __shfl_xor(rank, o);
  if (lane == 0) f.order[rank] = b;
}

// acc += v with the rounding error kept in err (Knuth's two-sum): the sums of
// tiles add up to the field's size many times over, and grouping the sources
// by distance can make them larger on the way than in the sources' order.
__device__ __forceinline__ void add_exact(double& acc, double& err, double v) {
  const double s = acc + v, b = s - acc;
  err += (acc - (s - b)) + (v - b);
  acc = s;
}
// The sum; its error term is no number where the sum is infinite.
__device__ __forceinline__ double exact_sum(double acc, double err) { return err == err ? acc + err : acc; }

// Far sources of a block at its nodes: one wave per 64 runs of 8 nodes and per
// part of the sources, so that a few hundred blocks still fill the chip.
constexpr int FAR_TS = 64, FAR_RUN = 8;
template <typename T, int N, bool FOLD>
__global__ __launch_bounds__(FAR_TS) void far_nodes_kernel(FarArgs f) {
  static_assert(N % FAR_RUN == 0 && N * N * N % (FAR_TS * FAR_RUN) == 0, "whole waves of whole runs");
  constexpr int G = N * N * N / (FAR_TS * FAR_RUN);
  __shared__ V8<T> tile[FAR_TS];
  V4<T>* tile4 = reinterpret_cast<V4<T>*>(tile);
  const int lane = threadIdx.x, run = (blockIdx.x % G) * FAR_TS + lane;
  const int64_t b = blockIdx.x / G, nb = (int64_t)f.b[0] * f.b[1] * f.b[2];
  const int split = blockIdx.y;
  double c[3], h[3];
  int64_t i0[3];
  far_box(f, b, c, h, i0);
  const int iz = run % (N / FAR_RUN) * FAR_RUN, iy = run / (N / FAR_RUN) % N, ix = run / (N / FAR_RUN * N);
  const T x0 = (T)(c[0] + h[0] * cheb_node(ix, N)), y0 = (T)(c[1] + h[1] * cheb_node(iy, N));
  TableRun<T, FAR_RUN> zr;
  double acc[FAR_RUN], err[FAR_RUN];
  T part[FAR_RUN], none[FAR_RUN][3];
#pragma unroll
  for (int q = 0; q < FAR_RUN; ++q) {
    zr.z[q] = (T)(c[2] + h[2] * cheb_node(iz + q, N));
    acc[q] = err[q] = 0.0;
    part[q] = T(0);
  }
  const V4<T>* pts = reinterpret_cast<const V4<T>*>(f.e.pts);
  const V8<T>* ori = reinterpret_cast<const V8<T>*>(f.e.ori);
  const int32_t* lp = f.lp + (b + 1) * f.e.n_pts - 1;          // far sources from the back
  const int32_t* lo = f.lo + (b + 1) * f.e.n_ori - 1;
  const int64_t np = f.cnt[4 * b + 1], no = f.cnt[4 * b + 3];
  const int64_t pe = np * (split + 1) / f.nsplit, oe = no * (split + 1) / f.nsplit;
  for (int64_t base = np * split / f.nsplit; base < pe; base += FAR_TS) {
    V4<T> v{};
    if (base + lane < pe) v = pts[lp[-(base + lane)]];
    __syncthreads();
    tile4[lane] = v;
    __syncthreads();
    lattice_pts_tile<T, false, false, FAR_RUN, FOLD>(tile4, FAR_TS, x0, y0, zr, part, none);
#pragma unroll
    for (int q = 0; q < FAR_RUN; ++q) { add_exact(acc[q], err[q], (double)part[q]); part[q] = T(0); }
  }
  for (int64_t base = no * split / f.nsplit; base < oe; base += FAR_TS) {
    V8<T> v{};
    if (base + lane < oe) v = ori[lo[-(base + lane)]];
    __syncthreads();
    tile[lane] = v;
    __syncthreads();
    lattice_ori_tile<T, false, false, FAR_RUN, FOLD>(tile, FAR_TS, x0, y0, zr, part, none);
#pragma unroll
    for (int q = 0; q < FAR_RUN; ++q) { add_exact(acc[q], err[q], (double)part[q]); part[q] = T(0); }
  }
  double* o = f.nodes + ((int64_t)split * nb + b) * (N * N * N) + ((int64_t)ix * N + iy) * N + iz;
#pragma unroll
  for (int q = 0; q < FAR_RUN; ++q) o[q] = exact_sum(acc[q], err[q]);
}

// Node sums to the points, one axis after the other: a workgroup takes up to
// FAR_PLANES x planes of a block; per plane the x contraction from registers,
// then z, then y through LDS.  The value at one node goes around the
// contractions (their weights sum to 1), which leaves their rounding the size
// of the field's variation over the block.
constexpr int FAR_PLANES = 8, FAR_MAX_P = 96;
template <int N>
__global__ __launch_bounds__(256) void far_interp_kernel(FarArgs f) {
  __shared__ double base, A[N * N], B[N * FAR_MAX_P], wy[FAR_MAX_P * (N + 1)], wz[FAR_MAX_P * (N + 1)];
  const int t = threadIdx.x;
  const int64_t b = blockIdx.y, nb = (int64_t)f.b[0] * f.b[1] * f.b[2];
  const int64_t i0 = b / ((int64_t)f.b[1] * f.b[2]) * f.p[0], j0 = b / f.b[2] % f.b[1] * f.p[1],
                k0 = b % f.b[2] * f.p[2];
  const int px = (int)min((int64_t)f.p[0], f.e.nx - i0), py = (int)min((int64_t)f.p[1], f.e.ny - j0),
            pz = (int)min((int64_t)f.p[2], f.e.nz - k0);
  const int x_lo = blockIdx.x * FAR_PLANES, x_hi = min(px, x_lo + FAR_PLANES);
  if (x_lo >= x_hi) return;
  for (int i = t; i < py * N; i += 256) wy[i / N * (N + 1) + i % N] = f.tab[(int64_t)f.p[0] * N + i];
  for (int i = t; i < pz * N; i += 256) wz[i / N * (N + 1) + i % N] = f.tab[((int64_t)f.p[0] + f.p[1]) * N + i];
  double v[N] = {};
  if (t < N * N) {
#pragma unroll
    for (int m = 0; m < N; ++m) v[m] = 0.0;
    for (int s = 0; s < f.nsplit; ++s) {
      const double* src = f.nodes + ((int64_t)s * nb + b) * (N * N * N) + t;
#pragma unroll
      for (int m = 0; m < N; ++m) v[m] += src[m * N * N];
    }
    if (t == N * N / 2 + N / 2) base = v[N / 2];
  }
  __syncthreads();
  const double mid = base;
#pragma unroll
  for (int m = 0; m < N; ++m) v[m] -= mid;
  for (int x = x_lo; x < x_hi; ++x) {
    if (t < N * N) {
      double a = 0.0;
#pragma unroll
      for (int m = 0; m < N; ++m) a = fma(f.tab[(int64_t)x * N + m], v[m], a);
      A[t] = a;
    }
    __syncthreads();                     // A written; the weights too, the first time
    for (int i = t; i < N * pz; i += 256) {
      const int j = i / pz, z = i % pz;
      double a = 0.0;
#pragma unroll
      for (int m = 0; m < N; ++m) a = fma(wz[z * (N + 1) + m], A[j * N + m], a);
      B[j * pz + z] = a;
    }
    __syncthreads();
    for (int i = t; i < py * pz; i += 256) {
      const int y = i / pz, z = i % pz;
      double a = 0.0;
#pragma unroll
      for (int m = 0; m < N; ++m) a = fma(wy[y * (N + 1) + m], B[m * pz + z], a);
      f.e.scalar[((i0 + x) * f.e.ny + j0 + y) * f.e.nz + k0 + z] = mid + a;
    }
  }
}

// Near sources at a block's points, added to the interpolated far field; then
// drift, ids and stores as in eval_kernel.  A workgroup takes 64 runs and its
// four waves a quarter of the sources each, added in order at the end: with 64
// runs a wave to itself a grid of 1e6 points gave each SIMD two or three waves
// of very different length (near part of 1e6 points, FP32: 351 us, 209 with
// quarters; 1.2e6 points, range 0.45 of the box: 2.78 ms and 1.86).  Each wave stages its sources in LDS of its own, so no
// barrier joins them before the end.
constexpr int NEAR_WAVES = 4;
template <typename T, bool GRAD, bool MASKED, int PPT>
__global__ __launch_bounds__(64 * NEAR_WAVES) void near_kernel(FarArgs f) {
  constexpr int VALS = GRAD ? 4 * PPT : PPT;
  constexpr size_t TILES = sizeof(V8<T>) * 64 * NEAR_WAVES, SUMS = sizeof(double) * VALS * 64 * (NEAR_WAVES - 1);
  __shared__ __align__(64) char lds[TILES > SUMS ? TILES : SUMS];
  const EvalArgs& a = f.e;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  V8<T>* tile = reinterpret_cast<V8<T>*>(lds) + 64 * wave;
  V4<T>* tile4 = reinterpret_cast<V4<T>*>(tile);
  const int64_t b = f.order[blockIdx.y];
  // the layers of runs one after the other, so that in the last, shorter
  // blocks of an axis whole workgroups have no points
  const int run = blockIdx.x * 64 + lane, ry = run % f.p[1], rx = run / f.p[1] % f.p[0], rz = run / (f.p[1] * f.p[0]);
  const int64_t ix = b / ((int64_t)f.b[1] * f.b[2]) * f.p[0] + rx, iy = b / f.b[2] % f.b[1] * f.p[1] + ry,
                iz0 = b % f.b[2] * f.p[2] + (int64_t)rz * PPT;
  const bool ok = rz < f.p[2] / PPT && ix < a.nx && iy < a.ny && iz0 < a.nz;
  if (!__any(ok)) return;              // the same lanes in all waves of the workgroup
  const T x0 = (T)((a.ox + ix * a.hx - a.cx) * a.inv_a), y0 = (T)((a.oy + iy * a.hy - a.cy) * a.inv_a);
  const SpacedRun<T> zr{(T)((a.oz + iz0 * a.hz - a.cz) * a.inv_a), (T)(a.hz * a.inv_a)};
  double acc[PPT], err[PPT], gacc[PPT][3];
  T part[PPT], gpart[PPT][3];
#pragma unroll
  for (int q = 0; q < PPT; ++q) {
    acc[q] = err[q] = 0.0;
    part[q] = T(0);
    gacc[q][0] = gacc[q][1] = gacc[q][2] = 0.0;
    gpart[q][0] = gpart[q][1] = gpart[q][2] = T(0);
  }
  auto flush = [&]() {
#pragma unroll
    for (int q = 0; q < PPT; ++q) {
      add_exact(acc[q], err[q], (double)part[q]);
      part[q] = T(0);
      if (GRAD)
        for (int u = 0; u < 3; ++u) { gacc[q][u] += (double)gpart[q][u]; gpart[q][u] = T(0); }
    }
  };
  const V4<T>* pts = reinterpret_cast<const V4<T>*>(a.pts);
  const V8<T>* ori = reinterpret_cast<const V8<T>*>(a.ori);
  const int32_t *lp = f.lp + b * a.n_pts, *lo = f.lo + b * a.n_ori;
  const int64_t np = f.cnt[4 * b], no = f.cnt[4 * b + 2];
  const int pe = (int)(np * (wave + 1) / NEAR_WAVES), oe = (int)(no * (wave + 1) / NEAR_WAVES);
  for (int base = (int)(np * wave / NEAR_WAVES); base < pe; base += 64) {
    const int nk = min(64, pe - base);
    V4<T> v{};
    if (lane < nk) v = pts[lp[base + lane]];
    __builtin_amdgcn_wave_barrier();
    tile4[lane] = v;
    __builtin_amdgcn_wave_barrier();
    lattice_pts_tile<T, GRAD, MASKED, PPT>(tile4, nk, x0, y0, zr, part, gpart);
    flush();
  }
  for (int base = (int)(no * wave / NEAR_WAVES); base < oe; base += 64) {
    const int nk = min(64, oe - base);
    V8<T> v{};
    if (lane < nk) v = ori[lo[base + lane]];
    __builtin_amdgcn_wave_barrier();
    tile[lane] = v;
    __builtin_amdgcn_wave_barrier();
    lattice_ori_tile<T, GRAD, MASKED, PPT>(tile, nk, x0, y0, zr, part, gpart);
    flush();
  }
#pragma unroll
  for (int q = 0; q < PPT; ++q) acc[q] = exact_sum(acc[q], err[q]);
  __syncthreads();                     // the tiles give way to the sums
  double* sums = reinterpret_cast<double*>(lds);
  if (wave > 0) {
    double* o = sums + (wave - 1) * VALS * 64 + lane;
#pragma unroll
    for (int q = 0; q < PPT; ++q) {
      o[64 * q] = acc[q];
      if (GRAD)
        for (int u = 0; u < 3; ++u) o[64 * (PPT + 3 * q + u)] = gacc[q][u];
    }
  }
  __syncthreads();
  if (wave > 0 || !ok) return;
  for (int w = 0; w < NEAR_WAVES - 1; ++w) {
    const double* o = sums + w * VALS * 64 + lane;
#pragma unroll
    for (int q = 0; q < PPT; ++q) {
      acc[q] += o[64 * q];
      if (GRAD)
        for (int u = 0; u < 3; ++u) gacc[q][u] += o[64 * (PPT + 3 * q + u)];
    }
  }
#pragma unroll
  for (int q = 0; q < PPT; ++q) {
    if (iz0 + q >= a.nz) continue;
    const int64_t p = (ix * a.ny + iy) * a.nz + iz0 + q;
    double s = acc[q], g[3] = {gacc[q][0] * a.inv_a, gacc[q][1] * a.inv_a, gacc[q][2] * a.inv_a};
    if (f.n > 0) s += a.scalar[p];       // the interpolated far field
    drift_terms(a, a.ox + ix * a.hx, a.oy + iy * a.hy, a.oz + (iz0 + q) * a.hz, p, s, GRAD ? g : nullptr);
    a.scalar[p] = s;
    if (GRAD && a.grad) { a.grad[3 * p] = g[0]; a.grad[3 * p + 1] = g[1]; a.grad[3 * p + 2] = g[2]; }
    if (a.ids) a.ids[p] = segment_id(a, s);
  }
}

// Sum the per-split partials, add drift, segment, store.  A block takes
// FIN_PTS points with FIN_LANES threads each: lane l adds splits l, l + 16,
// ... (its loads independent, so a hundred splits cost a few memory
// latencies), then a tree over the lanes in LDS; the order of the additions
// depends only on nsplit.
constexpr int FIN_PTS = 16, FIN_LANES = 16;
__global__ __launch_bounds__(FIN_PTS * FIN_LANES) void eval_finalize_kernel(EvalArgs a, int grad) {
  __shared__ double red[4][FIN_LANES][FIN_PTS];
  const int pl = threadIdx.x % FIN_PTS, lane = threadIdx.x / FIN_PTS;
  const int64_t p = (int64_t)blockIdx.x * FIN_PTS + pl;
  double s = 0.0, g[3] = {0.0, 0.0, 0.0};
  if (p < a.n_points) {
    for (int y = lane; y < a.nsplit; y += FIN_LANES) {
      const int64_t o = (int64_t)y * a.n_points + p;
      s += a.part_s[o];
      if (grad) { g[0] += a.part_g[3 * o]; g[1] += a.part_g[3 * o + 1]; g[2] += a.part_g[3 * o + 2]; }
    }
  }
  red[0][lane][pl] = s;
  red[1][lane][pl] = g[0];
  red[2][lane][pl] = g[1];
  red[3][lane][pl] = g[2];
  __syncthreads();
  for (int w = FIN_LANES / 2; w > 0; w >>= 1) {
    if (lane < w)
      for (int c = 0; c < 4; ++c) red[c][lane][pl] += red[c][lane + w][pl];
    __syncthreads();
  }
  if (lane != 0 || p >= a.n_points) return;
  s = red[0][0][pl];
  g[0] = red[1][0][pl] * a.inv_a; g[1] = red[2][0][pl] * a.inv_a; g[2] = red[3][0][pl] * a.inv_a;
  const double* P = a.xyz + 3 * p;
  drift_terms(a, P[0], P[1], P[2], p, s, grad ? g : nullptr);
  a.scalar[p] = s;
  if (grad && a.grad) { a.grad[3 * p] = g[0]; a.grad[3 * p + 1] = g[1]; a.grad[3 * p + 2] = g[2]; }
  if (a.ids) a.ids[p] = segment_id(a, s);
}

// ---------------------------------------------------------------- source prep
// Interface sources: rest points with weight i_res c_o w_i, reference points
// with weight -i_res c_o W_s (W_s = sum of w_i over the surface): the
// rest-minus-reference differencing of the interface covariance collapses
// into per-surface reference sources.
// One launch prepares everything an evaluation reads, the workgroups taking
// roles one after the other: a surface each (its sum of weights and its
// reference source), 1,024 rest points, 1,024 orientations; for the operator
// product also the data points' positions and the partial sums of its drift
// and fault rows, which depend on x alone.  These were four to six launches
// one after the other, each of them shorter than the gap between two: a
// product of 1,800 data took 49 us and takes 40 now, of 25,000 data 447 and
// 430.
//
// Drift and fault rows: workgroup (l, c) adds chunk c of row l's terms (the
// orientations and rest points split into DRIFT_CHUNKS ranges) into
// part[l DRIFT_CHUNKS + c]; matvec_combine_kernel adds the chunks in order.
constexpr int DRIFT_CHUNKS = 16, PREP = 1024;

__device__ __forceinline__ double block_sum(double acc, double* red) {   // PREP threads; valid in thread 0
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  double t = 0.0;
  if (threadIdx.x == 0)
    for (int w = 0; w < PREP / 64; ++w) t += red[w];
  return t;
}

__device__ __forceinline__ double drift_row_chunk(const gk_system& sys, const double* x, int l, int c) {
  const int64_t no = sys.n_ori, R = sys.n_rest, NG = 3 * no;
  const int L = sys.uni_degree == 0 ? 0 : (sys.uni_degree == 1 ? 3 : 9);
  const int64_t g0 = no * c / DRIFT_CHUNKS, g1 = no * (c + 1) / DRIFT_CHUNKS;
  const int64_t r0 = R * c / DRIFT_CHUNKS, r1 = R * (c + 1) / DRIFT_CHUNKS;
  double acc = 0.0;
  if (l < L) {
    for (int64_t g = g0 + threadIdx.x; g < g1; g += PREP) {
      const double* q = sys.ori_xyz + 3 * g;
#pragma unroll
      for (int u = 0; u < 3; ++u) {
        double df;
        if (l < 3) df = (l == u) ? 1.0 : 0.0;
        else if (l < 6) df = (l - 3 == u) ? 2.0 * q[u] : 0.0;
        else if (l == 6) df = (u == 0) ? q[1] : (u == 1 ? q[0] : 0.0);
        else if (l == 7) df = (u == 0) ? q[2] : (u == 2 ? q[0] : 0.0);
        else df = (u == 1) ? q[2] : (u == 2 ? q[1] : 0.0);
        acc += df * x[u * no + g];
      }
    }
    for (int64_t r = r0 + threadIdx.x; r < r1; r += PREP) {
      const double* p = sys.rest_xyz + 3 * r;
      const double* p0 = sys.ref_xyz + 3 * sys.rest_surf[r];
      double f1, f0;
      if (l < 3) { f1 = p[l]; f0 = p0[l]; }
      else if (l < 6) { f1 = p[l - 3] * p[l - 3]; f0 = p0[l - 3] * p0[l - 3]; }
      else if (l == 6) { f1 = p[0] * p[1]; f0 = p0[0] * p0[1]; }
      else if (l == 7) { f1 = p[0] * p[2]; f0 = p0[0] * p0[2]; }
      else { f1 = p[1] * p[2]; f0 = p0[1] * p0[2]; }
      acc += sys.gi_res * (f1 - f0) * x[NG + r];
    }
  } else {
    for (int64_t r = r0 + threadIdx.x; r < r1; r += PREP)
      acc += sys.gi_res * sys.fault_rest[r * sys.n_fault + (l - L)] * x[NG + r];
  }
  return acc;
}

// xyz, drift (nullable): the operator product's.  drift_rows of them.
// out (nullable): per workgroup of sources, whether one of them lies outside
// the sphere of half the range around the centre (or is no number).
template <typename T>
__global__ __launch_bounds__(PREP) void prep_kernel(gk_system sys, const double* w, V4<T>* pts, V8<T>* ori, double* xyz,
                                                    double* drift, int drift_rows, int32_t* out) {
  __shared__ double red[PREP / 64];
  const int64_t R = sys.n_rest, S = sys.n_surf, no = sys.n_ori;
  const double inv_a = 1.0 / sys.range;
  bool beyond = false;
  auto put = [&](int64_t i, const double* p, double wt) {
    V4<T> v;
    v.x = (T)((p[0] - sys.center[0]) * inv_a);
    v.y = (T)((p[1] - sys.center[1]) * inv_a);
    v.z = (T)((p[2] - sys.center[2]) * inv_a);
    v.w = (T)wt;
    pts[i] = v;
    beyond = !((double)v.x * v.x + (double)v.y * v.y + (double)v.z * v.z <= half_range2<T>());
    if (xyz) { xyz[3 * i] = p[0]; xyz[3 * i + 1] = p[1]; xyz[3 * i + 2] = p[2]; }
  };
  int64_t b = blockIdx.x;
  if (b < S) {                           // a surface
    double acc = 0.0;
#pragma unroll 4
    for (int64_t i = threadIdx.x; i < R; i += PREP) {
      const double wi = w[3 * no + i];
      acc += sys.rest_surf[i] == b ? wi : 0.0;
    }
    const double W = block_sum(acc, red);
    if (threadIdx.x == 0) {
      put(R + b, sys.ref_xyz + 3 * b, -sys.i_res * sys.c_o * W);
      if (out) out[blockIdx.x] = beyond;
    }
    return;
  }
  b -= S;
  const int64_t nr = (R + PREP - 1) / PREP, nq = (no + PREP - 1) / PREP;
  if (b < nr) {
    const int64_t i = b * PREP + threadIdx.x;
    if (i < R) put(i, sys.rest_xyz + 3 * i, sys.i_res * sys.c_o * w[3 * no + i]);
    const bool any = __syncthreads_or(beyond);
    if (out && threadIdx.x == 0) out[blockIdx.x] = any;
    return;
  }
  b -= nr;
  if (b < nq) {
    const int64_t g = b * PREP + threadIdx.x;
    if (g < no) {
      const double f = sys.gi_res * sys.c_o * inv_a;
      const double* q = sys.ori_xyz + 3 * g;
      V8<T> v;
      v.x = (T)((q[0] - sys.center[0]) * inv_a);
      v.y = (T)((q[1] - sys.center[1]) * inv_a);
      v.z = (T)((q[2] - sys.center[2]) * inv_a);
      v.pad0 = T(0);
      v.wx = (T)(f * w[g]);
      v.wy = (T)(f * w[no + g]);
      v.wz = (T)(f * w[2 * no + g]);
      v.pad1 = T(0);
      ori[g] = v;
      beyond = !((double)v.x * v.x + (double)v.y * v.y + (double)v.z * v.z <= half_range2<T>());
    }
    const bool any = __syncthreads_or(beyond);
    if (out && threadIdx.x == 0) out[blockIdx.x] = any;
    return;
  }
  b -= nq;
  if (b < (int64_t)drift_rows * DRIFT_CHUNKS) {
    const double t = block_sum(drift_row_chunk(sys, w, (int)(b / DRIFT_CHUNKS), (int)(b % DRIFT_CHUNKS)), red);
    if (threadIdx.x == 0) drift[b] = t;
  }
}

int n_drift_of(int deg) { return deg == 0 ? 0 : (deg == 1 ? 3 : 9); }

// Points per thread: a lattice z-run of 8 (FP64 with gradient or mask: 4);
// explicit points 4 (FP64 with gradient: 2, for its 24 accumulator registers).
constexpr int eval_ppt(bool lattice, bool f32, bool grad, bool masked) {
  return lattice ? ((f32 || (!grad && !masked)) ? 8 : 4) : ((f32 || !grad) ? 4 : 2);
}

template <typename T, bool LATTICE, bool GRAD, bool MASKED, bool SCALAR = true>
void launch_eval(const EvalArgs& a, int ppt_runs_div, hipStream_t st) {
  (void)ppt_runs_div;
  constexpr int PPT = eval_ppt(LATTICE, sizeof(T) == 4, GRAD, MASKED);
  EvalArgs b = a;
  if (LATTICE) {
    b.nzr = gk_ceil_div(a.nz, PPT);
    b.n_runs = a.nx * a.ny * b.nzr;
  } else {
    b.n_runs = gk_ceil_div(a.n_points, PPT);
  }
  const int64_t blocks = gk_ceil_div(b.n_runs, TS);
  if (blocks == 0) return;
  hipLaunchKernelGGL((eval_kernel<T, LATTICE, GRAD, MASKED, PPT, SCALAR>), dim3((unsigned)blocks, (unsigned)b.nsplit),
                     dim3(TS), 0, st, b);
  if (b.nsplit > 1)
    hipLaunchKernelGGL(eval_finalize_kernel, dim3((unsigned)gk_ceil_div(b.n_points, FIN_PTS)),
                       dim3(FIN_PTS * FIN_LANES), 0, st,
                       b, GRAD ? 1 : 0);
}

template <typename T>
void dispatch_eval(const EvalArgs& a, bool lattice, bool grad, bool masked, hipStream_t st, bool scalar = true) {
  if (lattice) {
    if (grad) { if (masked) launch_eval<T, true, true, true>(a, 0, st); else launch_eval<T, true, true, false>(a, 0, st); }
    else { if (masked) launch_eval<T, true, false, true>(a, 0, st); else launch_eval<T, true, false, false>(a, 0, st); }
  } else {
    if (grad && !scalar) {
      if (masked) launch_eval<T, false, true, true, false>(a, 0, st); else launch_eval<T, false, true, false, false>(a, 0, st);
    } else if (grad) { if (masked) launch_eval<T, false, true, true>(a, 0, st); else launch_eval<T, false, true, false>(a, 0, st); }
    else { if (masked) launch_eval<T, false, false, true>(a, 0, st); else launch_eval<T, false, false, false>(a, 0, st); }
  }
}

}  // namespace

// Workgroups of prep_kernel that hold sources.
static int64_t source_groups(const gk_system* sys) {
  return sys->n_surf + gk_ceil_div(sys->n_rest, PREP) + gk_ceil_div(sys->n_ori, PREP);
}

static size_t sources_bytes(const gk_system* sys) {
  const int64_t R = sys->n_rest, S = sys->n_surf, no = sys->n_ori;
  return gk_round_up((R + S) * 32, 256) + gk_round_up(no * 64, 256) + 256;
}

// The handle's workspace of packed sources, with the groups' flags behind them.
static int source_workspace(gk_handle h, const gk_system* sys, void** ws, int32_t** out) {
  const size_t at = gk_round_up(sources_bytes(sys), 256);
  GK_TRY(gk_workspace(h, WS_EVAL_SRC, at + source_groups(sys) * sizeof(int32_t) + 256, ws));
  *out = reinterpret_cast<int32_t*>(static_cast<char*>(*ws) + at);
  return GK_OK;
}

// Where the packed sources lie in a workspace: [pts V4<T> (R+S) | ori V8<T> (n_ori)].
static void source_layout(const gk_system* sys, int precision, void* ws, void** pts, void** ori) {
  const size_t tsz = precision == GK_F64 ? 8 : 4;
  *pts = ws;
  *ori = static_cast<char*>(ws) + gk_round_up((sys->n_rest + sys->n_surf) * 4 * tsz, 256);
}

// Prepare the packed sources for `weights` in the workspace ws; xyz, drift,
// drift_rows: see prep_kernel.
static int prepare_sources(const gk_system* sys, const double* weights, int precision, hipStream_t st, void* ws,
                           int32_t* out, double* xyz = nullptr, double* drift = nullptr, int drift_rows = 0) {
  const int64_t nb = source_groups(sys) + (int64_t)drift_rows * DRIFT_CHUNKS;
  void *p4, *p8;
  source_layout(sys, precision, ws, &p4, &p8);
  if (nb == 0) return GK_OK;
  if (precision == GK_F64)
    hipLaunchKernelGGL(prep_kernel<double>, dim3((unsigned)nb), dim3(PREP), 0, st, *sys, weights,
                       static_cast<V4<double>*>(p4), static_cast<V8<double>*>(p8), xyz, drift, drift_rows, out);
  else
    hipLaunchKernelGGL(prep_kernel<float>, dim3((unsigned)nb), dim3(PREP), 0, st, *sys, weights,
                       static_cast<V4<float>*>(p4), static_cast<V8<float>*>(p8), xyz, drift, drift_rows, out);
  GK_HIP(hipGetLastError());
  return GK_OK;
}

static int check_system(const gk_system* sys) {
  GK_REQUIRE(sys != nullptr, GK_ERR_ARG, "gk: system is NULL");
  GK_REQUIRE(sys->n_ori >= 0 && sys->n_rest >= 0 && sys->n_surf >= 0, GK_ERR_ARG,
             "gk: negative sizes in system");
  GK_REQUIRE(sys->uni_degree >= 0 && sys->uni_degree <= 2, GK_ERR_ARG,
             "gk: uni_degree must be 0, 1 or 2 (got %d)", sys->uni_degree);
  GK_REQUIRE(sys->n_fault >= 0 && sys->n_fault <= 8, GK_ERR_ARG, "gk: n_fault must be 0..8");
  GK_REQUIRE(sys->range > 0 && sys->c_o > 0, GK_ERR_ARG, "gk: range and c_o must be positive");
  GK_REQUIRE(sys->n_ori == 0 || (sys->ori_xyz && sys->ori_grad && sys->ori_nugget), GK_ERR_ARG,
             "gk: orientation arrays missing");
  GK_REQUIRE(sys->n_rest == 0 || (sys->rest_xyz && sys->rest_surf && sys->rest_nugget), GK_ERR_ARG,
             "gk: rest-point arrays missing");
  GK_REQUIRE(sys->n_surf == 0 || sys->ref_xyz, GK_ERR_ARG, "gk: reference points missing");
  GK_REQUIRE(sys->n_fault == 0 || sys->fault_rest, GK_ERR_ARG, "gk: fault_rest missing");
  return GK_OK;
}

// Largest distance between the sources and a box, in range units: when it is
// below 1 the cubic covariance needs no r < a mask (its polynomial is exact).
static bool needs_mask(const gk_system* sys, const double* lo, const double* hi, double src_lo[3],
                       double src_hi[3]) {
  double d2 = 0.0;
  for (int k = 0; k < 3; ++k) {
    double a = std::max(std::fabs(hi[k] - src_lo[k]), std::fabs(src_hi[k] - lo[k]));
    d2 += a * a;
  }
  return d2 >= (1.0 - 1e-9) * sys->range * sys->range;
}

// Split the sources over blockIdx.y when the points alone cannot fill the GPU,
// then launch the evaluation kernel for the requested variant.
static int run_eval(gk_handle h, EvalArgs& a, bool lattice, int precision, bool grad, bool masked,
                    hipStream_t st, bool external = false, char* part = nullptr, size_t part_bytes = 0,
                    bool grad_only = false) {
  const int64_t cost = a.n_pts * src_cost(grad, false) + a.n_ori * src_cost(grad, true);
  a.nsplit = 1;
  a.cost_chunk = std::max<int64_t>(cost, 1);
  if (!lattice) {
    const int ppt = eval_ppt(false, precision != GK_F64, grad, masked);
    const int64_t blocks = gk_ceil_div(gk_ceil_div(a.n_points, ppt), TS);
    // at most SPLIT_WGS workgroups in all (rounded down: a few more would
    // run as a nearly empty last round), each split at least 64 interface
    // sources' worth of work
    int64_t want = std::min<int64_t>(std::min<int64_t>(SPLIT_WGS / blocks, grad ? MAX_SPLIT : MAX_SPLIT_SCALAR),
                                     gk_ceil_div(cost, 64 * src_cost(grad, false)));
    if (external) {          // as many splits as the caller's scratch holds partials for
      const size_t per_split = (size_t)a.n_points * (grad ? 4 : 1) * sizeof(double);
      want = std::min<int64_t>(want, per_split > 0 ? (int64_t)((part_bytes > 512 ? part_bytes - 512 : 0) / per_split)
                                                   : 1);
    }
    if (want > 1) {
      a.cost_chunk = gk_ceil_div(cost, want);
      a.nsplit = (int32_t)gk_ceil_div(cost, a.cost_chunk);
      if (a.nsplit > 1) {
        void* pw = part;
        const size_t per = (size_t)a.n_points * (grad ? 4 : 1);
        if (!external) GK_TRY(gk_workspace(h, WS_EVAL_PART, per * a.nsplit * sizeof(double) + 512, &pw));
        a.part_s = static_cast<double*>(pw);
        a.part_g = grad ? a.part_s + (size_t)a.nsplit * a.n_points : nullptr;
      } else {
        a.cost_chunk = std::max<int64_t>(cost, 1);
      }
    }
  }
  if (precision == GK_F64) dispatch_eval<double>(a, lattice, grad, masked, st, !grad_only);
  else dispatch_eval<float>(a, lattice, grad, masked, st, !grad_only);
  GK_HIP(hipGetLastError());
  return GK_OK;
}

// Blocks of a lattice evaluation (see FarArgs), or false where the direct sum
// is expected to be as fast.  The estimate counts pairs at the rate of the
// direct kernel (f64 4.3e-13 s each, f32 3.1e-13, 1.4 times that with the
// mask) over the groups of 192 (block, source) pairs spread evenly (an R
// sequence) over the blocks and the source box.  Nodes are used without
// gradient: derivatives of the interpolant are 4,000 times less exact (8e-12 of
// an orientation's gradient with 16 nodes per axis, 4e-13 with 18, 6e-15 with
// 20), and a form with 20 nodes, for blocks of well more than 8,000 points, is
// not built.
//   8e6 points, 25,000 sources, f64: 86.9 ms direct, 22.5 in blocks (12.4 near, 10.0 nodes)
//   1e6 points, 6,000 sources, f32: 1.88 ms and 0.61
//   2.1e6 points, 1,920 sources, f64: 1.98 ms and 1.10
//   1.2e6 points, 6,000 sources, range 0.45 of the box: 4.28 ms and 1.76
// Below 0.2 ms of pairs the launches and their lists cost what they save.
static bool plan_blocks(FarArgs& f, int precision, bool grad, bool masked, const double* slo, const double* shi) {
  const EvalArgs& a = f.e;
  if ((grad && !masked) || a.n_pts + a.n_ori >= (int64_t)1 << 30) return false;
  const int64_t dim[3] = {a.nx, a.ny, a.nz}, nsrc = a.n_pts + a.n_ori;
  const double org[3] = {a.ox - a.cx, a.oy - a.cy, a.oz - a.cz}, sp[3] = {a.hx, a.hy, a.hz};
  const double ctr[3] = {a.cx, a.cy, a.cz};
  const bool f64 = precision == GK_F64;
  const double pair = (f64 ? 4.3e-13 : 3.1e-13) * (grad ? 2.0 : 1.0) * (masked ? 1.4 : 1.0);
  const double points = (double)a.nx * a.ny * gk_round_up(a.nz, 8), direct = pair * nsrc * points;
  if (!(direct > 2e-4)) return false;
  double ext[3], longest = 0.0;
  for (int k = 0; k < 3; ++k) {
    ext[k] = std::fabs(sp[k]) * dim[k] * a.inv_a;
    if (!(ext[k] > 0.0) || !std::isfinite(ext[k]) || !std::isfinite(org[k]) || !(shi[k] >= slo[k])) return false;
    longest = std::max(longest, ext[k]);
  }
  double best = 0.8 * direct;
  bool found = false;
  for (int use = grad ? 0 : 1; use >= (masked ? 0 : 1); --use) {
    const int64_t n = use ? (f64 ? 16 : 8) : 0, n3 = n * n * n;
    int32_t last[3] = {0, 0, 0};
    for (int cand = 0; cand < 24; ++cand) {
      constexpr int CUTS[12] = {2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16, 20};    // blocks along the longest side
      const int cut = CUTS[cand / 2];
      FarArgs c = f;
      int64_t nb = 1, pts = 1;
      double hmax = 0.0;
      float h[3];
      bool fits = true;
      for (int k = 0; k < 3; ++k) {
        const int64_t want = std::max<int64_t>(1, (int64_t)std::llround(cut * ext[k] / longest));
        int64_t p = gk_ceil_div(dim[k], want);
        if (k == 2) p = (cand & 1) ? std::max<int64_t>(8, p / 8 * 8) : gk_round_up(p, 8);     // whole runs
        fits = fits && p <= FAR_MAX_P && p >= 2;
        c.p[k] = (int32_t)p;
        c.b[k] = (int32_t)gk_ceil_div(dim[k], p);
        nb *= c.b[k];
        pts *= p;
        h[k] = (float)(0.5 * (p - 1) * std::fabs(sp[k]) * a.inv_a);
        hmax = std::max(hmax, (double)h[k]);
      }
      if (!fits || nb > 8192 || (c.p[0] == last[0] && c.p[1] == last[1] && c.p[2] == last[2])) continue;
      for (int k = 0; k < 3; ++k) last[k] = c.p[k];
      const double gap = n == 16 ? 3.0 + 0.8 * std::max(0.0, std::log(hmax / 0.036))
                                 : 2.5 + 0.9 * std::max(0.0, std::log(hmax / 0.036));
      c.n = (int32_t)n;
      c.masked = masked ? 1 : 0;
      c.amin = (float)std::sqrt(1.0 + gap * gap);
      c.nsplit = n ? (int32_t)std::min<int64_t>(std::max<int64_t>(8192 / (nb * n3 / (FAR_TS * FAR_RUN)), 1), 16) : 0;
      if (nb * nsrc * 4 + c.nsplit * nb * n3 * 8 > (int64_t)1 << 28) continue;      // workspace kept by the handle
      const double fixed = 8e-5 + 2e-12 * nb * nsrc + (n ? 5e-12 * nb * pts : 0.0);
      const double slots = points * gk_round_up(pts / 8, 64) * 8 / pts, node = (double)nb * n3 / (masked ? 1.4 : 1.0);
      if (fixed + pair * nsrc * std::min(slots, node) * (masked ? 0.0 : 1.0) >= best) continue;
      int near = 0, farc = 0;
      constexpr int SAMPLES = 192;
      for (int i = 1; i <= SAMPLES; ++i) {
        constexpr double R[6] = {0.8986537126286993, 0.8075784952213448, 0.7257334129697598,
                                 0.6521830259439717, 0.5860866974851957, 0.5266889867007451};
        float d[3];
        for (int k = 0; k < 3; ++k) {
          const double u = i * R[k] - std::floor(i * R[k]), v = i * R[k + 3] - std::floor(i * R[k + 3]);
          const double mid = org[k] + (std::floor(u * c.b[k]) * c.p[k] + 0.5 * (c.p[k] - 1)) * sp[k];
          d[k] = (float)(std::fabs(slo[k] + v * (shi[k] - slo[k]) - ctr[k] - mid) * a.inv_a);
        }
        const int g = far_group(d, h, masked, n > 0, c.amin);
        near += g == FAR_NEAR;
        farc += g == FAR_FAR;
      }
      const double t = fixed + pair * nsrc / SAMPLES * (near * slots + farc * node);
      if (t < best) {
        best = t;
        f = c;
        found = true;
      }
    }
  }
  return found;
}

template <typename T, int N>
static void launch_nodes(const FarArgs& f, int64_t nb, hipStream_t st) {
  const dim3 grid((unsigned)(nb * (N * N * N / (FAR_TS * FAR_RUN))), f.nsplit);
  if (f.masked) hipLaunchKernelGGL((far_nodes_kernel<T, N, false>), grid, dim3(FAR_TS), 0, st, f);
  else hipLaunchKernelGGL((far_nodes_kernel<T, N, true>), grid, dim3(FAR_TS), 0, st, f);
  hipLaunchKernelGGL(far_interp_kernel<N>, dim3((unsigned)gk_ceil_div(f.p[0], FAR_PLANES), (unsigned)nb), dim3(256), 0,
                     st, f);
}

template <typename T, bool GRAD, bool MASKED>
static void launch_near(const FarArgs& f, int64_t nb, hipStream_t st) {
  constexpr int PPT = sizeof(T) == 8 && GRAD ? 4 : 8;
  const int64_t runs = (int64_t)f.p[0] * f.p[1] * (f.p[2] / PPT);
  hipLaunchKernelGGL((near_kernel<T, GRAD, MASKED, PPT>), dim3((unsigned)gk_ceil_div(runs, 64), (unsigned)nb),
                     dim3(64 * NEAR_WAVES), 0, st, f);
}

// False, and nothing launched, where the workspace cannot be had: the direct
// sum needs none.
template <typename T>
static bool run_blocks(gk_handle h, FarArgs& f, bool grad, bool masked, hipStream_t st) {
  const int64_t nb = (int64_t)f.b[0] * f.b[1] * f.b[2], n3 = (int64_t)f.n * f.n * f.n;
  size_t need = 0;
  auto take = [&](size_t bytes) { const size_t o = need; need += gk_round_up(bytes, 256); return o; };
  const size_t o_n = take(f.nsplit * nb * n3 * 8), o_t = take((int64_t)(f.p[0] + f.p[1] + f.p[2]) * f.n * 8),
               o_c = take(nb * 16), o_r = take(nb * 4), o_p = take(nb * f.e.n_pts * 4), o_o = take(nb * f.e.n_ori * 4);
  void* ws = nullptr;
  if (gk_workspace(h, WS_EVAL_PART, need, &ws) != GK_OK) {
    (void)hipGetLastError();
    return false;
  }
  char* base = static_cast<char*>(ws);
  f.nodes = reinterpret_cast<double*>(base + o_n);
  f.tab = reinterpret_cast<double*>(base + o_t);
  f.cnt = reinterpret_cast<int32_t*>(base + o_c);
  f.order = reinterpret_cast<int32_t*>(base + o_r);
  f.lp = reinterpret_cast<int32_t*>(base + o_p);
  f.lo = reinterpret_cast<int32_t*>(base + o_o);
  hipLaunchKernelGGL(far_sort_kernel<T>, dim3((unsigned)(nb + (f.n > 0 ? 1 : 0))), dim3(1024), 0, st, f);
  hipLaunchKernelGGL(far_order_kernel, dim3((unsigned)gk_ceil_div(nb, 4)), dim3(256), 0, st, f, (int32_t)nb);
  if (f.n == 16) launch_nodes<T, 16>(f, nb, st);
  else if (f.n == 8) launch_nodes<T, 8>(f, nb, st);
  if (grad) launch_near<T, true, true>(f, nb, st);
  else if (masked) launch_near<T, false, true>(f, nb, st);
  else launch_near<T, false, false>(f, nb, st);
  return true;
}

// ext (nullable): caller-provided scratch for the packed sources and the
// split partials instead of the handle's workspaces (the no-allocation entry
// point); the split is then limited to what fits in it.
// grad_only (explicit points with gradient): the covariance part of the
// scalar is skipped; the scalar output then holds the drift terms alone.
static int eval_impl(gk_handle h, const gk_system* sys, const double* weights, gk_eval_desc* d, hipStream_t st,
                     bool force_mask, const double* src_box, bool reuse_sources, char* ext, size_t ext_bytes,
                     bool grad_only = false);

extern "C" int gk_eval_impl(gk_handle h, const gk_system* sys, const double* weights,
                            gk_eval_desc* d, hipStream_t st, bool force_mask,
                            const double* src_box /*6 or null*/, bool reuse_sources) {
  return eval_impl(h, sys, weights, d, st, force_mask, src_box, reuse_sources, nullptr, 0);
}

static int eval_impl(gk_handle h, const gk_system* sys, const double* weights, gk_eval_desc* d, hipStream_t st,
                     bool force_mask, const double* src_box, bool reuse_sources, char* ext, size_t ext_bytes,
                     bool grad_only) {
  GK_TRY(check_system(sys));
  GK_REQUIRE(!grad_only || (d && d->gradient && d->kind == GK_POINTS_EXPLICIT), GK_ERR_ARG,
             "gk_eval: a gradient-only evaluation needs explicit points and a gradient output");
  GK_REQUIRE(d && weights && d->scalar, GK_ERR_ARG, "gk_eval: desc, weights and scalar required");
  GK_REQUIRE(d->precision == GK_F32 || d->precision == GK_F64, GK_ERR_ARG, "gk_eval: bad precision");
  GK_REQUIRE(d->n_thresholds >= 0 && d->n_thresholds <= GK_MAX_THRESHOLDS, GK_ERR_ARG,
             "gk_eval: n_thresholds must be 0..%d", GK_MAX_THRESHOLDS);
  GK_REQUIRE(!d->ids || d->n_thresholds > 0, GK_ERR_ARG, "gk_eval: ids need thresholds");
  GK_REQUIRE(sys->n_fault == 0 || d->fault_values, GK_ERR_ARG,
             "gk_eval: fault_values required when the system has fault columns");
  EvalArgs a{};
  double lo[3], hi[3];
  if (d->kind == GK_POINTS_LATTICE) {
    GK_REQUIRE(d->res[0] > 0 && d->res[1] > 0 && d->res[2] > 0, GK_ERR_ARG, "gk_eval: bad lattice");
    a.nx = d->res[0]; a.ny = d->res[1]; a.nz = d->res[2];
    a.ox = d->origin[0]; a.oy = d->origin[1]; a.oz = d->origin[2];
    a.hx = d->spacing[0]; a.hy = d->spacing[1]; a.hz = d->spacing[2];
    d->n_points = a.nx * a.ny * a.nz;
    for (int k = 0; k < 3; ++k) {
      lo[k] = d->origin[k];
      hi[k] = d->origin[k] + (d->res[k] - 1) * d->spacing[k];
    }
  } else {
    GK_REQUIRE(d->kind == GK_POINTS_EXPLICIT, GK_ERR_ARG, "gk_eval: bad kind");
    GK_REQUIRE(d->n_points >= 0 && (d->n_points == 0 || d->xyz), GK_ERR_ARG, "gk_eval: points missing");
    for (int k = 0; k < 3; ++k) { lo[k] = -1e300; hi[k] = 1e300; }
  }
  a.n_points = d->n_points;
  if (a.n_points == 0) return GK_OK;
  a.xyz = d->xyz;
  a.cx = sys->center[0]; a.cy = sys->center[1]; a.cz = sys->center[2];
  a.inv_a = 1.0 / sys->range;
  a.n_pts = sys->n_rest + sys->n_surf;
  a.n_ori = sys->n_ori;
  a.uni_degree = sys->uni_degree;
  a.n_fault = sys->n_fault;
  a.lam = weights + 3 * sys->n_ori + sys->n_rest;
  a.gi_res = sys->gi_res;
  a.fault_values = d->fault_values;
  a.scalar = d->scalar;
  a.grad = d->gradient;
  a.ids = d->ids;
  a.n_thr = d->n_thresholds;
  a.thr_rev = (d->n_thresholds >= 2 && d->thresholds[0] < d->thresholds[d->n_thresholds - 1]) ? 1 : 0;
  for (int k = 0; k < d->n_thresholds; ++k) a.thr[k] = d->thresholds[k];

  void* ws = nullptr;
  int32_t* out = nullptr;
  char* part = nullptr;
  size_t part_bytes = 0;
  if (ext) {
    // 8 bytes a surface more than the sources take: the limit that gk.h states
    const size_t need = sources_bytes(sys) + gk_round_up(sys->n_surf * 8, 256);
    GK_REQUIRE(need <= ext_bytes, GK_ERR_ARG,
               "gk_eval_noalloc: the system's packed sources need %zu bytes, the scratch array holds %zu "
               "(GK_EVAL_SCRATCH_BYTES)", need, ext_bytes);
    ws = ext;
    part = ext + need;
    part_bytes = ext_bytes - need;
  } else {
    GK_TRY(source_workspace(h, sys, &ws, &out));
  }
  a.src_out = out;
  a.n_out = (int32_t)source_groups(sys);
  void *pts = nullptr, *ori = nullptr;
  source_layout(sys, d->precision, ws, &pts, &ori);
  a.pts = pts;
  a.ori = ori;
  if (!reuse_sources) GK_TRY(prepare_sources(sys, weights, d->precision, st, ws, out));
  bool masked = true;
  if (!force_mask && src_box) {
    // explicit points: only callers whose points lie inside the source box
    // (the data points themselves) pass a box for them
    double sl[3] = {src_box[0], src_box[1], src_box[2]}, sh[3] = {src_box[3], src_box[4], src_box[5]};
    if (d->kind == GK_POINTS_EXPLICIT)
      for (int k = 0; k < 3; ++k) { lo[k] = sl[k]; hi[k] = sh[k]; }
    masked = needs_mask(sys, lo, hi, sl, sh);
    if (d->kind == GK_POINTS_LATTICE && !ext) {
      FarArgs f{};
      f.e = a;
      const bool grad = d->gradient != nullptr;
      if (plan_blocks(f, d->precision, grad, masked, sl, sh) &&
          (d->precision == GK_F64 ? run_blocks<double>(h, f, grad, masked, st)
                                  : run_blocks<float>(h, f, grad, masked, st))) {
        GK_HIP(hipGetLastError());
        return GK_OK;
      }
    }
  }
  GK_TRY(run_eval(h, a, d->kind == GK_POINTS_LATTICE, d->precision, d->gradient != nullptr, masked, st, ext != nullptr,
                  part, part_bytes, grad_only));
  GK_HIP(hipGetLastError());
  return GK_OK;
}

// ------------------------------------------------------------------ matvec
namespace {
// y rows from the evaluated field at the data points (the fault drift enters
// the interface rows here); the last workgroup adds the chunks of the drift
// and fault rows.
__global__ void matvec_combine_kernel(gk_system sys, const double* x, const double* s_data, const double* g_ori,
                                      const double* drift, int drift_rows, double* y) {
  const int64_t no = sys.n_ori, R = sys.n_rest, NG = 3 * no;
  if (drift_rows > 0 && blockIdx.x + 1 == gridDim.x) {
    const int l = threadIdx.x;
    if (l >= drift_rows) return;
    double t = 0.0;
    for (int c = 0; c < DRIFT_CHUNKS; ++c) t += drift[l * DRIFT_CHUNKS + c];
    y[NG + R + l] = t;
    return;
  }
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < NG) {
    const int64_t u = i / no, g = i % no;
    y[i] = g_ori[3 * g + u] / sys.gi_res + sys.ori_nugget[g] * x[i];
  } else if (i < NG + R) {
    const int64_t r = i - NG;
    double v = s_data[r] - s_data[R + sys.rest_surf[r]] + sys.rest_nugget[r] * x[i];
    if (sys.n_fault > 0) {
      const int L = sys.uni_degree == 0 ? 0 : (sys.uni_degree == 1 ? 3 : 9);
      double t = 0.0;
      for (int f = 0; f < sys.n_fault; ++f)
        t += sys.gi_res * sys.fault_rest[r * sys.n_fault + f] * x[NG + R + L + f];
      v += t;
    }
    y[i] = v;
  }
}
}  // namespace

extern "C" int gk_matvec_impl(gk_handle h, const gk_system* sys, int32_t precision, const double* x,
                              double* y, hipStream_t st, void* scratch, const double* src_box) {
  // scratch: >= (R+S)*3 + (R+S) + n_ori*4 + 17 DRIFT_CHUNKS doubles
  const int64_t R = sys->n_rest, S = sys->n_surf, no = sys->n_ori;
  double* pts = static_cast<double*>(scratch);
  double* s_data = pts + 3 * (R + S);
  double* s_ori = s_data + (R + S);
  double* g_ori = s_ori + no;
  double* d_part = g_ori + 3 * no;          // drift / fault row chunks
  GK_TRY(check_system(sys));
  const int drift_rows = n_drift_of(sys->uni_degree) + sys->n_fault;
  void* ws = nullptr;
  int32_t* out = nullptr;
  GK_TRY(source_workspace(h, sys, &ws, &out));
  GK_TRY(prepare_sources(sys, x, precision, st, ws, out, pts, d_part, drift_rows));
  gk_system nofault = *sys;
  nofault.n_fault = 0;  // fault drift enters the interface rows separately
  if (R + S > 0) {
    gk_eval_desc d{};
    d.kind = GK_POINTS_EXPLICIT;
    d.precision = precision;
    d.n_points = R + S;
    d.xyz = pts;
    d.scalar = s_data;
    GK_TRY(gk_eval_impl(h, &nofault, x, &d, st, src_box == nullptr, src_box, true));
  }
  if (no > 0) {
    gk_eval_desc d{};
    d.kind = GK_POINTS_EXPLICIT;
    d.precision = precision;
    d.n_points = no;
    d.xyz = sys->ori_xyz;
    d.scalar = s_ori;             // drift terms only: the rows take the gradient
    d.gradient = g_ori;
    GK_TRY(eval_impl(h, &nofault, x, &d, st, src_box == nullptr, src_box, true, nullptr, 0, true));
  }
  const int64_t nb = gk_ceil_div(3 * no + R, 256) + (drift_rows > 0 ? 1 : 0);
  if (nb > 0)
    hipLaunchKernelGGL(matvec_combine_kernel, dim3((unsigned)nb), dim3(256), 0, st, *sys, x, s_data, g_ori, d_part,
                       drift_rows, y);
  GK_HIP(hipGetLastError());
  return GK_OK;
}

extern "C" size_t gk_matvec_scratch_doubles(const gk_system* sys) {
  return (size_t)(4 * (sys->n_rest + sys->n_surf) + 4 * sys->n_ori + 17 * DRIFT_CHUNKS + 64);
}

// ------------------------------------------------------------ stack combination
namespace {
// lith = global element id (offset per stack) of the stack that holds the
// point, basement otherwise.  ids: [n_stacks][n] int32, youngest stack
// first.  Stack s holds p when p is above its last surface
// (id <= nsurf[s]) and no younger stack holds it; an onlapping stack (rel ==
// GK_REL_ONLAP) additionally needs p above the first surface of the next
// older stack, whose top is preserved.  masks (nullable): [n_stacks][n],
// 1 where that stack holds the point.
__global__ void combine_lith_kernel(const int32_t* ids, int32_t n_stacks, int64_t n, const int32_t* nsurf,
                                    const int32_t* offset, const int32_t* rel, int32_t basement, int32_t* out,
                                    uint8_t* masks) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  int32_t v = basement;
  int owner = n_stacks - 1;          // the oldest stack holds the basement
  for (int s = 0; s < n_stacks; ++s) {
    const int32_t id = ids[(int64_t)s * n + p];
    if (id > nsurf[s]) continue;
    if (rel[s] == GK_REL_ONLAP && s + 1 < n_stacks && ids[(int64_t)(s + 1) * n + p] > 1) continue;
    v = id + offset[s];
    owner = s;
    break;
  }
  out[p] = v;
  if (masks)
    for (int s = 0; s < n_stacks; ++s) masks[(int64_t)s * n + p] = s == owner ? 1 : 0;
}
}  // namespace

static int combine_impl(gk_handle h, int32_t n_stacks, const int32_t* ids, int64_t n, const int32_t* n_surf,
                        const int32_t* relation, int32_t* lith, uint8_t* masks, hipStream_t st) {
  GK_REQUIRE(h && ids && lith && n_surf && n_stacks > 0 && n_stacks <= 64 && n >= 0, GK_ERR_ARG,
             "gk_combine_lith: bad arguments");
  int32_t hbuf[192];
  int32_t off = 0;
  for (int s = 0; s < n_stacks; ++s) {
    GK_REQUIRE(n_surf[s] > 0, GK_ERR_ARG, "gk_combine_lith: stack %d has no surface", s);
    const int32_t r = relation ? relation[s] : GK_REL_ERODE;
    GK_REQUIRE(r == GK_REL_ERODE || r == GK_REL_ONLAP, GK_ERR_ARG,
               "gk_combine_lith: stack %d: relation %d (erode or onlap expected)", s, r);
    hbuf[s] = n_surf[s];
    hbuf[64 + s] = off;
    hbuf[128 + s] = r;
    off += n_surf[s];
  }
  void* ws = nullptr;
  GK_TRY(gk_workspace(h, WS_SMALL, 192 * sizeof(int32_t), &ws));
  int32_t* d = static_cast<int32_t*>(ws);
  GK_HIP(hipMemcpyAsync(d, hbuf, sizeof(hbuf), hipMemcpyHostToDevice, st));
  if (n > 0)
    hipLaunchKernelGGL(combine_lith_kernel, dim3((unsigned)gk_ceil_div(n, 256)), dim3(256), 0, st, ids,
                       n_stacks, n, d, d + 64, d + 128, off + 1, lith, masks);
  GK_HIP(hipGetLastError());
  GK_HIP(hipStreamSynchronize(st));   // hbuf is a stack buffer
  return GK_OK;
}

extern "C" int gk_combine_lith(gk_handle h, int32_t n_stacks, const int32_t* ids, int64_t n,
                               const int32_t* n_surf, int32_t* lith, gk_stream stream) {
  return combine_impl(h, n_stacks, ids, n, n_surf, nullptr, lith, nullptr, (hipStream_t)stream);
}

extern "C" int gk_combine_stacks(gk_handle h, int32_t n_stacks, const int32_t* ids, int64_t n,
                                 const int32_t* n_surf, const int32_t* relation, int32_t* lith, uint8_t* masks,
                                 gk_stream stream) {
  return combine_impl(h, n_stacks, ids, n, n_surf, relation, lith, masks, (hipStream_t)stream);
}

// ------------------------------------------------------- raw-source fields
namespace {
__global__ void prep_raw_kernel(int64_t n, const double* xyz, const double* w, double c0, double c1, double c2,
                                double inv_a, double scale, V4<double>* out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  V4<double> v;
  v.x = (xyz[3 * i] - c0) * inv_a;
  v.y = (xyz[3 * i + 1] - c1) * inv_a;
  v.z = (xyz[3 * i + 2] - c2) * inv_a;
  v.w = scale * w[i];
  out[i] = v;
}
}  // namespace

// F(x) = sum_s w_s C(|x - s|) and grad F at explicit points (FP64), for
// sources given explicitly (e.g. observation points weighted by dL/dS).
extern "C" int gk_eval_sources(gk_handle h, double range, double c_o, const double* center, int64_t n_src,
                               const double* src_xyz, const double* src_w, int64_t n_points, const double* xyz,
                               double* scalar, double* gradient, gk_stream stream) {
  GK_REQUIRE(h && center && range > 0 && n_src >= 0 && n_points >= 0, GK_ERR_ARG, "gk_eval_sources: bad arguments");
  GK_REQUIRE((n_src == 0 || (src_xyz && src_w)) && (n_points == 0 || (xyz && scalar)), GK_ERR_ARG,
             "gk_eval_sources: NULL array");
  if (n_points == 0) return GK_OK;
  hipStream_t st = (hipStream_t)stream;
  void* ws = nullptr;
  GK_TRY(gk_workspace(h, WS_EVAL_SRC, (size_t)std::max<int64_t>(n_src, 1) * 32 + 256, &ws));
  V4<double>* src = static_cast<V4<double>*>(ws);
  if (n_src > 0)
    hipLaunchKernelGGL(prep_raw_kernel, dim3((unsigned)gk_ceil_div(n_src, 256)), dim3(256), 0, st, n_src, src_xyz,
                       src_w, center[0], center[1], center[2], 1.0 / range, c_o, src);
  EvalArgs a{};
  a.n_points = n_points;
  a.xyz = xyz;
  a.cx = center[0]; a.cy = center[1]; a.cz = center[2];
  a.inv_a = 1.0 / range;
  a.pts = src;
  a.n_pts = n_src;
  a.ori = nullptr;
  a.n_ori = 0;
  a.uni_degree = 0;
  a.n_fault = 0;
  a.scalar = scalar;
  a.grad = gradient;
  return run_eval(h, a, false, GK_F64, gradient != nullptr, true, st);
}

// Smooth ids (the engine's differentiable block, sigmoid_slope at
// 2-layers.approved.txt:181): the step 1 + #{k: S < t_k} (or S > t_k for a
// stack whose thresholds increase) with every unit step replaced by the
// logistic function of slope * (t_k - S) (or slope * (S - t_k)).
__global__ void block_values_kernel(const double* S, int64_t n, int32_t n_thr, const double* thr, int32_t rev,
                                    double slope, double* out) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const double s = S[p];
  double v = 1.0;
  for (int k = 0; k < n_thr; ++k) {
    const double z = rev ? slope * (s - thr[k]) : slope * (thr[k] - s);
    v += 1.0 / (1.0 + exp(-z));
  }
  out[p] = v;
}

extern "C" int gk_block_values(gk_handle h, const double* scalar, int64_t n, int32_t n_thresholds,
                               const double* thresholds, double sigmoid_slope, double* block, gk_stream stream) {
  GK_REQUIRE(h && scalar && block && thresholds && n >= 0 && n_thresholds >= 0 &&
             n_thresholds <= GK_MAX_THRESHOLDS, GK_ERR_ARG, "gk_block_values: bad arguments");
  hipStream_t st = (hipStream_t)stream;
  double hbuf[GK_MAX_THRESHOLDS];
  for (int k = 0; k < n_thresholds; ++k) hbuf[k] = thresholds[k];
  const int32_t rev = n_thresholds >= 2 && hbuf[0] < hbuf[n_thresholds - 1] ? 1 : 0;
  void* ws = nullptr;
  GK_TRY(gk_workspace(h, WS_SMALL, 192 * sizeof(int32_t) + GK_MAX_THRESHOLDS * sizeof(double), &ws));
  double* d = reinterpret_cast<double*>(static_cast<char*>(ws) + 192 * sizeof(int32_t));
  if (n_thresholds > 0) GK_HIP(hipMemcpyAsync(d, hbuf, n_thresholds * sizeof(double), hipMemcpyHostToDevice, st));
  if (n > 0)
    hipLaunchKernelGGL(block_values_kernel, dim3((unsigned)gk_ceil_div(n, 256)), dim3(256), 0, st, scalar, n,
                       n_thresholds, d, rev, sigmoid_slope, block);
  GK_HIP(hipGetLastError());
  GK_HIP(hipStreamSynchronize(st));   // hbuf is a stack buffer
  return GK_OK;
}

// ------------------------------------------------------ no-allocation entry
// Scratch of gk_eval_noalloc: the packed sources and the split partials live
// in this file-scope array (one copy per GPU, held until the process ends).
// Host code never uses the array's name as an address: gk_eval_scratch_init
// takes its device address once per handle (the device is current in
// gk_create) and the entry point passes that address to the kernels.
static __device__ __align__(256) unsigned char scratch[GK_EVAL_SCRATCH_BYTES];

int gk_eval_scratch_init(gk_handle h) {
  void* p = nullptr;
  GK_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  GK_REQUIRE(p != nullptr, GK_ERR_HIP, "gk_create: no device address for the evaluation scratch array");
  h->eval_scratch = static_cast<char*>(p);
  return GK_OK;
}

extern "C" int gk_eval_noalloc(gk_handle h, const gk_system* sys, const double* weights, gk_eval_desc* desc,
                               gk_stream stream) {
  GK_REQUIRE(h && h->eval_scratch, GK_ERR_ARG, "gk_eval_noalloc: handle without an evaluation scratch array");
  return eval_impl(h, sys, weights, desc, (hipStream_t)stream, false, nullptr, false, h->eval_scratch,
                   GK_EVAL_SCRATCH_BYTES);
}

// ------------------------------------------------------------ Hessians
// Second derivatives of a field at explicit points (FP64), for the adjoint
// with respect to the orientation positions.  In the frame X = (x - c)/a with
// unit polynomials (c_o folded into the source weights, as in the evaluation),
// d1 = c'/rho, d2 = (c'' - c'/rho)/rho^2 = 105/4 (1 - rho^2)^2 / rho and
// d3 = d2'/rho = -105/4 (1 - rho^2)(1 + 3 rho^2) / rho^3, H = X - source:
//   point source W:        W (delta d1 + H H^T d2)
//   orientation source V:  -(d2 (delta V.H + V H^T + H V^T) + H H^T (V.H) d3)
// (the orientation term at rho = 0 is odd and contributes 0).  Output per
// point: xx, yy, zz, xy, xz, yz of the Hessian in real coordinates.
namespace {
struct HessArgs {
  const V4<double>* pts;
  int64_t n_pts, pts_chunk;
  const V8<double>* ori;
  int64_t n_ori, ori_chunk;
  const double* xyz;
  int64_t n;
  double cx, cy, cz, inv_a;
  int32_t uni_degree;
  double gi_res;
  const double* lam;          // drift weights (degree 2 adds a constant Hessian)
  int32_t nsplit;
  double* part;               // [nsplit][n][6]
};

__global__ __launch_bounds__(256) void hessian_kernel(HessArgs a) {
  __shared__ V4<double> tp[256];
  __shared__ V8<double> to[256];
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const bool live = p < a.n;
  double X = 0.0, Y = 0.0, Z = 0.0;
  if (live) {
    X = (a.xyz[3 * p] - a.cx) * a.inv_a;
    Y = (a.xyz[3 * p + 1] - a.cy) * a.inv_a;
    Z = (a.xyz[3 * p + 2] - a.cz) * a.inv_a;
  }
  double h[6] = {0, 0, 0, 0, 0, 0};
  const int64_t p0 = (int64_t)blockIdx.y * a.pts_chunk;
  const int64_t p1 = p0 + a.pts_chunk < a.n_pts ? p0 + a.pts_chunk : a.n_pts;
  for (int64_t t0 = p0; t0 < p1; t0 += 256) {
    __syncthreads();
    if (t0 + threadIdx.x < p1) tp[threadIdx.x] = a.pts[t0 + threadIdx.x];
    __syncthreads();
    const int cnt = p1 - t0 < 256 ? (int)(p1 - t0) : 256;
    if (!live) continue;
    for (int k = 0; k < cnt; ++k) {
      const V4<double> sv = tp[k];
      const double hx = X - sv.x, hy = Y - sv.y, hz = Z - sv.z;
      const double r2 = hx * hx + hy * hy + hz * hz;
      if (r2 >= 1.0) continue;
      const double rho = sqrt(r2);
      const double d1 = -14.0 + rho * (26.25 + r2 * (-17.5 + 5.25 * r2));
      const double om = 1.0 - r2;
      const double d2 = rho > 0.0 ? 26.25 * om * om / rho : 0.0;
      const double w = sv.w, wd2 = w * d2;
      h[0] += w * d1 + wd2 * hx * hx;
      h[1] += w * d1 + wd2 * hy * hy;
      h[2] += w * d1 + wd2 * hz * hz;
      h[3] += wd2 * hx * hy;
      h[4] += wd2 * hx * hz;
      h[5] += wd2 * hy * hz;
    }
  }
  const int64_t q0 = (int64_t)blockIdx.y * a.ori_chunk;
  const int64_t q1 = q0 + a.ori_chunk < a.n_ori ? q0 + a.ori_chunk : a.n_ori;
  for (int64_t t0 = q0; t0 < q1; t0 += 256) {
    __syncthreads();
    if (t0 + threadIdx.x < q1) to[threadIdx.x] = a.ori[t0 + threadIdx.x];
    __syncthreads();
    const int cnt = q1 - t0 < 256 ? (int)(q1 - t0) : 256;
    if (!live) continue;
    for (int k = 0; k < cnt; ++k) {
      const V8<double> sv = to[k];
      const double hx = X - sv.x, hy = Y - sv.y, hz = Z - sv.z;
      const double r2 = hx * hx + hy * hy + hz * hz;
      if (r2 >= 1.0 || r2 == 0.0) continue;
      const double rho = sqrt(r2);
      const double om = 1.0 - r2;
      const double d2 = 26.25 * om * om / rho;
      const double d3 = -26.25 * om * (1.0 + 3.0 * r2) / (rho * r2);
      const double vx = sv.wx, vy = sv.wy, vz = sv.wz;
      const double vh = vx * hx + vy * hy + vz * hz;
      const double t = vh * d3;
      h[0] -= d2 * (vh + 2.0 * vx * hx) + hx * hx * t;
      h[1] -= d2 * (vh + 2.0 * vy * hy) + hy * hy * t;
      h[2] -= d2 * (vh + 2.0 * vz * hz) + hz * hz * t;
      h[3] -= d2 * (vx * hy + vy * hx) + hx * hy * t;
      h[4] -= d2 * (vx * hz + vz * hx) + hx * hz * t;
      h[5] -= d2 * (vy * hz + vz * hy) + hy * hz * t;
    }
  }
  if (live) {
    double* o = a.part + ((int64_t)blockIdx.y * a.n + p) * 6;
#pragma unroll
    for (int c = 0; c < 6; ++c) o[c] = h[c];
  }
}

__global__ void hessian_finalize_kernel(HessArgs a, double* out) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= a.n) return;
  double h[6] = {0, 0, 0, 0, 0, 0};
  for (int y = 0; y < a.nsplit; ++y)
#pragma unroll
    for (int c = 0; c < 6; ++c) h[c] += a.part[((int64_t)y * a.n + p) * 6 + c];
  const double s = a.inv_a * a.inv_a;
#pragma unroll
  for (int c = 0; c < 6; ++c) h[c] *= s;
  if (a.uni_degree >= 2 && a.lam) {       // x^2, y^2, z^2, xy, xz, yz drift terms
    const double* l = a.lam;
    h[0] += a.gi_res * 2.0 * l[3];
    h[1] += a.gi_res * 2.0 * l[4];
    h[2] += a.gi_res * 2.0 * l[5];
    h[3] += a.gi_res * l[6];
    h[4] += a.gi_res * l[7];
    h[5] += a.gi_res * l[8];
  }
#pragma unroll
  for (int c = 0; c < 6; ++c) out[p * 6 + c] = h[c];
}

int run_hessian(HessArgs& a, double* out, size_t part_cap, hipStream_t st) {
  const int64_t nsrc = a.n_pts + a.n_ori;
  int64_t ns = std::min<int64_t>(64, std::max<int64_t>(1, gk_ceil_div(nsrc, 2048)));
  ns = std::max<int64_t>(1, std::min<int64_t>(ns, (int64_t)(part_cap / ((size_t)std::max<int64_t>(a.n, 1) * 48))));
  a.nsplit = (int32_t)ns;
  a.pts_chunk = std::max<int64_t>(gk_ceil_div(a.n_pts, ns), 1);
  a.ori_chunk = std::max<int64_t>(gk_ceil_div(a.n_ori, ns), 1);
  if (a.n == 0) return GK_OK;
  hipLaunchKernelGGL(hessian_kernel, dim3((unsigned)gk_ceil_div(a.n, 256), (unsigned)ns), dim3(256), 0, st, a);
  hipLaunchKernelGGL(hessian_finalize_kernel, dim3((unsigned)gk_ceil_div(a.n, 256)), dim3(256), 0, st, a, out);
  GK_HIP(hipGetLastError());
  return GK_OK;
}
}  // namespace

// Hessian of the system's field for `weights` (covariance and drift terms; the
// fault block is piecewise constant) at n explicit points.  part: scratch of
// part_cap bytes (>= 48 n) for the source-split partials.
int gk_hessian_system(gk_handle h, const gk_system* sys, const double* weights, int64_t n, const double* xyz,
                      double* hess6, double* part, size_t part_cap, hipStream_t st) {
  GK_TRY(check_system(sys));
  GK_REQUIRE(part_cap >= (size_t)std::max<int64_t>(n, 1) * 48, GK_ERR_ARG, "hessian: partial buffer too small");
  void* ws = nullptr;
  GK_TRY(gk_workspace(h, WS_EVAL_SRC, sources_bytes(sys), &ws));
  void *pts = nullptr, *ori = nullptr;
  source_layout(sys, GK_F64, ws, &pts, &ori);
  GK_TRY(prepare_sources(sys, weights, GK_F64, st, ws, nullptr));
  HessArgs a{};
  a.pts = static_cast<const V4<double>*>(pts);
  a.n_pts = sys->n_rest + sys->n_surf;
  a.ori = static_cast<const V8<double>*>(ori);
  a.n_ori = sys->n_ori;
  a.xyz = xyz;
  a.n = n;
  a.cx = sys->center[0]; a.cy = sys->center[1]; a.cz = sys->center[2];
  a.inv_a = 1.0 / sys->range;
  a.uni_degree = sys->uni_degree;
  a.gi_res = sys->gi_res;
  a.lam = weights + 3 * sys->n_ori + sys->n_rest;
  a.part = part;
  return run_hessian(a, hess6, part_cap, st);
}

// Hessian of F(x) = sum_s w_s C(|x - s|) (explicit sources) at n points.
int gk_hessian_sources(gk_handle h, double range, double c_o, const double* center, int64_t n_src,
                       const double* src_xyz, const double* src_w, int64_t n, const double* xyz, double* hess6,
                       double* part, size_t part_cap, hipStream_t st) {
  GK_REQUIRE(part_cap >= (size_t)std::max<int64_t>(n, 1) * 48, GK_ERR_ARG, "hessian: partial buffer too small");
  void* ws = nullptr;
  GK_TRY(gk_workspace(h, WS_EVAL_SRC, (size_t)std::max<int64_t>(n_src, 1) * 32 + 256, &ws));
  V4<double>* src = static_cast<V4<double>*>(ws);
  if (n_src > 0)
    hipLaunchKernelGGL(prep_raw_kernel, dim3((unsigned)gk_ceil_div(n_src, 256)), dim3(256), 0, st, n_src, src_xyz,
                       src_w, center[0], center[1], center[2], 1.0 / range, c_o, src);
  HessArgs a{};
  a.pts = src;
  a.n_pts = n_src;
  a.ori = nullptr;
  a.n_ori = 0;
  a.xyz = xyz;
  a.n = n;
  a.cx = center[0]; a.cy = center[1]; a.cz = center[2];
  a.inv_a = 1.0 / range;
  a.uni_degree = 0;
  a.part = part;
  return run_hessian(a, hess6, part_cap, st);
}
