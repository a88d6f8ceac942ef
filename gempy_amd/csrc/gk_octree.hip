// Octree refinement of the evaluation grid (the engine's octree levels:
// _number_octree_levels, octree_error_threshold at fault.approved.txt:210-214;
// outputs per level at test_example_models_I.py:20; grid sizing
// resolution = base * 2^(levels-1) at regular_grid.py:36-43).
//
// A level holds a list of active voxels (linear index (ix*ny + iy)*nz + iz at
// that level's resolution).  Each voxel is probed at its centre and its 8
// corners; it is refined when any id field differs among those 9 points, and
// its 8 children (at twice the resolution) become the next level's voxels,
// written in voxel order (deterministic compaction: per-block counts, host
// exclusive scan, per-block LDS scan).
#include "gk_internal.h"

namespace {

__global__ void octree_points_kernel(double x0, double y0, double z0, double hx, double hy, double hz,
                                     int64_t ny, int64_t nz, const int64_t* vox, int64_t n, double* xyz) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n * 9) return;
  const int64_t v = vox[t / 9];
  const int k = (int)(t % 9);
  const int64_t iz = v % nz, iy = (v / nz) % ny, ix = v / (nz * ny);
  double fx, fy, fz;
  if (k == 0) { fx = 0.5; fy = 0.5; fz = 0.5; }
  else { const int c = k - 1; fx = (c >> 2) & 1; fy = (c >> 1) & 1; fz = c & 1; }
  xyz[3 * t + 0] = x0 + (ix + fx) * hx;
  xyz[3 * t + 1] = y0 + (iy + fy) * hy;
  xyz[3 * t + 2] = z0 + (iz + fz) * hz;
}

__global__ void octree_mark_kernel(const int32_t* ids, int32_t nf, int64_t n, uint8_t* refine, int32_t* counts) {
  __shared__ int32_t cnt;
  if (threadIdx.x == 0) cnt = 0;
  __syncthreads();
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int r = 0;
  if (v < n) {
    for (int f = 0; f < nf && !r; ++f) {
      const int32_t* p = ids + (int64_t)f * n * 9 + v * 9;
      for (int k = 1; k < 9; ++k) if (p[k] != p[0]) { r = 1; break; }
    }
    refine[v] = (uint8_t)r;
  }
  if (r) atomicAdd(&cnt, 1);
  __syncthreads();
  if (threadIdx.x == 0) counts[blockIdx.x] = cnt;
}

__global__ void octree_children_kernel(const uint8_t* refine, const int64_t* vox, int64_t n, const int64_t* offsets,
                                       int64_t ny, int64_t nz, int64_t* children) {
  __shared__ int32_t scan[256];
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int r = (v < n) ? refine[v] : 0;
  scan[threadIdx.x] = r;
  __syncthreads();
  for (int s = 1; s < 256; s <<= 1) {        // inclusive Hillis-Steele scan
    const int32_t add = threadIdx.x >= s ? scan[threadIdx.x - s] : 0;
    __syncthreads();
    scan[threadIdx.x] += add;
    __syncthreads();
  }
  if (!r) return;
  const int64_t pos = offsets[blockIdx.x] + scan[threadIdx.x] - 1;
  const int64_t w = vox[v];
  const int64_t iz = w % nz, iy = (w / nz) % ny, ix = w / (nz * ny);
  const int64_t NY = 2 * ny, NZ = 2 * nz;
  for (int c = 0; c < 8; ++c) {
    const int64_t cx = 2 * ix + ((c >> 2) & 1), cy = 2 * iy + ((c >> 1) & 1), cz = 2 * iz + (c & 1);
    children[8 * pos + c] = (cx * NY + cy) * NZ + cz;
  }
}

__global__ void octree_centres_kernel(double x0, double y0, double z0, double hx, double hy, double hz, int64_t ny,
                                      int64_t nz, const int64_t* vox, int64_t n, double* xyz) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int64_t v = vox[t];
  const int64_t iz = v % nz, iy = (v / nz) % ny, ix = v / (nz * ny);
  xyz[3 * t + 0] = x0 + (ix + 0.5) * hx;
  xyz[3 * t + 1] = y0 + (iy + 0.5) * hy;
  xyz[3 * t + 2] = z0 + (iz + 0.5) * hz;
}

// Probe points without repeats.  Voxels share their corners (a level whose
// voxels are all active has 9 probes a voxel but 2 points), and what a probe
// costs is the evaluation of every stack there, so each corner is evaluated
// once: flags over the level's corner lattice, ranks by a scan, points and the
// probes' map.  Octree part of a model of 128^3 points, four levels and four
// stacks: 7.2 ms of evaluations, 3.6 now.
struct ProbeArgs {
  double o[3], h[3];
  int64_t res[3];                        // voxels; corners: one more per axis
  const int64_t* vox;
  int64_t n, nc;                         // voxels, corners of the lattice
  uint8_t* flag;
  int32_t *rank, *sums;
  int32_t* total;                        // number of corners; then whether a voxel lies outside the level
  double* xyz;
  int32_t* map;
};

__device__ __forceinline__ bool probe_voxel(const ProbeArgs& a, int64_t v) {
  return v >= 0 && v < a.res[0] * a.res[1] * a.res[2];
}

__device__ __forceinline__ int64_t probe_corner(const ProbeArgs& a, int64_t v, int c, int64_t* at) {
  at[2] = v % a.res[2] + (c & 1);
  at[1] = v / a.res[2] % a.res[1] + ((c >> 1) & 1);
  at[0] = v / (a.res[2] * a.res[1]) + ((c >> 2) & 1);
  return (at[0] * (a.res[1] + 1) + at[1]) * (a.res[2] + 1) + at[2];
}

__global__ void probe_flags_kernel(ProbeArgs a) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t at[3];
  if (t >= 8 * a.n) return;
  const int64_t v = a.vox[t / 8];
  if (probe_voxel(a, v)) a.flag[probe_corner(a, v, (int)(t % 8), at)] = 1;
  else a.total[1] = 1;
}

// Ranks within blocks of 1,024 corners, and the blocks' totals.
__global__ __launch_bounds__(1024) void probe_rank_kernel(ProbeArgs a) {
  __shared__ int32_t s[16];
  const int64_t t = (int64_t)blockIdx.x * 1024 + threadIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bool set = t < a.nc && a.flag[t];
  const uint64_t m = __ballot(set);
  if (lane == 0) s[wave] = __popcll(m);
  __syncthreads();
  int32_t before = __popcll(m & ((1ull << lane) - 1)), all = 0;
  for (int w = 0; w < 16; ++w) {
    if (w < wave) before += s[w];
    all += s[w];
  }
  if (t < a.nc) a.rank[t] = before;
  if (threadIdx.x == 0) a.sums[blockIdx.x] = all;
}

// Block totals to sums over the earlier blocks (one workgroup).
__global__ __launch_bounds__(1024) void probe_scan_kernel(ProbeArgs a, int64_t nb) {
  __shared__ int32_t s[1024];
  const int t = threadIdx.x;
  const int64_t per = (nb + 1023) / 1024, b0 = t * per, b1 = b0 + per < nb ? b0 + per : nb;
  int32_t acc = 0;
  for (int64_t i = b0; i < b1; ++i) acc += a.sums[i];
  s[t] = acc;
  __syncthreads();
  for (int o = 1; o < 1024; o <<= 1) {
    const int32_t v = t >= o ? s[t - o] : 0;
    __syncthreads();
    s[t] += v;
    __syncthreads();
  }
  int32_t run = s[t] - acc;
  for (int64_t i = b0; i < b1; ++i) {
    const int32_t v = a.sums[i];
    a.sums[i] = run;
    run += v;
  }
  if (t == 1023) *a.total = s[1023];
}

// Points (centres, then corners in lattice order) and the map of the 9 probes
// of each voxel.  Corner positions are the same products for all voxels around.
__global__ void probe_points_kernel(ProbeArgs a) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 9 * a.n) return;
  const int64_t i = t / 9, v = a.vox[i];
  if (!probe_voxel(a, v)) return;
  const int k = (int)(t % 9);
  int64_t at[3], p = i;
  double f = 0.5;
  if (k == 0) {
    probe_corner(a, v, 0, at);
  } else {
    const int64_t c = probe_corner(a, v, k - 1, at);
    p = a.n + a.sums[c / 1024] + a.rank[c];
    f = 0.0;
  }
  a.map[t] = (int32_t)p;
  // voxels that share a corner write the same values
  for (int d = 0; d < 3; ++d) a.xyz[3 * p + d] = a.o[d] + (at[d] + f) * a.h[d];
}

}  // namespace

extern "C" int gk_octree_probes(gk_handle h, const double* extent, const int64_t* res, const int64_t* voxels,
                                int64_t n, double* xyz, int32_t* map, int64_t* n_points, gk_stream stream) {
  GK_REQUIRE(h && extent && res && n_points && n >= 0 && (n == 0 || (voxels && xyz && map)), GK_ERR_ARG,
             "gk_octree_probes: bad arguments");
  GK_REQUIRE(res[0] > 0 && res[1] > 0 && res[2] > 0, GK_ERR_ARG, "gk_octree_probes: bad resolution");
  *n_points = 0;
  if (n == 0) return GK_OK;
  hipStream_t st = (hipStream_t)stream;
  ProbeArgs a{};
  for (int d = 0; d < 3; ++d) {
    a.o[d] = extent[2 * d];
    a.h[d] = (extent[2 * d + 1] - extent[2 * d]) / res[d];
    a.res[d] = res[d];
  }
  a.vox = voxels;
  a.n = n;
  GK_REQUIRE(n < (int64_t)INT32_MAX / 9 && (res[0] + 1.0) * (res[1] + 1.0) * (res[2] + 1.0) < (double)INT32_MAX,
             GK_ERR_ARG, "gk_octree_probes: level too large");
  a.nc = (res[0] + 1) * (res[1] + 1) * (res[2] + 1);
  const int64_t nb = gk_ceil_div(a.nc, 1024);
  const size_t o_flag = 256, o_rank = o_flag + gk_round_up(a.nc, 256), o_sums = o_rank + gk_round_up(a.nc * 4, 256);
  void* ws = nullptr;
  GK_TRY(gk_workspace(h, WS_OCTREE, o_sums + gk_round_up(nb * 4, 256), &ws));
  char* b = static_cast<char*>(ws);
  a.total = reinterpret_cast<int32_t*>(b);
  a.flag = reinterpret_cast<uint8_t*>(b + o_flag);
  a.rank = reinterpret_cast<int32_t*>(b + o_rank);
  a.sums = reinterpret_cast<int32_t*>(b + o_sums);
  a.xyz = xyz;
  a.map = map;
  GK_HIP(hipMemsetAsync(b, 0, o_flag + a.nc, st));
  hipLaunchKernelGGL(probe_flags_kernel, dim3((unsigned)gk_ceil_div(8 * n, 256)), dim3(256), 0, st, a);
  hipLaunchKernelGGL(probe_rank_kernel, dim3((unsigned)nb), dim3(1024), 0, st, a);
  hipLaunchKernelGGL(probe_scan_kernel, dim3(1), dim3(1024), 0, st, a, nb);
  hipLaunchKernelGGL(probe_points_kernel, dim3((unsigned)gk_ceil_div(9 * n, 256)), dim3(256), 0, st, a);
  int32_t total[2] = {0, 0};
  GK_HIP(hipMemcpyAsync(total, a.total, sizeof(total), hipMemcpyDeviceToHost, st));
  GK_HIP(hipStreamSynchronize(st));
  GK_HIP(hipGetLastError());
  GK_REQUIRE(total[1] == 0, GK_ERR_ARG, "gk_octree_probes: a voxel index lies outside the level");
  *n_points = n + total[0];
  return GK_OK;
}

extern "C" int gk_octree_points(gk_handle h, const double* extent, const int64_t* res, const int64_t* voxels,
                                int64_t n, int32_t centres_only, double* xyz, gk_stream stream) {
  GK_REQUIRE(h && extent && res && (n == 0 || (voxels && xyz)) && n >= 0, GK_ERR_ARG,
             "gk_octree_points: bad arguments");
  GK_REQUIRE(res[0] > 0 && res[1] > 0 && res[2] > 0, GK_ERR_ARG, "gk_octree_points: bad resolution");
  if (n == 0) return GK_OK;
  hipStream_t st = (hipStream_t)stream;
  const double hx = (extent[1] - extent[0]) / res[0], hy = (extent[3] - extent[2]) / res[1],
               hz = (extent[5] - extent[4]) / res[2];
  if (centres_only)
    hipLaunchKernelGGL(octree_centres_kernel, dim3((unsigned)gk_ceil_div(n, 256)), dim3(256), 0, st, extent[0],
                       extent[2], extent[4], hx, hy, hz, res[1], res[2], voxels, n, xyz);
  else
    hipLaunchKernelGGL(octree_points_kernel, dim3((unsigned)gk_ceil_div(n * 9, 256)), dim3(256), 0, st, extent[0],
                       extent[2], extent[4], hx, hy, hz, res[1], res[2], voxels, n, xyz);
  GK_HIP(hipGetLastError());
  return GK_OK;
}

extern "C" int gk_octree_refine(gk_handle h, int32_t n_fields, const int32_t* ids, int64_t n, const int64_t* voxels,
                                const int64_t* res, uint8_t* refine, int64_t* children, int64_t* n_children,
                                gk_stream stream) {
  GK_REQUIRE(h && n_children && res && n >= 0 && n_fields >= 1, GK_ERR_ARG, "gk_octree_refine: bad arguments");
  *n_children = 0;
  if (n == 0) return GK_OK;
  GK_REQUIRE(ids && voxels && refine && children, GK_ERR_ARG, "gk_octree_refine: NULL array");
  hipStream_t st = (hipStream_t)stream;
  const int64_t nb = gk_ceil_div(n, 256);
  void* ws = nullptr;
  GK_TRY(gk_workspace(h, WS_SMALL, (size_t)nb * (sizeof(int32_t) + sizeof(int64_t)) + 512, &ws));
  int32_t* counts = static_cast<int32_t*>(ws);
  int64_t* offsets = reinterpret_cast<int64_t*>(static_cast<char*>(ws) + gk_round_up(nb * 4, 256));
  hipLaunchKernelGGL(octree_mark_kernel, dim3((unsigned)nb), dim3(256), 0, st, ids, n_fields, n, refine, counts);
  std::vector<int32_t> hc(nb);
  std::vector<int64_t> ho(nb);
  GK_HIP(hipMemcpyAsync(hc.data(), counts, nb * sizeof(int32_t), hipMemcpyDeviceToHost, st));
  GK_HIP(hipStreamSynchronize(st));
  int64_t total = 0;
  for (int64_t b = 0; b < nb; ++b) { ho[b] = total; total += hc[b]; }
  GK_HIP(hipMemcpyAsync(offsets, ho.data(), nb * sizeof(int64_t), hipMemcpyHostToDevice, st));
  if (total > 0)
    hipLaunchKernelGGL(octree_children_kernel, dim3((unsigned)nb), dim3(256), 0, st, refine, voxels, n, offsets,
                       res[1], res[2], children);
  GK_HIP(hipGetLastError());
  GK_HIP(hipStreamSynchronize(st));
  *n_children = 8 * total;
  return GK_OK;
}
