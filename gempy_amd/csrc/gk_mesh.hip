// Isosurface extraction (marching cubes) of a lattice field: the consumer of
// the evaluated scalar field that turns each surface's threshold into a
// triangle mesh (the reference calls skimage's marching cubes per element,
// gempy/modules/mesh_extranction/marching_cubes.py:59-101).
//
// One vertex per lattice edge whose end values straddle the level (a corner
// is "above" when its value > level), placed by linear interpolation along
// the edge; vertices are shared by all cubes that use the edge.  The
// triangulation of the 256 corner cases is built here from first principles:
// on every cube face the crossing points are joined by segments that cut off
// the face's "above" corners (so two cubes sharing a face always agree: the
// mesh is watertight), segments are directed along the face boundary taken
// counter-clockwise as seen from outside the cube (entering the "above" run
// -> leaving it), they chain into closed loops across the faces, and every
// loop is triangulated as a fan.  Triangles wind so that their normals
// (right-hand rule) point towards increasing field values.
//
// The field is read once: a first pass packs the points, in memory order, into
// words of 64 (above the level, NaN, masked), and everything that follows works
// on those words - an eighth of a byte per point and flag - until the crossed
// edges and the cubes with triangles, few and known, are written.  A neighbour
// along an axis is the same bit of the words shifted by that axis' step; words
// that began anew with every z row were mostly empty on lattices of few layers
// (2000 x 2000 x 2: 1,500 us, 170 now).  What it is bound
// by is that one read (8 bytes a point, 9 with a mask).  Per-point flags, edge
// ids and cube cases in memory with scans over them moved about 500 bytes a
// point: 200^3 cells with a mask took 400 us so and take 83 us now, of which the
// packing 22 us (75 MB, 3.4 TB/s) and the writing pass 32 us.
#include <algorithm>
#include <cmath>
#include <vector>
#include "gk_internal.h"

namespace {

constexpr int MC_MAX_TRI = 5;    // triangles per cube case, at most (the construction yields <= 5)

struct McTables {
  uint8_t ntri[256];
  int8_t tri[256][MC_MAX_TRI][3];      // local edges of each triangle
};

// corner c = x + 2y + 4z; local edge e = 4 * axis + k, k the two other
// coordinates (in increasing axis order) as bits
void edge_corners(int e, int* c0, int* c1) {
  const int axis = e / 4, k = e % 4;
  int o[3] = {0, 0, 0}, j = 0;
  for (int a = 0; a < 3; ++a)
    if (a != axis) o[a] = (k >> j++) & 1;
  *c0 = o[0] + 2 * o[1] + 4 * o[2];
  o[axis] = 1;
  *c1 = o[0] + 2 * o[1] + 4 * o[2];
}

int edge_of(int ca, int cb) {
  for (int e = 0; e < 12; ++e) {
    int c0, c1;
    edge_corners(e, &c0, &c1);
    if ((c0 == ca && c1 == cb) || (c0 == cb && c1 == ca)) return e;
  }
  return -1;
}

McTables build_tables() {
  McTables T{};
  // the six faces: corners in counter-clockwise order seen from outside
  int faces[6][4];
  for (int f = 0; f < 6; ++f) {
    const int axis = f / 2, side = f % 2;
    const double n[3] = {axis == 0 ? (side ? 1.0 : -1.0) : 0.0, axis == 1 ? (side ? 1.0 : -1.0) : 0.0,
                         axis == 2 ? (side ? 1.0 : -1.0) : 0.0};
    std::vector<int> cs;
    for (int c = 0; c < 8; ++c)
      if (((c >> axis) & 1) == side) cs.push_back(c);
    const int u = (axis + 1) % 3, v = (axis + 2) % 3;        // (u, v, axis) is right-handed
    std::sort(cs.begin(), cs.end(), [&](int a, int b) {
      const double au = ((a >> u) & 1) - 0.5, av = ((a >> v) & 1) - 0.5;
      const double bu = ((b >> u) & 1) - 0.5, bv = ((b >> v) & 1) - 0.5;
      return std::atan2(av, au) < std::atan2(bv, bu);        // counter-clockwise about +axis
    });
    if (n[axis] < 0) std::reverse(cs.begin(), cs.end());     // counter-clockwise about the outward normal
    for (int i = 0; i < 4; ++i) faces[f][i] = cs[i];
  }
  for (int cs = 0; cs < 256; ++cs) {
    int next[12];
    for (int& e : next) e = -1;
    for (int f = 0; f < 6; ++f) {
      int cross[4], dir[4], nc = 0;     // crossing edges in boundary order, +1 entering the "above" run
      for (int i = 0; i < 4; ++i) {
        const int a = faces[f][i], b = faces[f][(i + 1) % 4];
        const int ia = (cs >> a) & 1, ib = (cs >> b) & 1;
        if (ia != ib) {
          cross[nc] = edge_of(a, b);
          dir[nc] = ib ? 1 : -1;
          ++nc;
        }
      }
      // every entering crossing joins the next leaving one (cuts off the
      // "above" corners between them)
      for (int i = 0; i < nc; ++i) {
        if (dir[i] != 1) continue;
        for (int j = 1; j < nc; ++j) {
          const int k = (i + j) % nc;
          if (dir[k] == -1) {
            next[cross[i]] = cross[k];
            break;
          }
        }
      }
    }
    int nt = 0;
    bool seen[12] = {};
    for (int s = 0; s < 12; ++s) {
      if (next[s] < 0 || seen[s]) continue;
      std::vector<int> loop;
      for (int e = s; !seen[e]; e = next[e]) {
        seen[e] = true;
        loop.push_back(e);
      }
      // the loop runs clockwise about the direction of increasing values:
      // the fan is wound the other way round
      for (size_t i = 1; i + 1 < loop.size() && nt < MC_MAX_TRI; ++i) {
        T.tri[cs][nt][0] = (int8_t)loop[0];
        T.tri[cs][nt][1] = (int8_t)loop[i + 1];
        T.tri[cs][nt][2] = (int8_t)loop[i];
        ++nt;
      }
    }
    T.ntri[cs] = (uint8_t)nt;
  }
  return T;
}

struct McArgs {
  const double* f;
  const uint8_t* mask;
  int64_t nx, ny, nz, np, words;       // points, words of 64 points
  int64_t sx, sy;                      // points from one to the next along x and y
  double level;
  const McTables* T;
  uint64_t *above, *nan, *msk;         // bit of a point: value > level / NaN / mask set
  uint64_t *valid;                     // the cube at the point is meshed
  uint64_t *edge[3];                   // a meshed cube uses the edge from the point along the axis
  uint32_t *vpre, *tpre;               // vertices / triangles of the block's earlier words
  uint32_t *vsum, *tsum;               // vertices / triangles of each block of MC_WORDS words, then of the earlier ones
  uint32_t *total;                     // both, of all words
};

constexpr int MC_WORDS = 256;          // words (threads) per counting block
constexpr int MC_PER_WAVE = 8;         // words a wave packs: that many loads in flight

// One wave per word: lane l looks at point 64 w + l.
__global__ __launch_bounds__(256) void mc_bits_kernel(McArgs a) {
  const int lane = threadIdx.x & 63;
  const uint32_t w0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * MC_PER_WAVE;   // the points of a lattice fit 32 bits
  double v[MC_PER_WAVE];
  uint8_t m[MC_PER_WAVE];
#pragma unroll
  for (int i = 0; i < MC_PER_WAVE; ++i) {
    const int64_t p = (int64_t)(w0 + i) * 64 + lane;
    v[i] = p < a.np ? a.f[p] : a.level;                 // not above, and no cube reaches it
    m[i] = p < a.np && a.mask ? a.mask[p] : 1;
  }
#pragma unroll
  for (int i = 0; i < MC_PER_WAVE; ++i) {
    const uint64_t up = __ballot(v[i] > a.level), nn = __ballot(v[i] != v[i]), mk = __ballot(m[i] != 0);
    if (lane == 0 && w0 + i < a.words) {
      a.above[w0 + i] = up;
      a.nan[w0 + i] = nn;
      a.msk[w0 + i] = mk;
    }
  }
}

// The bits of points 64 i + step + (0 .. 63) and of the points one further
// along z; 0 before the lattice, of no use behind it.
struct McPair { uint64_t at, up; };
__device__ __forceinline__ McPair mc_pair(const McArgs& a, const uint64_t* b, int64_t i, int64_t step) {
  const int64_t j = i + (step >> 6), last = a.words - 1;        // floor, also of a negative step
  const int s = (int)(step & 63);                               // the same for all threads
  const uint64_t w0 = j < 0 ? 0 : b[min(j, last)], w1 = j + 1 < 0 ? 0 : b[min(j + 1, last)];
  McPair r;
  r.at = w0 >> s | w1 << 1 << (63 - s);
  r.up = r.at >> 1 | w1 >> s << 63;
  return r;
}

// Meshed cubes of a word: all corners on the lattice, the mask at the far
// corner (+1, +1, +1), no NaN at any corner.
__global__ __launch_bounds__(256) void mc_valid_kernel(McArgs a) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= a.words) return;
  const uint32_t nx = (uint32_t)a.nx, ny = (uint32_t)a.ny, nz = (uint32_t)a.nz, p = (uint32_t)i * 64, row = p / nz;
  uint32_t z = p - row * nz, x = row / ny, y = row - x * ny;
  uint64_t ok = 0;
  for (uint32_t at = 0; at < 64 && x + 1 < nx;) {       // the rows that reach into the word
    const uint32_t len = min(nz - z, 64 - at), cubes = min(len, nz - 1 - z);
    if (y + 1 < ny) ok |= (cubes < 64 ? (1ull << cubes) - 1 : ~0ull) << at;
    at += len;
    z = 0;
    if (++y == ny) { y = 0; ++x; }
  }
  if (ok) {
    ok &= mc_pair(a, a.msk, i, a.sx + a.sy).up;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const McPair n = mc_pair(a, a.nan, i, (k & 1) * a.sx + (k >> 1) * a.sy);
      ok &= ~(n.at | n.up);
    }
  }
  a.valid[i] = ok;
}

// Case of the cube at bit z of the four rows' words lo (z) and hi (z + 1).
__device__ __forceinline__ int mc_case(const uint64_t* lo, const uint64_t* hi, int z) {
  int cs = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k)
    cs |= (int)((lo[k] >> z) & 1) << k | (int)((hi[k] >> z) & 1) << (k + 4);
  return cs;
}

// The points x + (k & 1), y + (k >> 1) of the cubes of word i, at z and z + 1
// (what lies beyond a row's or the lattice's end belongs to no meshed cube).
__device__ __forceinline__ void mc_corner_words(const McArgs& a, int64_t i, uint64_t* lo, uint64_t* hi) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const McPair p = mc_pair(a, a.above, i, (k & 1) * a.sx + (k >> 1) * a.sy);
    lo[k] = p.at;
    hi[k] = p.up;
  }
}

__device__ __forceinline__ uint64_t mc_active(const uint64_t* lo, const uint64_t* hi, uint64_t valid) {
  const uint64_t any = lo[0] | lo[1] | lo[2] | lo[3] | hi[0] | hi[1] | hi[2] | hi[3];
  const uint64_t all = lo[0] & lo[1] & lo[2] & lo[3] & hi[0] & hi[1] & hi[2] & hi[3];
  return valid & any & ~all;
}

// Inclusive sums over the block's 256 threads of a pair of counts.
__device__ __forceinline__ uint2 block_scan(uint2 v, uint2* s) {
  const int t = threadIdx.x, n = blockDim.x;
  s[t] = v;
  __syncthreads();
  for (int o = 1; o < n; o <<= 1) {
    const uint2 u = t >= o ? s[t - o] : make_uint2(0, 0);
    __syncthreads();
    v.x += u.x;
    v.y += u.y;
    s[t] = v;
    __syncthreads();
  }
  return v;
}

// Used edges of each word, and the counts of the vertices and triangles
// before it in its block.  An edge is used when its ends differ and one of
// the (up to four) cubes around it is meshed.
__global__ __launch_bounds__(MC_WORDS) void mc_count_kernel(McArgs a) {
  __shared__ uint2 s[MC_WORDS];
  const int64_t i = (int64_t)blockIdx.x * MC_WORDS + threadIdx.x;
  uint2 n = make_uint2(0, 0);
  if (i < a.words) {
    uint64_t lo[4], hi[4];
    mc_corner_words(a, i, lo, hi);
    // cubes one back along x, y, both, and each of them one back along z (a
    // step across a row's or the lattice's start meets a cube that is not meshed)
    const McPair c00 = mc_pair(a, a.valid, i, -1), c10 = mc_pair(a, a.valid, i, -a.sx - 1),
                 c01 = mc_pair(a, a.valid, i, -a.sy - 1), c11 = mc_pair(a, a.valid, i, -a.sx - a.sy - 1);
    const uint64_t v00 = c00.up, v10 = c10.up, v01 = c01.up, v11 = c11.up, d00 = c00.at, d10 = c10.at, d01 = c01.at;
    const uint64_t e0 = (lo[0] ^ lo[1]) & (v00 | d00 | v01 | d01);
    const uint64_t e1 = (lo[0] ^ lo[2]) & (v00 | d00 | v10 | d10);
    const uint64_t e2 = (lo[0] ^ hi[0]) & (v00 | v10 | v01 | v11);
    a.edge[0][i] = e0;
    a.edge[1][i] = e1;
    a.edge[2][i] = e2;
    n.x = __popcll(e0) + __popcll(e1) + __popcll(e2);
    for (uint64_t left = mc_active(lo, hi, v00); left; left &= left - 1)
      n.y += a.T->ntri[mc_case(lo, hi, __ffsll((unsigned long long)left) - 1)];
  }
  const uint2 sum = block_scan(n, s);
  if (i < a.words) {
    a.vpre[i] = sum.x - n.x;
    a.tpre[i] = sum.y - n.y;
  }
  if (threadIdx.x == MC_WORDS - 1) {
    a.vsum[blockIdx.x] = sum.x;
    a.tsum[blockIdx.x] = sum.y;
  }
}

// Block sums to sums over the earlier blocks (one workgroup); the totals go
// to device memory, for the writing pass, and to the caller's pinned pair.
__global__ __launch_bounds__(1024) void mc_scan_kernel(McArgs a, int64_t nb, uint32_t* host) {
  __shared__ uint2 s[1024];
  const int64_t per = (nb + 1023) / 1024;
  const int64_t b0 = threadIdx.x * per, b1 = b0 + per < nb ? b0 + per : nb;
  uint2 acc = make_uint2(0, 0);
  for (int64_t i = b0; i < b1; ++i) { acc.x += a.vsum[i]; acc.y += a.tsum[i]; }
  const uint2 sum = block_scan(acc, s);
  uint2 run = make_uint2(sum.x - acc.x, sum.y - acc.y);
  for (int64_t i = b0; i < b1; ++i) {
    const uint32_t v = a.vsum[i], t = a.tsum[i];
    a.vsum[i] = run.x;
    a.tsum[i] = run.y;
    run.x += v;
    run.y += t;
  }
  if (threadIdx.x == 1023) {
    a.total[0] = host[0] = sum.x;
    a.total[1] = host[1] = sum.y;
  }
}

// Vertex of the edge from point p along axis: vertices are numbered by point, then axis.
__device__ __forceinline__ uint32_t mc_vertex(const McArgs& a, int64_t p, int axis) {
  const int64_t i = p >> 6;
  const int b = (int)(p & 63);
  const uint64_t e0 = a.edge[0][i], e1 = a.edge[1][i], e2 = a.edge[2][i], below = (1ull << b) - 1;
  uint32_t id = a.vsum[i / MC_WORDS] + a.vpre[i] + __popcll(e0 & below) + __popcll(e1 & below) + __popcll(e2 & below);
  if (axis > 0) id += (uint32_t)(e0 >> b) & 1u;
  if (axis > 1) id += (uint32_t)(e1 >> b) & 1u;
  return id;
}

// Writes the vertices and the triangles of EMIT words.  Both are few (a
// crossed word holds a handful) and reached through chains of dependent loads,
// so a block first lists them in LDS, LANES threads per word, and then gives
// every vertex and every triangle corner a thread of its own: as one lane per
// point, almost all idle, this pass took 75 us of 132 at 200^3, and takes 32 us
// now.  Up to MC_SMALL words the blocks alone decide, and they take 2 words
// (65^3 points, all of them crossed: the call 59 us, 70 with 16 words; 100^3,
// one surface: 45 and 38).  Writes nothing when the results exceed the caller's
// buffers.
constexpr int MC_SMALL = 4800;
template <int EMIT, int LANES>
__global__ __launch_bounds__(EMIT * LANES) void mc_emit_kernel(McArgs a, double ox, double oy, double oz,
                                                             double hx, double hy, double hz, double* verts,
                                                             int64_t max_verts, int32_t* faces, int64_t max_faces) {
  constexpr int BITS = 64 / LANES;                       // bits of a word per thread
  static_assert(MC_WORDS % EMIT == 0, "the words of a writing block lie in one counting block");
  __shared__ uint32_t list[EMIT * 64 * MC_MAX_TRI];      // vertices (at most 3 a point), then triangles
  __shared__ uint32_t count[2];
  if (a.total[0] > max_verts || a.total[1] > max_faces) return;
  const uint32_t t = threadIdx.x, w0 = blockIdx.x * EMIT, i = w0 + t / LANES;
  const int z0 = BITS * (int)(t % LANES);
  const bool live = i < a.words;
  // the first vertex and triangle of the block's words (one counting block holds them all)
  const uint32_t vbase = a.vsum[w0 / MC_WORDS] + a.vpre[w0], tbase = a.tsum[w0 / MC_WORDS] + a.tpre[w0];
  if (t < 2) count[t] = 0;
  __syncthreads();
  uint64_t e[3] = {0, 0, 0};
  uint32_t n = 0;
  if (live) {
#pragma unroll
    for (int u = 0; u < 3; ++u) {
      e[u] = a.edge[u][i];
      n += __popcll(e[u]);
    }
    uint32_t at = a.vpre[i] - a.vpre[w0];
    if (z0 == 0 && n) atomicMax(&count[0], at + n);
    const uint64_t below = (1ull << z0) - 1;
#pragma unroll
    for (int u = 0; u < 3; ++u) at += __popcll(e[u] & below);
#pragma unroll
    for (int z = z0; z < z0 + BITS; ++z)
#pragma unroll
      for (uint32_t u = 0; u < 3; ++u)
        if ((e[u] >> z) & 1) list[at++] = (i - w0) << 8 | (uint32_t)z << 2 | u;
  }
  __syncthreads();
  for (uint32_t k = t; k < count[0]; k += EMIT * LANES) {
    const uint32_t r = list[k], axis = r & 3, j = w0 + (r >> 8);
    const uint32_t p = j * 64 + ((r >> 2) & 63), row = p / (uint32_t)a.nz, z = p - row * (uint32_t)a.nz;
    const uint32_t x = row / (uint32_t)a.ny, y = row - x * (uint32_t)a.ny;
    const double v0 = a.f[p], v1 = a.f[p + (axis == 0 ? a.sx : (axis == 1 ? a.sy : 1))];
    const double s = (a.level - v0) / (v1 - v0);
    double P[3] = {(double)x, (double)y, (double)z};
#pragma unroll
    for (uint32_t u = 0; u < 3; ++u)
      if (u == axis) P[u] += s;
    double* o = verts + 3 * (int64_t)(vbase + k);
    o[0] = ox + P[0] * hx;
    o[1] = oy + P[1] * hy;
    o[2] = oz + P[2] * hz;
  }
  __syncthreads();
  int cs[BITS] = {};
  uint32_t nt = 0;
  if (live) {
    uint64_t lo[4], hi[4];
    mc_corner_words(a, i, lo, hi);
    const uint64_t act = mc_active(lo, hi, a.valid[i]);
#pragma unroll
    for (int b = 0; b < BITS; ++b)
      if ((act >> (z0 + b)) & 1) {
        cs[b] = mc_case(lo, hi, z0 + b);
        nt += a.T->ntri[cs[b]];
      }
  }
  uint32_t sum = nt;                     // of the word's threads up to this one
#pragma unroll
  for (int o = 1; o < LANES; o <<= 1) {
    const uint32_t v = __shfl_up(sum, o, LANES);
    if ((int)(t % LANES) >= o) sum += v;
  }
  if (live) {
    uint32_t at = a.tpre[i] - a.tpre[w0] + sum - nt;
    if (nt) atomicMax(&count[1], at + nt);
#pragma unroll
    for (int b = 0; b < BITS; ++b)
      if (cs[b])
        for (uint32_t q = 0; q < a.T->ntri[cs[b]]; ++q)
          list[at++] = (i - w0) << 17 | (uint32_t)(z0 + b) << 11 | (uint32_t)cs[b] << 3 | q;
  }
  __syncthreads();
  for (uint32_t k = t; k < 3 * count[1]; k += EMIT * LANES) {
    const uint32_t r = list[k / 3], j = w0 + (r >> 17);
    const int le = a.T->tri[(r >> 3) & 255][r & 7][k % 3], axis = le >> 2, q = le & 3;
    // the edge's start from the cube's corner: q's bits go to the other axes in order
    const int dx = axis == 0 ? 0 : q & 1, dy = axis == 1 ? 0 : (axis == 0 ? q & 1 : q >> 1),
              dz = axis == 2 ? 0 : q >> 1;
    const int64_t p = (int64_t)j * 64 + ((r >> 11) & 63) + dx * a.sx + dy * a.sy + dz;
    faces[3 * (int64_t)tbase + k] = (int32_t)mc_vertex(a, p, axis);
  }
}

}  // namespace

extern "C" int gk_marching_cubes(gk_handle h, const double* field, const int64_t* res, const uint8_t* mask,
                                 double level, const double* origin, const double* spacing, double* verts,
                                 int64_t max_verts, int32_t* faces, int64_t max_faces, int64_t* n_verts,
                                 int64_t* n_faces, gk_stream stream) {
  GK_REQUIRE(h && field && res && origin && spacing && n_verts && n_faces, GK_ERR_ARG,
             "gk_marching_cubes: NULL argument");
  const int64_t nx = res[0], ny = res[1], nz = res[2];
  GK_REQUIRE(nx >= 1 && ny >= 1 && nz >= 1, GK_ERR_ARG, "gk_marching_cubes: bad resolution");
  const int64_t np_ = nx * ny * nz;
  GK_REQUIRE(3 * np_ < (int64_t)UINT32_MAX, GK_ERR_ARG, "gk_marching_cubes: lattice too large");
  *n_verts = 0;
  *n_faces = 0;
  if (nx < 2 || ny < 2 || nz < 2) return GK_OK;
  hipStream_t st = (hipStream_t)stream;
  const int64_t words = gk_ceil_div(np_, 64), nb = gk_ceil_div(words, MC_WORDS);
  // workspace: totals | 7 word arrays | 2 counts per word | 2 sums per block
  size_t need = 0;
  auto take = [&](size_t bytes) { size_t o = need; need += gk_round_up(bytes, 256); return o; };
  const size_t o_tot = take(16);
  size_t o_w[7], o_n[4];
  for (size_t& o : o_w) o = take(words * 8);
  for (int k = 0; k < 4; ++k) o_n[k] = take((k < 2 ? words : nb) * 4);
  void* p = nullptr;
  GK_TRY(gk_workspace(h, WS_MESH, need, &p));
  char* b = static_cast<char*>(p);
  // The tables, once per handle, in memory of their own: a workspace that
  // grows may come back at the same address without its contents.
  if (!h->mesh_tables) {
    static const McTables host = build_tables();
    void* t = nullptr;
    GK_HIP(hipMalloc(&t, sizeof(McTables)));
    if (hipMemcpyAsync(t, &host, sizeof(McTables), hipMemcpyHostToDevice, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess) {
      (void)hipFree(t);
      GK_REQUIRE(false, GK_ERR_HIP, "gk_marching_cubes: the case tables could not be copied to the device");
    }
    h->mesh_tables = t;
  }
  if (!h->mesh_counts) GK_HIP(hipHostMalloc(reinterpret_cast<void**>(&h->mesh_counts), 64, hipHostMallocDefault));
  McArgs a{};
  a.f = field; a.mask = mask;
  a.nx = nx; a.ny = ny; a.nz = nz; a.np = np_; a.words = words;
  a.sx = ny * nz; a.sy = nz;
  a.level = level;
  a.T = static_cast<const McTables*>(h->mesh_tables);
  uint64_t** wp[7] = {&a.above, &a.nan, &a.msk, &a.valid, &a.edge[0], &a.edge[1], &a.edge[2]};
  for (int k = 0; k < 7; ++k) *wp[k] = reinterpret_cast<uint64_t*>(b + o_w[k]);
  uint32_t** np[4] = {&a.vpre, &a.tpre, &a.vsum, &a.tsum};
  for (int k = 0; k < 4; ++k) *np[k] = reinterpret_cast<uint32_t*>(b + o_n[k]);
  a.total = reinterpret_cast<uint32_t*>(b + o_tot);
  hipLaunchKernelGGL(mc_bits_kernel, dim3((unsigned)gk_ceil_div(words, 4 * MC_PER_WAVE)), dim3(256), 0, st, a);
  hipLaunchKernelGGL(mc_valid_kernel, dim3((unsigned)gk_ceil_div(words, 256)), dim3(256), 0, st, a);
  hipLaunchKernelGGL(mc_count_kernel, dim3((unsigned)nb), dim3(MC_WORDS), 0, st, a);
  hipLaunchKernelGGL(mc_scan_kernel, dim3(1), dim3(1024), 0, st, a, nb, h->mesh_counts);
  if (verts && faces) {
    auto emit = [&](auto kernel, int per, int threads) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)gk_ceil_div(words, per)), dim3(threads), 0, st, a, origin[0], origin[1],
                         origin[2], spacing[0], spacing[1], spacing[2], verts, max_verts, faces, max_faces);
    };
    if (words <= MC_SMALL) emit(mc_emit_kernel<2, 64>, 2, 128);
    else emit(mc_emit_kernel<16, 16>, 16, 256);
  }
  GK_HIP(hipGetLastError());
  GK_HIP(hipStreamSynchronize(st));
  const uint32_t counts[2] = {h->mesh_counts[0], h->mesh_counts[1]};
  *n_verts = counts[0];
  *n_faces = counts[1];
  if (!verts || !faces) return GK_OK;
  GK_REQUIRE(counts[0] <= max_verts && counts[1] <= max_faces, GK_ERR_ARG,
             "gk_marching_cubes: %u vertices / %u faces exceed the output capacity (%lld / %lld)", counts[0],
             counts[1], (long long)max_verts, (long long)max_faces);
  return GK_OK;
}
