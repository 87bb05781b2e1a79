// Exact point-mesh distance through a tree over the triangles, for the
// distance-map builder and the free-point signed distance.
//
// The results are those of the brute force over all triangles (k_mesh_sdf,
// distmap.hip), bit for bit:
//  - Distance and closest point.  Every triangle that can hold the smallest
//    computed squared distance goes through the same point_triangle_dist2;
//    among equal values the lowest triangle number wins, as the first one
//    does in the brute force.  A box is left out only when its distance
//    exceeds the best one by more than the rounding of both: the computed
//    closest point lies on the triangle up to a few roundings of the
//    coordinates (its barycentric weights are in [0, 1] in every region, or
//    NaN, which never wins), so the margin delta is 256 roundings of the
//    largest coordinate.
//  - Sign.  For a closed, consistently oriented mesh the winding number is
//    an integer away from the surface, and equal to the signed count of the
//    triangles a ray crosses (ray_cover, plane_side: mesh_distance.hpp).
//    Where rounding could decide it, on the surface or in a triangle's
//    plane, the brute force's own sum of solid angles is taken, in its
//    order.  Other meshes stay with the brute force (mesh_closed).
//
// Layout: triangles sorted along a Hilbert curve through their centroids,
// eight consecutive ones to a group, groups of groups above; no topology to
// build and no pointers, and a node's eight child boxes are 192 consecutive
// bytes, so one visit is twelve 16-byte loads in flight together (the traversal is
// a chain of dependent loads; wide nodes make it short).
#include "mesh_tree.hpp"

#include <cfloat>

#include "fc_internal.hpp"
#include "mesh_distance.hpp"

namespace fc {

namespace {

constexpr int kBlock = 256;
constexpr uint32_t kInfoBlocks = 64;
// Free points are sorted and taken this many at a time (bounds the scratch).
constexpr uint64_t kPointChunk = 1ull << 22;
// Fewer points share a wave (down to 8) until there are this many waves, four
// per SIMD: a wave's walk is a chain of dependent steps, longer the further
// apart its points lie.
constexpr uint32_t kPointWaves = 4096;

__device__ __forceinline__ unsigned long long mesh_key(double d) {
  const unsigned long long u = (unsigned long long)__double_as_longlong(d);
  return (u >> 63) ? ~u : (u | 0x8000000000000000ull);
}

// Finalizer of SplitMix64 (Steele, Lea, Flood 2014).
__device__ __forceinline__ unsigned long long mix64(unsigned long long z) {
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

__global__ void k_mesh_info_init(MeshInfo* I) {
  if (threadIdx.x < 3) {
    I->lo[threadIdx.x] = ~0ull;
    I->hi[threadIdx.x] = 0ull;
  }
  if (threadIdx.x < 2) I->edges[threadIdx.x] = 0ull;
  if (threadIdx.x == 0) I->bad = I->open = 0u;
}

__device__ __forceinline__ void load_corners(const double* __restrict__ verts, uint32_t nv,
                                             const uint32_t* __restrict__ tris, uint32_t t,
                                             double* v, uint32_t* vi) {
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    uint32_t i = tris[3 * (size_t)t + k];
    if (i >= nv) i = nv - 1;  // as the brute force reads it
    vi[k] = i;
#pragma unroll
    for (int a = 0; a < 3; ++a) v[3 * k + a] = verts[3 * (size_t)i + a];
  }
}

// At most kInfoBlocks blocks and one set of atomics a block, as all of them
// meet in one cache line, 10 ns each (6,144 triangles: 12.3 us with a set a
// wave, 5.0 with this).
__global__ __launch_bounds__(kBlock) void k_mesh_info(const double* __restrict__ verts,
                                                      uint32_t nv,
                                                      const uint32_t* __restrict__ tris,
                                                      uint32_t nt, MeshInfo* __restrict__ I) {
  __shared__ unsigned long long s_part[kBlock / 64][8];
  double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
  unsigned long long e0 = 0, e1 = 0;
  bool bad = false;
  for (uint32_t t = blockIdx.x * kBlock + threadIdx.x; t < nt; t += gridDim.x * kBlock) {
    double v[9];
    uint32_t vi[3];
    load_corners(verts, nv, tris, t, v, vi);
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      bad = bad || !(fabs(v[k]) <= DBL_MAX);
      lo[k % 3] = fmin(lo[k % 3], v[k]);
      hi[k % 3] = fmax(hi[k % 3], v[k]);
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const uint32_t a = vi[k], b = vi[(k + 1) % 3];
      const unsigned long long e =
          a < b ? ((unsigned long long)a << 32 | b) : ((unsigned long long)b << 32 | a);
      const unsigned long long h0 = mix64(e + 0x9E3779B97F4A7C15ull);
      const unsigned long long h1 = mix64(e ^ 0xD1B54A32D192ED03ull);
      if (a < b) {
        e0 += h0;
        e1 += h1;
      } else if (a > b) {
        e0 -= h0;
        e1 -= h1;
      }
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      lo[a] = fmin(lo[a], __shfl_xor(lo[a], off));
      hi[a] = fmax(hi[a], __shfl_xor(hi[a], off));
    }
    e0 += __shfl_xor(e0, off);
    e1 += __shfl_xor(e1, off);
  }
  const uint32_t w = threadIdx.x >> 6, lane = threadIdx.x & 63u;
  if (lane == 0u) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      s_part[w][a] = mesh_key(lo[a]);
      s_part[w][3 + a] = mesh_key(hi[a]);
    }
    s_part[w][6] = e0;
    s_part[w][7] = e1;
  }
  const bool anyBad = __syncthreads_or(bad ? 1 : 0) != 0;
  if (threadIdx.x < 8u) {
    unsigned long long r = s_part[0][threadIdx.x];
#pragma unroll
    for (int u = 1; u < kBlock / 64; ++u) {
      const unsigned long long o = s_part[u][threadIdx.x];
      r = threadIdx.x < 3u ? (o < r ? o : r) : (threadIdx.x < 6u ? (o > r ? o : r) : r + o);
    }
    if (threadIdx.x < 3u)
      atomicMin(&I->lo[threadIdx.x], r);
    else if (threadIdx.x < 6u)
      atomicMax(&I->hi[threadIdx.x - 3u], r);
    else
      atomicAdd(&I->edges[threadIdx.x - 6u], r);
    if (threadIdx.x == 0u && anyBad) atomicOr(&I->bad, 1u);
  }
}

// Place of a cell of a 256^3 grid along a Hilbert curve, by the coordinate
// transform of J. Skilling, "Programming the Hilbert curve" (AIP Conference
// Proceedings 707, 2004).  Neighbours along the curve are neighbours in space;
// in Morton order a group of eight may straddle one of its jumps, and a wave
// of the search below then visits a quarter more of them (64 against 52 nodes
// for 6,144 triangles; the lattice's search 354 against 287 us, that of
// 65,536 free points 353 against 236 us).
__device__ __forceinline__ uint32_t hilbert_key(uint32_t x, uint32_t y, uint32_t z) {
  uint32_t v[3] = {x, y, z};
#pragma unroll
  for (uint32_t bit = 128u; bit > 1u; bit >>= 1) {
    const uint32_t low = bit - 1u;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const uint32_t swap = (v[0] ^ v[a]) & low;
      const bool set = (v[a] & bit) != 0u;
      v[0] ^= set ? low : swap;  // (for a = 0 the swap is of nothing)
      if (a > 0) v[a] ^= set ? 0u : swap;
    }
  }
  v[1] ^= v[0];
  v[2] ^= v[1];
  uint32_t t = 0;
#pragma unroll
  for (uint32_t bit = 128u; bit > 1u; bit >>= 1) t ^= (v[2] & bit) ? bit - 1u : 0u;
  uint32_t key = 0;
#pragma unroll
  for (int k = 7; k >= 0; --k)
#pragma unroll
    for (int a = 0; a < 3; ++a) key = key << 1 | (((v[a] ^ t) >> k) & 1u);
  return key;
}

constexpr int kOrderBits = 24;

// Bits of the key that order nt triangles: the first five levels of the curve
// where they leave two or three of a mesh's triangles to a cell, which saves a
// pass of the sort (9 us; 6,144 triangles: 52.1 instead of 52.0 nodes visited).
inline int mesh_order_bits(uint32_t nt) { return nt <= (1u << 14) ? 15 : kOrderBits; }

__global__ __launch_bounds__(kBlock) void k_mesh_order(const double* __restrict__ verts,
                                                        uint32_t nv,
                                                        const uint32_t* __restrict__ tris,
                                                        uint32_t nt, MeshInfo* __restrict__ I,
                                                        int bits, uint32_t* __restrict__ keys) {
  const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
  // An open mesh is left to the brute force: the sorts and searches that follow
  // end at once (131 triangles, 200 points: 173 us a call with the whole tree
  // built in vain, 143 so; 65,536 points 198 and 155).
  if (t == 0 && !mesh_closed(*I)) I->open = 1u;
  if (t >= nt) return;
  double v[9];
  uint32_t vi[3];
  load_corners(verts, nv, tris, t, v, vi);
  uint32_t at[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const double lo = mesh_key_value(I->lo[a]), hi = mesh_key_value(I->hi[a]);
    const double c = (v[a] + v[3 + a] + v[6 + a]) * (1.0 / 3.0);
    // any value orders the triangles (a NaN reads 0)
    at[a] = (uint32_t)fmin(fmax((c - lo) / (hi - lo) * 256.0, 0.0), 255.0);
  }
  keys[t] = hilbert_key(at[0], at[1], at[2]) >> (kOrderBits - bits);
}

__device__ __forceinline__ uint32_t box_at(uint32_t node) {
  return (node >> 3) * 48u + (node & 7u);
}

// Triangles in sorted order with their boxes; the last group's spare boxes
// are never reached (count), but are written so that they hold no garbage.
__global__ __launch_bounds__(kBlock) void k_tree_leaves(const double* __restrict__ verts,
                                                        uint32_t nv,
                                                        const uint32_t* __restrict__ tris,
                                                        uint32_t nt,
                                                        const uint32_t* __restrict__ order,
                                                        TreeTri* __restrict__ tri,
                                                        float* __restrict__ box) {
  const uint32_t p = blockIdx.x * kBlock + threadIdx.x;
  if (p >= ((nt + 7u) & ~7u)) return;
  float* b = box + box_at(p);
  if (p >= nt) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      b[8 * a] = INFINITY;
      b[24 + 8 * a] = -INFINITY;
    }
    return;
  }
  TreeTri T;
  uint32_t vi[3];
  const uint32_t t = min(order[p], nt - 1u);  // (an open mesh's was not written)
  load_corners(verts, nv, tris, t, T.v, vi);
  T.id = t;
  tri[p] = T;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    b[8 * a] = __double2float_rd(fmin(T.v[a], fmin(T.v[3 + a], T.v[6 + a])));
    b[24 + 8 * a] = __double2float_ru(fmax(T.v[a], fmax(T.v[3 + a], T.v[6 + a])));
  }
}

struct TreeBuild {
  float* box[kTreeMaxLevels];
  uint32_t count[kTreeMaxLevels];
  int levels;
};

// The levels above the triangles, in one block (8192 boxes of level 1 for
// 65,536 triangles; a launch per level costs more).
__global__ __launch_bounds__(1024) void k_tree_levels(TreeBuild B) {
  for (int l = 1; l < B.levels; ++l) {
    const uint32_t cnt = B.count[l];
    for (uint32_t i = threadIdx.x; i < ((cnt + 7u) & ~7u); i += 1024u) {
      float* o = B.box[l] + box_at(i);
      const float* c = B.box[l - 1] + (size_t)i * 48u;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        float lo = INFINITY, hi = -INFINITY;
        if (i < cnt) {
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            lo = fminf(lo, c[8 * a + u]);
            hi = fmaxf(hi, c[24 + 8 * a + u]);
          }
        }
        o[8 * a] = lo;
        o[24 + 8 * a] = hi;
      }
    }
    __syncthreads();
  }
}

// Read-only memory at a wave-uniform address, through the scalar cache into
// scalar registers (the tree is written by earlier launches only).
template <typename E>
using Uniform = const E __attribute__((address_space(4)))*;
template <typename E>
__device__ __forceinline__ Uniform<E> uniform(const E* p) {
  return reinterpret_cast<Uniform<E>>(reinterpret_cast<uintptr_t>(p));
}

// The brute force's winding sum, in its order, for the lanes that `need` it,
// one such lane's point at a time: the wave takes 64 triangles' solid angles
// together and adds them one by one.
__device__ __forceinline__ double winding_sum(bool need, const double q[3],
                                              const double* __restrict__ verts, uint32_t nv,
                                              const uint32_t* __restrict__ tris, uint32_t nt) {
  const uint32_t lane = threadIdx.x & 63u;
  double mine = 0.0;
  uint64_t todo = __ballot(need);
  while (todo) {
    const int who = __ffsll((unsigned long long)todo) - 1;
    todo &= todo - 1ull;
    double p[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) p[a] = __shfl(q[a], who);
    double w = 0.0;
    for (uint32_t t0 = 0; t0 < nt; t0 += 64u) {
      const uint32_t cnt = nt - t0 < 64u ? nt - t0 : 64u;
      double sa = 0.0;
      if (lane < cnt) {
        double v[9];
        uint32_t vi[3];
        load_corners(verts, nv, tris, t0 + lane, v, vi);
        sa = solid_angle(p, v, v + 3, v + 6);
      }
      for (uint32_t j = 0; j < cnt; ++j) w += __shfl(sa, (int)j);
    }
    if ((int)lane == who) mine = w;
  }
  return mine;
}

__device__ __forceinline__ bool winds(double w) { return w / (4.0 * 3.14159265358979323846) > 0.5; }

// The closest triangles of a wave's 64 points, one per lane, found together.
// The points are neighbours, so the wave walks the tree once for all of them:
// a box is entered when any lane has to look into it, nearest first as seen
// from one lane, and its eight children's bounds are read once (uniform
// loads).  What a lane still has to test exactly, the triangles whose box is
// within its best distance and of which some corner lies in front of the
// plane through its best point (every point closer than that is), goes to a
// list of (lane, triangle) pairs that the wave takes 64 at a time, so that
// point_triangle_dist2, 300 instructions of binary64, runs with all lanes.
//
// Bound by issue: a wave takes about 52 boxes of eight, 60 triangles and 20
// rounds of pairs.  274,625 lattice points against 6,144 triangles: a search
// per lane, diverging at every step, took 1.02 ms; this 0.29 ms.
constexpr int kLanes = 64;  // one wave per block

// (4 waves per SIMD at 108 VGPRs: 598 us a build against 578, in Morton order)
constexpr int kTreeWavesPerSimd = 5;

struct TreeShared {
  double q[3][kLanes];
  double cp[3][kLanes];
  unsigned long long d2[kLanes];
  uint32_t id[kLanes];
  uint32_t pair[2 * kLanes];  // lane << 26 | triangle in tree order
  float lb[8][kLanes];
};

struct Nearest {
  double d2 = DBL_MAX;
  uint32_t id = 0xffffffffu;
  double cp[3] = {0.0, 0.0, 0.0};
};

__device__ __forceinline__ void tree_nearest(const MeshTree& T, const double q[3], double delta,
                                             bool active, int centre, uint32_t lanes,
                                             TreeShared& S, Nearest& best) {
  const int lane = (int)(threadIdx.x & 63u);
  float qf[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    qf[a] = (float)q[a];
    S.q[a][lane] = q[a];
  }
  S.d2[lane] = (unsigned long long)__double_as_longlong(best.d2);
  // (sqrt(d2) + delta)^2, with room for the float rounding of the boxes'
  // distances (2^-20 of the largest coordinate: delta is 2^-44 of it): a box
  // at least this far holds no winner
  const double deltaF = delta * 0x1p24;
  float limit = active ? FLT_MAX : -1.0f;
  // unit vector to the best point (0 before there is one), and where the
  // plane with this normal is too far: u . q + sqrt(d2) + delta
  double u[3] = {0.0, 0.0, 0.0}, front = INFINITY;
  uint32_t pairs = 0;
  // (fewer lanes test sooner, so that their bounds do not lag)
  const uint32_t full = min(2u * lanes, 64u);

  // Takes up to 64 pairs from the front of the list.
  auto test_pairs = [&]() {
    __syncthreads();
    const uint32_t cnt = pairs < 64u ? pairs : 64u;
    const bool on = (uint32_t)lane < cnt;
    const uint32_t e = S.pair[lane], l = on ? e >> 26 : 0u, at = on ? e & 0x03ffffffu : 0u;
    double p[3], c[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) p[a] = S.q[a][l];
    const TreeTri& R = T.tri[at];
    const uint32_t id = (uint32_t)R.id;
    const double d2 = point_triangle_dist2(p, R.v, R.v + 3, R.v + 6, c);
    // squared distances are not negative: their bits order as they do (a
    // NaN's above all of them)
    const unsigned long long key = (unsigned long long)__double_as_longlong(d2);
    if (on) atomicMin(&S.d2[l], key);
    __syncthreads();
    const unsigned long long mine = S.d2[lane];
    const bool closer = mine < (unsigned long long)__double_as_longlong(best.d2);
    S.id[lane] = closer ? 0xffffffffu : best.id;
    __syncthreads();
    const bool least = on && key == S.d2[l];
    if (least) atomicMin(&S.id[l], id);
    __syncthreads();
    if (least && S.id[l] == id) {
#pragma unroll
      for (int a = 0; a < 3; ++a) S.cp[a][l] = c[a];
    }
    __syncthreads();
    if (closer || S.id[lane] != best.id) {
      best.d2 = __longlong_as_double((long long)mine);
      best.id = S.id[lane];
#pragma unroll
      for (int a = 0; a < 3; ++a) best.cp[a] = S.cp[a][lane];
      const double dist = sqrt(best.d2), r = dist + delta, rf = dist + deltaF;
      limit = __double2float_ru(rf * rf * (1.0 + 0x1p-20));
      // (a little short of one, so that no rounding makes it longer)
      const double inv = dist > 0.0 ? (1.0 - 1e-12) / dist : 0.0;
      front = r;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        u[a] = (best.cp[a] - q[a]) * inv;
        front += u[a] * q[a];
      }
    }
    // what is left moves to the front
    const uint32_t rest = pairs - cnt;
    const uint32_t next = (uint32_t)lane < rest ? S.pair[64 + lane] : 0u;
    __syncthreads();
    if ((uint32_t)lane < rest) S.pair[lane] = next;
    pairs = rest;
  };

  // Lane L keeps level L's boxes still to be entered: three bits each, the
  // nearest lowest, and their number from bit 24 on.
  uint32_t todo = 0;
  int level = T.levels - 1;
  uint32_t group = 0;
  while (true) {
    // ---- the eight boxes of a group
    const Uniform<float> b = uniform(T.box[level] + (size_t)group * 48u);
    float lb[8] = {};
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const float d = fmaxf(fmaxf(b[8 * a + c] - qf[a], qf[a] - b[24 + 8 * a + c]), 0.0f);
        lb[c] = fmaf(d, d, lb[c]);
      }
    // the boxes some lane has to look into (a group's spare boxes are inside
    // out, infinitely far), and their distances from the centre lane
    uint32_t open = 0, key[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const uint32_t any = __ballot(!(lb[c] > limit)) != 0ull ? 1u : 0u;
      open |= any << c;
      // (the distance's sign bit is clear: its bits order as it does)
      const uint32_t at =
          ((uint32_t)__builtin_amdgcn_readlane(__float_as_int(lb[c]), centre) & ~7u) | (uint32_t)c;
      key[c] = any ? at : 0xffffffffu;
    }
    if (level == 0) {
#pragma unroll
      for (int c = 0; c < 8; ++c) S.lb[c][lane] = lb[c];
#pragma unroll 1
      for (uint32_t left = open; left != 0u; left &= left - 1u) {
        const uint32_t c = (uint32_t)__ffs((int)left) - 1u;
        const float x = S.lb[c][lane];
        if (__ballot(!(x > limit)) == 0ull) continue;
        const uint32_t at = group * 8u + c;
        const Uniform<double> v = uniform(T.tri[at].v);
        double s[3];
#pragma unroll
        for (int k = 0; k < 3; ++k)
          s[k] = fma(u[2], v[3 * k + 2], fma(u[1], v[3 * k + 1], u[0] * v[3 * k]));
        const bool test = !(x > limit) && !(fmin(s[0], fmin(s[1], s[2])) > front);
        const uint64_t m = __ballot(test);
        if (test)
          S.pair[pairs + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] =
              ((uint32_t)lane << 26) | at;
        pairs += (uint32_t)__popcll(m);
        if (pairs >= full) test_pairs();
      }
    } else {
      // nearest first (a network of 19 exchanges)
      constexpr int kNet[19][2] = {{0, 1}, {2, 3}, {4, 5}, {6, 7}, {0, 2}, {1, 3}, {4, 6},
                                   {5, 7}, {1, 2}, {5, 6}, {0, 4}, {3, 7}, {1, 5}, {2, 6},
                                   {1, 4}, {3, 6}, {2, 4}, {3, 5}, {3, 4}};
#pragma unroll
      for (int x = 0; x < 19; ++x) {
        const uint32_t lo = min(key[kNet[x][0]], key[kNet[x][1]]);
        const uint32_t hi = max(key[kNet[x][0]], key[kNet[x][1]]);
        key[kNet[x][0]] = lo;
        key[kNet[x][1]] = hi;
      }
      uint32_t word = (uint32_t)__popc(open) << 24;
#pragma unroll
      for (int c = 0; c < 8; ++c) word |= (key[c] & 7u) << (3 * c);
      if (lane == level) todo = word;
    }
    // ---- the next group: a box still to be entered, on this level or above
    uint32_t word = level == 0 ? 0u : (uint32_t)__builtin_amdgcn_readlane((int)todo, level);
    while ((word >> 24) == 0u) {
      group >>= 3;
      if (++level >= T.levels) break;
      word = (uint32_t)__builtin_amdgcn_readlane((int)todo, level);
    }
    if (level >= T.levels) break;
    if (lane == level) todo = (((word >> 24) - 1u) << 24) | ((word & 0xffffffu) >> 3);
    group = group * 8u + (word & 7u);
    --level;
  }
  while (pairs > 0u) test_pairs();
}

// The brute force's search for the lanes that `need` it (points beyond the
// float range that the tree's boxes are compared in), one such lane's point
// at a time, the wave over the triangles.
__device__ __forceinline__ void brute_nearest(bool need, const double q[3],
                                              const double* __restrict__ verts, uint32_t nv,
                                              const uint32_t* __restrict__ tris, uint32_t nt,
                                              Nearest& best) {
  const uint32_t lane = threadIdx.x & 63u;
  for (uint64_t todo = __ballot(need); todo != 0ull; todo &= todo - 1ull) {
    const int who = __ffsll((unsigned long long)todo) - 1;
    const double p[3] = {__shfl(q[0], who), __shfl(q[1], who), __shfl(q[2], who)};
    Nearest r;
    for (uint32_t t = lane; t < nt; t += 64u) {
      double v[9], c[3];
      uint32_t vi[3];
      load_corners(verts, nv, tris, t, v, vi);
      const double d2 = point_triangle_dist2(p, v, v + 3, v + 6, c);
      if (d2 < r.d2) {
        r.d2 = d2;
        r.id = t;
        r.cp[0] = c[0];
        r.cp[1] = c[1];
        r.cp[2] = c[2];
      }
    }
    for (int off = 32; off > 0; off >>= 1) {
      const double d2 = __shfl_xor(r.d2, off);
      const uint32_t id = (uint32_t)__shfl_xor((int)r.id, off);
      const double c[3] = {__shfl_xor(r.cp[0], off), __shfl_xor(r.cp[1], off),
                           __shfl_xor(r.cp[2], off)};
      if (d2 < r.d2 || (d2 == r.d2 && id < r.id)) {
        r.d2 = d2;
        r.id = id;
        r.cp[0] = c[0];
        r.cp[1] = c[1];
        r.cp[2] = c[2];
      }
    }
    if ((int)lane == who) best = r;
  }
}

__device__ __forceinline__ double rounding_margin(const MeshInfo& I, const double q[3]) {
  const double m = mesh_magnitude(I) + fmax(fabs(q[0]), fmax(fabs(q[1]), fabs(q[2])));
  return 256.0 * 2.220446049250313e-16 * m;
}

// The triangles whose boxes a ray from (x, y, z) along +x meets, 64 boxes (two
// levels of the tree) a step, one per lane: leaf(in, t) is called by the whole
// wave with up to 64 of them, lane by lane (`in`: the lane has one, number t
// in tree order).
template <class Leaf>
__device__ __forceinline__ void ray_boxes(const MeshTree& T, float x, float yLo, float yHi,
                                          float zLo, float zHi, Leaf leaf) {
  const int lane = (int)(threadIdx.x & 63u);
  // the top levels hold at most 8 and 64 boxes: start on an even one
  int level = (T.levels - 1) & ~1;
  const int top = level;
  uint32_t first = 0;  // of the 64 boxes
  // lane `level` keeps that level's boxes still to be opened, and their first
  uint32_t todoLo = 0, todoHi = 0, firstOf = 0;
  while (true) {
    const uint32_t i = first + (uint32_t)lane;
    bool in = i < T.count[level];
    if (in) {
      // (all five at once: one after the other, each waited for its load, 84
      // instead of 58 us for the rays of 65,536 points)
      const float* b = T.box[level] + box_at(i);
      const float hx = b[24], ly = b[8], hy = b[32], lz = b[16], hz = b[40];
      in = (hx >= x) & (ly <= yHi) & (hy >= yLo) & (lz <= zHi) & (hz >= zLo);
    }
    const uint64_t m = __ballot(in);
    if (level == 0) {
      if (m != 0ull) leaf(in, i);
    } else if (lane == level) {
      todoLo = (uint32_t)m;
      todoHi = (uint32_t)(m >> 32);
      firstOf = first;
    }
    // the next box to open, on this level or above
    uint64_t left = level == 0 ? 0ull : m;
    while (left == 0ull) {
      level += 2;
      if (level > top) return;
      left = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)todoHi, level) << 32 |
             (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)todoLo, level);
    }
    const uint32_t bit = (uint32_t)__ffsll((unsigned long long)left) - 1u;
    left &= left - 1ull;
    first = ((uint32_t)__builtin_amdgcn_readlane((int)firstOf, level) + bit) * 64u;
    if (lane == level) {
      todoLo = (uint32_t)left;
      todoHi = (uint32_t)(left >> 32);
    }
    level -= 2;
  }
}

// One wave per lattice line along x (all its vertices share the ray's y and
// z): the triangles that cover it are found once, each lane takes their
// sides for its vertices.  nrm[v].w receives 1 inside, 0 outside and 2 where
// rounding decides.
constexpr int kLineChunks = 4;  // vertices per lane

__global__ __launch_bounds__(kLanes) void k_tree_lines(MeshTree T, int nx, int ny, double bx,
                                                       double by, double bz, double cs,
                                                       float4* __restrict__ nrm) {
  if (!mesh_closed(*T.info)) return;
  const int lane = (int)threadIdx.x;
  const int x0 = (int)blockIdx.y * (kLanes * kLineChunks);
  const uint32_t iy = blockIdx.x % (uint32_t)ny, iz = blockIdx.x / (uint32_t)ny;
  const double qy = by + (double)iy * cs, qz = bz + (double)iz * cs;
  int wind[kLineChunks] = {};
  bool unsure[kLineChunks] = {};
  ray_boxes(T, -INFINITY, __double2float_rd(qy), __double2float_ru(qy), __double2float_rd(qz),
            __double2float_ru(qz), [&](bool in, uint32_t t) {
              double v[9] = {};
              int cover = 0;
              if (in) {
#pragma unroll
                for (int k = 0; k < 9; ++k) v[k] = T.tri[t].v[k];
                cover = ray_cover(qy, qz, v, v + 3, v + 6);
              }
              // each covering triangle in turn, for all the line's vertices
              for (uint64_t m = __ballot(cover != 0); m != 0ull; m &= m - 1ull) {
                const int who = __ffsll((unsigned long long)m) - 1;
                double c[9];
#pragma unroll
                for (int k = 0; k < 9; ++k) c[k] = __shfl(v[k], who);
                const int up = __builtin_amdgcn_readlane(cover, who);
#pragma unroll
                for (int h = 0; h < kLineChunks; ++h) {
                  if (x0 + h * kLanes < nx) {
                    const double q[3] = {bx + (double)(x0 + h * kLanes + lane) * cs, qy, qz};
                    const int side = plane_side(q, c, c + 3, c + 6);
                    if (side == up) wind[h] += up;
                    unsure[h] = unsure[h] || side == 0;
                  }
                }
              }
            });
#pragma unroll
  for (int h = 0; h < kLineChunks; ++h) {
    const int x = x0 + h * kLanes + lane;
    if (x < nx)
      nrm[((size_t)iz * ny + iy) * nx + x].w = unsure[h] ? 2.0f : (wind[h] > 0 ? 1.0f : 0.0f);
  }
}

// The same for free points, kRaysPerWave of them one after the other (those
// whose ray misses the mesh's box need none): sdf[v] receives what
// k_tree_lines leaves in nrm[v].w.  Bound by the latency of a ray's steps;
// 65,536 points against 6,144 triangles with 8, 4, 2 rays a wave: 100, 58,
// 37 us (400,000 points with 4, 2, 1: 1814, 1805, 1873 us a call).
constexpr uint32_t kRaysPerWave = 2;

__global__ __launch_bounds__(kLanes) void k_tree_signs(MeshTree T,
                                                       const double* __restrict__ pts, uint32_t n,
                                                       const uint32_t* __restrict__ order,
                                                       double* __restrict__ sdf) {
  const MeshInfo I = *T.info;
  if (!mesh_closed(I)) return;
  const int lane = (int)threadIdx.x;
  const uint32_t k = blockIdx.x * kRaysPerWave + (uint32_t)lane;
  const bool valid = (uint32_t)lane < kRaysPerWave && k < n;
  const size_t v = valid ? order[k] : 0;
  double q[3] = {0.0, 0.0, 0.0};
  bool meets = valid;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    if (valid) q[a] = pts[3 * v + a];
    // (false for a NaN, whose sums of solid angles are NaN: outside)
    meets = meets && q[a] <= mesh_key_value(I.hi[a]) && (a == 0 || q[a] >= mesh_key_value(I.lo[a]));
  }
  double where = 0.0;
  for (uint64_t m = __ballot(meets); m != 0ull; m &= m - 1ull) {
    const int who = __ffsll((unsigned long long)m) - 1;
    const double p[3] = {__shfl(q[0], who), __shfl(q[1], who), __shfl(q[2], who)};
    int wind = 0;
    bool unsure = false;
    ray_boxes(T, __double2float_rd(p[0]), __double2float_rd(p[1]), __double2float_ru(p[1]),
              __double2float_rd(p[2]), __double2float_ru(p[2]), [&](bool in, uint32_t t) {
                int cover = 0, side = 0;
                if (in) {
                  double c[9];
#pragma unroll
                  for (int j = 0; j < 9; ++j) c[j] = T.tri[t].v[j];
                  cover = ray_cover(p[1], p[2], c, c + 3, c + 6);
                  if (cover != 0) side = plane_side(p, c, c + 3, c + 6);
                }
                wind += (int)__popcll(__ballot(cover == 1 && side == 1)) -
                        (int)__popcll(__ballot(cover == -1 && side == -1));
                unsure = unsure || __ballot(cover != 0 && side == 0) != 0ull;
              });
    if (lane == who) where = unsure ? 2.0 : (wind > 0 ? 1.0 : 0.0);
  }
  if (valid) sdf[v] = where;
}

// A wave takes a 4 x 4 x 4 block of lattice vertices (4 x 4 x 2 and 4 x 4 x 1:
// 664 and 899 us a build against 626, in Morton order).
__global__ __launch_bounds__(kLanes, kTreeWavesPerSimd) void k_tree_lattice(
    MeshTree T, const double* __restrict__ verts, uint32_t nv, const uint32_t* __restrict__ tris,
    uint32_t nt, int nx, int ny, int nz, int kx, int ky, double bx, double by, double bz,
    double cs, float4* __restrict__ cpd, float4* __restrict__ nrm) {
  __shared__ TreeShared S;
  const MeshInfo I = *T.info;
  if (!mesh_closed(I)) return;
  const uint32_t b = blockIdx.x;
  const int ix = (int)(b % (uint32_t)kx) * 4 + (int)(threadIdx.x & 3u);
  const int iy = (int)(b / (uint32_t)kx % (uint32_t)ky) * 4 + (int)((threadIdx.x >> 2) & 3u);
  const int iz =
      (int)(b / ((uint32_t)kx * (uint32_t)ky)) * 4 + (int)(threadIdx.x >> 4);
  const bool valid = ix < nx && iy < ny && iz < nz;
  const size_t v = valid ? ((size_t)iz * ny + iy) * nx + ix : 0;
  const double q[3] = {bx + (double)ix * cs, by + (double)iy * cs, bz + (double)iz * cs};
  const double delta = rounding_margin(I, q);
  // lane 21 is the block's vertex (1, 1, 1); lane 0 is always a vertex
  const int centre = ((__ballot(valid) >> 21) & 1ull) != 0ull ? 21 : 0;
  Nearest r;
  tree_nearest(T, q, delta, valid, centre, kLanes, S, r);
  const float where = valid ? nrm[v].w : 0.0f;
  const double dist = sqrt(r.d2);
  bool inside = where == 1.0f;
  const bool need = valid && (where == 2.0f || dist <= delta);
  const double w = winding_sum(need, q, verts, nv, tris, nt);
  if (need) inside = winds(w);
  if (!valid) return;
  cpd[v] = make_float4((float)r.cp[0], (float)r.cp[1], (float)r.cp[2],
                       (float)(inside ? -dist : dist));
  nrm[v] = make_float4((float)(q[0] - r.cp[0]), (float)(q[1] - r.cp[1]), (float)(q[2] - r.cp[2]),
                       0.0f);
}

// Free points are taken along the Hilbert curve through their places in three times
// the mesh's box (any order gives the same results; a wave's points should
// be neighbours).
__global__ __launch_bounds__(kBlock) void k_point_order(const double* __restrict__ pts,
                                                         uint32_t n,
                                                         const MeshInfo* __restrict__ I,
                                                         uint32_t* __restrict__ keys) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  uint32_t at[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const double lo = mesh_key_value(I->lo[a]), hi = mesh_key_value(I->hi[a]), ext = hi - lo;
    const double u = (pts[3 * (size_t)i + a] - (lo - ext)) / (3.0 * ext) * 256.0;
    at[a] = (uint32_t)fmin(fmax(u, 0.0), 255.0);  // (a NaN reads 0)
  }
  keys[i] = hilbert_key(at[0], at[1], at[2]);
}

__global__ __launch_bounds__(kLanes, kTreeWavesPerSimd) void k_tree_points(
    MeshTree T, const double* __restrict__ verts, uint32_t nv, const uint32_t* __restrict__ tris,
    uint32_t nt, const double* __restrict__ pts, uint32_t n, const uint32_t* __restrict__ order,
    uint32_t perWave, double* __restrict__ sdf, double* __restrict__ cp) {
  __shared__ TreeShared S;
  const MeshInfo I = *T.info;
  if (!mesh_closed(I)) return;
  const uint32_t k = blockIdx.x * perWave + threadIdx.x;
  const bool valid = threadIdx.x < perWave && k < n;
  const size_t v = valid ? order[k] : 0;
  double q[3] = {0.0, 0.0, 0.0};
  bool finite = valid;
  if (valid) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      q[a] = pts[3 * v + a];
      finite = finite && fabs(q[a]) <= kTreeRange;
    }
  }
  const double delta = rounding_margin(I, q);
  const uint64_t on = __ballot(finite);
  const int mid = (int)(perWave / 2);
  const int centre =
      ((on >> mid) & 1ull) != 0ull || on == 0ull ? mid : __ffsll((unsigned long long)on) - 1;
  Nearest r;
  if (on != 0ull) tree_nearest(T, q, delta, finite, centre, perWave, S, r);
  brute_nearest(valid && !finite, q, verts, nv, tris, nt, r);
  const double where = valid ? sdf[v] : 0.0;
  const double dist = sqrt(r.d2);
  bool inside = where == 1.0;
  const bool need = valid && (where == 2.0 || dist <= delta);
  const double w = winding_sum(need, q, verts, nv, tris, nt);
  if (need) inside = winds(w);
  if (!valid) return;
  sdf[v] = inside ? -dist : dist;
  if (cp) {
#pragma unroll
    for (int a = 0; a < 3; ++a) cp[3 * v + a] = r.cp[a];
  }
}

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

// Boxes of every level, in floats, and the levels' sizes.
size_t tree_levels(uint32_t nt, uint32_t count[kTreeMaxLevels], int* levels) {
  size_t floats = 0;
  uint32_t c = nt;
  int l = 0;
  while (true) {
    count[l++] = c;
    floats += (size_t)((c + 7) / 8) * 48;
    if (c <= 8u) break;
    c = (c + 7) / 8;
  }
  *levels = l;
  return floats;
}

}  // namespace

// The brute force costs 1.1 us a triangle however few the points (a wave
// walks all of them) and 7.7 ps a pair at full load; the tree's build and its
// searches' fixed cost are about 110 us.
bool mesh_tree_pays(uint32_t nt, uint64_t npts) {
  return nt >= 128u && nt <= (1u << 22) && npts < (1ull << 31);
}

bool tree_lattice_fits(const int cells[3], const double bmin[3], double cs) {
  for (int a = 0; a < 3; ++a) {
    const double lo = bmin[a], hi = bmin[a] + (double)cells[a] * cs;
    if (!(lo >= -kTreeRange && lo <= kTreeRange && hi <= kTreeRange)) return false;
  }
  const uint64_t nx = (uint64_t)cells[0] + 1, ny = (uint64_t)cells[1] + 1,
                 nz = (uint64_t)cells[2] + 1;
  // threads of one launch dimension stay below 2^32
  return ny * nz < (1ull << 26) && ((nx + 3) / 4) * ((ny + 3) / 4) * ((nz + 3) / 4) < (1ull << 26) &&
         nx < (1ull << 23);
}

size_t mesh_tree_bytes(uint32_t nt) {
  uint32_t count[kTreeMaxLevels];
  int levels;
  const size_t floats = tree_levels(nt, count, &levels);
  return align256(sizeof(MeshInfo)) + align256((size_t)nt * sizeof(TreeTri)) +
         align256(floats * sizeof(float)) + 2 * align256((size_t)nt * sizeof(uint32_t));
}

hipError_t launch_mesh_tree(fc_context* ctx, const double* verts, uint32_t nv,
                            const uint32_t* tris, uint32_t nt, void* block, MeshTree* out) {
  hipStream_t s = ctx->stream;
  TreeBuild B = {};
  const size_t floats = tree_levels(nt, B.count, &B.levels);
  char* at = static_cast<char*>(block);
  MeshInfo* info = reinterpret_cast<MeshInfo*>(at);
  at += align256(sizeof(MeshInfo));
  TreeTri* tri = reinterpret_cast<TreeTri*>(at);
  at += align256((size_t)nt * sizeof(TreeTri));
  float* box = reinterpret_cast<float*>(at);
  at += align256(floats * sizeof(float));
  uint32_t* keys = reinterpret_cast<uint32_t*>(at);
  at += align256((size_t)nt * sizeof(uint32_t));
  uint32_t* order = reinterpret_cast<uint32_t*>(at);
  for (int l = 0; l < B.levels; ++l) {
    B.box[l] = box;
    box += (size_t)((B.count[l] + 7) / 8) * 48;
  }
  const unsigned blocks = (nt + kBlock - 1) / kBlock;
  hipLaunchKernelGGL(k_mesh_info_init, dim3(1), dim3(64), 0, s, info);
  hipLaunchKernelGGL(k_mesh_info, dim3(blocks < kInfoBlocks ? blocks : kInfoBlocks), dim3(kBlock),
                     0, s, verts, nv, tris, nt, info);
  const int bits = mesh_order_bits(nt);
  hipLaunchKernelGGL(k_mesh_order, dim3(blocks), dim3(kBlock), 0, s, verts, nv, tris, nt, info,
                     bits, keys);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess)
    e = radix_sort_pairs(s, ctx->sort, ctx->devFlags, keys, nullptr, keys, order, nt, bits,
                         nullptr, false, 1, nullptr, nullptr, nullptr, nullptr, &info->open);
  if (e != hipSuccess) return e;
  const uint32_t padded = (nt + 7u) & ~7u;
  hipLaunchKernelGGL(k_tree_leaves, dim3((padded + kBlock - 1) / kBlock), dim3(kBlock), 0, s,
                     verts, nv, tris, nt, order, tri, B.box[0]);
  if (B.levels > 1) hipLaunchKernelGGL(k_tree_levels, dim3(1), dim3(1024), 0, s, B);
  e = hipGetLastError();
  out->tri = tri;
  for (int l = 0; l < B.levels; ++l) {
    out->box[l] = B.box[l];
    out->count[l] = B.count[l];
  }
  out->levels = B.levels;
  out->info = info;
  return e;
}

hipError_t launch_tree_lattice(hipStream_t s, const MeshTree& T, const double* verts, uint32_t nv,
                               const uint32_t* tris, uint32_t nt, const int cells[3],
                               const double bmin[3], double cs, float4* cpd, float4* nrm) {
  const int nx = cells[0] + 1, ny = cells[1] + 1, nz = cells[2] + 1;
  hipLaunchKernelGGL(k_tree_lines,
                     dim3((unsigned)ny * (unsigned)nz,
                          (unsigned)((nx + kLanes * kLineChunks - 1) / (kLanes * kLineChunks))),
                     dim3(kLanes), 0, s, T, nx, ny, bmin[0], bmin[1], bmin[2], cs, nrm);
  const int kx = (nx + 3) / 4, ky = (ny + 3) / 4, kz = (nz + 3) / 4;
  hipLaunchKernelGGL(k_tree_lattice, dim3((unsigned)kx * (unsigned)ky * (unsigned)kz),
                     dim3(kLanes), 0, s, T, verts, nv, tris, nt, nx, ny, nz, kx, ky, bmin[0],
                     bmin[1], bmin[2], cs, cpd, nrm);
  return hipGetLastError();
}

size_t tree_points_bytes(uint64_t np) {
  const uint64_t chunk = np < kPointChunk ? np : kPointChunk;
  return 2 * align256((size_t)chunk * sizeof(uint32_t));
}

uint32_t tree_sort_pairs(uint32_t nt, uint64_t np) {
  const uint64_t chunk = np < kPointChunk ? np : kPointChunk;
  return chunk > nt ? (uint32_t)chunk : nt;
}

hipError_t launch_tree_points(fc_context* ctx, const MeshTree& T, const double* verts,
                              uint32_t nv, const uint32_t* tris, uint32_t nt, const double* pts,
                              uint64_t np, void* block, double* sdf, double* cp) {
  hipStream_t s = ctx->stream;
  const uint64_t chunk = np < kPointChunk ? np : kPointChunk;
  uint32_t* keys = static_cast<uint32_t*>(block);
  uint32_t* order =
      reinterpret_cast<uint32_t*>(static_cast<char*>(block) + align256((size_t)chunk * 4));
  for (uint64_t at = 0; at < np; at += chunk) {
    const uint32_t n = (uint32_t)(np - at < chunk ? np - at : chunk);
    const double* p = pts + 3 * at;
    hipLaunchKernelGGL(k_point_order, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, p, n,
                       T.info, keys);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess)
      e = radix_sort_pairs(s, ctx->sort, ctx->devFlags, keys, nullptr, keys, order, n,
                           kOrderBits, nullptr, false, 1, nullptr, nullptr, nullptr, nullptr,
                           &T.info->open);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_tree_signs, dim3((n + kRaysPerWave - 1) / kRaysPerWave), dim3(kLanes), 0,
                       s, T, p, n, order, sdf + at);
    uint32_t perWave = 8;
    while (perWave < (uint32_t)kLanes && n / perWave > kPointWaves) perWave *= 2;
    hipLaunchKernelGGL(k_tree_points, dim3((n + perWave - 1) / perWave), dim3(kLanes), 0, s, T,
                       verts, nv, tris, nt, p, n, order, perWave, sdf + at,
                       cp ? cp + 3 * at : nullptr);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace fc
