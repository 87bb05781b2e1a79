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
// Layout: triangles sorted by the Morton code of their centroids, eight
// consecutive ones to a group, groups of groups above; no topology to build
// and no pointers, and a node's eight child boxes are 192 consecutive bytes,
// so one visit is twelve 16-byte loads in flight together (the traversal is
// a chain of dependent loads; wide nodes make it short).
#include "mesh_tree.hpp"

#include <cfloat>

#include "fc_internal.hpp"
#include "mesh_distance.hpp"

namespace fc {

namespace {

constexpr int kBlock = 256;
constexpr uint32_t kInfoBlocks = 64;

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
  if (threadIdx.x == 0) I->bad = I->pad = 0u;
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

// At most kInfoBlocks blocks, so that the atomics on the one result stay few.
__global__ __launch_bounds__(kBlock) void k_mesh_info(const double* __restrict__ verts,
                                                      uint32_t nv,
                                                      const uint32_t* __restrict__ tris,
                                                      uint32_t nt, MeshInfo* __restrict__ I) {
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
  const bool anyBad = __ballot(bad) != 0ull;
  if ((threadIdx.x & 63u) == 0u) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      atomicMin(&I->lo[a], mesh_key(lo[a]));
      atomicMax(&I->hi[a], mesh_key(hi[a]));
    }
    atomicAdd(&I->edges[0], e0);
    atomicAdd(&I->edges[1], e1);
    if (anyBad) atomicOr(&I->bad, 1u);
  }
}

// The low 8 bits of x, spread to every third bit.
__device__ __forceinline__ uint32_t spread3(uint32_t x) {
  x &= 0xffu;
  x = (x | (x << 8)) & 0x00f00fu;
  x = (x | (x << 4)) & 0x0c30c3u;
  return (x | (x << 2)) & 0x249249u;
}

constexpr int kMortonBits = 24;

__global__ __launch_bounds__(kBlock) void k_mesh_morton(const double* __restrict__ verts,
                                                        uint32_t nv,
                                                        const uint32_t* __restrict__ tris,
                                                        uint32_t nt,
                                                        const MeshInfo* __restrict__ I,
                                                        uint32_t* __restrict__ keys) {
  const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
  if (t >= nt) return;
  double v[9];
  uint32_t vi[3];
  load_corners(verts, nv, tris, t, v, vi);
  uint32_t key = 0;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const double lo = mesh_key_value(I->lo[a]), hi = mesh_key_value(I->hi[a]);
    const double c = (v[a] + v[3 + a] + v[6 + a]) * (1.0 / 3.0);
    // any value orders the triangles (a NaN reads 0)
    const double u = fmin(fmax((c - lo) / (hi - lo) * 256.0, 0.0), 255.0);
    key |= spread3((uint32_t)u) << a;
  }
  keys[t] = key;
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
  const uint32_t t = order[p];
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

// The smallest (squared distance, triangle number) of q.  s_lb: this lane's
// column of the block's [levels][8][lanes] child distances.
struct Nearest {
  double d2;
  uint32_t id;
  double cp[3];
};

constexpr int kLanes = 64;  // one wave per block: no barriers, any balance

__device__ __forceinline__ Nearest tree_nearest(const MeshTree& T, const double q[3],
                                                double delta, float (*s_lb)[8][kLanes]) {
  Nearest best;
  best.d2 = DBL_MAX;
  best.id = 0xffffffffu;
  best.cp[0] = best.cp[1] = best.cp[2] = 0.0;
  float qlo[3], qhi[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    qlo[a] = __double2float_rd(q[a]);
    qhi[a] = __double2float_ru(q[a]);
  }
  const int lane = (int)(threadIdx.x & 63u);
  // (sqrt(d2) + delta)^2, rounded up: a box at least this far holds no winner
  float limit = INFINITY;
  uint64_t todo = 0;  // a byte per level: the children still to be taken
  int level = T.levels - 1;
  uint32_t group = 0;
  bool enter = true;
  while (true) {
    if (enter) {
      const float4* b = reinterpret_cast<const float4*>(T.box[level] + (size_t)group * 48u);
      float lb[8] = {};
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const float4 l0 = b[2 * a], l1 = b[2 * a + 1], h0 = b[6 + 2 * a], h1 = b[7 + 2 * a];
        const float lo[8] = {l0.x, l0.y, l0.z, l0.w, l1.x, l1.y, l1.z, l1.w};
        const float hi[8] = {h0.x, h0.y, h0.z, h0.w, h1.x, h1.y, h1.z, h1.w};
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const float d = fmaxf(fmaxf(lo[u] - qhi[a], qlo[a] - hi[u]), 0.0f);
          lb[u] += d * d;
        }
      }
      uint32_t m = 0;
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        // below the exact box distance by more than its few roundings
        const float x = lb[u] * (1.0f - 0x1p-20f);
        s_lb[level][u][lane] = x;
        if (!(x > limit) && group * 8u + (uint32_t)u < T.count[level]) m |= 1u << u;
      }
      todo = (todo & ~(0xffull << (8 * level))) | ((uint64_t)m << (8 * level));
      enter = false;
    }
    // the nearest child still to be taken
    uint32_t m = (uint32_t)(todo >> (8 * level)) & 0xffu;
    float near = INFINITY;
    int pick = -1;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      if ((m >> u) & 1u) {
        const float x = s_lb[level][u][lane];
        if (!(x > limit) && (pick < 0 || x < near)) {
          near = x;
          pick = u;
        }
      }
    }
    if (pick < 0) {  // none left within reach
      if (++level == T.levels) break;
      group >>= 3;
      continue;
    }
    todo &= ~(1ull << (8 * level + pick));
    const uint32_t child = group * 8u + (uint32_t)pick;
    if (level > 0) {
      group = child;
      --level;
      enter = true;
      continue;
    }
    const TreeTri& R = T.tri[child];
    double v[9], c[3];
#pragma unroll
    for (int k = 0; k < 9; ++k) v[k] = R.v[k];
    const uint32_t id = (uint32_t)R.id;
    const double d2 = point_triangle_dist2(q, v, v + 3, v + 6, c);
    if (d2 < best.d2 || (d2 == best.d2 && id < best.id)) {
      best.d2 = d2;
      best.id = id;
      best.cp[0] = c[0];
      best.cp[1] = c[1];
      best.cp[2] = c[2];
      const double r = sqrt(d2) + delta;
      limit = __double2float_ru(r * r * (1.0 + 1e-12));
    }
  }
  return best;
}

__device__ __forceinline__ double rounding_margin(const MeshInfo& I, const double q[3]) {
  const double m = mesh_magnitude(I) + fmax(fabs(q[0]), fmax(fabs(q[1]), fabs(q[2])));
  return 256.0 * 2.220446049250313e-16 * m;
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
  const float qyLo = __double2float_rd(qy), qyHi = __double2float_ru(qy);
  const float qzLo = __double2float_rd(qz), qzHi = __double2float_ru(qz);
  int wind[kLineChunks] = {};
  bool unsure[kLineChunks] = {};
  uint64_t todo = 0;
  int level = T.levels - 1;
  uint32_t group = 0;
  bool enter = true;
  while (true) {
    if (enter) {
      // lanes 0-7 take a child each
      const int u = lane & 7;
      const float* b = T.box[level] + (size_t)group * 48u + u;
      const bool in = lane < 8 && group * 8u + (uint32_t)u < T.count[level] && b[8] <= qyHi &&
                      b[32] >= qyLo && b[16] <= qzHi && b[40] >= qzLo;
      const uint64_t m = __ballot(in);
      todo = (todo & ~(0xffull << (8 * level))) | (m << (8 * level));
      enter = false;
    }
    const uint32_t m = (uint32_t)(todo >> (8 * level)) & 0xffu;
    if (m == 0u) {
      if (++level == T.levels) break;
      group >>= 3;
      continue;
    }
    const uint32_t child = group * 8u + (uint32_t)(__ffs((int)m) - 1);
    todo &= ~(1ull << (8 * level + (__ffs((int)m) - 1)));
    if (level > 0) {
      group = child;
      --level;
      enter = true;
      continue;
    }
    const TreeTri& R = T.tri[child];
    double v[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) v[k] = R.v[k];
    const int cover = ray_cover(qy, qz, v, v + 3, v + 6);
    if (cover == 0) continue;
#pragma unroll
    for (int c = 0; c < kLineChunks; ++c) {
      if (x0 + c * kLanes < nx) {
        const double q[3] = {bx + (double)(x0 + c * kLanes + lane) * cs, qy, qz};
        const int side = plane_side(q, v, v + 3, v + 6);
        if (side == cover) wind[c] += cover;
        unsure[c] = unsure[c] || side == 0;
      }
    }
  }
#pragma unroll
  for (int c = 0; c < kLineChunks; ++c) {
    const int x = x0 + c * kLanes + lane;
    if (x < nx)
      nrm[((size_t)iz * ny + iy) * nx + x].w = unsure[c] ? 2.0f : (wind[c] > 0 ? 1.0f : 0.0f);
  }
}

// The same for one point per lane.
__device__ __forceinline__ int tree_inside(const MeshTree& T, const double q[3]) {
  float qlo[3], qhi[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    qlo[a] = __double2float_rd(q[a]);
    qhi[a] = __double2float_ru(q[a]);
  }
  int wind = 0;
  bool unsure = false;
  uint64_t todo = 0;
  int level = T.levels - 1;
  uint32_t group = 0;
  bool enter = true;
  while (true) {
    if (enter) {
      const float4* b = reinterpret_cast<const float4*>(T.box[level] + (size_t)group * 48u);
      uint32_t m = 0;
      float lo[3][8], hi[3][8];
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const float4 l0 = b[2 * a], l1 = b[2 * a + 1], h0 = b[6 + 2 * a], h1 = b[7 + 2 * a];
        const float l[8] = {l0.x, l0.y, l0.z, l0.w, l1.x, l1.y, l1.z, l1.w};
        const float h[8] = {h0.x, h0.y, h0.z, h0.w, h1.x, h1.y, h1.z, h1.w};
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          lo[a][u] = l[u];
          hi[a][u] = h[u];
        }
      }
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (hi[0][u] >= qlo[0] && lo[1][u] <= qhi[1] && hi[1][u] >= qlo[1] &&
            lo[2][u] <= qhi[2] && hi[2][u] >= qlo[2] && group * 8u + (uint32_t)u < T.count[level])
          m |= 1u << u;
      todo = (todo & ~(0xffull << (8 * level))) | ((uint64_t)m << (8 * level));
      enter = false;
    }
    const uint32_t m = (uint32_t)(todo >> (8 * level)) & 0xffu;
    if (m == 0u) {
      if (++level == T.levels) break;
      group >>= 3;
      continue;
    }
    const uint32_t child = group * 8u + (uint32_t)(__ffs((int)m) - 1);
    todo &= ~(1ull << (8 * level + (__ffs((int)m) - 1)));
    if (level > 0) {
      group = child;
      --level;
      enter = true;
      continue;
    }
    const TreeTri& R = T.tri[child];
    double v[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) v[k] = R.v[k];
    const int cover = ray_cover(q[1], q[2], v, v + 3, v + 6);
    if (cover != 0) {
      const int side = plane_side(q, v, v + 3, v + 6);
      if (side == cover) wind += cover;
      unsure = unsure || side == 0;
    }
  }
  return unsure ? 2 : (wind > 0 ? 1 : 0);
}

// A wave takes a 4 x 4 x 4 block of lattice vertices, whose searches visit
// mostly the same boxes.
__global__ __launch_bounds__(kLanes) void k_tree_lattice(
    MeshTree T, const double* __restrict__ verts, uint32_t nv, const uint32_t* __restrict__ tris,
    uint32_t nt, int nx, int ny, int nz, int kx, int ky, double bx, double by, double bz,
    double cs, float4* __restrict__ cpd, float4* __restrict__ nrm) {
  extern __shared__ float s_mem[];
  const MeshInfo I = *T.info;
  if (!mesh_closed(I)) return;
  const uint32_t b = blockIdx.x;
  const int ix = (int)(b % (uint32_t)kx) * 4 + (int)(threadIdx.x & 3u);
  const int iy = (int)(b / (uint32_t)kx % (uint32_t)ky) * 4 + (int)((threadIdx.x >> 2) & 3u);
  const int iz = (int)(b / ((uint32_t)kx * (uint32_t)ky)) * 4 + (int)(threadIdx.x >> 4);
  const bool valid = ix < nx && iy < ny && iz < nz;
  const size_t v = valid ? ((size_t)iz * ny + iy) * nx + ix : 0;
  const double q[3] = {bx + (double)ix * cs, by + (double)iy * cs, bz + (double)iz * cs};
  const double delta = rounding_margin(I, q);
  Nearest r;
  r.d2 = DBL_MAX;
  float where = 0.0f;
  if (valid) {
    where = nrm[v].w;
    r = tree_nearest(T, q, delta, reinterpret_cast<float(*)[8][kLanes]>(s_mem));
  }
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

__global__ __launch_bounds__(kLanes) void k_tree_points(
    MeshTree T, const double* __restrict__ verts, uint32_t nv, const uint32_t* __restrict__ tris,
    uint32_t nt, const double* __restrict__ pts, uint64_t np, double* __restrict__ sdf,
    double* __restrict__ cp) {
  extern __shared__ float s_mem[];
  const MeshInfo I = *T.info;
  if (!mesh_closed(I)) return;
  const uint64_t v = (uint64_t)blockIdx.x * kLanes + threadIdx.x;
  const bool valid = v < np;
  double q[3] = {0.0, 0.0, 0.0};
  Nearest r;
  r.d2 = DBL_MAX;
  int where = 0;
  if (valid) {
#pragma unroll
    for (int a = 0; a < 3; ++a) q[a] = pts[3 * v + a];
  }
  const double delta = rounding_margin(I, q);
  if (valid) {
    r = tree_nearest(T, q, delta, reinterpret_cast<float(*)[8][kLanes]>(s_mem));
    where = tree_inside(T, q);
  }
  const double dist = sqrt(r.d2);
  bool inside = where == 1;
  const bool need = valid && (where == 2 || dist <= delta);
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

// The brute force costs about 7.7 ps per point-triangle pair at full load;
// the tree's build and its searches' fixed cost are about 100 us.  Below
// 256 triangles the tree has two levels and saves little.
bool mesh_tree_pays(uint32_t nt, uint64_t npts) {
  return nt >= 256u && nt <= (1u << 22) && npts < (1ull << 31) &&
         npts * (uint64_t)nt >= (1ull << 24);
}

bool tree_lattice_fits(const int cells[3]) {
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
  hipLaunchKernelGGL(k_mesh_morton, dim3(blocks), dim3(kBlock), 0, s, verts, nv, tris, nt, info,
                     keys);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess)
    e = radix_sort_pairs(s, ctx->sort, ctx->devFlags, keys, nullptr, keys, order, nt, kMortonBits,
                         nullptr);
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
                     dim3(kLanes), (size_t)T.levels * 8 * kLanes * sizeof(float), s, T, verts, nv,
                     tris, nt, nx, ny, nz, kx, ky, bmin[0], bmin[1], bmin[2], cs, cpd, nrm);
  return hipGetLastError();
}

hipError_t launch_tree_points(hipStream_t s, const MeshTree& T, const double* verts, uint32_t nv,
                              const uint32_t* tris, uint32_t nt, const double* pts, uint64_t np,
                              double* sdf, double* cp) {
  hipLaunchKernelGGL(k_tree_points, dim3((unsigned)((np + kLanes - 1) / kLanes)), dim3(kLanes),
                     (size_t)T.levels * 8 * kLanes * sizeof(float), s, T, verts, nv, tris, nt, pts,
                     np, sdf, cp);
  return hipGetLastError();
}

}  // namespace fc
