// Distance-map boundary on gfx950: upload of a reference-layout map, map
// queries (plain and rigidly transformed), and the exact point-mesh builder.
#include "fc_internal.hpp"
#include "distmap.hpp"
#include "mesh_distance.hpp"
#include "mesh_tree.hpp"

#include <cfloat>
#include <charconv>
#include <cmath>
#include <cstdio>
#include <fstream>
#include <iterator>
#include <new>
#include <string>
#include <vector>

namespace fc {

namespace {

constexpr int kBlock = 256;

inline unsigned grid_for(size_t n, int block) {
  size_t g = (n + (size_t)block - 1) / (size_t)block;
  return (unsigned)(g == 0 ? 1 : g);
}

// Batched queryMap over float[3] points (the reference's vector3 arrays).
// queryFBM (distancemap.cuh:195-225): 1 where the interpolated distance of
// a point inside the box is <= 0, else 0 (0 outside the box).
__global__ __launch_bounds__(kBlock) void k_distmap_query_fbm(DistMapView m,
                                                              const float* __restrict__ pts,
                                                              uint32_t n,
                                                              int32_t* __restrict__ out) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const v3f q = make_v3(pts[3 * i], pts[3 * i + 1], pts[3 * i + 2]);
  float d = 0.0f;
  v3f c = make_v3(0.0f, 0.0f, 0.0f);
  const bool inside = distmap_query(m, q, d, c, nullptr);
  out[i] = (inside && d <= 0.0f) ? 1 : 0;
}

__global__ __launch_bounds__(kBlock) void k_distmap_query(DistMapView m,
                                                          const float* __restrict__ pts,
                                                          uint32_t n, float* __restrict__ dist,
                                                          float* __restrict__ cp,
                                                          float* __restrict__ nrm) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const v3f q = make_v3(pts[3 * i], pts[3 * i + 1], pts[3 * i + 2]);
  float d = 0.0f;
  v3f c = make_v3(0.0f, 0.0f, 0.0f), nn = make_v3(0.0f, 0.0f, 0.0f);
  distmap_query(m, q, d, c, &nn);
  dist[i] = d;
  if (cp) {
    cp[3 * i] = c.x;
    cp[3 * i + 1] = c.y;
    cp[3 * i + 2] = c.z;
  }
  if (nrm) {
    nrm[3 * i] = nn.x;
    nrm[3 * i + 1] = nn.y;
    nrm[3 * i + 2] = nn.z;
  }
}

// The value of the other lane of a pair (2 k, 2 k + 1).
__device__ __forceinline__ float other_of_pair(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0xB1, 0xf, 0xf, true));
}
__device__ __forceinline__ double other_of_pair(double x) {
  const long long u = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)u, 0xB1, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(u >> 32), 0xB1, 0xf, 0xf, true);
  return __longlong_as_double((long long)hi << 32 | (uint32_t)lo);
}

// distmap_query with the normal, two lanes a point: lane p of the pair takes
// the corners of x plane p, so that one load brings the 32 adjacent bytes of
// an edge; each lane multiplies its corners by their x weight, and the pair's
// products are added across (the same two addends, hence the same sums).
// Scattered points are bound by the requests that a CU's L1 keeps in flight
// (about 116, 520 cycles each; the edge's corners in two loads of one lane
// also took two passes through its tags, 15 a point against 10 here).
// 1,000,003 points in a map of 64^3 cells: 49.6 us with a lane a point, 47.1
// with two (vertices in bricks of 2 x 2 x 2, a lane a point: 53.1; fewer
// L2 misses, more requests).
__global__ __launch_bounds__(kBlock) void k_distmap_query_pairs(DistMapView m,
                                                          const float* __restrict__ pts,
                                                          uint32_t n, float* __restrict__ dist,
                                                          float* __restrict__ cp,
                                                          float* __restrict__ nrm) {
  const uint32_t i = blockIdx.x * (kBlock / 2) + (threadIdx.x >> 1);
  const int p = (int)(threadIdx.x & 1u);
  if (i >= n) return;
  const v3f q = make_v3(pts[3 * (size_t)i], pts[3 * (size_t)i + 1], pts[3 * (size_t)i + 2]);
  float d = 5.0f;
  v3f c = make_v3(0.0f, 0.0f, 0.0f);
  if (m.bmin[0] <= q.x && q.x <= m.bmax[0] && m.bmin[1] <= q.y && q.y <= m.bmax[1] &&
      m.bmin[2] <= q.z && q.z <= m.bmax[2]) {
    const float inv = (float)(1.0 / (double)m.cellSize);
    const int x = dm_clamp_cell((int)(fabsf(q.x - m.bmin[0]) * inv), m.cx);
    const int y = dm_clamp_cell((int)(fabsf(q.y - m.bmin[1]) * inv), m.cy);
    const int z = dm_clamp_cell((int)(fabsf(q.z - m.bmin[2]) * inv), m.cz);
    const int64_t ix = m.cx + 1, islice = (int64_t)(m.cx + 1) * (m.cy + 1);
    const int64_t base = (int64_t)z * islice + (int64_t)y * ix + x;
    const float4* at = m.cpd + base + p;
    const float4 v00 = at[0], v10 = at[ix], v01 = at[islice], v11 = at[ix + islice];
    float4 n0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (p != 0 && nrm != nullptr) n0 = m.nrm[base];
    auto place = [&](const float* axis, int cell, float v) {
      const float mine = axis[cell + p], yours = other_of_pair(mine);
      const float lo = p ? yours : mine, hi = p ? mine : yours;
      return (v - lo) / (hi - lo);
    };
    const float xd = place(m.xs, x, q.x), yd = place(m.ys, y, q.y), zd = place(m.zs, z, q.z);
    const double ox = 1.0 - (double)xd, oy = 1.0 - (double)yd, oz = 1.0 - (double)zd;
    const float wx = p ? xd : (float)ox, wy = (float)oy, wz = (float)oz;
    auto across = [&](float v) {
      const double t = p ? (double)(v * xd) : (double)v * ox;
      return (float)(t + other_of_pair(t));
    };
    const float c00 = across(v00.w), c10 = across(v10.w), c01 = across(v01.w), c11 = across(v11.w);
    const float c0 = (float)((double)c00 * oy + (double)(c10 * yd));
    const float c1 = (float)((double)c01 * oy + (double)(c11 * yd));
    d = (float)((double)c0 * oz + (double)(c1 * zd));
    auto mix = [&](float a, float b, float e, float f) {
      const float ta = a * wx, tb = b * wx, te = e * wx, tf = f * wx;
      const float p00 = ta + other_of_pair(ta), p10 = tb + other_of_pair(tb);
      const float p01 = te + other_of_pair(te), p11 = tf + other_of_pair(tf);
      return (p00 * wy + p10 * yd) * wz + (p01 * wy + p11 * yd) * zd;
    };
    c = make_v3(mix(v00.x, v10.x, v01.x, v11.x), mix(v00.y, v10.y, v01.y, v11.y),
                mix(v00.z, v10.z, v01.z, v11.z));
    if (p) c = make_v3(n0.x, n0.y, n0.z);
  }
  if (p == 0) dist[i] = d;
  float* out = p ? nrm : cp;  // the second lane stores the normal
  if (out != nullptr) {
    out[3 * (size_t)i] = c.x;
    out[3 * (size_t)i + 1] = c.y;
    out[3 * (size_t)i + 2] = c.z;
  }
}

// Matrix3x3<T> * Vector3<T> (math/matrix3x3.h:313-321): row major,
// accumulated from zero.
__device__ __forceinline__ v3f mat3_mul(const float* M, v3f v) {
  float r[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    float s = 0.0f;
    s += M[i * 3 + 0] * v.x;
    s += M[i * 3 + 1] * v.y;
    s += M[i * 3 + 2] * v.z;
    r[i] = s;
  }
  return make_v3(r[0], r[1], r[2]);
}

// eval_distmap_kernel (difi.cu:427-474).
// eval_distmap for one vertex p of body 1 (difi.cu:427-474): to world space
// by body 1's pose, into body 0's model frame, queryMap there, then the
// world closest point, the unit normal from the vertex to it and the
// midpoint contact.  Returns false outside body 0's box (distance 1000).
__device__ __forceinline__ bool eval_vertex(const DistMapView& m, const fc_trans_info& T, v3f p,
                                            float& d, v3f& contact, v3f& normal) {
  v3f qw = mat3_mul(T.m2w1, p);
  qw = make_v3(qw.x + T.origin1.x, qw.y + T.origin1.y, qw.z + T.origin1.z);
  const v3f q = mat3_mul(T.w2m0, make_v3(qw.x - T.origin0.x, qw.y - T.origin0.y, qw.z - T.origin0.z));
  if (!(m.bmin[0] <= q.x && q.x <= m.bmax[0] && m.bmin[1] <= q.y && q.y <= m.bmax[1] &&
        m.bmin[2] <= q.z && q.z <= m.bmax[2])) {
    d = 1000.0f;
    return false;
  }
  d = 1000.0f;
  v3f cp = make_v3(0.0f, 0.0f, 0.0f);
  distmap_query(m, q, d, cp, nullptr);
  v3f c0 = mat3_mul(T.m2w0, cp);
  c0 = make_v3(c0.x + T.origin0.x, c0.y + T.origin0.y, c0.z + T.origin0.z);
  // Vector3::normalize (math/vector3.h:159-167): scale by (float)(1.0/|n|).
  const v3f nn = make_v3(c0.x - qw.x, c0.y - qw.y, c0.z - qw.z);
  const float mag = sqrtf(dot3(nn, nn));
  const float invMag = (float)(1.0 / (double)mag);
  normal = make_v3(nn.x * invMag, nn.y * invMag, nn.z * invMag);
  contact = make_v3((c0.x + qw.x) * 0.5f, (c0.y + qw.y) * 0.5f, (c0.z + qw.z) * 0.5f);
  return true;
}

__global__ __launch_bounds__(kBlock) void k_distmap_eval(DistMapView m, fc_trans_info T,
                                                         const float* __restrict__ v, uint32_t n,
                                                         float* __restrict__ cps,
                                                         float* __restrict__ normals,
                                                         float* __restrict__ distance) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  float d;
  v3f c, nn;
  if (eval_vertex(m, T, make_v3(v[3 * i], v[3 * i + 1], v[3 * i + 2]), d, c, nn)) {
    normals[3 * i] = nn.x;
    normals[3 * i + 1] = nn.y;
    normals[3 * i + 2] = nn.z;
    cps[3 * i] = c.x;
    cps[3 * i + 1] = c.y;
    cps[3 * i + 2] = c.z;
  }
  distance[i] = d;
}

// ColliderMeshMesh<gpu>::collide (collidermeshmesh.cuh:89-172) keeps the
// vertices with eval distance < threshold as contacts, in vertex order.
// Pass 1 counts them per block; pass 2 writes each at its block's offset
// plus its rank in the block (ballots), so the list is in vertex order.
__global__ __launch_bounds__(kBlock) void k_mesh_contacts_count(DistMapView m, fc_trans_info T,
                                                                const float* __restrict__ v,
                                                                uint32_t n, float threshold,
                                                                uint32_t* __restrict__ blockCounts) {
  __shared__ uint32_t s_w[kBlock / 64];
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  bool hit = false;
  if (i < n) {
    float d;
    v3f c, nn;
    eval_vertex(m, T, make_v3(v[3 * i], v[3 * i + 1], v[3 * i + 2]), d, c, nn);
    hit = d < threshold;
  }
  const uint64_t b = __ballot(hit);
  if ((threadIdx.x & 63u) == 0u) s_w[threadIdx.x >> 6] = (uint32_t)__popcll(b);
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t t = 0;
    for (int w = 0; w < kBlock / 64; ++w) t += s_w[w];
    blockCounts[blockIdx.x] = t;
  }
}

__global__ __launch_bounds__(kBlock) void k_mesh_contacts_write(
    DistMapView m, fc_trans_info T, const float* __restrict__ v, uint32_t n, float threshold,
    const uint32_t* __restrict__ blockOffsets, uint32_t capacity, float* __restrict__ cps,
    float* __restrict__ normals, uint32_t* __restrict__ ids) {
  __shared__ uint32_t s_w[kBlock / 64];
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  bool hit = false;
  float d = 1000.0f;
  v3f c = make_v3(0.0f, 0.0f, 0.0f), nn = c;
  if (i < n) {
    eval_vertex(m, T, make_v3(v[3 * i], v[3 * i + 1], v[3 * i + 2]), d, c, nn);
    hit = d < threshold;
  }
  const uint64_t b = __ballot(hit);
  if (lane == 0u) s_w[wave] = (uint32_t)__popcll(b);
  __syncthreads();
  uint32_t rank = blockOffsets[blockIdx.x] + (uint32_t)__popcll(b & ((1ull << lane) - 1ull));
  for (uint32_t w = 0; w < wave; ++w) rank += s_w[w];
  if (hit && rank < capacity) {
    cps[3 * (size_t)rank] = c.x;
    cps[3 * (size_t)rank + 1] = c.y;
    cps[3 * (size_t)rank + 2] = c.z;
    normals[3 * (size_t)rank] = nn.x;
    normals[3 * (size_t)rank + 1] = nn.y;
    normals[3 * (size_t)rank + 2] = nn.z;
    ids[rank] = i;
  }
}

// integrateSystem with the distance-map boundary on caller arrays.
__global__ __launch_bounds__(kBlock) void k_integrate_distmap(fc_sim_params P, DistMapView m,
                                                              float4* __restrict__ pos,
                                                              float4* __restrict__ vel, float dt,
                                                              uint32_t n) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const float4 p4 = pos[i], v4 = vel[i];
  v3f p = xyz(p4), v = xyz(v4);
  integrate_distmap(P, m, P.particleRadius, dt, p, v);
  pos[i] = make_float4(p.x, p.y, p.z, p4.w);
  vel[i] = make_float4(v.x, v.y, v.z, v4.w);
}

// ---------------------------------------------------------------------------
// Builder: exact signed distance of every lattice vertex to a closed mesh.
// ---------------------------------------------------------------------------

constexpr int kTriTile = 128;

// One lane per query point (lattice vertex or free point); triangles are
// streamed through LDS in tiles that every lane of the block reads
// (broadcast reads, no bank conflicts).  Minimum over triangles in order
// (first minimum wins), sign from the generalized winding number.
// For small problems, and for meshes that the triangle tree does not take:
// with `info` the kernel leaves those that it does take (mesh_closed).
// Blocks walk the points with the grid's stride, so that a launch that finds
// nothing to do is short.
constexpr unsigned kSdfMaxBlocks = 4096;
// A builder's copy of its mesh of up to so many bytes stays in the context's
// scratch for the next one.
constexpr size_t kMeshCopyKept = (size_t)256 << 20;

template <bool kLattice>
__global__ __launch_bounds__(kBlock) void k_mesh_sdf(
    const MeshInfo* __restrict__ info, const double* __restrict__ verts, uint32_t nv,
    const uint32_t* __restrict__ tris, uint32_t nt, uint64_t npts, const double* __restrict__ pts,
    int cx, int cy, double bx, double by, double bz, double cs, float4* __restrict__ cpd,
    float4* __restrict__ nrm, double* __restrict__ sdfOut, double* __restrict__ cpOut) {
  __shared__ double s_tri[kTriTile][9];
  if (info != nullptr && mesh_closed(*info)) return;
  for (uint64_t base = (uint64_t)blockIdx.x * kBlock; base < npts;
       base += (uint64_t)gridDim.x * kBlock) {
    const uint64_t v = base + threadIdx.x;
    const bool valid = v < npts;
    double q[3] = {0.0, 0.0, 0.0};
    if (valid) {
      if (kLattice) {
        const uint64_t ix = (uint64_t)cx + 1, islice = ix * ((uint64_t)cy + 1);
        const uint64_t iz = v / islice, rem = v - iz * islice, iy = rem / ix, ixx = rem - iy * ix;
        q[0] = bx + (double)ixx * cs;
        q[1] = by + (double)iy * cs;
        q[2] = bz + (double)iz * cs;
      } else {
        q[0] = pts[3 * v];
        q[1] = pts[3 * v + 1];
        q[2] = pts[3 * v + 2];
      }
    }
    double best = DBL_MAX, bcp[3] = {0.0, 0.0, 0.0}, w = 0.0;
    for (uint32_t t0 = 0; t0 < nt; t0 += kTriTile) {
      __syncthreads();
      for (int k = threadIdx.x; k < kTriTile * 3; k += kBlock) {
        const uint32_t t = t0 + k / 3;
        if (t < nt) {
          uint32_t vi = tris[3 * t + k % 3];
          if (vi >= nv) vi = nv - 1;  // out-of-range indices must not read past the mesh
          s_tri[k / 3][3 * (k % 3)] = verts[3 * vi];
          s_tri[k / 3][3 * (k % 3) + 1] = verts[3 * vi + 1];
          s_tri[k / 3][3 * (k % 3) + 2] = verts[3 * vi + 2];
        }
      }
      __syncthreads();
      if (!valid) continue;
      const uint32_t cnt = (nt - t0) < (uint32_t)kTriTile ? (nt - t0) : (uint32_t)kTriTile;
      for (uint32_t t = 0; t < cnt; ++t) {
        const double* T = s_tri[t];
        double c3[3];
        const double d2 = point_triangle_dist2(q, T, T + 3, T + 6, c3);
        if (d2 < best) {
          best = d2;
          bcp[0] = c3[0];
          bcp[1] = c3[1];
          bcp[2] = c3[2];
        }
        w += solid_angle(q, T, T + 3, T + 6);
      }
    }
    if (!valid) continue;
    w /= 4.0 * 3.14159265358979323846;
    const double dist = sqrt(best);
    const double sd = (w > 0.5) ? -dist : dist;
    if (kLattice) {
      cpd[v] = make_float4((float)bcp[0], (float)bcp[1], (float)bcp[2], (float)sd);
      nrm[v] = make_float4((float)(q[0] - bcp[0]), (float)(q[1] - bcp[1]), (float)(q[2] - bcp[2]),
                           0.0f);
    } else {
      sdfOut[v] = sd;
      if (cpOut) {
        cpOut[3 * v] = bcp[0];
        cpOut[3 * v + 1] = bcp[1];
        cpOut[3 * v + 2] = bcp[2];
      }
    }
  }
}

unsigned sdf_blocks(uint64_t npts) {
  const unsigned g = grid_for(npts, kBlock);
  return g < kSdfMaxBlocks ? g : kSdfMaxBlocks;
}

// Grows the context's mesh scratch to `need` bytes (the tree: about 130 a
// triangle, 8 more per free point up to 2^22; a builder's copy of its mesh)
// and its sort scratch to `sorted` pairs.  False when there is no memory, or
// inside a graph capture, where they could not grow.  The callers then take
// the brute force alone.
bool tree_scratch(fc_context* ctx, uint32_t sorted, size_t need) {
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(ctx->stream, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone)
    return false;
  if (sorted > 0 && ensure_sort_capacity(ctx, sorted) != FC_SUCCESS) {
    (void)hipGetLastError();
    return false;
  }
  if (ctx->meshCapacity >= need) return true;
  if (hipStreamSynchronize(ctx->stream) != hipSuccess) return false;
  (void)hipFree(ctx->meshScratch);
  ctx->meshScratch = nullptr;
  ctx->meshCapacity = 0;
  if (hipMalloc(&ctx->meshScratch, need) != hipSuccess) {
    (void)hipGetLastError();
    ctx->meshScratch = nullptr;
    return false;
  }
  ctx->meshCapacity = need;
  return true;
}

}  // namespace

hipError_t launch_integrate_distmap(hipStream_t s, const fc_sim_params& P, const DistMapView& m,
                                    float4* pos, float4* vel, float dt, uint32_t n) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_integrate_distmap, dim3(grid_for(n, kBlock)), dim3(kBlock), 0, s, P, m,
                     pos, vel, dt, n);
  return hipGetLastError();
}

hipError_t launch_mesh_sdf_points(fc_context* ctx, const double* verts, uint32_t nv,
                                  const uint32_t* tris, uint32_t nt, const double* pts,
                                  uint64_t np, double* sdf, double* cp) {
  if (np == 0) return hipSuccess;
  hipStream_t s = ctx->stream;
  MeshTree T;
  if (mesh_tree_pays(nt, np) &&
      tree_scratch(ctx, tree_sort_pairs(nt, np), mesh_tree_bytes(nt) + tree_points_bytes(np))) {
    hipError_t e = launch_mesh_tree(ctx, verts, nv, tris, nt, ctx->meshScratch, &T);
    if (e == hipSuccess)
      e = launch_tree_points(ctx, T, verts, nv, tris, nt, pts, np,
                             static_cast<char*>(ctx->meshScratch) + mesh_tree_bytes(nt), sdf, cp);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(k_mesh_sdf<false>, dim3(sdf_blocks(np)), dim3(kBlock), 0, s, T.info, verts,
                     nv, tris, nt, np, pts, 0, 0, 0.0, 0.0, 0.0, 0.0, nullptr, nullptr, sdf, cp);
  return hipGetLastError();
}

}  // namespace fc

using namespace fc;

struct fc_distmap {
  fc_context* ctx = nullptr;
  int cells[3] = {0, 0, 0};
  float cellSize = 0.0f;
  float bmin[3] = {0, 0, 0};
  float bmax[3] = {0, 0, 0};
  void* block = nullptr;  // the allocation that the arrays below lie in
  float* xs = nullptr;
  float* ys = nullptr;
  float* zs = nullptr;
  float4* cpd = nullptr;
  float4* nrm = nullptr;
  size_t V = 0;
  std::vector<int32_t> fbm;  // stateFBM_ per vertex (host; empty = all 0)
};

namespace fc {

namespace {
// Smallest and largest vertex distance of each block of 8^3 cells (its
// 9^3 vertices); a NaN distance makes the block's bounds NaN.
__global__ __launch_bounds__(kBlock) void k_distmap_block_bounds(DistMapView m,
                                                                 float2* __restrict__ out,
                                                                 int bz) {
  const int nb = m.bx * m.by * bz;
  const int c = blockIdx.x * kBlock + threadIdx.x;
  if (c >= nb) return;
  const int ix = c % m.bx, iy = (c / m.bx) % m.by, iz = c / (m.bx * m.by);
  const int x0 = ix << kMapBlockShift, y0 = iy << kMapBlockShift, z0 = iz << kMapBlockShift;
  const int x1 = min(x0 + (1 << kMapBlockShift), m.cx), y1 = min(y0 + (1 << kMapBlockShift), m.cy),
            z1 = min(z0 + (1 << kMapBlockShift), m.cz);
  const int64_t sx = m.cx + 1, sxy = (int64_t)(m.cx + 1) * (m.cy + 1);
  float lo = INFINITY, hi = -INFINITY;
  bool nan = false;
  for (int z = z0; z <= z1; ++z)
    for (int y = y0; y <= y1; ++y)
      for (int x = x0; x <= x1; ++x) {
        const float d = m.cpd[z * sxy + y * sx + x].w;
        nan = nan || d != d;
        lo = fminf(lo, d);
        hi = fmaxf(hi, d);
      }
  out[c] = nan ? make_float2(NAN, NAN) : make_float2(lo, hi);
}
}  // namespace

fc_status distmap_block_bounds(const fc_distmap* m, hipStream_t s, float2** out, int* bx,
                               int* by) {
  *out = nullptr;
  *bx = *by = 0;
  // only on the uniform lattice bmin + i cellSize (see distmap_far)
  const float* coords[3] = {m->xs, m->ys, m->zs};
  for (int a = 0; a < 3; ++a) {
    std::vector<float> c((size_t)m->cells[a] + 1);
    FC_HIP_TRY(hipMemcpy(c.data(), coords[a], c.size() * sizeof(float), hipMemcpyDeviceToHost));
    for (size_t i = 0; i < c.size(); ++i) {
      const double want = (double)m->bmin[a] + (double)i * (double)m->cellSize;
      if (!(std::fabs((double)c[i] - want) <= 1e-5 * (double)m->cellSize)) return FC_SUCCESS;
    }
  }
  const int nbx = (m->cells[0] + (1 << kMapBlockShift) - 1) >> kMapBlockShift;
  const int nby = (m->cells[1] + (1 << kMapBlockShift) - 1) >> kMapBlockShift;
  const int nbz = (m->cells[2] + (1 << kMapBlockShift) - 1) >> kMapBlockShift;
  const size_t nb = (size_t)nbx * nby * nbz;
  float2* d = nullptr;
  FC_HIP_TRY(hipMalloc(&d, nb * sizeof(float2)));
  DistMapView v = distmap_view(m);
  v.bx = nbx;
  v.by = nby;
  hipLaunchKernelGGL(k_distmap_block_bounds, dim3((unsigned)((nb + kBlock - 1) / kBlock)),
                     dim3(kBlock), 0, s, v, d, nbz);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) {
    (void)hipFree(d);
    return hip_error(e, "distance-map block bounds");
  }
  *out = d;
  *bx = nbx;
  *by = nby;
  return FC_SUCCESS;
}

DistMapView distmap_view(const fc_distmap* m) {
  DistMapView v;
  v.cx = m->cells[0];
  v.cy = m->cells[1];
  v.cz = m->cells[2];
  v.cellSize = m->cellSize;
  for (int a = 0; a < 3; ++a) {
    v.bmin[a] = m->bmin[a];
    v.bmax[a] = m->bmax[a];
  }
  v.xs = m->xs;
  v.ys = m->ys;
  v.zs = m->zs;
  v.cpd = m->cpd;
  v.nrm = m->nrm;
  return v;
}

}  // namespace fc

namespace {

// Where the coordinates of axis a start in the map's allocation, in floats
// (a = 3: their end).
size_t axis_offset(const fc_distmap* m, int a) {
  size_t at = 0;
  for (int k = 0; k < a; ++k) at += ((size_t)m->cells[k] + 1 + 63) / 64 * 64;
  return at;
}

// Uploads the lattice coordinates of the three axes in one copy.
hipError_t upload_axes(fc_distmap* m, const std::vector<float> ax[3], hipStream_t s) {
  std::vector<float> host(axis_offset(m, 3), 0.0f);
  for (int a = 0; a < 3; ++a) std::copy(ax[a].begin(), ax[a].end(), host.begin() + axis_offset(m, a));
  hipError_t e = hipMemcpyAsync(m->block, host.data(), host.size() * sizeof(float),
                                hipMemcpyHostToDevice, s);
  return e == hipSuccess ? hipStreamSynchronize(s) : e;
}

fc_status alloc_map(fc_context* ctx, const int32_t cells[3], fc_distmap** out) {
  for (int a = 0; a < 3; ++a)
    if (cells[a] < 1) return set_error(FC_ERROR_INVALID_VALUE, "cells must be >= 1 per axis");
  const size_t V = (size_t)(cells[0] + 1) * (cells[1] + 1) * (cells[2] + 1);
  if (V > ((size_t)1 << 33)) return set_error(FC_ERROR_CAPACITY, "distance map too large");
  fc_distmap* m = new fc_distmap();
  m->ctx = ctx;
  for (int a = 0; a < 3; ++a) m->cells[a] = cells[a];
  m->V = V;
  // one allocation: the axes (axis_offset's layout), then the vertices' arrays
  const size_t axes = axis_offset(m, 3);
  const hipError_t e = hipMalloc(&m->block, axes * sizeof(float) + 2 * V * sizeof(float4));
  if (e == hipSuccess) {
    float* at = static_cast<float*>(m->block);
    m->xs = at;
    m->ys = at + axis_offset(m, 1);
    m->zs = at + axis_offset(m, 2);
    m->cpd = reinterpret_cast<float4*>(at + axes);
    m->nrm = m->cpd + V;
  }
  if (e != hipSuccess) {
    fc_distmap_destroy(m);
    return hip_error(e, "distance map allocation");
  }
  *out = m;
  return FC_SUCCESS;
}

// Text map file of RigidBody::buildDistanceMapFromFile /
// storeDistanceMapToFile (rigidbody.cpp:1214-1376): "dim0 dim1", "cx cy cz",
// "cellSize", then (cx+1)(cy+1)(cz+1) lines each of vertex coordinates,
// closest points, normals (3 values), distances and FBM states (1 value).
// Like the reference's stream reads, each record's numbers are read across
// whitespace and line breaks and the rest of its last line is skipped.
struct MapFileReader {
  std::string text;
  size_t at = 0;
  bool ok = true;

  void skip_space() {
    while (at < text.size() && (text[at] == ' ' || text[at] == '\t' || text[at] == '\n' ||
                                text[at] == '\r' || text[at] == '\v' || text[at] == '\f'))
      ++at;
  }
  void end_line() {
    while (at < text.size() && text[at] != '\n') ++at;
    if (at < text.size()) ++at;
  }
  double real() {
    skip_space();
    if (at >= text.size()) { ok = false; return 0.0; }
    double v = 0.0;
    const char* b = text.data() + at;
    const char* e = text.data() + text.size();
    if (*b == '+') ++b;  // from_chars takes no leading plus; stream extraction does
    auto r = std::from_chars(b, e, v);
    if (r.ec != std::errc() && r.ec != std::errc::result_out_of_range) { ok = false; return 0.0; }
    at = (size_t)(r.ptr - text.data());
    return v;
  }
  long long integer() {
    skip_space();
    if (at >= text.size()) { ok = false; return 0; }
    long long v = 0;
    const char* b = text.data() + at;
    const char* e = text.data() + text.size();
    if (*b == '+') ++b;
    auto r = std::from_chars(b, e, v);
    if (r.ec != std::errc()) { ok = false; return 0; }
    at = (size_t)(r.ptr - text.data());
    return v;
  }
};

struct MapFileData {
  int32_t dim[2] = {0, 0};
  int32_t cells[3] = {0, 0, 0};
  double cellSize = 0.0;
  std::vector<double> coords, cps, normals, dist;  // 3, 3, 3, 1 per vertex
  std::vector<int32_t> fbm;
};

fc_status read_map_file(const char* path, bool headerOnly, MapFileData& d) {
  std::ifstream f(path, std::ios::binary);
  if (!f.is_open()) return set_error(FC_ERROR_INVALID_VALUE, std::string("cannot open ") + path);
  MapFileReader r;
  try {
    r.text.assign(std::istreambuf_iterator<char>(f), std::istreambuf_iterator<char>());
  } catch (const std::bad_alloc&) {
    return set_error(FC_ERROR_OUT_OF_MEMORY, "map file: text buffer");
  }
  d.dim[0] = (int32_t)r.integer();
  d.dim[1] = (int32_t)r.integer();
  r.end_line();
  for (int a = 0; a < 3; ++a) d.cells[a] = (int32_t)r.integer();
  r.end_line();
  d.cellSize = r.real();
  r.end_line();
  if (!r.ok) return set_error(FC_ERROR_INVALID_VALUE, "map file: bad header");
  for (int a = 0; a < 3; ++a)
    if (d.cells[a] < 1 || d.cells[a] > 4096)
      return set_error(FC_ERROR_INVALID_VALUE, "map file: cell counts outside [1, 4096]");
  if (headerOnly) return FC_SUCCESS;
  const size_t V = (size_t)(d.cells[0] + 1) * (d.cells[1] + 1) * (d.cells[2] + 1);
  if (V > (size_t(1) << 27)) return set_error(FC_ERROR_CAPACITY, "map file: more than 2^27 vertices");
  try {
    d.coords.resize(3 * V);
    d.cps.resize(3 * V);
    d.normals.resize(3 * V);
    d.dist.resize(V);
    d.fbm.resize(V);
  } catch (const std::bad_alloc&) {
    return set_error(FC_ERROR_OUT_OF_MEMORY, "map file: host arrays");
  }
  std::vector<double>* tri[3] = {&d.coords, &d.cps, &d.normals};
  for (auto* t : tri) {
    for (size_t v = 0; v < V && r.ok; ++v) {
      (*t)[3 * v] = r.real();
      (*t)[3 * v + 1] = r.real();
      (*t)[3 * v + 2] = r.real();
      r.end_line();
    }
  }
  for (size_t v = 0; v < V && r.ok; ++v) {
    d.dist[v] = r.real();
    r.end_line();
  }
  for (size_t v = 0; v < V && r.ok; ++v) {
    d.fbm[v] = (int32_t)r.integer();
    r.end_line();
  }
  if (!r.ok) return set_error(FC_ERROR_INVALID_VALUE, "map file: truncated or malformed data");
  return FC_SUCCESS;
}

}  // namespace

extern "C" {

fc_status fc_distmap_file_read(const char* path, int32_t cells[3], double* cellSize,
                               int32_t dim[2], double* vertexCoords, double* contactPoints,
                               double* normals, double* distance, int32_t* stateFBM) {
  if (!path || !cells || !cellSize) return set_error(FC_ERROR_INVALID_VALUE, "NULL argument");
  const bool headerOnly =
      !vertexCoords && !contactPoints && !normals && !distance && !stateFBM;
  MapFileData d;
  FC_TRY(read_map_file(path, headerOnly, d));
  for (int a = 0; a < 3; ++a) cells[a] = d.cells[a];
  *cellSize = d.cellSize;
  if (dim) {
    dim[0] = d.dim[0];
    dim[1] = d.dim[1];
  }
  if (headerOnly) return FC_SUCCESS;
  const size_t V = d.dist.size();
  if (vertexCoords) std::copy(d.coords.begin(), d.coords.end(), vertexCoords);
  if (contactPoints) std::copy(d.cps.begin(), d.cps.end(), contactPoints);
  if (normals) std::copy(d.normals.begin(), d.normals.end(), normals);
  if (distance) std::copy(d.dist.begin(), d.dist.end(), distance);
  if (stateFBM) std::copy(d.fbm.begin(), d.fbm.begin() + V, stateFBM);
  return FC_SUCCESS;
}

fc_status fc_distmap_load(fc_context* ctx, const char* path, const float bmin[3],
                          const float bmax[3], fc_distmap** out) {
  if (!ctx || !path || !out) return set_error(FC_ERROR_INVALID_VALUE, "NULL argument");
  if ((bmin == nullptr) != (bmax == nullptr))
    return set_error(FC_ERROR_INVALID_VALUE, "give both box corners or neither");
  *out = nullptr;
  MapFileData d;
  FC_TRY(read_map_file(path, false, d));
  const size_t V = d.dist.size();
  // binary64 -> binary32 as the conversion constructor does
  // (DistanceMap<float,cpu>(DistanceMap<Real,cpu>*), distancemap.cpp:129-178)
  std::vector<float> c, p, nn, ds;
  try {
    c.resize(3 * V);
    p.resize(3 * V);
    nn.resize(3 * V);
    ds.resize(V);
  } catch (const std::bad_alloc&) {
    return set_error(FC_ERROR_OUT_OF_MEMORY, "map file: float arrays");
  }
  for (size_t i = 0; i < 3 * V; ++i) {
    c[i] = (float)d.coords[i];
    p[i] = (float)d.cps[i];
    nn[i] = (float)d.normals[i];
  }
  for (size_t v = 0; v < V; ++v) ds[v] = (float)d.dist[v];
  float lo[3], hi[3];
  for (int a = 0; a < 3; ++a) {
    lo[a] = bmin ? bmin[a] : c[a];
    hi[a] = bmax ? bmax[a] : c[3 * (V - 1) + a];
  }
  fc_distmap* m = nullptr;
  FC_TRY(fc_distmap_create(ctx, d.cells, (float)d.cellSize, lo, hi, c.data(), nn.data(), p.data(),
                           ds.data(), &m));
  m->fbm = std::move(d.fbm);
  *out = m;
  return FC_SUCCESS;
}

fc_status fc_distmap_save(fc_context* ctx, const fc_distmap* m, const char* path) {
  if (!ctx || !m || !path) return set_error(FC_ERROR_INVALID_VALUE, "NULL argument");
  const size_t V = m->V;
  std::vector<float> c(3 * V), p(3 * V), nn(3 * V), ds(V);
  FC_TRY(fc_distmap_download(ctx, m, c.data(), nn.data(), p.data(), ds.data()));
  std::FILE* f = std::fopen(path, "w");
  if (!f) return set_error(FC_ERROR_INVALID_VALUE, std::string("cannot write ") + path);
  // %.9g: nine significant digits give every binary32 value back exactly
  // (the reference writes six).
  std::fprintf(f, "%d %d\n", m->cells[0] + 1, (m->cells[1] + 1) * (m->cells[2] + 1));
  std::fprintf(f, "%d %d %d\n", m->cells[0], m->cells[1], m->cells[2]);
  std::fprintf(f, "%.9g\n", (double)m->cellSize);
  const float* tri[3] = {c.data(), p.data(), nn.data()};
  for (const float* t : tri)
    for (size_t v = 0; v < V; ++v)
      std::fprintf(f, "%.9g %.9g %.9g\n", (double)t[3 * v], (double)t[3 * v + 1],
                   (double)t[3 * v + 2]);
  for (size_t v = 0; v < V; ++v) std::fprintf(f, "%.9g\n", (double)ds[v]);
  for (size_t v = 0; v < V; ++v) std::fprintf(f, "%d\n", m->fbm.empty() ? 0 : (int)m->fbm[v]);
  const bool bad = std::ferror(f) != 0;
  if (std::fclose(f) != 0 || bad) return set_error(FC_ERROR_INVALID_VALUE, "map file write failed");
  return FC_SUCCESS;
}

fc_status fc_distmap_get_fbm(const fc_distmap* m, int32_t* stateFBM) {
  if (!m || !stateFBM) return set_error(FC_ERROR_INVALID_VALUE, "NULL argument");
  for (size_t v = 0; v < m->V; ++v) stateFBM[v] = m->fbm.empty() ? 0 : m->fbm[v];
  return FC_SUCCESS;
}

fc_status fc_distmap_set_fbm(fc_distmap* m, const int32_t* stateFBM) {
  if (!m) return set_error(FC_ERROR_INVALID_VALUE, "NULL argument");
  if (!stateFBM) {
    m->fbm.clear();
    return FC_SUCCESS;
  }
  m->fbm.assign(stateFBM, stateFBM + m->V);
  return FC_SUCCESS;
}

fc_status fc_distmap_query_fbm(fc_context* ctx, const fc_distmap* m, const float* points,
                               uint32_t n, int32_t* out) {
  if (!ctx || !m) return set_error(FC_ERROR_INVALID_VALUE, "NULL argument");
  if (n == 0) return FC_SUCCESS;
  if (!points || !out) return set_error(FC_ERROR_INVALID_VALUE, "NULL array");
  hipLaunchKernelGGL(k_distmap_query_fbm, dim3(grid_for(n, kBlock)), dim3(kBlock), 0,
                     ctx->stream, distmap_view(m), points, n, out);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_error(e, "distmap queryFBM");
  return FC_SUCCESS;
}

fc_status fc_distmap_create(fc_context* ctx, const int32_t cells[3], float cellSize,
                            const float bmin[3], const float bmax[3], const float* vertexCoords,
                            const float* normals, const float* contactPoints,
                            const float* distance, fc_distmap** out) {
  if (!ctx || !cells || !bmin || !bmax || !vertexCoords || !normals || !contactPoints ||
      !distance || !out)
    return set_error(FC_ERROR_INVALID_VALUE, "NULL argument");
  *out = nullptr;
  fc_distmap* m = nullptr;
  FC_TRY(alloc_map(ctx, cells, &m));
  const int cx = cells[0], cy = cells[1], cz = cells[2];
  const size_t ix = cx + 1, islice = ix * (cy + 1), V = m->V;
  std::vector<float> ax[3] = {std::vector<float>(cx + 1), std::vector<float>(cy + 1),
                              std::vector<float>(cz + 1)};
  std::vector<float>&xs = ax[0], &ys = ax[1], &zs = ax[2];
  for (int i = 0; i <= cx; ++i) xs[i] = vertexCoords[3 * i];
  for (int i = 0; i <= cy; ++i) ys[i] = vertexCoords[3 * (i * ix) + 1];
  for (int i = 0; i <= cz; ++i) zs[i] = vertexCoords[3 * (i * islice) + 2];
  std::vector<float4> cpd(V), nrm(V);
  for (size_t v = 0; v < V; ++v) {
    const size_t z = v / islice, y = (v % islice) / ix, x = v % ix;
    if (vertexCoords[3 * v] != xs[x] || vertexCoords[3 * v + 1] != ys[y] ||
        vertexCoords[3 * v + 2] != zs[z]) {
      fc_distmap_destroy(m);
      return set_error(FC_ERROR_INVALID_VALUE,
                       "vertex coordinates are not a tensor-product lattice");
    }
    cpd[v] = make_float4(contactPoints[3 * v], contactPoints[3 * v + 1],
                         contactPoints[3 * v + 2], distance[v]);
    nrm[v] = make_float4(normals[3 * v], normals[3 * v + 1], normals[3 * v + 2], 0.0f);
  }
  m->cellSize = cellSize;
  for (int a = 0; a < 3; ++a) {
    m->bmin[a] = bmin[a];
    m->bmax[a] = bmax[a];
  }
  hipStream_t st = ctx->stream;
  hipError_t e = upload_axes(m, ax, st);
  if (e == hipSuccess) e = hipMemcpyAsync(m->cpd, cpd.data(), V * 16, hipMemcpyHostToDevice, st);
  if (e == hipSuccess) e = hipMemcpyAsync(m->nrm, nrm.data(), V * 16, hipMemcpyHostToDevice, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  if (e != hipSuccess) {
    fc_distmap_destroy(m);
    return hip_error(e, "distance map upload");
  }
  *out = m;
  return FC_SUCCESS;
}

fc_status fc_distmap_build(fc_context* ctx, const double* vertices, uint32_t numVertices,
                           const uint32_t* triangles, uint32_t numTriangles,
                           const int32_t cells[3], float cellSize, const float bmin[3],
                           fc_distmap** out) {
  if (!ctx || !vertices || !triangles || !cells || !bmin || !out)
    return set_error(FC_ERROR_INVALID_VALUE, "NULL argument");
  if (numTriangles == 0 || numVertices == 0)
    return set_error(FC_ERROR_INVALID_VALUE, "empty mesh");
  if (!(cellSize > 0.0f)) return set_error(FC_ERROR_INVALID_VALUE, "cellSize must be positive");
  for (uint64_t i = 0; i < 3ull * numTriangles; ++i)
    if (triangles[i] >= numVertices)
      return set_error(FC_ERROR_INVALID_VALUE, "triangle index out of range");
  *out = nullptr;
  fc_distmap* m = nullptr;
  FC_TRY(alloc_map(ctx, cells, &m));
  const double cs = cellSize, b[3] = {bmin[0], bmin[1], bmin[2]};
  std::vector<float> ax[3];
  for (int a = 0; a < 3; ++a) {
    ax[a].resize(cells[a] + 1);
    for (int i = 0; i <= cells[a]; ++i) ax[a][i] = (float)(b[a] + (double)i * cs);
    m->bmin[a] = bmin[a];
    m->bmax[a] = (float)(b[a] + (double)cells[a] * cs);
  }
  m->cellSize = cellSize;
  hipStream_t st = ctx->stream;
  // the mesh's copy lies in the context's scratch, after the tree; a large one
  // (the tree's own part is bounded by its 2^22 triangles) is not kept there
  const size_t vb = (size_t)numVertices * 3 * sizeof(double),
               tb = (size_t)numTriangles * 3 * sizeof(uint32_t);
  const bool keep = vb + tb <= kMeshCopyKept;
  const bool tree = mesh_tree_pays(numTriangles, m->V) && tree_lattice_fits(cells, b, cs);
  const size_t at = tree ? mesh_tree_bytes(numTriangles) : 0;
  hipError_t e = hipSuccess;
  void* own = nullptr;
  const bool scratch = tree_scratch(ctx, tree ? numTriangles : 0, at + (keep ? vb + tb : 0));
  const bool kept = scratch && keep;
  if (!kept) e = hipMalloc(&own, vb + tb);
  double* dv = reinterpret_cast<double*>(kept ? static_cast<char*>(ctx->meshScratch) + at
                                              : static_cast<char*>(own));
  uint32_t* dt = reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(dv) + vb);
  if (e == hipSuccess) e = hipMemcpyAsync(dv, vertices, vb, hipMemcpyHostToDevice, st);
  if (e == hipSuccess) e = hipMemcpyAsync(dt, triangles, tb, hipMemcpyHostToDevice, st);
  if (e == hipSuccess) e = upload_axes(m, ax, st);
  MeshTree T;
  if (e == hipSuccess && tree && scratch) {
    e = launch_mesh_tree(ctx, dv, numVertices, dt, numTriangles, ctx->meshScratch, &T);
    if (e == hipSuccess)
      e = launch_tree_lattice(st, T, dv, numVertices, dt, numTriangles, m->cells, b, cs, m->cpd,
                              m->nrm);
  }
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_mesh_sdf<true>, dim3(sdf_blocks(m->V)), dim3(kBlock), 0, st, T.info, dv,
                       numVertices, dt, numTriangles, (uint64_t)m->V, nullptr, cells[0], cells[1],
                       b[0], b[1], b[2], cs, m->cpd, m->nrm, nullptr, nullptr);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  hipFree(own);
  if (e != hipSuccess) {
    fc_distmap_destroy(m);
    return hip_error(e, "distance map build");
  }
  *out = m;
  return FC_SUCCESS;
}

fc_status fc_distmap_destroy(fc_distmap* m) {
  if (!m) return FC_SUCCESS;
  // No use of m->ctx: the context may already be gone; hipFree waits for
  // the device.
  hipFree(m->block);
  delete m;
  return FC_SUCCESS;
}

fc_status fc_distmap_info(const fc_distmap* m, int32_t cells[3], float* cellSize, float bmin[3],
                          float bmax[3]) {
  if (!m) return set_error(FC_ERROR_INVALID_VALUE, "map is NULL");
  for (int a = 0; a < 3; ++a) {
    if (cells) cells[a] = m->cells[a];
    if (bmin) bmin[a] = m->bmin[a];
    if (bmax) bmax[a] = m->bmax[a];
  }
  if (cellSize) *cellSize = m->cellSize;
  return FC_SUCCESS;
}

fc_status fc_distmap_download(fc_context* ctx, const fc_distmap* m, float* vertexCoords,
                              float* normals, float* contactPoints, float* distance) {
  if (!ctx || !m) return set_error(FC_ERROR_INVALID_VALUE, "NULL argument");
  const size_t V = m->V, ix = m->cells[0] + 1, islice = ix * (m->cells[1] + 1);
  std::vector<float4> cpd(V), nrm(V);
  std::vector<float> ax[3];
  const float* src[3] = {m->xs, m->ys, m->zs};
  hipStream_t st = ctx->stream;
  hipError_t e = hipSuccess;
  for (int a = 0; a < 3 && e == hipSuccess; ++a) {
    ax[a].resize(m->cells[a] + 1);
    e = hipMemcpyAsync(ax[a].data(), src[a], ax[a].size() * 4, hipMemcpyDeviceToHost, st);
  }
  if (e == hipSuccess) e = hipMemcpyAsync(cpd.data(), m->cpd, V * 16, hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipMemcpyAsync(nrm.data(), m->nrm, V * 16, hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  if (e != hipSuccess) return hip_error(e, "distance map download");
  for (size_t v = 0; v < V; ++v) {
    const size_t z = v / islice, y = (v % islice) / ix, x = v % ix;
    if (vertexCoords) {
      vertexCoords[3 * v] = ax[0][x];
      vertexCoords[3 * v + 1] = ax[1][y];
      vertexCoords[3 * v + 2] = ax[2][z];
    }
    if (contactPoints) {
      contactPoints[3 * v] = cpd[v].x;
      contactPoints[3 * v + 1] = cpd[v].y;
      contactPoints[3 * v + 2] = cpd[v].z;
    }
    if (distance) distance[v] = cpd[v].w;
    if (normals) {
      normals[3 * v] = nrm[v].x;
      normals[3 * v + 1] = nrm[v].y;
      normals[3 * v + 2] = nrm[v].z;
    }
  }
  return FC_SUCCESS;
}

fc_status fc_distmap_query(fc_context* ctx, const fc_distmap* m, const float* points, uint32_t n,
                           float* dist, float* cp, float* normal) {
  if (!ctx || !m) return set_error(FC_ERROR_INVALID_VALUE, "NULL argument");
  if (n == 0) return FC_SUCCESS;
  if (!points || !dist) return set_error(FC_ERROR_INVALID_VALUE, "NULL array");
  // From 2^17 points on two threads take a point (k_distmap_query_pairs);
  // fewer do not fill the card, and a thread each is up to 7 % faster: 100,000
  // points in 32^3 / 64^3 cells 5.3 / 7.5 us against 5.6 / 7.3, 200,000 in 32^3
  // 8.5 against 8.3.
  if (n < (1u << 17)) {
    hipLaunchKernelGGL(k_distmap_query, dim3(grid_for(n, kBlock)), dim3(kBlock), 0, ctx->stream,
                       distmap_view(m), points, n, dist, cp, normal);
  } else {
    constexpr uint64_t kMost = 1ull << 30;  // points of one launch
    for (uint64_t at = 0; at < n; at += kMost) {
      const uint32_t count = (uint32_t)std::min<uint64_t>(n - at, kMost);
      hipLaunchKernelGGL(k_distmap_query_pairs, dim3(grid_for(2 * (uint64_t)count, kBlock)),
                         dim3(kBlock), 0, ctx->stream, distmap_view(m), points + 3 * at, count,
                         dist + at, cp ? cp + 3 * at : nullptr,
                         normal ? normal + 3 * at : nullptr);
    }
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_error(e, "distmap query");
  return FC_SUCCESS;
}

fc_status fc_distmap_eval(fc_context* ctx, const fc_distmap* m, const float* v, uint32_t n,
                          const fc_trans_info* info, float* cps, float* normals,
                          float* distance) {
  if (!ctx || !m || !info) return set_error(FC_ERROR_INVALID_VALUE, "NULL argument");
  if (n == 0) return FC_SUCCESS;
  if (!v || !cps || !normals || !distance) return set_error(FC_ERROR_INVALID_VALUE, "NULL array");
  hipLaunchKernelGGL(k_distmap_eval, dim3(grid_for(n, kBlock)), dim3(kBlock), 0, ctx->stream,
                     distmap_view(m), *info, v, n, cps, normals, distance);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_error(e, "eval_distmap");
  return FC_SUCCESS;
}

fc_status fc_mesh_mesh_contacts(fc_context* ctx, const fc_distmap* m, const float* v, uint32_t n,
                                const fc_trans_info* info, float threshold, float* cps,
                                float* normals, uint32_t* vertexIds, uint32_t capacity,
                                uint32_t* numContacts) {
  if (!ctx || !m || !info || !numContacts) return set_error(FC_ERROR_INVALID_VALUE, "NULL argument");
  *numContacts = 0;
  if (n == 0) return FC_SUCCESS;
  if (!v || (capacity > 0 && (!cps || !normals || !vertexIds)))
    return set_error(FC_ERROR_INVALID_VALUE, "NULL array");
  const uint32_t blocks = grid_for(n, kBlock);
  uint32_t* dCounts = nullptr;
  hipError_t e = hipMalloc(&dCounts, (size_t)blocks * sizeof(uint32_t));
  if (e != hipSuccess) return hip_error(e, "contact counts");
  hipStream_t st = ctx->stream;
  const DistMapView view = distmap_view(m);
  hipLaunchKernelGGL(k_mesh_contacts_count, dim3(blocks), dim3(kBlock), 0, st, view, *info, v, n,
                     threshold, dCounts);
  e = hipGetLastError();
  std::vector<uint32_t> counts(blocks);
  if (e == hipSuccess)
    e = hipMemcpyAsync(counts.data(), dCounts, (size_t)blocks * 4, hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  uint64_t total = 0;
  for (uint32_t b = 0; b < blocks; ++b) {
    const uint32_t c = counts[b];
    counts[b] = (uint32_t)total;
    total += c;
  }
  if (e == hipSuccess && total > 0 && capacity > 0) {
    e = hipMemcpyAsync(dCounts, counts.data(), (size_t)blocks * 4, hipMemcpyHostToDevice, st);
    if (e == hipSuccess) {
      hipLaunchKernelGGL(k_mesh_contacts_write, dim3(blocks), dim3(kBlock), 0, st, view, *info, v,
                         n, threshold, dCounts, capacity, cps, normals, vertexIds);
      e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipStreamSynchronize(st);
  }
  hipFree(dCounts);
  if (e != hipSuccess) return hip_error(e, "mesh-mesh contacts");
  *numContacts = (uint32_t)total;
  return FC_SUCCESS;
}

fc_status fc_integrate_system_distmap(fc_context* ctx, const fc_distmap* m, float* pos, float* vel,
                                      float deltaTime, uint32_t numParticles) {
  if (!ctx || !m) return set_error(FC_ERROR_INVALID_VALUE, "NULL argument");
  if (numParticles == 0) return FC_SUCCESS;
  if (!pos || !vel) return set_error(FC_ERROR_INVALID_VALUE, "NULL array");
  hipError_t e = launch_integrate_distmap(ctx->stream, ctx->params, distmap_view(m), (float4*)pos,
                                          (float4*)vel, deltaTime, numParticles);
  if (e != hipSuccess) return hip_error(e, "integrate (distance map)");
  return FC_SUCCESS;
}

fc_status fc_mesh_signed_distance(fc_context* ctx, const double* vertices, uint32_t numVertices,
                                  const uint32_t* triangles, uint32_t numTriangles,
                                  const double* points, uint32_t numPoints, double* sdf,
                                  double* closest) {
  if (!ctx || !vertices || !triangles || !points || !sdf)
    return set_error(FC_ERROR_INVALID_VALUE, "NULL argument");
  if (numPoints == 0) return FC_SUCCESS;
  if (numTriangles == 0) return set_error(FC_ERROR_INVALID_VALUE, "empty mesh");
  if (numVertices == 0) return set_error(FC_ERROR_INVALID_VALUE, "empty mesh");
  hipError_t e = launch_mesh_sdf_points(ctx, vertices, numVertices, triangles, numTriangles,
                                        points, numPoints, sdf, closest);
  if (e != hipSuccess) return hip_error(e, "mesh signed distance");
  return FC_SUCCESS;
}

}  // extern "C"
