// Tree over a mesh's triangles for the exact point-mesh distance
// (mesh_tree.hip): eight-wide, implicit, rebuilt on the device per call.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

struct fc_context;

namespace fc {

// What one pass over the triangles finds, on the device: the corners'
// bounds (as order-preserving keys), two sums over the directed edges that
// are zero when every edge (a, b) is matched by an edge (b, a), and whether
// any corner is not finite.
struct MeshInfo {
  unsigned long long lo[3], hi[3];
  unsigned long long edges[2];
  uint32_t bad;
  uint32_t open;  // 1 when mesh_closed is false (k_mesh_order)
};

// A triangle in tree order: its corners and its number in the mesh.
struct TreeTri {
  double v[9];
  unsigned long long id;
};

constexpr int kTreeMaxLevels = 8;  // 8^8 triangles
// Level l holds count[l] boxes (level 0 one per triangle), eight to a group:
// float lo.x[8] lo.y[8] lo.z[8] hi.x[8] hi.y[8] hi.z[8], rounded outwards.
// Box g of level l + 1 bounds group g of level l.
struct MeshTree {
  const TreeTri* tri = nullptr;
  const float* box[kTreeMaxLevels] = {};
  uint32_t count[kTreeMaxLevels] = {};
  int levels = 0;
  const MeshInfo* info = nullptr;
};

__device__ __forceinline__ double mesh_key_value(unsigned long long k) {
  const unsigned long long u = (k >> 63) ? (k & 0x7fffffffffffffffull) : ~k;
  return __longlong_as_double((long long)u);
}

// The tree's boxes are compared in binary32: squared distances of points and
// meshes within this range stay in its range.
constexpr double kTreeRange = 1e15;

// Largest corner coordinate by magnitude.
__device__ __forceinline__ double mesh_magnitude(const MeshInfo& I) {
  double m = 0.0;
#pragma unroll
  for (int a = 0; a < 3; ++a)
    m = fmax(m, fmax(fabs(mesh_key_value(I.lo[a])), fabs(mesh_key_value(I.hi[a]))));
  return m;
}

// Whether the tree's signs hold: the mesh is closed and consistently
// oriented (every directed edge matched by its opposite, by two 64-bit
// sums), finite, and of a magnitude whose squares stay in range.  The
// brute-force kernel takes the meshes for which it is false.
__device__ __forceinline__ bool mesh_closed(const MeshInfo& I) {
  const double m = mesh_magnitude(I);
  return I.bad == 0u && I.edges[0] == 0ull && I.edges[1] == 0ull && m < kTreeRange &&
         m > 1.0 / kTreeRange;
}

// Meshes of fewer triangles take the brute force: see mesh_tree.hip.
bool mesh_tree_pays(uint32_t nt, uint64_t npts);
// Whether the lattice's launches stay within the grid limits, and its
// coordinates within kTreeRange.
bool tree_lattice_fits(const int cells[3], const double bmin[3], double cs);
// Device bytes the tree of nt triangles needs.
size_t mesh_tree_bytes(uint32_t nt);
// Builds the tree of the mesh (device arrays; triangle indices are clamped
// below nv) in `block` (mesh_tree_bytes(nt) bytes) on the context's stream;
// the context's sort scratch must hold nt pairs.
hipError_t launch_mesh_tree(fc_context* ctx, const double* verts, uint32_t nv,
                            const uint32_t* tris, uint32_t nt, void* block, MeshTree* out);
// Distance maps' vertices (cpd, nrm as in DistMapView) or free points; does
// nothing when mesh_closed is false.
hipError_t launch_tree_lattice(hipStream_t s, const MeshTree& T, const double* verts, uint32_t nv,
                               const uint32_t* tris, uint32_t nt, const int cells[3],
                               const double bmin[3], double cs, float4* cpd, float4* nrm);
hipError_t launch_tree_points(fc_context* ctx, const MeshTree& T, const double* verts,
                              uint32_t nv, const uint32_t* tris, uint32_t nt, const double* pts,
                              uint64_t np, void* block, double* sdf, double* cp);
// Device bytes the free points' order needs in `block`, and the pairs the
// context's sort scratch must hold for a mesh and its points.
size_t tree_points_bytes(uint64_t np);
uint32_t tree_sort_pairs(uint32_t nt, uint64_t np);

}  // namespace fc
