// Exact point-triangle geometry in binary64, shared by the brute-force mesh
// distance (distmap.hip) and the triangle tree (mesh_tree.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <cmath>
#include <cstdint>

namespace fc {

// Squared distance from q to triangle (B, V1, V2) and the closest point, by
// the region method of D. Eberly, "Distance Between Point and Triangle in
// 3D" (Geometric Tools), in binary64.  (The reference's variant,
// distance/distancetriangle.cpp:55-190, departs from it in regions 4 and 6.)
__host__ __device__ __forceinline__ double point_triangle_dist2(const double q[3],
                                                                const double* B, const double* V1,
                                                                const double* V2, double cp[3]) {
  double E0[3], E1[3], D[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    E0[k] = V1[k] - B[k];
    E1[k] = V2[k] - B[k];
    D[k] = B[k] - q[k];
  }
  const double a = E0[0] * E0[0] + E0[1] * E0[1] + E0[2] * E0[2];
  const double b = E0[0] * E1[0] + E0[1] * E1[1] + E0[2] * E1[2];
  const double c = E1[0] * E1[0] + E1[1] * E1[1] + E1[2] * E1[2];
  const double d = E0[0] * D[0] + E0[1] * D[1] + E0[2] * D[2];
  const double e = E1[0] * D[0] + E1[1] * D[1] + E1[2] * D[2];
  const double det = a * c - b * b;
  double s = b * e - c * d, t = b * d - a * e;
  // The regions differ in the edge they clamp to, all with one quotient: on
  // E0 (t = 0) -d / a, on E1 (s = 0) -e / c, on the third edge s or t =
  // (difference of its ends' slopes) / |E1 - E0|^2, each within [0, 1]; inside,
  // 1 / det.  The operands are picked first, so that a wave whose lanes lie in
  // different regions divides once.
  const bool inner = s + t <= det, sNeg = s < 0.0, tNeg = t < 0.0;
  const double ce = c + e, bd = b + d, ad = a + d, be = b + e;
  const bool inside = inner && !sNeg && !tNeg;                      // region 0
  const bool third2 = !inner && sNeg && ce > bd;                    // region 2
  const bool third6 = !inner && !sNeg && tNeg && ad > be;           // region 6
  const bool third = third2 || third6 || (!inner && !sNeg && !tNeg);  // region 1
  // regions 4 (one side), 5 and 6 (rest); else 4 (other side), 3 and 2 (rest)
  const bool first = inner ? (sNeg ? tNeg && d < 0.0 : tNeg) : !sNeg && tNeg && !third6;
  const double num = inside ? 1.0 : (third6 ? ad - be : (third ? ce - bd : (first ? -d : -e)));
  const double den = inside ? det : (third ? a - 2.0 * b + c : (first ? a : c));
  double x = num / den;
  if (num >= den) x = 1.0;
  if (num <= 0.0) x = 0.0;
  if (inside) {
    const double inv = num / den;
    s *= inv;
    t *= inv;
  } else if (third) {
    s = third6 ? 1.0 - x : x;
    t = third6 ? x : 1.0 - x;
  } else {
    s = first ? x : 0.0;
    t = first ? 0.0 : x;
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) cp[k] = (B[k] + s * E0[k]) + t * E1[k];
  double r2 = 0.0;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const double diff = cp[k] - q[k];
    r2 += diff * diff;
  }
  return r2;
}

// Solid angle of a triangle seen from q (Van Oosterom & Strackee 1983).
__host__ __device__ __forceinline__ double solid_angle(const double q[3], const double* A,
                                                       const double* B, const double* C) {
  double a[3], b[3], c[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    a[k] = A[k] - q[k];
    b[k] = B[k] - q[k];
    c[k] = C[k] - q[k];
  }
  const double la = sqrt(a[0] * a[0] + a[1] * a[1] + a[2] * a[2]);
  const double lb = sqrt(b[0] * b[0] + b[1] * b[1] + b[2] * b[2]);
  const double lc = sqrt(c[0] * c[0] + c[1] * c[1] + c[2] * c[2]);
  const double det = a[0] * (b[1] * c[2] - b[2] * c[1]) - a[1] * (b[0] * c[2] - b[2] * c[0]) +
                     a[2] * (b[0] * c[1] - b[1] * c[0]);
  const double ab = a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
  const double bc = b[0] * c[0] + b[1] * c[1] + b[2] * c[2];
  const double ca = c[0] * a[0] + c[1] * a[1] + c[2] * a[2];
  const double den = la * lb * lc + ab * lc + bc * la + ca * lb;
  return 2.0 * atan2(det, den);
}

// Where a ray from q along +x meets a closed triangle mesh, exact in its
// bookkeeping: the winding number of the projections on the (y, z) plane.
//
// ray_cover: +1 or -1 when the projected triangle covers (q.y, q.z), with the
// sign of its normal's x component, else 0.  An edge counts when exactly one
// of its ends has z <= q.z (an exact comparison), on the side of q that one
// expression of its lower and upper end gives, the same for both triangles
// that share the edge.  So the covers of a closed, consistently oriented mesh
// cancel exactly, whatever that expression rounds to, and a ray through an
// edge or a vertex needs no special case.
__host__ __device__ __forceinline__ int ray_cover(double qy, double qz, const double* A,
                                                  const double* B, const double* C) {
  const double* P[4] = {A, B, C, A};
  int cover = 0;
#pragma unroll
  for (int e = 0; e < 3; ++e) {
    const double* from = P[e];
    const double* to = P[e + 1];
    const bool lowF = from[2] <= qz, lowT = to[2] <= qz;
    if (lowF != lowT) {
      const double ly = lowF ? from[1] : to[1], lz = lowF ? from[2] : to[2];
      const double uy = lowF ? to[1] : from[1], uz = lowF ? to[2] : from[2];
      if ((uy - ly) * (qz - lz) > (uz - lz) * (qy - ly)) cover += lowF ? 1 : -1;
    }
  }
  return cover;
}

// Which side of the triangle's plane q lies on: the sign of
// det(A - q, B - q, C - q), or 0 when its rounding could have decided it
// (then q is within rounding of the plane).
__host__ __device__ __forceinline__ int plane_side(const double q[3], const double* A,
                                                   const double* B, const double* C) {
  double a[3], b[3], c[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    a[k] = A[k] - q[k];
    b[k] = B[k] - q[k];
    c[k] = C[k] - q[k];
  }
  const double x0 = b[1] * c[2], x1 = b[2] * c[1], y0 = b[0] * c[2], y1 = b[2] * c[0],
               z0 = b[0] * c[1], z1 = b[1] * c[0];
  const double det = a[0] * (x0 - x1) - a[1] * (y0 - y1) + a[2] * (z0 - z1);
  // about 8 roundings of relative 2^-53 on each product; the bound takes 45
  const double mag = fabs(a[0]) * (fabs(x0) + fabs(x1)) + fabs(a[1]) * (fabs(y0) + fabs(y1)) +
                     fabs(a[2]) * (fabs(z0) + fabs(z1));
  if (!(fabs(det) > 1e-14 * mag)) return 0;
  return det > 0.0 ? 1 : -1;
}

}  // namespace fc
