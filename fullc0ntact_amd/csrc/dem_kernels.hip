// Particle-step kernels for gfx950: integrate, calcHash, reorder /
// find-cell-start and the 27-cell collide.
//
// Layout in HBM: positions and velocities are float4[N] arrays (x, y, z, w),
// read and written as one 16-byte vector per particle per lane, so a wave64
// touches 1 KiB of consecutive memory per access.  Hash, index and cell
// tables are uint32 arrays.  Parameters arrive by value as kernel arguments.
#include "fc_internal.hpp"
#include "fc_device.hpp"
#include "radix_common.hpp"
#include "distmap.hpp"
#include "collide.hpp"
#include "row_resort.hpp"

#include <cmath>
#include <cstring>

namespace fc {

namespace {

constexpr int kBlock = 256;

inline unsigned grid_for(size_t n, int block) {
  size_t g = (n + (size_t)block - 1) / (size_t)block;
  return (unsigned)(g == 0 ? 1 : g);
}

// Fills p (blockIdx.y 0) and p2 (blockIdx.y 1) with value.
__global__ __launch_bounds__(kBlock) void k_fill_u32(uint32_t* __restrict__ p0,
                                                     uint32_t* __restrict__ p2, uint32_t value,
                                                     size_t count) {
  uint32_t* __restrict__ p = blockIdx.y == 0 ? p0 : p2;
  size_t tid = (size_t)blockIdx.x * kBlock + threadIdx.x;
  size_t stride = (size_t)gridDim.x * kBlock;
  // 16-byte stores over the aligned body, scalar stores for the ragged ends.
  size_t head = ((16 - ((uintptr_t)p & 15)) & 15) / 4;
  if (head > count) head = count;
  if (tid < head) p[tid] = value;
  uint32_t* body = p + head;
  size_t nvec = (count - head) / 4;
  uint4 v = make_uint4(value, value, value, value);
  for (size_t i = tid; i < nvec; i += stride) reinterpret_cast<uint4*>(body)[i] = v;
  size_t tail = head + nvec * 4;
  if (tid < count - tail) p[tail + tid] = value;
}

// Plain 16-byte-per-lane copy (bandwidth probe).  Launched with one lane per
// element: on MI355X a capped grid that strides over 1 GiB (2048 or 8192
// blocks) copies at 4.5-4.8 TB/s, one element per lane at 6.2 TB/s.
__global__ __launch_bounds__(kBlock) void k_copy16(uint4* __restrict__ dst,
                                                   const uint4* __restrict__ src, size_t count) {
  size_t stride = (size_t)gridDim.x * kBlock;
  for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < count; i += stride) dst[i] = src[i];
}

// integrate_functor (particles_kernel.cu:39-75) over zip(pos, vel).
__global__ __launch_bounds__(kBlock) void k_integrate(fc_sim_params P, float4* __restrict__ pos,
                                                      float4* __restrict__ vel, float dt,
                                                      uint32_t n) {
  uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  float4 p4 = pos[i];
  float4 v4 = vel[i];
  v3f p = xyz(p4), v = xyz(v4);
  integrate_box(P, P.particleRadius, dt, p, v);
  pos[i] = make_float4(p.x, p.y, p.z, p4.w);
  vel[i] = make_float4(v.x, v.y, v.z, v4.w);
}

// calcHashD (particles_kernel.cu:97-115).
__global__ __launch_bounds__(kBlock) void k_calc_hash(fc_sim_params P, uint32_t* __restrict__ hash,
                                                      uint32_t* __restrict__ index,
                                                      const float4* __restrict__ pos, uint32_t n) {
  uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  float4 p = pos[i];
  hash[i] = hash_of(P, p.x, p.y, p.z);
  index[i] = i;
}

// The state the row-range collide reads, built from the reference-style
// sorted arrays of fc_collide / fc_eval_forces, which carry neither: each
// sorted sphere's velocity with the bits of its cell hash in w (the hash of
// its position, as calcHash computes it, so the hash it was sorted by when
// the arrays come from reorderDataAndFindCellStart of those hashes), and its
// 16-bit coordinates in `frame`; *outside = epoch when a sphere's cell index
// lies outside the grid.
__global__ __launch_bounds__(kBlock) void k_rows_state(fc_sim_params P, QuantFrame frame,
                                                       const float4* __restrict__ sortedPos,
                                                       const float4* __restrict__ sortedVel,
                                                       uint32_t n, float4* __restrict__ velOut,
                                                       uint2* __restrict__ qOut,
                                                       uint32_t* __restrict__ outside,
                                                       uint32_t epoch) {
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const float4 p = sortedPos[i], v = sortedVel[i];
  const int gx = cell_coord(p.x, P.worldOrigin.x, P.cellSize.x);
  const int gy = cell_coord(p.y, P.worldOrigin.y, P.cellSize.y);
  const int gz = cell_coord(p.z, P.worldOrigin.z, P.cellSize.z);
  if ((uint32_t)gx >= P.gridSize.x || (uint32_t)gy >= P.gridSize.y || (uint32_t)gz >= P.gridSize.z)
    *outside = epoch;
  velOut[i] = make_float4(v.x, v.y, v.z, __uint_as_float(grid_hash(gx, gy, gz, P.gridSize)));
  qOut[i] = quantize_pos(frame, p.x, p.y, p.z);
}

// integrate + calcHash in one pass (the update order runs them back to back
// on the same arrays, so fusing them changes no value), with two more jobs
// folded into the same read of the particles:
//  * when prevSortedHash is given, the cells occupied after the previous
//    update are reset to EMPTY: cell h was written iff h starts a run in the
//    sorted hash array, so exactly those entries are cleared (instead of the
//    reference's memset of the whole table, particleSystem.cu:198);
//  * the digit histogram of the new keys for the radix sort's passes.
// Each thread handles kIhPer particles strided by the block size.
constexpr int kIhPer = 4;

__global__ __launch_bounds__(kBlock) void k_integrate_hash(
    fc_sim_params P, BoundaryArg B, float4* __restrict__ pos, float4* __restrict__ vel, float dt,
    uint32_t* __restrict__ keysOut, const uint32_t* __restrict__ prevSortedHash,
    uint32_t* __restrict__ cellStart, uint32_t* __restrict__ cellEnd, uint32_t n, int passes,
    uint32_t* gHist, uint32_t* counters) {
  __shared__ uint32_t s_hist[RS_RADIX];
  for (int i = threadIdx.x; i < RS_RADIX; i += kBlock) s_hist[i] = 0u;
  histogram_producer_prologue(gHist, passes, counters);
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kIhPer; ++u) {
    const uint32_t i = blockIdx.x * (kBlock * kIhPer) + u * kBlock + threadIdx.x;
    uint32_t key = 0;
    if (i < n) {
    if (prevSortedHash != nullptr) {
      const uint32_t h = prevSortedHash[i];
      if (i == 0 || prevSortedHash[i - 1] != h) {
        cellStart[h] = CELL_EMPTY;
        cellEnd[h] = CELL_EMPTY;
      }
    }
    const float4 p4 = pos[i];
    const float4 v4 = vel[i];
    v3f p = xyz(p4), v = xyz(v4);
    integrate_with(P, B, p4.w, dt, p, v);
    pos[i] = make_float4(p.x, p.y, p.z, p4.w);
    vel[i] = make_float4(v.x, v.y, v.z, v4.w);
    key = hash_of(P, p.x, p.y, p.z);
    keysOut[i] = key;
    }
    histogram_add_digit(s_hist, key & (RS_RADIX - 1), i < n);
  }
  __syncthreads();
  histogram_flush(s_hist, gHist, 0);
}

// k_integrate_hash for systems whose sort counts ranks (launch_sort_small) and
// reads no digit histogram: one sphere per thread over many small blocks, no
// LDS, no atomics.  Bound by one round of loads; with the histogram (whose
// first block also clears 48 KB of it) 1331 spheres took 8.3 us, this 2.9.
constexpr int kSmallBlock = 64;

__global__ __launch_bounds__(kSmallBlock) void k_integrate_hash_small(
    fc_sim_params P, BoundaryArg B, float4* __restrict__ pos, float4* __restrict__ vel, float dt,
    uint32_t* __restrict__ keysOut, const uint32_t* __restrict__ prevSortedHash,
    uint32_t* __restrict__ cellStart, uint32_t* __restrict__ cellEnd, uint32_t n) {
  const uint32_t i = blockIdx.x * kSmallBlock + threadIdx.x;
  if (i >= n) return;
  const float4 p4 = pos[i], v4 = vel[i];
  if (prevSortedHash != nullptr) {
    const uint32_t h = prevSortedHash[i];
    if (i == 0 || prevSortedHash[i - 1] != h) {
      cellStart[h] = CELL_EMPTY;
      cellEnd[h] = CELL_EMPTY;
    }
  }
  v3f p = xyz(p4), v = xyz(v4);
  integrate_with(P, B, p4.w, dt, p, v);
  pos[i] = make_float4(p.x, p.y, p.z, p4.w);
  vel[i] = make_float4(v.x, v.y, v.z, v4.w);
  keysOut[i] = hash_of(P, p.x, p.y, p.z);
}

// reorderDataAndFindCellStartD (particles_kernel.cu:119-182).  The
// neighbour's hash comes from the previous lane through a cross-lane
// shuffle; lane 0 of each wave reads it from memory.
// vals are the sorted values: particle ids, or -- with idOfSlot, in the
// sorted-slot layout kept between the fused steps of a run -- the slots of
// oldPos/oldVel that hold each particle, whose ids idOfSlot gives; then the
// ids are written to indexOut.
__global__ __launch_bounds__(kBlock) void k_reorder(
    uint32_t* __restrict__ cellStart, uint32_t* __restrict__ cellEnd,
    float4* __restrict__ sortedPos, float4* __restrict__ sortedVel,
    const uint32_t* __restrict__ hash, const uint32_t* __restrict__ vals,
    const uint32_t* __restrict__ idOfSlot, uint32_t* __restrict__ indexOut,
    const float4* __restrict__ oldPos, const float4* __restrict__ oldVel, uint32_t n,
    uint32_t numCells) {
  uint32_t k = blockIdx.x * kBlock + threadIdx.x;
  uint32_t h = (k < n) ? hash[k] : 0u;
  uint32_t hprev = __shfl_up(h, 1);
  if (k >= n) return;
  if ((threadIdx.x & 63u) == 0u && k > 0) hprev = hash[k - 1];
  // Hashes produced by calcHash are < numCells; the guards only keep
  // caller-supplied out-of-range hashes from writing outside the tables.
  if (k == 0 || h != hprev) {
    if (h < numCells) cellStart[h] = k;
    if (k > 0 && hprev < numCells) cellEnd[hprev] = k;
  }
  if (k == n - 1 && h < numCells) cellEnd[h] = k + 1;
  const uint32_t src = vals[k];
  sortedPos[k] = oldPos[src];
  sortedVel[k] = oldVel[src];
  if (idOfSlot) indexOut[k] = idOfSlot[src];
}

// The cell-table half of k_reorder (the gather done by the sort's last
// pass).
__global__ __launch_bounds__(kBlock) void k_cell_bounds(uint32_t* __restrict__ cellStart,
                                                        uint32_t* __restrict__ cellEnd,
                                                        const uint32_t* __restrict__ hash,
                                                        uint32_t n, uint32_t numCells) {
  uint32_t k = blockIdx.x * kBlock + threadIdx.x;
  uint32_t h = (k < n) ? hash[k] : 0u;
  uint32_t hprev = __shfl_up(h, 1);
  if (k >= n) return;
  if ((threadIdx.x & 63u) == 0u && k > 0) hprev = hash[k - 1];
  if (k == 0 || h != hprev) {
    if (h < numCells) cellStart[h] = k;
    if (k > 0 && hprev < numCells) cellEnd[hprev] = k;
  }
  if (k == n - 1 && h < numCells) cellEnd[h] = k + 1;
}

// Sum of the pair forces of cells [s, e) on particle k, in index order,
// with a one-ahead prefetch of the next neighbour's position and velocity.
__device__ __forceinline__ v3f cell_sum(const fc_sim_params& P, v3f pos, v3f vel, uint32_t k,
                                        uint32_t s, uint32_t e, const float4* __restrict__ sp,
                                        const float4* __restrict__ sv, float rA, bool poly) {
  v3f cf = make_v3(0.0f, 0.0f, 0.0f);
  if (s >= e) return cf;
  float4 pn = sp[s], vn = sv[s];
  for (uint32_t j = s; j < e; ++j) {
    const float4 pc = pn, vc = vn;
    if (j + 1 < e) {
      pn = sp[j + 1];
      vn = sv[j + 1];
    }
    if (j != k) {
      v3f f = collide_spheres(pos, xyz(pc), vel, xyz(vc), rA, poly ? pc.w : rA, P.spring,
                              P.damping, P.shear, P.attraction);
      cf = make_v3(cf.x + f.x, cf.y + f.y, cf.z + f.z);
    }
  }
  return cf;
}

// collideD / collideCell (particles_kernel.cu:223-293): one lane per sorted
// particle; for z, y, x in {-1,0,1} (that nesting is the summation order),
// each neighbour cell's forces are summed into a per-cell partial that is
// then added to the total, then the collider sphere is added, and
// vel + force is scattered to the particle's original slot.  The 9
// cell-table entries of one z-plane of
// the neighbourhood (start and end) are loaded together before any
// neighbour is visited, so each plane costs one table latency instead of a
// chain of 9-18 dependent loads.  Empty cells contribute nothing: their
// partial sum is +0 and the running total is never -0, so skipping the add
// leaves every bit unchanged.
// forceOut != nullptr is evalForces_launcher (particledem_um.cu:538-589):
// no cursor sphere, and the force also stored as float3 at the original
// index.
__global__ __launch_bounds__(kBlock) void k_collide_v2(
    fc_sim_params P, float4* __restrict__ newVel, const float4* __restrict__ sortedPos,
    const float4* __restrict__ sortedVel, const uint32_t* __restrict__ index,
    const uint32_t* __restrict__ cellStart, const uint32_t* __restrict__ cellEnd, uint32_t n,
    int poly, uint32_t* devFlags, float* __restrict__ forceOut) {
  const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
  if (k >= n) return;
  const float4 p4 = sortedPos[k];
  const v3f pos = xyz(p4);
  const v3f vel = xyz(sortedVel[k]);
  const int gx = cell_coord(pos.x, P.worldOrigin.x, P.cellSize.x);
  const int gy = cell_coord(pos.y, P.worldOrigin.y, P.cellSize.y);
  const int gz = cell_coord(pos.z, P.worldOrigin.z, P.cellSize.z);
  const float r = poly ? p4.w : P.particleRadius;
  if (poly && !(r <= P.particleRadius)) atomicOr(devFlags, DEVERR_RADIUS);
  v3f force = make_v3(0.0f, 0.0f, 0.0f);
#pragma unroll 1
  for (int dz = -1; dz <= 1; ++dz) {
    uint32_t st[9], en[9];
#pragma unroll
    for (int c = 0; c < 9; ++c) {
      const uint32_t h = grid_hash(gx + (c % 3) - 1, gy + (c / 3) - 1, gz + dz, P.gridSize);
      st[c] = cellStart[h];
      en[c] = cellEnd[h];
    }
#pragma unroll
    for (int c = 0; c < 9; ++c) {
      if (st[c] != CELL_EMPTY) {
        const uint32_t e = en[c] > n ? n : en[c];
        v3f cf = cell_sum(P, pos, vel, k, st[c], e, sortedPos, sortedVel, r, poly != 0);
        force = make_v3(force.x + cf.x, force.y + cf.y, force.z + cf.z);
      }
    }
  }
  const uint32_t orig = index[k];
  if (forceOut == nullptr) {
    force = add_collider(P, pos, vel, r, force);
  } else {  // evalForces: no cursor sphere, the force stored as float3
    forceOut[3 * (size_t)orig] = force.x;
    forceOut[3 * (size_t)orig + 1] = force.y;
    forceOut[3 * (size_t)orig + 2] = force.z;
  }
  newVel[orig] = make_float4(vel.x + force.x, vel.y + force.y, vel.z + force.z, 0.0f);
}

// The collide stage.  newVel[index[k]] = (vel + force, 0), and with posOut
// also posOut[index[k]] = sortedPos[k] (the last step of a multi-step run
// returns the positions to id order).
// With kFuse the kernel also performs the next update's first stage for the
// same particle, which the update order would run next: integrate (from the
// collided velocity and the unchanged position), the cell hash and the
// radix sort's digit histogram of the hashes.  The integrated state is
// written at the sorted slot k (pos[k], newVel[k], coalesced), the hash at
// the particle's id (keysOut[id], so that the stable sort still orders ties
// by id), slotOf[id] = k (the value the sort carries) and idOfSlot[k] = id
// (for the next reorder).  Every value is the one the separate stages would
// compute.
// kPoly takes each sphere's radius from pos.w (a radius above
// particleRadius raises DEVERR_RADIUS: the neighbour search and the contact
// pre-filter are sized by particleRadius).
// kRows selects the row-range neighbour walk (collide_one_rows), which
// needs the sorted hashes in sortedVel.w and the fixed-point coordinates
// sortedQ with their filter bounds, and leaves out the cells reached by
// wrapping where `wraps` allows it.
// forceOut != nullptr (not fused) is evalForces_launcher
// (particledem_um.cu:538-589): no cursor sphere, and the force also stored
// as float3 at the original index.
// slotKeys (fused): the next key is stored at the sorted slot k (coalesced)
// instead of the key at the id and the slot map, for the row resort
// (row_resort.hip), with kMovedBit when the cell changes; the per-row
// counts it needs are accumulated here (rows) instead of the radix digit
// histogram.
// At least kCollideWavesPerSimd waves per SIMD: the register budget this
// sets (96 VGPRs, a few values spilled to scratch) beats 4 waves at 104
// VGPRs; the fused launch on the settled 1M-sphere bed measured 91.0 us
// against 94.3 us.
constexpr int kCollideWavesPerSimd = 5;

// What follows the 27 cells' sum for one sphere: the cursor sphere, the new
// velocity at the sphere's id, and with kFuse the next update's integrate and
// hash (its key returned).
template <bool kFuse>
__device__ __forceinline__ uint32_t collide_finish(
    const fc_sim_params& P, const BoundaryArg& B, const float4& p4, v3f pos0, v3f vel0, float rA,
    v3f force, uint32_t k, uint32_t orig, float4* __restrict__ newVel, float4* __restrict__ pos,
    float dt, v3f invCell, uint32_t oldKey, uint32_t* __restrict__ keysOut,
    uint32_t* __restrict__ slotOf, uint32_t* __restrict__ idOfSlot, bool slotKeys,
    float* __restrict__ forceOut) {
  if (kFuse || forceOut == nullptr) {
    force = add_collider(P, pos0, vel0, rA, force);
  } else {  // evalForces: no cursor sphere, the force stored as float3
    forceOut[3 * (size_t)orig] = force.x;
    forceOut[3 * (size_t)orig + 1] = force.y;
    forceOut[3 * (size_t)orig + 2] = force.z;
  }
  const v3f nv = make_v3(vel0.x + force.x, vel0.y + force.y, vel0.z + force.z);
  if (!kFuse) {
    newVel[orig] = make_float4(nv.x, nv.y, nv.z, 0.0f);
    if (pos) pos[orig] = p4;
    return 0u;
  }
  v3f p = pos0, v = nv;
  integrate_with(P, B, p4.w, dt, p, v);
  pos[k] = make_float4(p.x, p.y, p.z, p4.w);
  newVel[k] = make_float4(v.x, v.y, v.z, 0.0f);
  const uint32_t key = hash_of_q(P, cell_quotients(P, invCell, p));
  if (slotKeys) {
    // at the slot, with whether the sphere changed cell, for the row resort
    keysOut[k] = key != oldKey ? (key | kMovedBit) : key;
  } else {
    keysOut[orig] = key;
    slotOf[orig] = k;
  }
  idOfSlot[k] = orig;
  return key;
}

// Whether the wrapped cells may be cut (collide_one_rows): known by the
// launch, or unless the arrays' check wrote `epoch` (GatheredState).
struct WrapCut {
  uint32_t cut = 0, epoch = 0;
  const uint32_t* outside = nullptr;
};

template <bool kFuse, bool kPoly, bool kRows>
__global__ __launch_bounds__(kBlock, kCollideWavesPerSimd) void k_collide_v3(
    fc_sim_params P, BoundaryArg B, float contactD2, float4* __restrict__ newVel,
    const float4* __restrict__ sortedPos, const float4* __restrict__ sortedVel,
    const uint32_t* __restrict__ index, const uint32_t* __restrict__ cellStart,
    const uint32_t* __restrict__ cellEnd, uint32_t n, uint32_t xcdGroup, float4* __restrict__ pos,
    float dt, uint32_t* __restrict__ keysOut, int passes, uint32_t* gHist, uint32_t* counters,
    uint32_t* devFlags, uint32_t* __restrict__ slotOf, uint32_t* __restrict__ idOfSlot,
    v3f invCell, const uint2* __restrict__ sortedQ, RowFilter filter, WrapCut wraps,
    float* __restrict__ forceOut, int slotKeys, RowHists rows, uint32_t* __restrict__ piles) {
  __shared__ uint32_t s_list[kListCap + 1][kBlock];
  const bool cutWraps =
      wraps.cut != 0u && (wraps.outside == nullptr || *wraps.outside != wraps.epoch);
  __shared__ uint32_t s_hist[kFuse ? RS_RADIX : 1];
  const uint32_t k = xcd_grouped_block(blockIdx.x, gridDim.x, xcdGroup) * kBlock + threadIdx.x;
  const bool valid = k < n;
  // rows.rowHist: the next sort is a row resort, which takes per-row counts
  // instead of the radix digit histogram; without either, it counts ranks
  // (up to RS_TILE spheres); the same for every block
  const bool digitHist = kFuse && rows.rowHist == nullptr && gHist != nullptr;
  if (digitHist) {
    for (int i = threadIdx.x; i < RS_RADIX; i += kBlock) s_hist[i] = 0u;
    histogram_producer_prologue(gHist, passes, counters);
  }
  uint32_t key = 0, oldKey = 0;
  bool left = false;
  if (valid) {
    const float4 p4 = sortedPos[k];
    const float rA = kPoly ? p4.w : P.particleRadius;
    if (kPoly && !(rA <= P.particleRadius)) atomicOr(devFlags, DEVERR_RADIUS);
    const float4 v4 = sortedVel[k];
    oldKey = __float_as_uint(v4.w);  // the gather keeps the sorted hash in w
    const v3f pos0 = xyz(p4), vel0 = xyz(v4);
    v3f force =
        kRows ? collide_one_rows<kPoly, kBlock>(P, invCell, contactD2, k, pos0, vel0, rA,
                                                sortedPos, sortedVel, sortedQ, filter, cutWraps,
                                                cellStart, cellEnd, n, s_list, left)
              : collide_one_v3<kPoly, kBlock>(P, contactD2, k, pos0, vel0, rA, sortedPos,
                                              sortedVel, cellStart, cellEnd, n, s_list);
    if (kPoly && kRows && left) {
      piles[kPilesList + atomicAdd(&piles[0], 1u)] = k;
    } else {
      key = collide_finish<kFuse>(P, B, p4, pos0, vel0, rA, force, k, index[k], newVel, pos, dt,
                                  invCell, oldKey, keysOut, slotOf, idOfSlot, slotKeys != 0,
                                  forceOut);
    }
  }
  if (digitHist) {
    __syncthreads();
    histogram_add_digit(s_hist, key & (RS_RADIX - 1), valid && !left);
    __syncthreads();
    histogram_flush(s_hist, gHist, 0);
  } else if (kFuse && rows.rowHist != nullptr) {
    row_histograms(rows, k, key, oldKey, valid && !left);
  }
}

// The spheres that a polydisperse k_collide_v3 left (their lists overflowed,
// or a row of theirs has two runs), one wave each: lanes 0-26 take a
// neighbour cell each (those out of reach cut, as collide_one_rows does),
// then the wave takes the cells' spheres 64 at a time through the exact pair
// force, and each cell's lane adds its own contacts in index order, so the 27
// partials and their order are the reference's.  Bound by the latency of the
// rounds: the next 64 states are loaded while a round is worked on, and only
// the contacts' forces are added.  A sphere with 300 candidates is a chain of
// about five rounds here and of 90 in a lane of its own, which was the launch's
// tail: 120,011 log-normal spheres settled on a knot, fused collide 189 us
// with every candidate through the pair force in the lane, 133 us with lists
// refilled in the lane, 61 us with this launch; 50 us (36 + 14) with its
// shorter rounds, the spheres of many candidates left unread and its blocks
// reporting to 32 counters (to one: 5 us more for 512 blocks).
// Equal radii keep the lane's own path: their lists overflow only while a
// bed is compressed, and an empty launch costs about 1 us a step of a run and
// 2 an update (its blocks return at once; with their reports 2: 40,000 spheres
// of 0.6 to 1 radii at random in a 128^3 grid 55.5 us a step without the
// launch, 57.0 with it, 58.0 with the reports).
constexpr unsigned kPileBlocks = 768;  // three waves per SIMD (152 VGPRs)
static_assert(kPileBlocks >= kPilesParts, "every part has a block");

template <bool kFuse>
__global__ __launch_bounds__(kBlock) void k_collide_piles(
    fc_sim_params P, BoundaryArg B, float contactD2, float4* __restrict__ newVel,
    const float4* __restrict__ sortedPos, const float4* __restrict__ sortedVel,
    const uint32_t* __restrict__ index, const uint32_t* __restrict__ cellStart,
    const uint32_t* __restrict__ cellEnd, uint32_t n, float4* __restrict__ pos, float dt,
    uint32_t* __restrict__ keysOut, uint32_t* gHist, uint32_t* __restrict__ slotOf,
    uint32_t* __restrict__ idOfSlot, v3f invCell, int slotKeys, RowHists rows,
    uint32_t* __restrict__ piles) {
  __shared__ float s_f[kBlock / 64][3][64];
  __shared__ uint32_t s_first[kBlock / 64][32], s_end[kBlock / 64][32];
  const int lane = (int)(threadIdx.x & 63u), w = (int)(threadIdx.x >> 6);
  const uint32_t count = min(piles[0], n);
  if (count == 0u) return;  // (the same for every block, and nothing to report)
  for (uint32_t i = blockIdx.x * (kBlock / 64) + (uint32_t)w; i < count;
       i += gridDim.x * (kBlock / 64)) {
    const uint32_t k = piles[kPilesList + i];
    const float4 p4 = sortedPos[k], v4 = sortedVel[k];
    const v3f pos0 = xyz(p4), vel0 = xyz(v4);
    const float rA = p4.w, reach = rA + P.particleRadius;
    const v3f q = cell_quotients(P, invCell, pos0);
    uint32_t first = 0, len = 0;
    if (lane < 27) {
      const int d[3] = {lane % 3 - 1, lane / 3 % 3 - 1, lane / 9 - 1};
      const float qa[3] = {q.x, q.y, q.z};
      const float cs[3] = {P.cellSize.x, P.cellSize.y, P.cellSize.z};
      float g = 0.0f;  // lower bound on the squared distance to the cell
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const float f = qa[a] - floorf(qa[a]), u = fmaf(fabsf(qa[a]), 0x1p-20f, 0x1p-20f);
        const float e = fmaxf((d[a] < 0 ? f : 1.0f - f) - u, 0.0f) * cs[a];
        g += d[a] == 0 ? 0.0f : e * e;
      }
      const float d2 = fminf(contactD2, reach * reach * (1.0f + 0x1p-20f));
      const float thr = fmaxf(d2 * (1.0f + 0x1p-18f), d2 + 0x1p-140f) * (1.0f + 0x1p-16f);
      const uint32_t h = grid_hash(cell_of_quotient(q.x) + d[0], cell_of_quotient(q.y) + d[1],
                                   cell_of_quotient(q.z) + d[2], P.gridSize);
      const uint32_t s = cellStart[h], e = min(cellEnd[h], n);
      if (s != CELL_EMPTY && s < e && !(g >= thr)) {
        first = s;
        len = e - s;
      }
    }
    uint32_t end = len;  // inclusive sum over the cells
#pragma unroll
    for (int off = 1; off < 32; off <<= 1) {
      const uint32_t t = __shfl_up(end, off);
      if (lane >= off) end += t;
    }
    const uint32_t begin = end - len, total = __shfl(end, 26);
    if (lane < 27) {
      s_first[w][lane] = first - begin;  // modulo 2^32: candidate t is sphere t + this
      s_end[w][lane] = end;
    }
    __builtin_amdgcn_wave_barrier();
    v3f cf = make_v3(0.0f, 0.0f, 0.0f);
    float4 pj, vj;
    bool other = false;
    auto fetch = [&](uint32_t t) {
      other = false;
      if (t < total) {
        int c = 0;  // the first cell that ends past t
#pragma unroll
        for (int step = 16; step > 0; step >>= 1)
          if (c + step <= 26 && s_end[w][c + step - 1] <= t) c += step;
        const uint32_t j = t + s_first[w][c];
        other = j != k;
        pj = sortedPos[j];
        vj = sortedVel[j];
      }
    };
    fetch((uint32_t)lane);
    for (uint32_t t0 = 0; t0 < total; t0 += 64u) {
      v3f f = make_v3(0.0f, 0.0f, 0.0f);
      const float4 pn = pj, vn = vj;
      const bool pair = other;
      fetch(t0 + 64u + (uint32_t)lane);  // the next round's, while this one is worked on
      if (pair)
        f = collide_spheres_fast(pos0, xyz(pn), vel0, xyz(vn), rA, pn.w, P.spring, P.damping,
                                 P.shear, P.attraction);
      s_f[w][0][lane] = f.x;
      s_f[w][1][lane] = f.y;
      s_f[w][2][lane] = f.z;
      // (a zero force adds nothing to a partial, which is never -0)
      const uint64_t contacts = __ballot(f.x != 0.0f || f.y != 0.0f || f.z != 0.0f);
      __builtin_amdgcn_wave_barrier();
      if (lane < 27) {
        const uint32_t a = begin > t0 ? begin : t0, b = end < t0 + 64u ? end : t0 + 64u;
        uint64_t mine = a < b ? contacts & lanes_from(a - t0) & ~lanes_from(b - t0) : 0ull;
        while (mine != 0ull) {
          const uint32_t u = lowest_lane(mine);
          mine &= mine - 1ull;
          cf = make_v3(cf.x + s_f[w][0][u], cf.y + s_f[w][1][u], cf.z + s_f[w][2][u]);
        }
      }
      __builtin_amdgcn_wave_barrier();
    }
    v3f force = make_v3(0.0f, 0.0f, 0.0f);
    for (int c = 0; c < 27; ++c)
      force = make_v3(force.x + __shfl(cf.x, c), force.y + __shfl(cf.y, c),
                      force.z + __shfl(cf.z, c));
    if (lane == 0) {
      const uint32_t oldKey = __float_as_uint(v4.w);
      const uint32_t key = collide_finish<kFuse>(
          P, B, p4, pos0, vel0, rA, force, k, index[k], newVel, pos, dt, invCell, oldKey, keysOut,
          slotOf, idOfSlot, slotKeys != 0, nullptr);
      if (kFuse && rows.rowHist != nullptr) {
        const uint32_t r = key >> rows.shift, at = r * kRowCopies + row_copy(k);
        atomicAdd(&rows.rowHist[at], 1u);
        if (r != (oldKey >> rows.shift)) atomicAdd(&rows.chgHist[at], 1u);
      } else if (kFuse && gHist != nullptr) {
        atomicAdd(&hist_buffer(gHist, 0)[(blockIdx.x % RS_HIST_COPIES) * RS_RADIX +
                                         (key & (RS_RADIX - 1))],
                  1u);
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
  // every block has read the count before it reports here: to a counter that
  // few share (one for all took 10 ns a block), whose last one reports on
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint32_t part = blockIdx.x % kPilesParts;
    uint32_t* done = piles + 16u * (1u + part);
    if (atomicAdd(done, 1u) == (gridDim.x - part + kPilesParts - 1u) / kPilesParts - 1u) {
      *done = 0u;
      if (atomicAdd(&piles[1], 1u) == kPilesParts - 1u) {
        piles[0] = 0u;
        piles[1] = 0u;
      }
    }
  }
}

// The collide of small systems (few spheres: the per-lane walk of
// k_collide_v3 is then bound by the latency of its chain of dependent
// loads, not by throughput), with each sphere's nine neighbour rows on nine
// lanes of a wave (collide_row_cells: seven spheres per wave, lane 63
// idle).  Three of its lanes add the rows' 27 cell partials in the reference
// order (z, then y, then x), a component each, then the row-0 lane the cursor
// sphere; the rest is k_collide_v3's tail (the scatter, or with
// kFuse the next update's integrate, hash and histogram), with the same
// arguments and results (oldKey, for slotKeys and rows, is the hash that the
// gather left in sortedVel.w).
constexpr int kSplitSpheresPerWave = 7;

template <bool kFuse, bool kPoly>
__global__ __launch_bounds__(kBlock) void k_collide_split(
    fc_sim_params P, BoundaryArg B, float contactD2, float4* __restrict__ newVel,
    const float4* __restrict__ sortedPos, const float4* __restrict__ sortedVel,
    const uint32_t* __restrict__ index, const uint32_t* __restrict__ cellStart,
    const uint32_t* __restrict__ cellEnd, uint32_t n, float4* __restrict__ pos, float dt,
    uint32_t* __restrict__ keysOut, int passes, uint32_t* gHist, uint32_t* counters,
    uint32_t* devFlags, uint32_t* __restrict__ slotOf, uint32_t* __restrict__ idOfSlot,
    v3f invCell, float* __restrict__ forceOut, int slotKeys, RowHists rows) {
  __shared__ uint32_t s_hist[kFuse ? RS_RADIX : 1];
  __shared__ float s_cells[kBlock / 64][9 * 64];
  const int lane = (int)(threadIdx.x & 63u);
  const uint32_t wave = (blockIdx.x * kBlock + threadIdx.x) >> 6;
  const int sl = lane / 9, r = lane - 9 * (lane / 9);
  const uint32_t k = wave * kSplitSpheresPerWave + (uint32_t)sl;
  const bool valid = lane < 9 * kSplitSpheresPerWave && k < n;
  const bool digitHist = kFuse && rows.rowHist == nullptr && gHist != nullptr;
  if (digitHist) {
    for (int i = threadIdx.x; i < RS_RADIX; i += kBlock) s_hist[i] = 0u;
    histogram_producer_prologue(gHist, passes, counters);
  }
  v3f cf[3];
  float4 p4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  v3f vel0 = make_v3(0.0f, 0.0f, 0.0f);
  float rA = P.particleRadius;
  uint32_t orig = 0;  // (read with the state: a round trip less at the end)
  uint32_t oldKey = 0;
  if (valid) {
    p4 = sortedPos[k];
    orig = index[k];
    const float4 v4 = sortedVel[k];
    vel0 = xyz(v4);
    oldKey = __float_as_uint(v4.w);
    rA = kPoly ? p4.w : P.particleRadius;
    collide_row_cells<kPoly>(P, invCell, contactD2, k, xyz(p4), vel0, rA, r, sortedPos,
                             sortedVel, cellStart, cellEnd, n, cf);
  } else {
#pragma unroll
    for (int c = 0; c < 3; ++c) cf[c] = make_v3(0.0f, 0.0f, 0.0f);
  }
  // lanes 0-2 of each sphere add the 27 cell partials in order, a component
  // each (through LDS: lane shuffles would take 81 and as many adds)
  const int base = 9 * sl;
  float* cells = s_cells[threadIdx.x >> 6];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    cells[9 * lane + 3 * c] = cf[c].x;
    cells[9 * lane + 3 * c + 1] = cf[c].y;
    cells[9 * lane + 3 * c + 2] = cf[c].z;
  }
  __builtin_amdgcn_wave_barrier();
  float sum = 0.0f;
  if (r < 3 && lane < 9 * kSplitSpheresPerWave) {
#pragma unroll
    for (int c = 0; c < 27; ++c) sum += cells[9 * base + 3 * c + r];
  }
  const v3f force = make_v3(sum, __shfl(sum, base + 1 < 64 ? base + 1 : 63),
                            __shfl(sum, base + 2 < 64 ? base + 2 : 63));
  uint32_t key = 0;
  const bool owner = valid && r == 0;
  if (owner) {
    if (kPoly && !(rA <= P.particleRadius)) atomicOr(devFlags, DEVERR_RADIUS);
    key = collide_finish<kFuse>(P, B, p4, xyz(p4), vel0, rA, force, k, orig, newVel, pos, dt,
                                invCell, oldKey, keysOut, slotOf, idOfSlot, slotKeys != 0,
                                forceOut);
  }
  if (digitHist) {
    __syncthreads();
    histogram_add_digit(s_hist, key & (RS_RADIX - 1), owner);
    __syncthreads();
    histogram_flush(s_hist, gHist, 0);
  } else if (kFuse && rows.rowHist != nullptr) {
    // the wave's spheres side by side, so that a row's run is counted at once
    const int from = lane < kSplitSpheresPerWave ? 9 * lane : 0;
    const uint32_t keyL = (uint32_t)__shfl((int)key, from),
                   oldL = (uint32_t)__shfl((int)oldKey, from);
    const bool mine = __shfl(owner ? 1 : 0, from) != 0 && lane < kSplitSpheresPerWave;
    row_histograms(rows, wave * kSplitSpheresPerWave + (uint32_t)lane, keyL, oldL, mine);
  }
}

}  // namespace

hipError_t launch_fill_u32(hipStream_t s, uint32_t* p, uint32_t value, size_t count,
                           uint32_t* p2) {
  if (count == 0) return hipSuccess;
  size_t vec = count / 4 + 2;
  unsigned grid = grid_for(vec, kBlock);
  if (grid > 2048u) grid = 2048u;
  hipLaunchKernelGGL(k_fill_u32, dim3(grid, p2 ? 2 : 1), dim3(kBlock), 0, s, p, p2, value, count);
  return hipGetLastError();
}

hipError_t launch_copy16(hipStream_t s, void* dst, const void* src, size_t bytes) {
  const size_t count = bytes / 16;
  if (count == 0) return hipSuccess;
  const size_t blocks = (count + kBlock - 1) / kBlock;
  const unsigned grid = blocks < (1u << 30) ? (unsigned)blocks : (1u << 30);
  hipLaunchKernelGGL(k_copy16, dim3(grid), dim3(kBlock), 0, s, (uint4*)dst, (const uint4*)src,
                     count);
  return hipGetLastError();
}

hipError_t launch_integrate(hipStream_t s, const fc_sim_params& P, float4* pos, float4* vel,
                            float dt, uint32_t n) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_integrate, dim3(grid_for(n, kBlock)), dim3(kBlock), 0, s, P, pos, vel, dt,
                     n);
  return hipGetLastError();
}

hipError_t launch_rows_state(hipStream_t s, const fc_sim_params& P, const QuantFrame& frame,
                             const float4* sortedPos, const float4* sortedVel, uint32_t n,
                             float4* velOut, uint2* qOut, uint32_t* outside, uint32_t epoch) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_rows_state, dim3(grid_for(n, kBlock)), dim3(kBlock), 0, s, P, frame,
                     sortedPos, sortedVel, n, velOut, qOut, outside, epoch);
  return hipGetLastError();
}

hipError_t launch_calc_hash(hipStream_t s, const fc_sim_params& P, uint32_t* hash,
                            uint32_t* index, const float4* pos, uint32_t n) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_calc_hash, dim3(grid_for(n, kBlock)), dim3(kBlock), 0, s, P, hash, index,
                     pos, n);
  return hipGetLastError();
}

hipError_t launch_integrate_hash(hipStream_t s, const fc_sim_params& P, const BoundaryArg& B,
                                 float4* pos, float4* vel, float dt, uint32_t* keysOut,
                                 const uint32_t* prevSortedHash, uint32_t* cellStart,
                                 uint32_t* cellEnd, uint32_t n, SortScratch& sort, int passes,
                                 uint32_t* devFlags) {
  (void)devFlags;
  if (n == 0) return hipSuccess;
  if (n <= (uint32_t)RS_TILE) {
    hipLaunchKernelGGL(k_integrate_hash_small, dim3(grid_for(n, kSmallBlock)), dim3(kSmallBlock),
                       0, s, P, B, pos, vel, dt, keysOut, prevSortedHash, cellStart, cellEnd, n);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(k_integrate_hash, dim3(grid_for(n, kBlock * kIhPer)), dim3(kBlock), 0, s, P, B,
                     pos, vel, dt, keysOut, prevSortedHash, cellStart, cellEnd, n, passes,
                     sort.histogram, sort.counters);
  return hipGetLastError();
}

hipError_t launch_reorder(hipStream_t s, uint32_t* cellStart, uint32_t* cellEnd, float4* sortedPos,
                          float4* sortedVel, const uint32_t* hash, const uint32_t* index,
                          const float4* oldPos, const float4* oldVel, uint32_t n,
                          uint32_t numCells, const uint32_t* idOfSlot, uint32_t* indexOut) {
  if (n == 0) return hipSuccess;
  if (idOfSlot && !indexOut) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_reorder, dim3(grid_for(n, kBlock)), dim3(kBlock), 0, s, cellStart, cellEnd,
                     sortedPos, sortedVel, hash, index, idOfSlot, indexOut, oldPos, oldVel, n,
                     numCells);
  return hipGetLastError();
}

hipError_t launch_cell_bounds(hipStream_t s, uint32_t* cellStart, uint32_t* cellEnd,
                              const uint32_t* hash, uint32_t n, uint32_t numCells) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_cell_bounds, dim3(grid_for(n, kBlock)), dim3(kBlock), 0, s, cellStart,
                     cellEnd, hash, n, numCells);
  return hipGetLastError();
}

// Smallest float t with sqrtf(t) >= R: every d2 >= t has sqrtf(d2) >= R
// (sqrtf is correctly rounded and monotone), so d2 < t is a lossless
// pre-test for the contact condition sqrtf(d2) < R.
float contact_d2_threshold(float R) {
  if (!(R > 0.0f)) return 0.0f;
  if (std::isinf(R)) return INFINITY;
  float t = R * R;
  while (t > 0.0f && std::sqrt(std::nextafter(t, 0.0f)) >= R) t = std::nextafter(t, 0.0f);
  while (std::sqrt(t) < R) t = std::nextafter(t, INFINITY);
  return t;
}

// The row-range walk needs the sorted hash in sortedVel.w and the
// fixed-point coordinates with kSortedPosPad entries of padding
// (GatheredState: a system's arrays gathered by its sort, or the ones
// k_rows_state builds), 27 distinct neighbour cells (every grid dimension
// >= 4 here) and cell byte offsets below 2^32.
static bool rows_walk_ok(const fc_sim_params& P) {
  return P.gridSize.x >= 4 && P.gridSize.y >= 4 && P.gridSize.z >= 4 &&
         P.numCells <= (1u << 30);
}

// Exact reciprocal of c when c is a positive normal power of two whose
// reciprocal is normal too, else 0.
static float pow2_reciprocal(float c) {
  uint32_t b;
  std::memcpy(&b, &c, 4);
  const uint32_t ex = (b >> 23) & 0xffu;
  return ((b & 0x807fffffu) == 0u && ex >= 1u && ex <= 253u) ? 1.0f / c : 0.0f;
}

// Reciprocal cell sizes for cell_quotients: all three or none.
v3f inv_cell(const fc_sim_params& P) {
  const float ix = pow2_reciprocal(P.cellSize.x), iy = pow2_reciprocal(P.cellSize.y),
              iz = pow2_reciprocal(P.cellSize.z);
  if (ix == 0.0f || iy == 0.0f || iz == 0.0f) return v3f{0.0f, 0.0f, 0.0f};
  return v3f{ix, iy, iz};
}

// Bound on the squared fixed-point distance (in units of 1/scale) of every
// pair closer than R, for the row-range collide's candidate filter: each
// coordinate lies within 0.51 units of (p - lo) * scale after the float
// rounding of that product and rint, so a pair's difference vector is
// within 1.02 * sqrt(3) < 1.8 units of the scaled true one; the bound adds
// 2.5 units, which also covers the rounding of the reference's own distance
// (~1e-7 relative).  Every pair is a candidate when the bound leaves the
// int16 range of the coordinate differences.
uint32_t quant_threshold(float R, float scale) {
  const double b = (double)R * (double)scale + 2.5;
  if (!(b < 32000.0)) return 0xffffffffu;
  return (uint32_t)std::ceil(b * b);
}

bool wraps_out_of_reach(const fc_sim_params& P) {
  const uint32_t G[3] = {P.gridSize.x, P.gridSize.y, P.gridSize.z};
  const float cs[3] = {P.cellSize.x, P.cellSize.y, P.cellSize.z};
  for (int a = 0; a < 3; ++a) {
    if (G[a] < 4u) return false;
    // relative margin for the rounding of the spheres' cell quotients (2^-24
    // of up to G cells each) and of their distance
    const double apart = ((double)G[a] - 2.0 - 1e-6 * (double)G[a]) * (double)cs[a];
    if (!(apart > 2.0 * (double)P.particleRadius * (1.0 + 1e-6))) return false;
  }
  return true;
}

bool walls_inside_grid(const fc_sim_params& P) {
  // integrate_box's bounds, and the quotients of cell_coord: both ends in
  // the same float operations, monotone in between
  const float hi = 1.0f - P.particleRadius, lo = -1.0f + P.particleRadius;
  const float top = hi > lo ? hi : lo, low = hi > lo ? lo : hi;
  const float org[3] = {P.worldOrigin.x, P.worldOrigin.y, P.worldOrigin.z};
  const float cs[3] = {P.cellSize.x, P.cellSize.y, P.cellSize.z};
  const uint32_t G[3] = {P.gridSize.x, P.gridSize.y, P.gridSize.z};
  for (int a = 0; a < 3; ++a)
    if (!((low - org[a]) / cs[a] >= 0.0f && (top - org[a]) / cs[a] < (float)G[a])) return false;
  return true;
}

static WrapCut wrap_cut(const fc_sim_params& P, const GatheredState& gs) {
  WrapCut w;
  if (!wraps_out_of_reach(P)) return w;
  if (gs.walled && walls_inside_grid(P)) {
    w.cut = 1u;
  } else if (gs.outside != nullptr) {
    w.cut = 1u;
    w.outside = gs.outside;
    w.epoch = gs.epoch;
  }
  return w;
}

// Systems up to this many spheres take the row-split collide
// (k_collide_split): a step of a run of 20,000 / 32,000 / 48,000 spheres of
// one radius with it 26.7 / 30.5 / 35.4 us, with the row-range kernel 31.7 /
// 33.8 / 33.5; with radii of their own, piled on the knot, 20,000 / 26,000
// 67.9 / 79.5 against 70.2 / 70.6.
constexpr uint32_t kSplitMaxSpheres = 32768, kSplitMaxPoly = 16384;

template <bool kFuse, bool kPoly>
static void launch_v3(hipStream_t s, const GatheredState* gs, dim3 g, dim3 b,
                      const fc_sim_params& P,
                      const BoundaryArg& B, float d2, float4* newVel, const float4* sortedPos,
                      const float4* sortedVel, const uint32_t* index, const uint32_t* cellStart,
                      const uint32_t* cellEnd, uint32_t n, float4* pos, float dt,
                      uint32_t* keysOut, int passes, uint32_t* gHist, uint32_t* counters,
                      uint32_t* devFlags, uint32_t* slotOf, uint32_t* idOfSlot,
                      float* forceOut = nullptr, bool slotKeys = false,
                      const RowHists* rows = nullptr) {
  // up to RS_TILE spheres the next sort counts ranks: no digit histogram
  if (n <= (uint32_t)RS_TILE) gHist = nullptr;
  if (rows_walk_ok(P) && n <= (kPoly ? kSplitMaxPoly : kSplitMaxSpheres)) {
    const uint32_t waves = (n + kSplitSpheresPerWave - 1) / kSplitSpheresPerWave;
    hipLaunchKernelGGL((k_collide_split<kFuse, kPoly>), dim3((waves + 3) / 4), b, 0, s, P, B, d2,
                       newVel, sortedPos, sortedVel, index, cellStart, cellEnd, n, pos, dt,
                       keysOut, passes, gHist, counters, devFlags, slotOf, idOfSlot, inv_cell(P),
                       forceOut, slotKeys ? 1 : 0, rows ? *rows : RowHists{});
  } else if (gs != nullptr && rows_walk_ok(P)) {
    hipLaunchKernelGGL((k_collide_v3<kFuse, kPoly, true>), g, b, 0, s, P, B, d2, newVel,
                       sortedPos, sortedVel, index, cellStart, cellEnd, n, kCollideXcdGroup, pos,
                       dt, keysOut, passes, gHist, counters, devFlags, slotOf, idOfSlot,
                       inv_cell(P), gs->sortedQ,
                       RowFilter{quant_threshold(P.particleRadius + P.particleRadius,
                                                 gs->frame.scale),
                                 gs->frame.scale},
                       wrap_cut(P, *gs), forceOut, slotKeys ? 1 : 0, rows ? *rows : RowHists{},
                       gs->piles);
    if (kPoly)
      hipLaunchKernelGGL(k_collide_piles<kFuse>, dim3(kPileBlocks), b, 0, s, P, B, d2, newVel,
                         sortedPos, sortedVel, index, cellStart, cellEnd, n, pos, dt, keysOut,
                         gHist, slotOf, idOfSlot, inv_cell(P), slotKeys ? 1 : 0,
                         rows ? *rows : RowHists{}, gs->piles);
  } else
    hipLaunchKernelGGL((k_collide_v3<kFuse, kPoly, false>), g, b, 0, s, P, B, d2, newVel,
                       sortedPos, sortedVel, index, cellStart, cellEnd, n, kCollideXcdGroup, pos,
                       dt, keysOut, passes, gHist, counters, devFlags, slotOf, idOfSlot,
                       inv_cell(P), nullptr, RowFilter{}, WrapCut{}, forceOut, 0, RowHists{},
                       nullptr);
}

hipError_t launch_collide(hipStream_t s, const fc_sim_params& P, bool poly, uint32_t* devFlags,
                          float4* newVel, const float4* sortedPos, const float4* sortedVel,
                          const uint32_t* index, const uint32_t* cellStart,
                          const uint32_t* cellEnd, uint32_t n, float4* posOut,
                          const GatheredState* gathered, float* forceOut) {
  if (n == 0) return hipSuccess;
  dim3 g(grid_for(n, kBlock)), b(kBlock);
  const float d2 = contact_d2_threshold(P.particleRadius + P.particleRadius);
  // The contact-list kernel packs a sorted index into 27 bits and assumes
  // the three cells of a neighbour row are distinct (G.x >= 4).
  if (n >= (1u << 27) || P.gridSize.x < 4) {
    if (posOut) return hipErrorInvalidValue;  // only the multi-step run asks for positions
    hipLaunchKernelGGL(k_collide_v2, g, b, 0, s, P, newVel, sortedPos, sortedVel, index,
                       cellStart, cellEnd, n, poly ? 1 : 0, devFlags, forceOut);
    return hipGetLastError();
  }
  if (poly)
    launch_v3<false, true>(s, gathered, g, b, P, BoundaryArg{}, d2, newVel, sortedPos, sortedVel,
                           index, cellStart, cellEnd, n, posOut, 0.0f, nullptr, 0, nullptr,
                           nullptr, devFlags, nullptr, nullptr, forceOut);
  else
    launch_v3<false, false>(s, gathered, g, b, P, BoundaryArg{}, d2, newVel, sortedPos, sortedVel,
                            index, cellStart, cellEnd, n, posOut, 0.0f, nullptr, 0, nullptr,
                            nullptr, devFlags, nullptr, nullptr, forceOut);
  return hipGetLastError();
}

// Whether a run's fused collide stores the next key at the sorted slot for a
// row resort, on a grid whose row tables fit; up to RS_TILE spheres a step
// sorts by counting ranks.  Small systems leave grids of many rows (the scan
// reads every row) and of few (their rows are beyond the resort's LDS and go
// to it in parts) to the radix sort, which carries the key at the id and the
// slot map.  A step of 8,000 / 16,000 spheres at random with the resort against
// the radix sort: 64^3 grid 29 / 30 us against 48 / 48, 64 x 512 x 512 38 / 40
// against 48 / 49, 64 x 1024 x 1024 70 / 72 against 55 / 56, 64 x 8 x 8
// 26 / 32 against 38 / 43, 64 x 4 x 4 35 / 80 against 43 / 60, 8^3 44 / 75
// against 56 / 87, 4^3 165 / 462 against 174 / 391; all on the floor of an 8^3
// grid 160 / 334 against 157 / 317.
bool collide_slot_keys(const fc_sim_params& P, uint32_t n) {
  if (!rows_walk_ok(P) || !row_resort_grid_ok(P)) return false;
  if (!collide_rows_optional(n)) return true;
  const uint64_t rows = (uint64_t)P.gridSize.y * P.gridSize.z;
  return n > (uint32_t)RS_TILE && rows <= (1u << 18) && n <= 256u * rows;
}

bool collide_rows_optional(uint32_t n) { return n <= 16384u; }

bool collide_rows_state_pays(const fc_sim_params& P, uint32_t n) {
  return rows_walk_ok(P) && n > kSplitMaxSpheres && n < (1u << 27);
}

bool collide_can_fuse(const fc_sim_params& P, uint32_t n) {
  return n > 0 && n < (1u << 27) && P.gridSize.x >= 4;
}

hipError_t launch_collide_fused(hipStream_t s, const fc_sim_params& P, const BoundaryArg& B,
                                float4* pos, float4* vel,
                                const float4* sortedPos, const float4* sortedVel,
                                const uint32_t* index, const uint32_t* cellStart,
                                const uint32_t* cellEnd, uint32_t n, float dt, uint32_t* keysOut,
                                SortScratch& sort, int passes, uint32_t* devFlags,
                                uint32_t* slotOf, uint32_t* idOfSlot,
                                const GatheredState* gathered, bool slotKeys,
                                const RowHists* rows) {
  if (!collide_can_fuse(P, n)) return hipErrorInvalidValue;
  // slot keys go with the row counts, for the row resort
  if (slotKeys != (rows != nullptr)) return hipErrorInvalidValue;
  if (slotKeys && !(gathered != nullptr && collide_slot_keys(P, n))) return hipErrorInvalidValue;
  const float d2 = contact_d2_threshold(P.particleRadius + P.particleRadius);
  const dim3 g(grid_for(n, kBlock)), b(kBlock);
  if (B.poly)
    launch_v3<true, true>(s, gathered, g, b, P, B, d2, vel, sortedPos, sortedVel, index, cellStart,
                          cellEnd, n, pos, dt, keysOut, passes, sort.histogram, sort.counters,
                          devFlags, slotOf, idOfSlot, nullptr, slotKeys, rows);
  else
    launch_v3<true, false>(s, gathered, g, b, P, B, d2, vel, sortedPos, sortedVel, index, cellStart,
                           cellEnd, n, pos, dt, keysOut, passes, sort.histogram, sort.counters,
                           devFlags, slotOf, idOfSlot, nullptr, slotKeys, rows);
  return hipGetLastError();
}

}  // namespace fc
