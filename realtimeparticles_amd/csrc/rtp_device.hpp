// Device-side helpers shared by the gfx950 kernels.
//
// Floating-point contract of every kernel in this library (build flags: -ffp-contract=off,
// correctly rounded fp32 division and square root, IEEE denormals):
//   * each OpenCL expression of the reference is evaluated in its written order;
//   * dot(a,b)        = ((a.x*b.x + a.y*b.y) + a.z*b.z)   (the w lanes are 0, so the
//                       reference's "+ a.w*b.w" adds +0 and changes nothing);
//   * length(v)       = sqrtf(dot(v,v));  normalize(v) = v / length(v), 0 for v == 0;
//   * pow(x, n)       = ((x*x)*x)... with n-1 products for the integral exponents the
//                       reference uses (3 and 2 in sph.cl, artPressureExp in fluids.cl:56);
//   * clamp(x,lo,hi)  = fminf(fmaxf(x, lo), hi).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "rtp_internal.hpp"

namespace rtp {

constexpr float kFloatEps = 0.00000001f;  // FLOAT_EPS, define.cl:6

__device__ __forceinline__ float clampf(float x, float lo, float hi)
{
  return fminf(fmaxf(x, lo), hi);
}

__device__ __forceinline__ float pown(float x, uint32_t n)
{
  if (n == 0)
    return 1.0f;
  float r = x;
  for (uint32_t k = 1; k < n; ++k)
    r = r * x;
  return r;
}

__device__ __forceinline__ float cube(float x) { return (x * x) * x; }

// getCell3DIndexFromPos, grid.cl:14-23.
__device__ __forceinline__ void cell3d(float4 p, const GridConsts& g, uint32_t& cx, uint32_t& cy,
                                       uint32_t& cz)
{
  cx = (uint32_t)floorf((clampf(p.x, -g.absWall[0], g.absWall[0]) + g.absWall[0]) / g.cellSize);
  cy = (uint32_t)floorf((clampf(p.y, -g.absWall[1], g.absWall[1]) + g.absWall[1]) / g.cellSize);
  cz = (uint32_t)floorf((clampf(p.z, -g.absWall[2], g.absWall[2]) + g.absWall[2]) / g.cellSize);
}

// getCell1DIndexFromPos, grid.cl:28-38.
__device__ __forceinline__ uint32_t cell1d(float4 p, const GridConsts& g)
{
  uint32_t cx, cy, cz;
  cell3d(p, g, cx, cy, cz);
  const uint32_t ry = (uint32_t)g.res[1], rz = (uint32_t)g.res[2];
  return cx * rz * ry + cy * rz + cz;
}

// The thread-order key of the cell of q under RTP_LAUNCH_BRICKS: (y, z) tile of kBrick x kBrick
// cells (cell coordinates 0..res), then x, then the cell's place in its tile, so that the
// order runs along x through one pencil of tiles after another.
__device__ __forceinline__ uint32_t brick_key(float4 q, const GridConsts& g)
{
  uint32_t cx, cy, cz;
  cell3d(q, g, cx, cy, cz);
  const uint32_t nTz = ((uint32_t)g.res[2] + kBrick) / kBrick;
  const uint32_t tile = (cy / kBrick) * nTz + cz / kBrick;
  return ((tile * ((uint32_t)g.res[0] + 1u) + cx) * kBrick + cy % kBrick) * kBrick + cz % kBrick;
}

// (c + o + res) % res for c in [0, res] and o in {-1, 0, 1} (fluids.cl:107).
__device__ __forceinline__ int32_t wrap(int32_t v, int32_t res)
{
  v = v < 0 ? v + res : v;
  return v >= res ? v - res : v;
}

// Logical block index that hands every XCD a contiguous run of particle blocks, so the
// neighbour data of consecutive (spatially adjacent) blocks shares one L2.  Workgroups are
// dispatched to the 8 XCDs round-robin by blockIdx.
__device__ __forceinline__ uint32_t logical_block(int remap)
{
  const uint32_t b = blockIdx.x;
  if (!remap)
    return b;
  const uint32_t nb = gridDim.x;
  const uint32_t q = nb / 8u, r = nb % 8u;
  const uint32_t x = b % 8u, slot = b / 8u;
  return x * q + (x < r ? x : r) + slot;
}

__device__ __forceinline__ float4 ld4(const float4* p) { return *p; }

// ------------------------------------------------------------------- quads of lanes
// Walks that give a particle a quad of four lanes (lanes 4q .. 4q + 3 of a wave) exchange
// their terms within the quad and queue survivors in LDS that the quad's other lanes read.

// Orders the wave's LDS accesses on both sides (a quad's lanes read what the others wrote).
__device__ __forceinline__ void wave_sync()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// v of lane K of the quad.
template <int K>
__device__ __forceinline__ float quad_lane(float v)
{
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v),
                                                               K * 0x55, 0xF, 0xF, false));
}

// ((((s + t0) + t1) + t2) + t3) for t_k the t of quad lane k: four terms added to a sum
// in the order of the quad's lanes.
__device__ __forceinline__ float quad_add(float s, float t)
{
  s = s + quad_lane<0>(t);
  s = s + quad_lane<1>(t);
  s = s + quad_lane<2>(t);
  return s + quad_lane<3>(t);
}

// x of the quad's lane A in lane 0, B in lane 1, C in lane 2 and D in lane 3.
template <int A, int B, int C, int D>
__device__ __forceinline__ uint32_t quad_perm(uint32_t x)
{
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, A | B << 2 | C << 4 | D << 6, 0xF, 0xF, true);
}

// Sum of x over the quad's lanes below this one, and over all four.
struct QuadSum {
  uint32_t below, all;
};
__device__ __forceinline__ QuadSum quad_sum(uint32_t x)
{
  const uint32_t u = threadIdx.x & 3u;
  const uint32_t a = quad_perm<0, 0, 1, 2>(x);
  uint32_t s = x + (u >= 1u ? a : 0u);
  const uint32_t b = quad_perm<0, 0, 0, 1>(s);
  s += u >= 2u ? b : 0u;
  return QuadSum{ s - x, quad_perm<3, 3, 3, 3>(s) };
}

// Places for what a quad keeps of sixteen items, item u + 4 j being lane u's k[j], in the items'
// order: the four counts of each lane as bytes of one word, summed over the quad's lanes below
// and over the bytes below.
struct QuadSlots {
  uint32_t at, sum;  // bytes: place of item j, items kept up to and with group j
  __device__ __forceinline__ uint32_t slot(uint32_t j) const { return (at >> (8u * j)) & 0xffu; }
  __device__ __forceinline__ uint32_t all() const { return sum >> 24; }
};
__device__ __forceinline__ QuadSlots quad_slots(const bool k[4])
{
  uint32_t x[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    x[j] = k[j] ? 1u << (8 * j) : 0u;
    asm("" : "+v"(x[j]));  // one selection each
  }
  const QuadSum s = quad_sum(x[0] | x[1] | x[2] | x[3]);
  uint32_t t = s.all + (s.all << 8);
  t = t + (t << 16);
  return QuadSlots{ (t << 8) + s.below, t };
}

// The index ranges of each lane's column of three cells (first, last; empty: first > last), the
// quad's columns in lane order, into out with `tag` in the first indices: one range when the
// non-empty cells are back to back, else one each.  Returns the quad's number of ranges.
__device__ __forceinline__ uint32_t quad_column(const uint2 cells[3], uint2* out, uint32_t tag)
{
  uint32_t lo = 1u, hi = 0u, cnt = 0;
  bool ok = true;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const uint2 r = cells[k];
    if (r.x > r.y)
      continue;
    ++cnt;
    if (lo > hi) {
      lo = r.x;
      hi = r.y;
    } else if (r.x == hi + 1u) {
      hi = r.y;
    } else {
      ok = false;
    }
  }
  if (ok)
    cnt = min(cnt, 1u);
  const QuadSum at = quad_sum(cnt);
  uint2* w = out + at.below;
  if (ok) {
    if (cnt != 0u)
      *w = make_uint2(lo | tag, hi);
  } else {
#pragma unroll
    for (int k = 0; k < 3; ++k)
      if (cells[k].x <= cells[k].y)
        *w++ = make_uint2(cells[k].x | tag, cells[k].y);
  }
  return at.all;
}

// The quad's four bits of a wave ballot, lane 0 lowest.
__device__ __forceinline__ uint32_t quad_bits(bool x)
{
  return (uint32_t)(__builtin_amdgcn_ballot_w64(x) >> (threadIdx.x & 60u)) & 0xFu;
}

}  // namespace rtp
