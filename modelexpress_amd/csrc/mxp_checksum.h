// Device-side checksum algebra and wavefront reductions shared by the placement kernels
// (mxp_kernels.hip) and the transpose kernels (mxp_permute.hip).  Device code only.
#pragma once
#include "mxp_device.h"

namespace mxp {

// ---------------------------------------------------------------------------
// Checksum algebra.  The per-tensor fingerprint is
//     sum_i  byte[i] * ((i * 2654435761 + 1) mod 2^32)   mod 2^32
// (reference: modelexpress/tensor_utils.py:27-44).  For a group of bytes starting at
// position i with local offsets j:
//     sum_j b_j * ((i + j) K + 1) = K * (i * S0 + S1) + S0,   S0 = sum b_j, S1 = sum j b_j
// so three wrapping 32-bit accumulators P = sum i*S0, R = sum S1, Q = sum S0 are kept
// per lane and folded once at the end as K * (P + R) + Q.  S0 and S1 come from the
// unsigned 8-bit dot-product instruction, four bytes at a time.
// ---------------------------------------------------------------------------
struct Csum {
  uint32_t P = 0, Q = 0, R = 0;
  __device__ __forceinline__ void add16(const uint4& x, uint32_t i) {
    uint32_t s0 = __builtin_amdgcn_udot4(x.x, 0x01010101u, 0u, false);
    s0 = __builtin_amdgcn_udot4(x.y, 0x01010101u, s0, false);
    s0 = __builtin_amdgcn_udot4(x.z, 0x01010101u, s0, false);
    s0 = __builtin_amdgcn_udot4(x.w, 0x01010101u, s0, false);
    R = __builtin_amdgcn_udot4(x.x, 0x03020100u, R, false);
    R = __builtin_amdgcn_udot4(x.y, 0x07060504u, R, false);
    R = __builtin_amdgcn_udot4(x.z, 0x0b0a0908u, R, false);
    R = __builtin_amdgcn_udot4(x.w, 0x0f0e0d0cu, R, false);
    Q += s0;
    P += i * s0;
  }
  __device__ __forceinline__ void add8(uint32_t lo, uint32_t hi, uint32_t i) {
    uint32_t s0 = __builtin_amdgcn_udot4(lo, 0x01010101u, 0u, false);
    s0 = __builtin_amdgcn_udot4(hi, 0x01010101u, s0, false);
    R = __builtin_amdgcn_udot4(lo, 0x03020100u, R, false);
    R = __builtin_amdgcn_udot4(hi, 0x07060504u, R, false);
    Q += s0;
    P += i * s0;
  }
  // Up to four bytes packed little-endian in x (missing bytes zero).
  __device__ __forceinline__ void add4(uint32_t x, uint32_t i) {
    uint32_t s0 = __builtin_amdgcn_udot4(x, 0x01010101u, 0u, false);
    R = __builtin_amdgcn_udot4(x, 0x03020100u, R, false);
    Q += s0;
    P += i * s0;
  }
  // One unit of UNIT <= 4 bytes (the narrow paths).
  template <int UNIT>
  __device__ __forceinline__ void addn(uint32_t x, uint32_t i) { add4(x, i); }
  // One byte at position i.
  __device__ __forceinline__ void add_byte(uint32_t b, uint32_t i) {
    Q += b;
    P += i * b;
  }
  // Units at evenly spaced positions: `step` takes them from the last to the first, then `close_steps` is called
  // once, with the position of the first and the spacing, before anything else is added.  sum i*S0 is first * Q +
  // spacing * (sum of k * S0 of the k-th unit), and that sum is the sum of the running Q: one add a unit, where a
  // position of its own costs each unit a 32-bit multiply (four times an add) and the address it multiplies by.
  __device__ __forceinline__ void step(const uint4& x, bool first) {
    step(make_uint2(x.x, x.y), true);
    Q = __builtin_amdgcn_udot4(x.z, 0x01010101u, Q, false);
    Q = __builtin_amdgcn_udot4(x.w, 0x01010101u, Q, false);
    R = __builtin_amdgcn_udot4(x.z, 0x0b0a0908u, R, false);
    R = __builtin_amdgcn_udot4(x.w, 0x0f0e0d0cu, R, false);
    if (!first) P += Q;
  }
  __device__ __forceinline__ void step(const uint2& x, bool first) {
    Q = __builtin_amdgcn_udot4(x.x, 0x01010101u, Q, false);
    Q = __builtin_amdgcn_udot4(x.y, 0x01010101u, Q, false);
    R = __builtin_amdgcn_udot4(x.x, 0x03020100u, R, false);
    R = __builtin_amdgcn_udot4(x.y, 0x07060504u, R, false);
    if (!first) P += Q;
  }
  __device__ __forceinline__ bool steps_fit(uint32_t, uint32_t) const { return true; }
  __device__ __forceinline__ void close_steps(uint32_t first_pos, uint32_t spacing) { P = spacing * P + first_pos * Q; }
  __device__ __forceinline__ uint32_t fold() const { return kKnuth * (P + R) + Q; }
};

// Sums over a whole wavefront (all 64 lanes active), the same in every lane.  Data-parallel primitives move the
// partial sums from lane to lane: row_shr 1, 2, 4, 8 inside a row of sixteen, then the last lane of a row into the
// next row and of the second row into the last two.  A step is one or two VALU instructions where a shuffle is a
// trip through LDS, which a kernel that waits for the sum (finish_kernel: 60 of them in a row) pays in full.
template <uint32_t CTRL, uint32_t ROWS>
__device__ __forceinline__ uint32_t lane_move(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xF, false);
}
template <uint32_t CTRL, uint32_t ROWS = 0xF>
__device__ __forceinline__ uint64_t lane_add(uint64_t v) {
  return v + ((uint64_t)lane_move<CTRL, ROWS>((uint32_t)v) | ((uint64_t)lane_move<CTRL, ROWS>((uint32_t)(v >> 32)) << 32));
}
constexpr uint32_t kRowShr1 = 0x111, kRowShr2 = 0x112, kRowShr4 = 0x114, kRowShr8 = 0x118, kRowBcast15 = 0x142, kRowBcast31 = 0x143;

__device__ __forceinline__ uint32_t wave_sum_u32(uint32_t v) {
  v += lane_move<kRowShr1, 0xF>(v);
  v += lane_move<kRowShr2, 0xF>(v);
  v += lane_move<kRowShr4, 0xF>(v);
  v += lane_move<kRowShr8, 0xF>(v);
  v += lane_move<kRowBcast15, 0xA>(v);
  v += lane_move<kRowBcast31, 0xC>(v);
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

__device__ __forceinline__ unsigned long long wave_sum_u64(unsigned long long x) {
  uint64_t v = x;
  v = lane_add<kRowShr1>(v);
  v = lane_add<kRowShr2>(v);
  v = lane_add<kRowShr4>(v);
  v = lane_add<kRowShr8>(v);
  v = lane_add<kRowBcast15, 0xA>(v);
  v = lane_add<kRowBcast31, 0xC>(v);
  return (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, 63) |
         ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), 63) << 32);
}

}  // namespace mxp
