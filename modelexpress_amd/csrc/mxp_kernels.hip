// CDNA4 (gfx950) kernels for the weight-placement path.
//
// All of them are HBM-bound byte movers or reducers; none is a contraction, so there
// is no MFMA here.  What matters is: 128-bit accesses that are contiguous across the
// 64 lanes of a wavefront, thousands of workgroups per launch (256 CUs in 8 XCDs),
// and one launch for a whole batch of tensors instead of one launch per tensor.
//
//  place_kernel   pitched box copy / fp32->bf16 cast with the position-weighted
//                 checksum of every byte written fused in (reads each output byte's
//                 source once, writes it once: 2 x output bytes of traffic for a
//                 copy, 6 bytes per element for the cast)
//  digest_kernel  int32-word row sums for the blake2b-hashed tensor digest
//                 (reads each byte once), with the checksum of the same bytes where both
//                 are wanted
//  checksum_kernel the checksum alone over existing buffers (reads each byte once)
//  finish_kernel  adds up the copies the accumulators are kept in (mxp_device.h: Fan), hashes
//                 digests and hands the results to the host
#include "mxp_device.h"
#include "mxp_checksum.h"
#include "mxp_convert.h"
#include <atomic>
#include <type_traits>

namespace mxp {

// Checksum plus the tensor_digest sums of the bytes being stored (reference:
// modelexpress/refit/reshard/verify.py:112-150), for launches that verify what they place
// without a second pass over the finished buffers.  The digest reads a buffer as little-endian
// signed 32-bit words: whole 1024-word rows contribute sum(w) and sum(w) * (row + 1), the
// words after the last whole row sum(w) and sum(w * (k + 1)), the 1..3 bytes after the last
// whole word their unsigned sum - every term is linear in the stored bytes, so each lane adds
// the share of the bytes it stores, weighted by where they land in the destination buffer,
// and the sums wrap mod 2^64 exactly as the reference's int64 arithmetic does.
struct DigestAcc {
  Csum cs;
  unsigned long long S = 0, SW = 0, T = 0, TW = 0, RG = 0;
  // Whole-row words of this tile, kept as 32-bit sums until the tile is done: low halves
  // (unsigned) and high halves (signed) of the words apart, plain and weighted by the row's
  // distance from the tile's first row.  A lane adds at most 64 units of at most 4 words at
  // distances below 64, so nothing wraps; rows further away take the 64-bit route.
  uint32_t a_lo = 0, b_lo = 0;
  int32_t a_hi = 0, b_hi = 0;
  uint64_t row0 = 0;        // row (4 KiB of the buffer) the tile starts in
  uint64_t base = 0;        // position of the tile's first destination byte inside its buffer
  uint32_t base32 = 0;      // the 32-bit checksum position the callers count from
  uint64_t tail_byte0 = 0;  // first byte after the last whole row
  uint64_t body_end = 0;    // first ragged byte
  __device__ __forceinline__ void init(uint64_t buffer_bytes, uint64_t tile_pos, uint32_t tile_pos32) {
    base = tile_pos;
    base32 = tile_pos32;
    row0 = tile_pos >> 12;
    body_end = buffer_bytes & ~3ull;
    tail_byte0 = buffer_bytes / (4ull * kDigestRowWords) * (4ull * kDigestRowWords);
  }
  static_assert(kDigestRowWords == 1024, "rows are 4 KiB: the row of byte p is p >> 12");
  typedef short s16x2 __attribute__((ext_vector_type(2)));
  typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
  static __device__ __forceinline__ uint32_t lo_add(uint32_t w, uint32_t acc) {
    u16x2 v;
    __builtin_memcpy(&v, &w, 4);
    const u16x2 one_zero = {1, 0};
    return __builtin_amdgcn_udot2(v, one_zero, acc, false);
  }
  static __device__ __forceinline__ int32_t hi_add(uint32_t w, int32_t acc) {
    s16x2 v;
    __builtin_memcpy(&v, &w, 4);
    const s16x2 zero_one = {0, 1};
    return __builtin_amdgcn_sdot2(v, zero_one, acc, false);
  }
  // Words after the last whole row: `sum` of the words and `ramp` = sum of word k times k.
  __device__ __forceinline__ void tail_words(long long sum, long long ramp, uint64_t p) {
    T += (unsigned long long)sum;
    TW += (unsigned long long)sum * (unsigned long long)(((p - tail_byte0) >> 2) + 1) + (unsigned long long)ramp;
  }
  // Whole-row words far from the tile's first row (pitched boxes with a large pitch).
  __device__ __forceinline__ void far_words(long long sum, uint64_t p) {
    S += (unsigned long long)sum;
    SW += (unsigned long long)sum * (unsigned long long)((p >> 12) + 1);
  }
  __device__ __forceinline__ void add16(const uint4& x, uint32_t i) {
    cs.add16(x, i);
    const uint64_t p = base + (uint32_t)(i - base32);
    const uint64_t dr = (p >> 12) - row0;
    if (p < tail_byte0 && dr < 64) {
      const uint32_t lo = lo_add(x.w, lo_add(x.z, lo_add(x.y, lo_add(x.x, 0u))));
      const int32_t hi = hi_add(x.w, hi_add(x.z, hi_add(x.y, hi_add(x.x, 0))));
      a_lo += lo;
      a_hi += hi;
      b_lo += lo * (uint32_t)dr;
      b_hi += hi * (int32_t)dr;
    } else {
      const long long a = (int32_t)x.x, b = (int32_t)x.y, c = (int32_t)x.z, d = (int32_t)x.w;
      if (p < tail_byte0) far_words(a + b + c + d, p);
      else tail_words(a + b + c + d, b + 2 * c + 3 * d, p);
    }
  }
  __device__ __forceinline__ void add8(uint32_t lo_w, uint32_t hi_w, uint32_t i) {
    cs.add8(lo_w, hi_w, i);
    const uint64_t p = base + (uint32_t)(i - base32);
    const uint64_t dr = (p >> 12) - row0;
    if (p < tail_byte0 && dr < 64) {
      const uint32_t lo = lo_add(hi_w, lo_add(lo_w, 0u));
      const int32_t hi = hi_add(hi_w, hi_add(lo_w, 0));
      a_lo += lo;
      a_hi += hi;
      b_lo += lo * (uint32_t)dr;
      b_hi += hi * (int32_t)dr;
    } else {
      const long long a = (int32_t)lo_w, b = (int32_t)hi_w;
      if (p < tail_byte0) far_words(a + b, p);
      else tail_words(a + b, b, p);
    }
  }
  // Units whose positions are `spacing` (a whole number of rows) apart, all in whole rows of one tile: taken from the
  // last to the first, closed before anything else is added (Csum::step).  Units of one lane are k * spacing >> 12 rows
  // after its first, so the row weights come out of running sums too: 10 instructions a 16-byte unit beside the
  // checksum's 9, where finding each unit's row, 64-bit compares and weighting by it took some 60 and a tile 4 us of
  // its compute unit.  1.4 GB of fp32 rows placed as 0.7 GB of bf16 with digests: 373 us, 349 this way.
  __device__ __forceinline__ bool steps_fit(uint32_t tile_bytes, uint32_t spacing) const {
    return (spacing & 4095u) == 0 && base + tile_bytes <= tail_byte0;
  }
  __device__ __forceinline__ void step(const uint4& x, bool first) {
    cs.step(x, first);
    a_lo = lo_add(x.w, lo_add(x.z, lo_add(x.y, lo_add(x.x, a_lo))));
    a_hi = hi_add(x.w, hi_add(x.z, hi_add(x.y, hi_add(x.x, a_hi))));
    if (!first) { b_lo += a_lo; b_hi += a_hi; }
  }
  __device__ __forceinline__ void step(const uint2& x, bool first) {
    cs.step(x, first);
    a_lo = lo_add(x.y, lo_add(x.x, a_lo));
    a_hi = hi_add(x.y, hi_add(x.x, a_hi));
    if (!first) { b_lo += a_lo; b_hi += a_hi; }
  }
  __device__ __forceinline__ void close_steps(uint32_t first_pos, uint32_t spacing) {
    cs.close_steps(first_pos, spacing);
    const uint32_t dr = (((uint32_t)base & 4095u) + (first_pos - base32)) >> 12, rows = spacing >> 12;
    b_lo = b_lo * rows + a_lo * dr;
    b_hi = b_hi * (int32_t)rows + a_hi * (int32_t)dr;
  }
  // Folds the tile's 32-bit sums into the 64-bit ones; call once, after the last add.
  __device__ __forceinline__ void flush() {
    const long long s = (long long)a_hi * 65536 + (long long)a_lo;
    const long long sw = (long long)b_hi * 65536 + (long long)b_lo;
    S += (unsigned long long)s;
    SW += (unsigned long long)sw + (unsigned long long)s * (unsigned long long)(row0 + 1);
  }
  template <int UNIT>
  __device__ __forceinline__ void addn(uint32_t x, uint32_t i) {
    cs.add4(x, i);
    const uint64_t p = base + (uint32_t)(i - base32);
    if constexpr (UNIT == 4) {
      const uint64_t dr = (p >> 12) - row0;
      if (p < tail_byte0 && dr < 64) {
        const uint32_t lo = lo_add(x, 0u);
        const int32_t hi = hi_add(x, 0);
        a_lo += lo;
        a_hi += hi;
        b_lo += lo * (uint32_t)dr;
        b_hi += hi * (int32_t)dr;
      } else if (p < tail_byte0) {
        far_words((long long)(int32_t)x, p);
      } else {
        tail_words((long long)(int32_t)x, 0, p);
      }
    } else {  // part of a word, or ragged bytes: byte by byte
#pragma unroll
      for (int e = 0; e < UNIT; ++e) {
        const uint32_t b = (x >> (8 * e)) & 0xFFu;
        const uint64_t q = p + e;
        if (q >= body_end) {
          RG += b;
          continue;
        }
        const uint32_t j = (uint32_t)q & 3u;
        const long long v = j == 3u ? (long long)(int32_t)(b << 24) : (long long)(b << (8u * j));
        if (q < tail_byte0) far_words(v, q);
        else tail_words(v, 0, q & ~3ull);
      }
    }
  }
};

// 128-bit non-temporal accesses: every byte is touched exactly once, so nothing is worth
// keeping in L2 / Infinity Cache (measured: +3..4% over plain accesses on this copy).
// Loads carry no alignment promise (the `_u` types): the source of a box only has to be element
// aligned - a tensor's offset in a safetensors file is - while stores are always whole and aligned.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 u32x4_u __attribute__((aligned(1)));
__device__ __forceinline__ uint4 ld16(const uint8_t* p) {
  const u32x4 t = __builtin_nontemporal_load(reinterpret_cast<const u32x4_u*>(p));
  return make_uint4(t.x, t.y, t.z, t.w);
}
__device__ __forceinline__ void st16(uint8_t* p, const uint4& v) {
  u32x4 t;
  t.x = v.x; t.y = v.y; t.z = v.z; t.w = v.w;
  __builtin_nontemporal_store(t, reinterpret_cast<u32x4*>(p));
}
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef u32x2 u32x2_u __attribute__((aligned(1)));
typedef uint32_t u32_u __attribute__((aligned(1)));
typedef uint16_t u16_u __attribute__((aligned(1)));
__device__ __forceinline__ uint2 ld8(const uint8_t* p) {
  const u32x2 t = __builtin_nontemporal_load(reinterpret_cast<const u32x2_u*>(p));
  return make_uint2(t.x, t.y);
}
__device__ __forceinline__ void st8(uint8_t* p, const uint2& v) {
  u32x2 t;
  t.x = v.x; t.y = v.y;
  __builtin_nontemporal_store(t, reinterpret_cast<u32x2*>(p));
}

// The first n bytes of a (0 < n < their size) and the rest of b.
__device__ __forceinline__ uint32_t join_word(uint32_t a, uint32_t b, int n) {
  const uint32_t from_a = n >= 4 ? ~0u : n <= 0 ? 0u : (1u << (8 * n)) - 1u;
  return (a & from_a) | (b & ~from_a);
}
__device__ __forceinline__ uint4 join(const uint4& a, const uint4& b, uint32_t n) {
  return make_uint4(join_word(a.x, b.x, (int)n), join_word(a.y, b.y, (int)n - 4), join_word(a.z, b.z, (int)n - 8),
                    join_word(a.w, b.w, (int)n - 12));
}
__device__ __forceinline__ uint2 join(const uint2& a, const uint2& b, uint32_t n) {
  return make_uint2(join_word(a.x, b.x, (int)n), join_word(a.y, b.y, (int)n - 4));
}

// One tile of one segment.  UNIT = destination bytes handled per lane access.
// Lanes walk the tile in flattened (row, unit) order, so neighbouring lanes touch
// neighbouring 16-byte units of the same row: every wavefront access is a run of
// contiguous 1 KiB pieces in both the source and the destination.
//
// RAGGED (mxp_device.h: Seg): the destination is one contiguous run of aligned units and the source rows are
// `row_bytes` destination bytes long, whatever that is.  A unit that begins less than a unit before the end of its
// row reads past that end - into the row's own pitch, or the next row - and takes the rest from a second read that
// ends where the next row's share ends; both lie inside the box (rows are at least a unit long, and the last unit
// of a box ends where its last row does).  `col0`: the byte of its row at which the tile starts; `src` is that row.
// Bound by HBM as the plain copy is: 65536 rows of 5735 bf16 out of a pitch of 11470 take 278 us = 5.4 TB/s, where the
// row-wise form, one 2-byte element per lane and access, takes 478; 262144 rows of 1433 out of 11464: 293 against 454.
template <int OP, int UNIT, bool RAGGED = false, class ACC>
__device__ __forceinline__ void run_tile(const Seg& s, const uint8_t* __restrict__ src,
                                         uint8_t* __restrict__ dst, uint32_t csum_base,
                                         uint32_t n_units, uint32_t nan_bits, ACC& cs, uint32_t first, uint32_t col0 = 0) {
  constexpr bool NARROW = op_narrows(OP), WIDEN = op_widens(OP);
  constexpr int SRC_UNIT = NARROW ? 2 * UNIT : WIDEN ? UNIT / 2 : UNIT;
  const uint32_t upr = s.units_per_row;
  const uint32_t magic = s.div_magic;
  const uint32_t sp = (uint32_t)s.src_pitch, dp = (uint32_t)s.dst_pitch;
  // Within a tile the row offsets fit 32 bits (the planner bounds rows_per_tile * pitch).
  auto locate = [&](uint32_t v, uint32_t& so, uint32_t& d_o) {
    const uint32_t row = (upr == 1u) ? v : __umulhi(v, magic);
    const uint32_t col = v - row * upr;
    so = row * sp + col * (uint32_t)SRC_UNIT;
    d_o = row * dp + col * (uint32_t)UNIT;
  };

  constexpr bool BATCHED = (NARROW && UNIT == 8) || (!NARROW && UNIT == 16);
  static_assert(BATCHED || !RAGGED, "ragged segments move in whole units");
  // Ragged: the row of unit v, and its bytes left in that row.
  auto locate_ragged = [&](uint32_t v, uint32_t& so, uint32_t& d_o, uint32_t& room) {
    const uint32_t at = col0 + v * (uint32_t)UNIT;
    uint32_t row = __umulhi(at, magic);  // the quotient, or one more
    if (row * s.row_bytes > at) --row;
    const uint32_t col = at - row * s.row_bytes;
    so = row * sp + (NARROW ? 2u * col : WIDEN ? col / 2u : col);
    d_o = v * (uint32_t)UNIT;
    room = s.row_bytes - col;
  };
  if constexpr (BATCHED) {
    // The wide paths.  A lane moves kPlaceBatch units: 16 bytes in and out for a copy, 16 in /
    // 8 out for a narrowing cast, 8 in / 16 out for a widening one, so a wavefront access is
    // 1 KiB (512 B on the narrow side) of contiguous memory.  A tile is at most one batch (the
    // host bounds it): a single pass in four phases that the scheduler may not interleave -
    // all addresses, all loads, all stores, then the checksum arithmetic - so the workgroup
    // presents the memory system with one burst of reads over a contiguous region followed by
    // one burst of writes over another.  Measured on the Llama rank: 256 lanes x 4 loads
    // 5.16 TB/s, 1024 x 8 5.98 TB/s; sixteen loads per lane are slower.
    constexpr int U = kPlaceBatch;
    using In = typename std::conditional<WIDEN, uint2, uint4>::type;
    using Out = typename std::conditional<NARROW, uint2, uint4>::type;
    auto load = [&](uint32_t off) -> In {
      if constexpr (WIDEN) return ld8(src + off);
      else return ld16(src + off);
    };
    auto convert = [&](const In& a) -> Out {
      if constexpr (NARROW) return narrow4<OP>(a, nan_bits);
      else if constexpr (WIDEN) return widen4<OP>(a);
      else if constexpr (op_recodes16(OP))
        return make_uint4(recode2<OP>(a.x, nan_bits), recode2<OP>(a.y, nan_bits), recode2<OP>(a.z, nan_bits),
                          recode2<OP>(a.w, nan_bits));
      else return a;
    };
    auto store = [&](uint32_t off, const Out& x) {
      if constexpr (OP == kOpChecksumOnly) return;
      else if constexpr (NARROW) st8(dst + off, x);
      else st16(dst + off, x);
    };
    auto sum = [&](uint32_t off, const Out& x) {
      if constexpr (NARROW) cs.add8(x.x, x.y, csum_base + off);
      else cs.add16(x, csum_base + off);
    };
    // A lane's units are a fixed stride apart, also in a bundle, whose wavefronts have one unit a lane at most.  (A stride
    // in a register, for bundles one of 64, took the kernel to 19 spilled scalar registers and 64 VGPRs.)
    constexpr uint32_t STRIDE = OP == kOpChecksumOnly && !std::is_same<ACC, DigestAcc>::value ? 64u : (uint32_t)kPlaceThreads;
    auto unit_of = [&](int k) -> uint32_t { return first + (uint32_t)k * STRIDE; };
    uint32_t so[U], d_o[U];
    In a[U];
    Out x[U];
    // A tile whose destination is one run has its lanes' units evenly spaced (Csum::step); the others, and for digests
    // those that reach into the words after a buffer's last whole row, find each unit's position on its own.
    constexpr uint32_t spacing = STRIDE * (uint32_t)UNIT;
    const bool steps = (RAGGED || dp == upr * (uint32_t)UNIT || n_units <= upr) && cs.steps_fit(n_units * (uint32_t)UNIT, spacing);
    const bool unasked = !std::is_same<ACC, DigestAcc>::value && s.csum_slot == 0xFFFFFFFFu;  // nobody reads the sums
    auto add_steps = [&](auto whole) {
#pragma unroll
      for (int k = U - 1; k >= 0; --k)  // a k-th unit that no lane of the wavefront has is zero and adds nothing: 0.5 us of a small tile
        if (decltype(whole)::value || __builtin_amdgcn_ballot_w64(unit_of(k) < n_units)) cs.step(x[k], k == 0);
      cs.close_steps(csum_base + first * (uint32_t)UNIT, spacing);
    };
    if constexpr (RAGGED) {
      uint32_t room[U];
      In b[U];
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const uint32_t v = unit_of(k);
        locate_ragged(v < n_units ? v : 0u, so[k], d_o[k], room[k]);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < U; ++k)
        if (unit_of(k) < n_units) a[k] = load(so[k]);
#pragma unroll
      for (int k = 0; k < U; ++k)
        if (unit_of(k) < n_units && room[k] < (uint32_t)UNIT) {
          // the next row starts src_pitch after this one: back by the source bytes this row still gives
          const uint32_t taken = NARROW ? 2u * room[k] : WIDEN ? room[k] / 2u : room[k];
          const uint32_t row_src = NARROW ? 2u * s.row_bytes : WIDEN ? s.row_bytes / 2u : s.row_bytes;
          b[k] = load(so[k] + sp - row_src);
          room[k] = taken;
        } else {
          room[k] = 16u;  // the unit lies in one row
        }
#pragma unroll
      for (int k = 0; k < U; ++k)
        if (room[k] < 16u) a[k] = join(a[k], b[k], room[k]);
      __builtin_amdgcn_sched_barrier(0);
    } else if (n_units == (uint32_t)(U * kPlaceThreads)) {  // full tile: nothing is predicated
#pragma unroll
      for (int k = 0; k < U; ++k) locate(unit_of(k), so[k], d_o[k]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < U; ++k) a[k] = load(so[k]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < U; ++k) {
        x[k] = convert(a[k]);
        store(d_o[k], x[k]);
      }
      if constexpr (OP != kOpChecksumOnly) __builtin_amdgcn_sched_barrier(0);
      if (unasked) return;
      if (steps) {
        add_steps(std::true_type{});
      } else {
#pragma unroll
        for (int k = 0; k < U; ++k) sum(d_o[k], x[k]);
      }
      return;
    } else {
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const uint32_t v = unit_of(k);
        locate(v < n_units ? v : 0u, so[k], d_o[k]);
      }
#pragma unroll
      for (int k = 0; k < U; ++k)
        if (unit_of(k) < n_units) a[k] = load(so[k]);
    }
    // a partial tile, or a ragged one
#pragma unroll
    for (int k = 0; k < U; ++k) {
      x[k] = Out{};
      if (unit_of(k) < n_units) {
        x[k] = convert(a[k]);
        store(d_o[k], x[k]);
      }
    }
    if (unasked) return;
    if (steps) {
      add_steps(std::false_type{});
    } else {
#pragma unroll
      for (int k = 0; k < U; ++k)
        if (unit_of(k) < n_units) sum(d_o[k], x[k]);
    }
  } else {
    // The narrow paths (boxes the 16-byte grid does not fit): one unit of at most four bytes per
    // lane and step, eight steps at a time - all their loads first, then the stores - so a lane
    // keeps eight loads in flight here too.
    auto load_raw = [&](uint32_t so) -> uint32_t {
      if constexpr (NARROW) {
        static_assert(UNIT == 2, "the element-wise cast path moves one element per lane");
        return *reinterpret_cast<const uint32_t*>(src + so);
      } else if constexpr (op_recodes16(OP)) {
        static_assert(UNIT == 4 || UNIT == 2, "two elements or one per lane");
        if constexpr (UNIT == 4) return *reinterpret_cast<const u32_u*>(src + so);
        else return *reinterpret_cast<const uint16_t*>(src + so);
      } else if constexpr (OP == kOpCastF8E4M3Bf16) {
        static_assert(UNIT == 4 || UNIT == 2, "two elements or one per lane");
        if constexpr (UNIT == 4) return *reinterpret_cast<const u16_u*>(src + so);
        else return src[so];
      } else if constexpr (WIDEN) {
        static_assert(UNIT == 4, "the element-wise cast path moves one element per lane");
        return *reinterpret_cast<const uint16_t*>(src + so);
      } else if constexpr (UNIT == 4) {
        return *reinterpret_cast<const u32_u*>(src + so);
      } else if constexpr (UNIT == 2) {
        return *reinterpret_cast<const u16_u*>(src + so);
      } else {
        return src[so];
      }
    };
    auto finish = [&](uint32_t raw, uint32_t d_o) {
      uint32_t x;
      if constexpr (NARROW) x = narrow1<OP>(raw, nan_bits);
      else if constexpr (op_recodes16(OP)) x = UNIT == 4 ? recode2<OP>(raw, nan_bits) : recode1<OP>(raw, nan_bits);
      else if constexpr (OP == kOpCastF8E4M3Bf16)
        x = UNIT == 4 ? (f8e4m3_to_bf16_bits(raw & 0xFFu) | (f8e4m3_to_bf16_bits(raw >> 8) << 16)) : f8e4m3_to_bf16_bits(raw);
      else if constexpr (WIDEN) x = widen1<OP>(raw);
      else x = raw;
      if constexpr (OP != kOpChecksumOnly) {
        if constexpr (UNIT == 4) *reinterpret_cast<uint32_t*>(dst + d_o) = x;
        else if constexpr (UNIT == 2) *reinterpret_cast<uint16_t*>(dst + d_o) = (uint16_t)x;
        else dst[d_o] = (uint8_t)x;
      }
      cs.template addn<UNIT>(x, csum_base + d_o);
    };
    constexpr uint32_t G = 8;
    constexpr uint32_t lanes = kPlaceThreads;
    for (uint32_t v0 = first; v0 < n_units; v0 += G * lanes) {
      uint32_t so[G], d_o[G], raw[G];
#pragma unroll
      for (uint32_t k = 0; k < G; ++k) {
        const uint32_t v = v0 + k * lanes;
        locate(v < n_units ? v : v0, so[k], d_o[k]);  // a step past the end re-reads the lane's first unit and drops it
      }
#pragma unroll
      for (uint32_t k = 0; k < G; ++k) raw[k] = load_raw(so[k]);
#pragma unroll
      for (uint32_t k = 0; k < G; ++k)
        if (v0 + k * lanes < n_units) finish(raw[k], d_o[k]);
    }
  }
}

// RAGGED: the table may hold ragged segments (mxp_device.h: Seg).  Their second load takes the kernel from 63 to 92
// VGPRs, so tables without them have kernels of their own: with the ragged branch in it the plain kernel had room for one
// workgroup per compute unit only, and bf16 -> fp32 of 2^24 elements took 34 us, not 30.  With digests (108 and 114) a
// unit holds one either way; large launches take the same through both, small ones up to 0.8 us more through the ragged one
// (8.5 and 9.0 us for 23 MB read and written).
template <bool CHECKSUM_ONLY, bool RAGGED, bool DIGEST = false>
__device__ __forceinline__ void place_body(
    const Seg* __restrict__ segs, const WorkItem* __restrict__ work,
    const void* const* __restrict__ src_bases, void* const* __restrict__ dst_bases,
    uint32_t* __restrict__ sums, Fan fan, uint32_t nan_bits, const unsigned long long* __restrict__ dst_sizes = nullptr,
    unsigned long long* __restrict__ digest_sums = nullptr, uint32_t* __restrict__ zero = nullptr, uint32_t zero_words = 0) {
  // Housekeeping for the launch after this one: its accumulators are cleared here, a slice per
  // workgroup, so it needs no clearing launch of its own.
  for (uint64_t i = (uint64_t)blockIdx.x * kPlaceThreads + threadIdx.x; i < zero_words; i += (uint64_t)gridDim.x * kPlaceThreads) zero[i] = 0u;
  // This workgroup's copy of the accumulators.
  const uint32_t lane_first = (blockIdx.x & fan.mask) * fan.pitch;
  const WorkItem w = work[blockIdx.x];
  const bool bundle = (w.tile & kBundle) != 0;  // every wavefront has a segment to itself
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63u;
  if (bundle && wave >= (w.tile & ~kBundle)) return;
  const Seg s = segs[w.seg + (bundle ? wave : 0u)];
  // rows_per_tile is read either way: read for one of them only it is a trip to memory of its own ahead of the segment, and
  // a launch of 3 MB (read and written) takes 5.2 us, 5.0 this way
  const uint32_t r0 = (bundle ? 0u : w.tile) * s.rows_per_tile;
  const uint32_t nrows = min(s.rows - r0, s.rows_per_tile);
  const uint32_t n_units = nrows * s.units_per_row;
  uint64_t src_row = r0;
  uint32_t col0 = 0;
  if (RAGGED && s.ragged) {
    const uint64_t at = s.ragged - 1u + (uint64_t)r0 * s.unit;
    src_row = at / s.row_bytes;
    col0 = (uint32_t)(at - src_row * s.row_bytes);
  }
  const void* src_base = s.src_buf == kSrcIsDestination ? dst_bases[s.dst_buf] : src_bases[s.src_buf];
  const uint8_t* src = static_cast<const uint8_t*>(src_base) + s.src_off + src_row * s.src_pitch;
  uint8_t* dst = nullptr;
  if (s.op != kOpChecksumOnly)
    dst = static_cast<uint8_t*>(dst_bases[s.dst_buf]) + s.dst_off + (uint64_t)r0 * s.dst_pitch;
  // Checksum positions are taken mod 2^32, exactly as the weights are.
  const uint32_t csum_base = (uint32_t)(s.dst_off + (uint64_t)r0 * s.dst_pitch) + s.csum_bias;

  typename std::conditional<DIGEST, DigestAcc, Csum>::type cs;
  if constexpr (DIGEST) cs.init(dst_sizes[s.dst_buf], s.dst_off + (uint64_t)r0 * s.dst_pitch, csum_base);
  // A copy interleaves the wavefronts (load k of the whole workgroup covers 16 KiB in a row); a read-only pass gives
  // every wavefront its own contiguous 8 KiB instead - measured 3-4% faster when nothing is written, 2-5% slower
  // when the same tile is also stored.
  uint32_t first = bundle ? lane : threadIdx.x;
  if (!DIGEST && !bundle && s.op == kOpChecksumOnly && s.unit == 16u) first = wave * (64u * kPlaceBatch) + lane;
  bool placed = false;
  if constexpr (RAGGED) {
    placed = s.ragged != 0;
    if (placed) switch (s.op) {
      case kOpCopy: run_tile<kOpCopy, 16, true>(s, src, dst, csum_base, n_units, nan_bits, cs, first, col0); break;
      case kOpCastF32Bf16: run_tile<kOpCastF32Bf16, 8, true>(s, src, dst, csum_base, n_units, nan_bits, cs, first, col0); break;
      case kOpCastF32F16: run_tile<kOpCastF32F16, 8, true>(s, src, dst, csum_base, n_units, nan_bits, cs, first, col0); break;
      case kOpCastBf16F32: run_tile<kOpCastBf16F32, 16, true>(s, src, dst, csum_base, n_units, nan_bits, cs, first, col0); break;
      case kOpCastF16F32: run_tile<kOpCastF16F32, 16, true>(s, src, dst, csum_base, n_units, nan_bits, cs, first, col0); break;
      case kOpCastF8E4M3Bf16: run_tile<kOpCastF8E4M3Bf16, 16, true>(s, src, dst, csum_base, n_units, nan_bits, cs, first, col0); break;
      case kOpCastF16Bf16: run_tile<kOpCastF16Bf16, 16, true>(s, src, dst, csum_base, n_units, nan_bits, cs, first, col0); break;
      case kOpCastBf16F16: run_tile<kOpCastBf16F16, 16, true>(s, src, dst, csum_base, n_units, nan_bits, cs, first, col0); break;
      default: break;
    }
  }
  if constexpr (CHECKSUM_ONLY) {
    switch (s.unit) {
      case 16u: run_tile<kOpChecksumOnly, 16>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
      case 4u: run_tile<kOpChecksumOnly, 4>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
      case 2u: run_tile<kOpChecksumOnly, 2>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
      case 1u: run_tile<kOpChecksumOnly, 1>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
      default: break;
    }
  } else if (placed) {
  } else if (s.op * 32u + s.unit == kOpCopy * 32u + 16u) {
    // ahead of the switch, whose branches lie far apart and are not in the instruction cache when a small launch starts: 3 MB in 11.1 us, 10.7
    run_tile<kOpCopy, 16>(s, src, dst, csum_base, n_units, nan_bits, cs, first);
  } else
  switch (s.op * 32u + s.unit) {
    case kOpCopy * 32u + 4u: run_tile<kOpCopy, 4>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
    case kOpCopy * 32u + 2u: run_tile<kOpCopy, 2>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
    case kOpCopy * 32u + 1u: run_tile<kOpCopy, 1>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
    case kOpCastF32Bf16 * 32u + 8u: run_tile<kOpCastF32Bf16, 8>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
    case kOpCastF32Bf16 * 32u + 2u: run_tile<kOpCastF32Bf16, 2>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
    case kOpCastF32F16 * 32u + 8u: run_tile<kOpCastF32F16, 8>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
    case kOpCastF32F16 * 32u + 2u: run_tile<kOpCastF32F16, 2>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
    case kOpCastBf16F32 * 32u + 16u: run_tile<kOpCastBf16F32, 16>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
    case kOpCastBf16F32 * 32u + 4u: run_tile<kOpCastBf16F32, 4>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
    case kOpCastF16F32 * 32u + 16u: run_tile<kOpCastF16F32, 16>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
    case kOpCastF16F32 * 32u + 4u: run_tile<kOpCastF16F32, 4>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
    case kOpCastF8E4M3Bf16 * 32u + 16u: run_tile<kOpCastF8E4M3Bf16, 16>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
    case kOpCastF8E4M3Bf16 * 32u + 4u: run_tile<kOpCastF8E4M3Bf16, 4>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
    case kOpCastF8E4M3Bf16 * 32u + 2u: run_tile<kOpCastF8E4M3Bf16, 2>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
    case kOpCastF16Bf16 * 32u + 16u: run_tile<kOpCastF16Bf16, 16>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
    case kOpCastF16Bf16 * 32u + 4u: run_tile<kOpCastF16Bf16, 4>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
    case kOpCastF16Bf16 * 32u + 2u: run_tile<kOpCastF16Bf16, 2>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
    case kOpCastBf16F16 * 32u + 16u: run_tile<kOpCastBf16F16, 16>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
    case kOpCastBf16F16 * 32u + 4u: run_tile<kOpCastBf16F16, 4>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
    case kOpCastBf16F16 * 32u + 2u: run_tile<kOpCastBf16F16, 2>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
    case kOpChecksumOnly * 32u + 16u: run_tile<kOpChecksumOnly, 16>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
    case kOpChecksumOnly * 32u + 4u: run_tile<kOpChecksumOnly, 4>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
    case kOpChecksumOnly * 32u + 2u: run_tile<kOpChecksumOnly, 2>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
    case kOpChecksumOnly * 32u + 1u: run_tile<kOpChecksumOnly, 1>(s, src, dst, csum_base, n_units, nan_bits, cs, first); break;
    default: break;  // the host validates (op, unit) before upload
  }

  if constexpr (DIGEST) {
    // five 64-bit sums and the checksum per workgroup: wavefront reductions, then one lane adds them up
    __shared__ unsigned long long dpart[kPlaceThreads / 64][5];
    __shared__ uint32_t part[kPlaceThreads / 64];
    // whether some of what the tile stored lies after the buffer's last whole row
    const bool tail = s.dst_off + (uint64_t)(r0 + nrows - 1u) * s.dst_pitch + (uint64_t)s.units_per_row * s.unit > cs.tail_byte0;
    cs.flush();
    if (bundle) {
      const unsigned long long sums5[5] = {wave_sum_u64(cs.S), wave_sum_u64(cs.SW), wave_sum_u64(cs.T), wave_sum_u64(cs.TW), wave_sum_u64(cs.RG)};
      const uint32_t wsum = wave_sum_u32(cs.cs.fold());
      const unsigned long long t = lane == 0 ? sums5[0] : lane == 1 ? sums5[1] : lane == 2 ? sums5[2] : lane == 3 ? sums5[3] : sums5[4];
      if (lane < 5u && t) atomicAdd(&digest_sums[5ull * (lane_first + s.dst_buf) + lane], t);
      if (lane == 0 && s.csum_slot != 0xFFFFFFFFu) atomicAdd(&sums[lane_first + s.csum_slot], wsum);
      return;
    }
    unsigned long long v[5] = {cs.S, cs.SW, cs.T, cs.TW, cs.RG};
    const uint32_t n_sums = tail ? 5u : 2u;
#pragma unroll
    for (uint32_t q = 0; q < 5; ++q)
      if (q < n_sums) {
        v[q] = wave_sum_u64(v[q]);
        if ((threadIdx.x & 63) == 0) dpart[threadIdx.x >> 6][q] = v[q];
      }
    const uint32_t wsum = wave_sum_u32(cs.cs.fold());
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = wsum;
    __syncthreads();
    if (threadIdx.x < n_sums) {
      unsigned long long t = 0;
#pragma unroll
      for (int k = 0; k < kPlaceThreads / 64; ++k) t += dpart[k][threadIdx.x];
      if (t) atomicAdd(&digest_sums[5ull * (lane_first + s.dst_buf) + threadIdx.x], t);
    } else if (threadIdx.x == 64 && s.csum_slot != 0xFFFFFFFFu) {
      uint32_t t = 0;
#pragma unroll
      for (int k = 0; k < kPlaceThreads / 64; ++k) t += part[k];
      atomicAdd(&sums[lane_first + s.csum_slot], t);
    }
  } else if (s.csum_slot != 0xFFFFFFFFu) {
    __shared__ uint32_t part[kPlaceThreads / 64];
    const uint32_t wsum = wave_sum_u32(cs.fold());
    if (bundle) {
      if (lane == 0) atomicAdd(&sums[lane_first + s.csum_slot], wsum);
      return;
    }
    if (lane == 0) part[wave] = wsum;
    __syncthreads();
    if (threadIdx.x == 0) {
      uint32_t t = 0;
#pragma unroll
      for (int k = 0; k < kPlaceThreads / 64; ++k) t += part[k];
      atomicAdd(&sums[lane_first + s.csum_slot], t);
    }
  }
}

// Writes parameter bytes (copy, cast) and accumulates their checksums.  Eight wavefronts to a SIMD (64 VGPRs): a launch
// that only widens runs two workgroups per compute unit (launch_place).
__global__ __launch_bounds__(kPlaceThreads, 8) void place_kernel(
    const Seg* __restrict__ segs, const WorkItem* __restrict__ work,
    const void* const* __restrict__ src_bases, void* const* __restrict__ dst_bases,
    uint32_t* __restrict__ sums, Fan fan, uint32_t nan_bits, uint32_t* __restrict__ zero, uint32_t zero_words) {
  place_body<false, false>(segs, work, src_bases, dst_bases, sums, fan, nan_bits, nullptr, nullptr, zero, zero_words);
}
__global__ __launch_bounds__(kPlaceThreads) void place_ragged_kernel(
    const Seg* __restrict__ segs, const WorkItem* __restrict__ work,
    const void* const* __restrict__ src_bases, void* const* __restrict__ dst_bases,
    uint32_t* __restrict__ sums, Fan fan, uint32_t nan_bits, uint32_t* __restrict__ zero, uint32_t zero_words) {
  place_body<false, true>(segs, work, src_bases, dst_bases, sums, fan, nan_bits, nullptr, nullptr, zero, zero_words);
}

// place_kernel that also accumulates the tensor_digest sums of every destination buffer
// (five 64-bit words per buffer in `digest_sums`; `dst_sizes` holds the buffers' byte sizes).
__global__ __launch_bounds__(kPlaceThreads) void place_digest_kernel(
    const Seg* __restrict__ segs, const WorkItem* __restrict__ work,
    const void* const* __restrict__ src_bases, void* const* __restrict__ dst_bases,
    uint32_t* __restrict__ sums, Fan fan, uint32_t nan_bits, const unsigned long long* __restrict__ dst_sizes,
    unsigned long long* __restrict__ digest_sums, uint32_t* __restrict__ zero, uint32_t zero_words) {
  place_body<false, false, true>(segs, work, src_bases, dst_bases, sums, fan, nan_bits, dst_sizes, digest_sums, zero, zero_words);
}
__global__ __launch_bounds__(kPlaceThreads) void place_digest_ragged_kernel(
    const Seg* __restrict__ segs, const WorkItem* __restrict__ work,
    const void* const* __restrict__ src_bases, void* const* __restrict__ dst_bases,
    uint32_t* __restrict__ sums, Fan fan, uint32_t nan_bits, const unsigned long long* __restrict__ dst_sizes,
    unsigned long long* __restrict__ digest_sums, uint32_t* __restrict__ zero, uint32_t zero_words) {
  place_body<false, true, true>(segs, work, src_bases, dst_bases, sums, fan, nan_bits, dst_sizes, digest_sums, zero, zero_words);
}

// Read-only variant for batches made of checksum-only segments.
__global__ __launch_bounds__(kPlaceThreads) void checksum_kernel(
    const Seg* __restrict__ segs, const WorkItem* __restrict__ work,
    const void* const* __restrict__ src_bases, uint32_t* __restrict__ sums, Fan fan) {
  place_body<true, false>(segs, work, src_bases, nullptr, sums, fan, 0u);
}

// One workgroup per compute unit: a unit then alternates between one 128 KiB read burst and
// one 128 KiB write burst instead of mixing the two.  Two resident workgroups measured 3-5%
// slower on every configuration.  The limit is imposed with an otherwise unused dynamic LDS
// allocation of more than half a unit's LDS, which needs the attribute below once per device.
// A launch that only reads (checksum_kernel) is the other way round: two resident workgroups, one
// loading while the other adds up, read a tenth faster than one.
constexpr uint32_t kOnePerCu = 96 * 1024;
constexpr uint32_t kTwoPerCu = 48 * 1024;

hipError_t configure_place_kernels() {
  static std::atomic<uint64_t> configured{0};  // bit per device
  int dev = 0;
  if (hipError_t e = hipGetDevice(&dev); e != hipSuccess) return e;
  const uint64_t bit = 1ull << (dev & 63);
  if (configured.load(std::memory_order_acquire) & bit) return hipSuccess;
  const void* const kernels[] = {reinterpret_cast<const void*>(place_kernel), reinterpret_cast<const void*>(place_ragged_kernel),
                                 reinterpret_cast<const void*>(place_digest_kernel),
                                 reinterpret_cast<const void*>(place_digest_ragged_kernel),
                                 reinterpret_cast<const void*>(checksum_kernel)};
  hipError_t e = hipSuccess;
  for (const void* k : kernels)
    if (e == hipSuccess) e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kOnePerCu);
  if (e == hipSuccess) configured.fetch_or(bit, std::memory_order_release);
  return e;
}

hipError_t launch_place(const Seg* segs_dev, const WorkItem* work_dev, uint32_t n_work,
                        const void* const* src_bases_dev, void* const* dst_bases_dev,
                        uint32_t* sums_dev, Fan fan, uint16_t nan_bits, hipStream_t stream, bool checksum_only,
                        uint32_t* zero_dev, uint32_t zero_words, bool widening_only, bool ragged) {
  if (n_work == 0) return hipSuccess;
  if (hipError_t e = configure_place_kernels(); e != hipSuccess) return e;
  const uint32_t lds_place = widening_only ? kTwoPerCu : kOnePerCu, lds_csum = kTwoPerCu;
  if (checksum_only) {
    hipLaunchKernelGGL(checksum_kernel, dim3(n_work), dim3(kPlaceThreads), lds_csum, stream, segs_dev, work_dev,
                       src_bases_dev, sums_dev, fan);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(ragged ? place_ragged_kernel : place_kernel, dim3(n_work), dim3(kPlaceThreads), lds_place, stream, segs_dev,
                     work_dev, src_bases_dev, dst_bases_dev, sums_dev, fan, (uint32_t)nan_bits, zero_dev, zero_words);
  return hipGetLastError();
}

hipError_t launch_place_digest(const Seg* segs_dev, const WorkItem* work_dev, uint32_t n_work,
                               const void* const* src_bases_dev, void* const* dst_bases_dev, uint32_t* sums_dev, Fan fan,
                               const unsigned long long* dst_sizes_dev, unsigned long long* digest_sums_dev,
                               uint16_t nan_bits, hipStream_t stream, uint32_t* zero_dev, uint32_t zero_words, bool ragged) {
  if (n_work == 0) return hipSuccess;
  if (hipError_t e = configure_place_kernels(); e != hipSuccess) return e;
  hipLaunchKernelGGL(ragged ? place_digest_ragged_kernel : place_digest_kernel, dim3(n_work), dim3(kPlaceThreads), kOnePerCu, stream,
                     segs_dev, work_dev, src_bases_dev, dst_bases_dev, sums_dev, fan, (uint32_t)nan_bits, dst_sizes_dev, digest_sums_dev, zero_dev, zero_words);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// tensor_digest row sums (reference: modelexpress/refit/reshard/verify.py:112-150).
// Bytes are read as little-endian signed int32 words; whole 1024-word rows give
// sum_r rs[r] and sum_r rs[r]*(r+1); the words after the last whole row give
// sum_k t[k] and sum_k t[k]*(k+1); the 1..3 bytes after the last whole word are summed
// unsigned.  All sums wrap mod 2^64.  The index weight is applied per lane before any
// reduction (sum_r (sum_lane p)*(r+1) == sum_lane sum_r p*(r+1)), so there is a single
// reduction per workgroup.
//
// With CSUM the checksum of the same bytes comes out of the same pass: a manifest needs both, the kernel is bound
// by the read (22 VALU instructions per 16 bytes are a quarter of what a compute unit issues meanwhile), and two
// passes read every buffer twice.  195 buffers, 2.008 GB: 291 us = 6.9 TB/s for both, where checksum_kernel takes
// 289 and the digest alone 285.
// Loads carry no alignment promise, so a buffer at any address takes this path.
// ---------------------------------------------------------------------------
template <bool CSUM>
__global__ __launch_bounds__(kDigestThreads) void digest_kernel(
    const DigestJob* __restrict__ jobs, uint32_t n_jobs, uint32_t rows_per_block, unsigned long long* __restrict__ out,
    uint32_t* __restrict__ sums, Fan fan) {
  // Workgroup-uniform binary search for the job that owns this workgroup.
  uint32_t lo = 0, hi = n_jobs;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (jobs[mid].first_block <= blockIdx.x) lo = mid; else hi = mid;
  }
  const DigestJob j = jobs[lo];
  const uint64_t blk = blockIdx.x - j.first_block;
  const uint64_t body_words = j.nbytes >> 2;
  const uint64_t rows = body_words / kDigestRowWords;
  const uint64_t n_blocks = rows ? (rows + rows_per_block - 1) / rows_per_block : 1;
  const uint64_t row_begin = blk * rows_per_block;
  const uint64_t row_end = min(rows, row_begin + rows_per_block);
  const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  constexpr uint32_t kWaves = kDigestThreads / 64, kRowBytes = kDigestRowWords * 4;

  unsigned long long A = 0, B = 0, At = 0, Bt = 0, Rg = 0;
  Csum cs;
  auto lane_sum = [](const uint4& x) {
    return (long long)(int32_t)x.x + (long long)(int32_t)x.y + (long long)(int32_t)x.z + (long long)(int32_t)x.w;
  };
  // Two rows per wavefront: eight 16-byte loads per lane in flight, a 128 KiB read burst per workgroup, the
  // shape that measured fastest for the copy kernel.  A batch too small to give every compute unit two such
  // workgroups is cut into workgroups of one row per wavefront (digest_jobs).
  const uint32_t per_wave = rows_per_block / kWaves;
  for (uint64_t r = row_begin + per_wave * wave; r < row_end; r += per_wave * kWaves) {
    const bool two = per_wave == 2u && r + 1 < row_end;
    const uint8_t* row0 = j.ptr + r * (uint64_t)kRowBytes;
    uint4 x[8];
#pragma unroll
    for (int k = 0; k < 4; ++k) x[k] = ld16(row0 + 16u * (lane + 64u * k));
    if (two) {
#pragma unroll
      for (int k = 0; k < 4; ++k) x[4 + k] = ld16(row0 + kRowBytes + 16u * (lane + 64u * k));
    }
    long long a0 = 0, a1 = 0;
    const uint32_t pos = (uint32_t)(r * kRowBytes) + 16u * lane;  // checksum positions are taken mod 2^32
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      a0 += lane_sum(x[k]);
      if constexpr (CSUM) cs.add16(x[k], pos + 1024u * k);
    }
    if (two) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        a1 += lane_sum(x[4 + k]);
        if constexpr (CSUM) cs.add16(x[4 + k], pos + kRowBytes + 1024u * k);
      }
    }
    A += (unsigned long long)a0 + (unsigned long long)a1;
    B += (unsigned long long)a0 * (unsigned long long)(r + 1) + (unsigned long long)a1 * (unsigned long long)(r + 2);
  }
  if (blk == n_blocks - 1) {
    const uint8_t* tail = j.ptr + rows * (uint64_t)kRowBytes;
    const uint32_t tw = (uint32_t)(body_words - rows * kDigestRowWords), pos = (uint32_t)(rows * kRowBytes);
    for (uint32_t k = threadIdx.x; k < tw; k += kDigestThreads) {
      const uint32_t u = *reinterpret_cast<const u32_u*>(tail + 4u * k);
      const long long w = (long long)(int32_t)u;
      At += (unsigned long long)w;
      Bt += (unsigned long long)w * (unsigned long long)(k + 1);
      if constexpr (CSUM) cs.add4(u, pos + 4u * k);
    }
    if (threadIdx.x == 0) {
      const uint32_t rag = (uint32_t)(j.nbytes & 3u);
      for (uint32_t k = 0; k < rag; ++k) {
        const uint32_t byte = j.ptr[body_words * 4 + k];
        Rg += byte;
        if constexpr (CSUM) cs.add_byte(byte, (uint32_t)(body_words * 4) + k);
      }
    }
  }

  __shared__ unsigned long long part[kDigestThreads / 64][5];
  __shared__ uint32_t csum_part[kDigestThreads / 64];
  unsigned long long v[5] = {A, B, At, Bt, Rg};
#pragma unroll
  for (int q = 0; q < 5; ++q) {
    const unsigned long long wsum = wave_sum_u64(v[q]);
    if (lane == 0) part[wave][q] = wsum;
  }
  if constexpr (CSUM) {
    const uint32_t wsum = wave_sum_u32(cs.fold());
    if (lane == 0) csum_part[wave] = wsum;
  }
  __syncthreads();
  const uint64_t copy = (uint64_t)(blockIdx.x & fan.mask) * fan.pitch;
  if (threadIdx.x < 5) {
    unsigned long long t = 0;
#pragma unroll
    for (int k = 0; k < kDigestThreads / 64; ++k) t += part[k][threadIdx.x];
    if (t) atomicAdd(&out[5ull * (copy + lo) + threadIdx.x], t);
  } else if (CSUM && threadIdx.x == 64) {
    uint32_t t = 0;
#pragma unroll
    for (int k = 0; k < kDigestThreads / 64; ++k) t += csum_part[k];
    atomicAdd(&sums[copy + lo], t);
  }
}

hipError_t launch_digest(const DigestJob* jobs_dev, uint32_t n_jobs, uint32_t n_blocks, uint32_t rows_per_block,
                         unsigned long long* out_dev, uint32_t* sums_dev, Fan fan, hipStream_t stream) {
  if (n_jobs == 0 || n_blocks == 0) return hipSuccess;
  if (sums_dev)
    hipLaunchKernelGGL(digest_kernel<true>, dim3(n_blocks), dim3(kDigestThreads), 0, stream, jobs_dev, n_jobs, rows_per_block, out_dev,
                       sums_dev, fan);
  else
    hipLaunchKernelGGL(digest_kernel<false>, dim3(n_blocks), dim3(kDigestThreads), 0, stream, jobs_dev, n_jobs, rows_per_block, out_dev,
                       nullptr, fan);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Results to the host.  One wavefront per accumulator: lane l reads copy l (a fan has at most 64 copies), so the
// loads of an accumulator are all in flight at once.  BLAKE2b (RFC 7693) of the scalar list runs in the same
// wavefront, four lanes a column each (every group of four does the same work), the diagonal step being three
// quad permutations; the message waits in LDS.  Each record ends with a word that carries the caller's sequence
// number: the host spins on that instead of waiting for an event behind the launch, 6.5 against 12 us for a
// launch and its result, and of the hashes nothing is left on the host (195 of them: 30 us).
// ---------------------------------------------------------------------------
constexpr uint32_t quad_perm(uint32_t a, uint32_t b, uint32_t c, uint32_t d) { return a | (b << 2) | (c << 4) | (d << 6); }
template <uint32_t CTRL>
__device__ __forceinline__ uint64_t quad_permute(uint64_t v) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)v, CTRL, 0xF, 0xF, true);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(v >> 32), CTRL, 0xF, 0xF, true);
  return (uint64_t)lo | ((uint64_t)hi << 32);
}
template <int N>
__device__ __forceinline__ uint64_t rotr64(uint64_t x) {
  return (x >> N) | (x << (64 - N));
}
__device__ __forceinline__ void blake2b_g(uint64_t& a, uint64_t& b, uint64_t& c, uint64_t& d, uint64_t x, uint64_t y) {
  a = a + b + x;
  d = rotr64<32>(d ^ a);
  c = c + d;
  b = rotr64<24>(b ^ c);
  a = a + b + y;
  d = rotr64<16>(d ^ a);
  c = c + d;
  b = rotr64<63>(b ^ c);
}
// RFC 7693 section 2.7: the message word order of the ten rounds, sixteen 4-bit indices each, first index lowest.
constexpr uint64_t kBlakeOrder[10] = {0xFEDCBA9876543210ull, 0x357B20C16DF984AEull, 0x491763EADF250C8Bull, 0x8F04A562EBCD1397ull,
                                      0xD386CB1EFA427509ull, 0x91EF57D438B0A6C2ull, 0xB8293670A4DEF15Cull, 0xA2684F05931CE7BDull,
                                      0x5A417D2C803B9EF6ull, 0x0DC3E9BF5167482Aull};
// The first 128 bits of BLAKE2b-128 of the `words` (1..7) 64-bit words in `m` (sixteen words of LDS, zero beyond
// them), in lane 0 of every group of four lanes (low word) and lane 1 (high word).  All lanes of the wavefront
// must be active.
__device__ __forceinline__ uint64_t blake2b_quad(const uint64_t* m, uint32_t words) {
  constexpr uint64_t iv[8] = {0x6a09e667f3bcc908ull, 0xbb67ae8584caa73bull, 0x3c6ef372fe94f82bull, 0xa54ff53a5f1d36f1ull,
                              0x510e527fade682d1ull, 0x9b05688c2b3e6c1full, 0x1f83d9abfb41bd6bull, 0x5be0cd19137e2179ull};
  const uint32_t q = threadIdx.x & 3u;
  auto pick = [&](uint64_t w0, uint64_t w1, uint64_t w2, uint64_t w3) { return q == 0 ? w0 : q == 1 ? w1 : q == 2 ? w2 : w3; };
  const uint64_t h0 = pick(iv[0] ^ 0x01010010ull, iv[1], iv[2], iv[3]);  // unkeyed, 16 bytes out
  uint64_t a = h0, b = pick(iv[4], iv[5], iv[6], iv[7]), c = pick(iv[0], iv[1], iv[2], iv[3]);
  uint64_t d = pick(iv[4] ^ (uint64_t)(words * 8u), iv[5], ~iv[6], iv[7]);  // byte count; the last block
#pragma unroll
  for (int r = 0; r < 12; ++r) {
    const uint64_t order = kBlakeOrder[r % 10] >> (8u * q);
    const uint64_t x0 = m[order & 15u], x1 = m[(order >> 4) & 15u], x2 = m[(order >> 32) & 15u], x3 = m[(order >> 36) & 15u];
    blake2b_g(a, b, c, d, x0, x1);
    b = quad_permute<quad_perm(1, 2, 3, 0)>(b);
    c = quad_permute<quad_perm(2, 3, 0, 1)>(c);
    d = quad_permute<quad_perm(3, 0, 1, 2)>(d);
    blake2b_g(a, b, c, d, x2, x3);
    b = quad_permute<quad_perm(3, 0, 1, 2)>(b);
    c = quad_permute<quad_perm(2, 3, 0, 1)>(c);
    d = quad_permute<quad_perm(1, 2, 3, 0)>(d);
  }
  return h0 ^ a ^ c;
}

constexpr int kFinishWaves = 4;
__global__ __launch_bounds__(kFinishWaves * 64) void finish_kernel(uint32_t* __restrict__ sums, unsigned long long* __restrict__ dsums,
                                                                   Fan fan, uint64_t n, const uint8_t* __restrict__ sizes,
                                                                   uint32_t sizes_stride, FinishRec* __restrict__ out, uint32_t seq,
                                                                   bool clear) {
  static_assert(kFanLanes <= 64, "one lane of a wavefront per copy");
  __shared__ uint64_t message[kFinishWaves][16];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const bool mine = lane <= fan.mask;
  for (uint64_t k = (uint64_t)blockIdx.x * kFinishWaves + wave; k < n; k += (uint64_t)gridDim.x * kFinishWaves) {
    uint32_t csum = 0;
    if (sums && mine) {
      uint32_t* p = sums + (uint64_t)lane * fan.pitch + k;
      csum = *p;
      if (clear) *p = 0;
    }
    unsigned long long s[5] = {0, 0, 0, 0, 0};
    if (dsums && mine) {
      unsigned long long* p = dsums + 5ull * ((uint64_t)lane * fan.pitch + k);
#pragma unroll
      for (int i = 0; i < 5; ++i) s[i] = p[i];
      if (clear) {
#pragma unroll
        for (int i = 0; i < 5; ++i) p[i] = 0;
      }
    }
    csum = wave_sum_u32(csum);
    if (dsums) {
#pragma unroll
      for (int i = 0; i < 5; ++i) s[i] = wave_sum_u64(s[i]);
      const uint64_t bytes = *reinterpret_cast<const uint64_t*>(sizes + k * sizes_stride);
      // the scalar list: the size, then the sums of what the buffer has - whole rows, words after them, ragged bytes
      const uint64_t words = bytes / 4, rows = words / kDigestRowWords;
      const bool has_tail = words != rows * kDigestRowWords, has_ragged = (bytes & 3u) != 0;
      const uint32_t at_tail = rows ? 3u : 1u, at_ragged = at_tail + (has_tail ? 2u : 0u), count = at_ragged + (has_ragged ? 2u : 0u);
      if (lane < 16u) {
        uint64_t w = 0;
        if (lane == 0u) w = bytes;
        else if (lane < at_tail) w = lane == 1u ? s[0] : s[1];
        else if (lane < at_ragged) w = lane == at_tail ? s[2] : s[3];
        else if (lane < count) w = lane == at_ragged ? s[4] : (bytes & 3u);
        message[wave][lane] = w;
      }
      // one wavefront's own LDS words: its accesses complete in issue order
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      const uint64_t h = blake2b_quad(message[wave], count);
      const uint64_t w = lane < 2u ? h : lane == 2u ? s[0] : lane == 3u ? s[1] : lane == 4u ? s[2] : lane == 5u ? s[3] : s[4];
      if (lane < 7u) __hip_atomic_store(&out[k].w[lane], w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    // The record's other words have left before its last one does.  They are stored through every cache (system
    // scope), so waiting for the wavefront's own stores is all the order they need on this hardware (the language's
    // memory model would ask for a release); a release, which also writes back whatever else the cache holds, is for
    // the accumulators cleared here, which the next run adds to.
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_s_waitcnt(0);
    const uint64_t last = (uint64_t)csum | ((uint64_t)seq << 32);
    if (lane == 0u) {
      if (clear) __hip_atomic_store(&out[k].w[7], last, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
      else __hip_atomic_store(&out[k].w[7], last, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
}

hipError_t launch_finish(uint32_t* sums_dev, unsigned long long* dsums_dev, Fan fan, uint64_t n, const uint8_t* sizes_dev,
                         uint32_t sizes_stride, FinishRec* out_dev, uint32_t seq, bool clear, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  const uint64_t blocks = (n + kFinishWaves - 1) / kFinishWaves;
  hipLaunchKernelGGL(finish_kernel, dim3((uint32_t)(blocks > 4096 ? 4096 : blocks)), dim3(kFinishWaves * 64), 0, stream, sums_dev,
                     dsums_dev, fan, n, sizes_dev, sizes_stride, out_dev, seq, clear);
  return hipGetLastError();
}

// Plain vector-store fill; used instead of a memset node so callers may capture it.
__global__ __launch_bounds__(256) void fill_u32_kernel(uint32_t* __restrict__ p, uint64_t n,
                                                       uint32_t value) {
  for (uint64_t i = blockIdx.x * 256ull + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256ull)
    p[i] = value;
}

hipError_t launch_fill_u32(uint32_t* ptr, uint64_t n, uint32_t value, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  const uint64_t blocks = (n + 255) / 256;
  hipLaunchKernelGGL(fill_u32_kernel, dim3((uint32_t)(blocks > 4096 ? 4096 : blocks)), dim3(256), 0,
                     stream, ptr, n, value);
  return hipGetLastError();
}

// Table copy by plain 16-byte loads and stores (no memcpy node: callers may capture it), and the clearing of the
// accumulators the next launch adds to: a launch of their own cost every operator call 3 us.
__global__ __launch_bounds__(256) void copy_table_kernel(uint4* __restrict__ dst, const uint4* __restrict__ src, uint64_t n16,
                                                         uint32_t* __restrict__ zero, uint64_t zero_words) {
  for (uint64_t i = blockIdx.x * 256ull + threadIdx.x; i < n16; i += (uint64_t)gridDim.x * 256ull) dst[i] = src[i];
  for (uint64_t i = blockIdx.x * 256ull + threadIdx.x; i < zero_words; i += (uint64_t)gridDim.x * 256ull) zero[i] = 0u;
}

hipError_t launch_copy_table(void* dst, const void* src, size_t bytes, hipStream_t stream, uint32_t* zero_dev, uint64_t zero_words) {
  if (bytes == 0 && zero_words == 0) return hipSuccess;
  if ((bytes & 15u) || (reinterpret_cast<uintptr_t>(dst) & 15u) || (reinterpret_cast<uintptr_t>(src) & 15u)) return hipErrorInvalidValue;
  const uint64_t n16 = bytes / 16, n = n16 > zero_words / 4 ? n16 : zero_words / 4, blocks = (n + 255) / 256;
  hipLaunchKernelGGL(copy_table_kernel, dim3((uint32_t)(blocks > 1024 ? 1024 : blocks ? blocks : 1)), dim3(256), 0, stream,
                     static_cast<uint4*>(dst), static_cast<const uint4*>(src), n16, zero_dev, zero_words);
  return hipGetLastError();
}

}  // namespace mxp
