// CPU stand-ins for the kernel launches the host engine issues (declared in csrc/mxp_device.h), queued on the
// CPU streams of cpu_hip.cpp.  Test infrastructure: they exist so that the engine's ring, reader threads, descriptor
// arenas, results and stream ordering run under ThreadSanitizer / AddressSanitizer with every "device" access a real memory access.
// A segment is executed by its meaning (a pitched box, a conversion, a position-weighted checksum of the bytes
// written), not by the kernel's lane arithmetic - that is checked elsewhere (tests/c/lower_check.cpp, the GPU tests).
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <utility>
#include <vector>

#include "mxp.h"
#include "mxp_device.h"

namespace mxp {

// Views launched so far as wavefront-autonomous transposes, as panels and woven.
int launched_forms[3];

namespace {

int form_of(const TransposeDesc& d) { return d.weave_chunks ? 2 : d.panel_rows_log2 ? 1 : 0; }

uint32_t f32_to_bf16(uint32_t u, uint32_t nan_bits) {
  if ((u & 0x7FFFFFFFu) > 0x7F800000u) return nan_bits;
  return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}

[[noreturn]] void unsupported(const char* what) {
  std::fprintf(stderr, "cpu stand-in: %s is not implemented\n", what);
  std::abort();
}

// The share of `n` bytes at position `pos` of a buffer of `nbytes` in its five digest sums: little-endian signed words in
// rows of 1024, the words after the last whole row, the bytes after the last whole word.
void add_digest(unsigned long long* sums, uint64_t nbytes, uint64_t pos, const uint8_t* bytes, uint64_t n) {
  const uint64_t body_end = nbytes / 4 * 4, tail = nbytes / 4096 * 4096;
  unsigned long long add[5] = {};
  for (uint64_t p = pos; p < pos + n; ++p) {
    const uint32_t b = bytes[p - pos];
    if (p >= body_end) {
      add[4] += b;
      continue;
    }
    const long long v = p % 4 == 3 ? (long long)(int32_t)(b << 24) : (long long)b << (8 * (p % 4));
    if (p < tail) {
      add[0] += (unsigned long long)v;
      add[1] += (unsigned long long)v * (p / 4096 + 1);
    } else {
      add[2] += (unsigned long long)v;
      add[3] += (unsigned long long)v * ((p - tail) / 4 + 1);
    }
  }
  for (int q = 0; q < 5; ++q) __atomic_fetch_add(&sums[q], add[q], __ATOMIC_RELAXED);
}

struct DigestSums {
  const unsigned long long* sizes;  // byte size of every destination buffer
  unsigned long long* sums;         // fanned, five to a buffer
};

void run_item(const Seg* segs, const WorkItem& w, uint32_t block, const void* const* src_bases, void* const* dst_bases,
              uint32_t* sums, Fan fan, uint32_t nan_bits, const DigestSums* digests = nullptr) {
  if (w.tile & kBundle) {  // a segment of one tile for every wavefront
    for (uint32_t k = 0; k < (w.tile & ~kBundle); ++k) {
      if (segs[w.seg + k].rows > segs[w.seg + k].rows_per_tile) unsupported("a segment of several tiles in a bundle");
      run_item(segs, WorkItem{w.seg + k, 0}, block, src_bases, dst_bases, sums, fan, nan_bits, digests);
    }
    return;
  }
  const Seg& seg = segs[w.seg];
  if (seg.ragged) {  // the pieces of rows a tile of a contiguous destination takes, each as a row of its own
    const uint64_t u0 = (uint64_t)w.tile * seg.rows_per_tile;
    if (u0 >= seg.rows) unsupported("a work item past the end of its segment");
    const uint64_t n = seg.rows - u0 < seg.rows_per_tile ? seg.rows - u0 : seg.rows_per_tile;
    uint64_t at = seg.ragged - 1u + u0 * seg.unit;
    const uint64_t end = at + n * seg.unit, at0 = seg.ragged - 1u;
    while (at < end) {
      const uint64_t row = at / seg.row_bytes, col = at % seg.row_bytes;
      const uint64_t take = seg.row_bytes - col < end - at ? seg.row_bytes - col : end - at;
      Seg piece = seg;
      piece.ragged = 0;
      piece.rows = piece.rows_per_tile = 1;
      piece.src_off = seg.src_off + row * seg.src_pitch + op_src_bytes(seg.op, col);
      piece.dst_off = seg.dst_off + (at - at0);
      piece.row_bytes = (uint32_t)take;
      run_item(&piece, WorkItem{0, 0}, block, src_bases, dst_bases, sums, fan, nan_bits, digests);
      at += take;
    }
    return;
  }
  const Seg& s = seg;
  const uint64_t r0 = (uint64_t)w.tile * s.rows_per_tile;
  if (r0 >= s.rows) unsupported("a work item past the end of its segment");
  const uint64_t nrows = s.rows - r0 < s.rows_per_tile ? s.rows - r0 : s.rows_per_tile;
  const uint8_t* src_base = static_cast<const uint8_t*>(s.src_buf == kSrcIsDestination ? dst_bases[s.dst_buf] : src_bases[s.src_buf]);
  uint8_t* dst_base = s.op == kOpChecksumOnly ? nullptr : static_cast<uint8_t*>(dst_bases[s.dst_buf]);
  uint32_t sum = 0;
  for (uint64_t r = r0; r < r0 + nrows; ++r) {
    const uint8_t* sp = src_base + s.src_off + r * s.src_pitch;
    uint8_t* dp = dst_base ? dst_base + s.dst_off + r * s.dst_pitch : nullptr;
    const uint8_t* written = nullptr;
    switch (s.op) {
      case kOpCopy:
        std::memcpy(dp, sp, s.row_bytes);
        written = dp;
        break;
      case kOpChecksumOnly:
        written = sp;
        break;
      case kOpCastF32Bf16:
        for (uint32_t e = 0; e < s.row_bytes / 2; ++e) {
          uint32_t u;
          std::memcpy(&u, sp + 4ull * e, 4);
          const uint16_t h = (uint16_t)f32_to_bf16(u, nan_bits);
          std::memcpy(dp + 2ull * e, &h, 2);
        }
        written = dp;
        break;
      case kOpCastBf16F32:
        for (uint32_t e = 0; e < s.row_bytes / 4; ++e) {
          uint16_t h;
          std::memcpy(&h, sp + 2ull * e, 2);
          const uint32_t u = (uint32_t)h << 16;
          std::memcpy(dp + 4ull * e, &u, 4);
        }
        written = dp;
        break;
      default:
        unsupported("this conversion");
    }
    if (digests)
      add_digest(digests->sums + 5 * ((uint64_t)(block & fan.mask) * fan.pitch + s.dst_buf), digests->sizes[s.dst_buf],
                 s.dst_off + r * s.dst_pitch, written, s.row_bytes);
    if (s.csum_slot != 0xFFFFFFFFu) {
      const uint32_t pos0 = (uint32_t)(s.dst_off + r * s.dst_pitch) + s.csum_bias;
      for (uint32_t i = 0; i < s.row_bytes; ++i) sum += written[i] * ((pos0 + i) * kKnuth + 1u);
    }
  }
  if (s.csum_slot != 0xFFFFFFFFu)
    __atomic_fetch_add(&sums[(block & fan.mask) * fan.pitch + s.csum_slot], sum, __ATOMIC_RELAXED);
}

}  // namespace

hipError_t configure_place_kernels() { return hipSuccess; }

hipError_t launch_place(const Seg* segs_dev, const WorkItem* work_dev, uint32_t n_work, const void* const* src_bases_dev,
                        void* const* dst_bases_dev, uint32_t* sums_dev, Fan fan, uint16_t nan_bits, hipStream_t stream, bool,
                        uint32_t* zero_dev, uint32_t zero_words, bool, bool) {
  if (n_work == 0 && zero_words == 0) return hipSuccess;
  cpu_hip::enqueue(stream, [=] {
    for (uint32_t i = 0; i < zero_words; ++i) zero_dev[i] = 0u;
    for (uint32_t b = 0; b < n_work; ++b) run_item(segs_dev, work_dev[b], b, src_bases_dev, dst_bases_dev, sums_dev, fan, nan_bits);
  });
  return hipSuccess;
}

hipError_t launch_fill_u32(uint32_t* ptr, uint64_t n, uint32_t value, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  cpu_hip::enqueue(stream, [=] {
    for (uint64_t i = 0; i < n; ++i) ptr[i] = value;
  });
  return hipSuccess;
}

hipError_t launch_copy_table(void* dst, const void* src, size_t bytes, hipStream_t stream, uint32_t* zero_dev, uint64_t zero_words) {
  if (bytes == 0 && zero_words == 0) return hipSuccess;
  cpu_hip::enqueue(stream, [=] {
    std::memcpy(dst, src, bytes);
    for (uint64_t i = 0; i < zero_words; ++i) zero_dev[i] = 0u;
  });
  return hipSuccess;
}

// The release is what the kernel's wait for its own stores, which go past every cache, comes to.
hipError_t launch_finish(uint32_t* sums_dev, unsigned long long* dsums_dev, Fan fan, uint64_t n, const uint8_t* sizes_dev,
                         uint32_t sizes_stride, FinishRec* out_dev, uint32_t seq, bool clear, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  cpu_hip::finish_queued();
  cpu_hip::enqueue(stream, [=] {
    cpu_hip::finish_starts();
    for (uint64_t k = 0; k < n; ++k) {
      uint32_t t = 0;
      unsigned long long d[5] = {};
      for (uint32_t l = 0; l < fan.lanes(); ++l) {
        const uint64_t at = (uint64_t)l * fan.pitch + k;
        if (sums_dev) {
          t += sums_dev[at];
          if (clear) sums_dev[at] = 0;
        }
        for (int q = 0; dsums_dev && q < 5; ++q) {
          d[q] += dsums_dev[5 * at + q];
          if (clear) dsums_dev[5 * at + q] = 0;
        }
      }
      if (dsums_dev) {
        uint64_t nbytes;
        std::memcpy(&nbytes, sizes_dev + k * sizes_stride, 8);
        const uint64_t scalars[7] = {nbytes, d[0], d[1], d[2], d[3], d[4], nbytes % 4};
        uint8_t hash[16];
        if (mxp_digest_from_scalars(scalars, hash) != MXP_OK) unsupported("hashing these scalars");
        std::memcpy(out_dev[k].w, hash, 16);
        for (int q = 0; q < 5; ++q) out_dev[k].w[2 + q] = d[q];
      }
      __atomic_store_n(&out_dev[k].w[7], (uint64_t)t | ((uint64_t)seq << 32), __ATOMIC_RELEASE);
    }
  });
  return hipSuccess;
}

hipError_t launch_place_digest(const Seg* segs_dev, const WorkItem* work_dev, uint32_t n_work, const void* const* src_bases_dev,
                               void* const* dst_bases_dev, uint32_t* sums_dev, Fan fan, const unsigned long long* dst_sizes_dev,
                               unsigned long long* digest_sums_dev, uint16_t nan_bits, hipStream_t stream, uint32_t* zero_dev,
                               uint32_t zero_words, bool) {
  if (n_work == 0 && zero_words == 0) return hipSuccess;
  cpu_hip::enqueue(stream, [=] {
    for (uint32_t i = 0; i < zero_words; ++i) zero_dev[i] = 0u;
    const DigestSums digests{dst_sizes_dev, digest_sums_dev};
    for (uint32_t b = 0; b < n_work; ++b) run_item(segs_dev, work_dev[b], b, src_bases_dev, dst_bases_dev, sums_dev, fan, nan_bits, &digests);
  });
  return hipSuccess;
}

// Workgroup by workgroup, as the jobs say which rows of their buffer a workgroup takes.
hipError_t launch_digest(const DigestJob* jobs_dev, uint32_t n_jobs, uint32_t n_blocks, uint32_t rows_per_block,
                         unsigned long long* out_dev, uint32_t* sums_dev, Fan fan, hipStream_t stream) {
  if (n_jobs == 0 || n_blocks == 0) return hipSuccess;
  cpu_hip::enqueue(stream, [=] {
    for (uint32_t b = 0; b < n_blocks; ++b) {
      uint32_t k = 0;
      while (k + 1 < n_jobs && jobs_dev[k + 1].first_block <= b) ++k;
      const DigestJob& j = jobs_dev[k];
      const uint64_t rows = j.nbytes / 4096, first = (b - j.first_block) * rows_per_block;
      const uint64_t blocks = rows ? (rows + rows_per_block - 1) / rows_per_block : 1;
      if (b - j.first_block >= blocks) unsupported("a workgroup past the end of its buffer");
      const uint64_t begin = first * 4096, end = b - j.first_block == blocks - 1 ? j.nbytes : begin + rows_per_block * 4096ull;
      const uint64_t at = (uint64_t)(b & fan.mask) * fan.pitch + k;
      add_digest(out_dev + 5 * at, j.nbytes, begin, j.ptr + begin, end - begin);
      uint32_t sum = 0;
      for (uint64_t p = begin; sums_dev && p < end; ++p) sum += j.ptr[p] * ((uint32_t)p * kKnuth + 1u);
      if (sums_dev) __atomic_fetch_add(&sums_dev[at], sum, __ATOMIC_RELAXED);
    }
  });
  return hipSuccess;
}

// Not exercised by the sanitizer driver: refused, so that a call that reached it is noticed.
hipError_t launch_probe_gather(const void*, void*, uint32_t, uint32_t, uint32_t, uint32_t, bool, hipStream_t) { return hipErrorNotSupported; }
namespace {

// One converted element, out of memory and into memory.
void convert_element(const uint8_t* sp, uint8_t* dp, int es, uint32_t op, uint32_t nan_bits) {
  if (op == kOpCopy) {
    std::memcpy(dp, sp, (size_t)es);
  } else if (op == kOpCastF32Bf16) {
    uint32_t u;
    std::memcpy(&u, sp, 4);
    const uint16_t h = (uint16_t)f32_to_bf16(u, nan_bits);
    std::memcpy(dp, &h, 2);
  } else if (op == kOpCastBf16F32) {
    uint16_t h;
    std::memcpy(&h, sp, 2);
    const uint32_t u = (uint32_t)h << 16;
    std::memcpy(dp, &u, 4);
  } else if (op == kOpCastF8E4M3Bf16 && (*sp & 0x7Fu) != 0x7Fu) {  // any value but NaN: exact
    const int exponent = *sp >> 3 & 15, mantissa = *sp & 7;
    const float f = (*sp & 0x80 ? -1.0f : 1.0f) * std::ldexp(exponent ? 8.0f + (float)mantissa : (float)mantissa, (exponent ? exponent : 1) - 10);
    uint32_t u;
    std::memcpy(&u, &f, 4);
    const uint16_t h = (uint16_t)(u >> 16);
    std::memcpy(dp, &h, 2);
  } else {
    unsupported("this conversion in a transpose");
  }
}

struct Batches {
  const TransposeDesc& d;
  uint64_t n = 1;
  explicit Batches(const TransposeDesc& desc) : d(desc) {
    for (int k = 0; k < kMaxBatchDims; ++k) n *= d.batch_size[k];
  }
  void offsets(uint64_t b, uint64_t& s_off, uint64_t& d_off) const {
    s_off = d_off = 0;
    for (int k = kMaxBatchDims - 1; k >= 0; --k) {
      s_off += b % d.batch_size[k] * d.batch_sstride[k];
      d_off += b % d.batch_size[k] * d.batch_dstride[k];
      b /= d.batch_size[k];
    }
  }
};

// A woven tile lane by lane, with the kernel's chunks, steps back, LDS rows and gathers: `lds` is a block of exactly the bytes
// the launch asks for, and the sources are the caller's own blocks, so the address sanitizer sees an access off either.
void run_woven(const uint8_t* src, uint8_t* dst, const TransposeDesc& d, int es, uint32_t op, uint32_t nan_bits, uint32_t* sum_out,
               uint32_t lds_bytes) {
  const uint32_t eo = op == kOpCopy ? (uint32_t)es : (uint32_t)op_dst_elem(op), V = 16 / eo;
  if (!weave_desc_ok(d, (uint32_t)es, eo) || lds_bytes > 64u * 1024u) unsupported("a woven descriptor of this kind");
  const uint32_t C = d.weave_chunks, pitch = (C << 4) + kWeavePad, ni = (uint32_t)d.ni, threads = d.waves * 64u, cols = (C << 4) / (uint32_t)es;
  const Batches batches(d);
  uint32_t sum = 0;
  std::vector<uint8_t> written;
  for (uint64_t tile = 0; tile < d.n_tiles; ++tile) {
    const uint64_t b = tile / d.tiles_j, j0 = tile % d.tiles_j * cols;
    if (b >= batches.n) unsupported("a tile past the last batch");
    uint64_t s_off, d_off;
    batches.offsets(b, s_off, d_off);
    const uint32_t nj = (uint32_t)(d.nj - j0 < cols ? d.nj - j0 : cols), row_bytes = nj * (uint32_t)es;
    const uint8_t* sp = src + (s_off + j0) * (uint64_t)es;
    uint8_t* dp = dst + (d_off + j0 * ni) * eo;
    const std::unique_ptr<uint8_t[]> lds(new uint8_t[lds_bytes]());
    if (ni * C > kWeaveLoads * threads) unsupported("a chunk that no lane loads");
    for (uint32_t q = 0; q < ni * C; ++q) {
      const uint32_t row = q / C, at = q % C * 16u, back = at + 16u > row_bytes ? at + 16u - row_bytes : 0u;
      if (at >= row_bytes) continue;
      uint8_t x[16], shifted[16] = {};
      std::memcpy(x, sp + row * d.si * (uint64_t)es + at - back, 16);  // the row's own bytes, or those of the tile before
      std::memcpy(shifted, x + back, 16 - back);
      std::memcpy(lds.get() + row * pitch + at, shifted, 16);
    }
    const uint32_t elems = ni * nj;
    written.assign(elems, 0);
    for (uint32_t e0 = 0; e0 < elems; e0 += V) {
      const uint32_t j = (uint32_t)(((uint64_t)e0 * d.weave_magic) >> 32);
      uint32_t i = e0 - j * ni, col = j;
      for (uint32_t v = 0; v < V; ++v) {
        uint8_t raw[4];
        std::memcpy(raw, lds.get() + i * pitch + col * (uint32_t)es, (size_t)es);  // past the tile's last element: in the block all the same
        if (e0 + v < elems) {
          uint8_t* o = dp + (uint64_t)(e0 + v) * eo;
          convert_element(raw, o, es, op, nan_bits);
          if (col * ni + i >= elems || written[col * ni + i]++) unsupported("an element that is stored twice");
          const uint32_t pos0 = (uint32_t)((d_off + j0 * ni + e0 + v) * eo) + d.csum_bias;
          for (uint32_t k = 0; k < eo; ++k) sum += o[k] * ((pos0 + k) * kKnuth + 1u);
        }
        if (++i == ni) {
          i = 0;
          ++col;
        }
      }
    }
  }
  if (sum_out) __atomic_fetch_add(sum_out, sum, __ATOMIC_RELAXED);
}

// dst[b..., j, i] = convert(src[b..., i, j]) for every batch index, as the descriptor says it (strides in elements).
void run_transpose(const uint8_t* src, uint8_t* dst, const TransposeDesc& d, int es, uint32_t op, uint32_t nan_bits, uint32_t* sum_out,
                   uint32_t woven_lds = 0) {
  if (d.weave_chunks) return run_woven(src, dst, d, es, op, nan_bits, sum_out, woven_lds);
  const int eo = op == kOpCopy ? es : (int)op_dst_elem(op);
  const Batches batches(d);
  uint32_t sum = 0;
  for (uint64_t b = 0; b < batches.n; ++b) {
    uint64_t s_off, d_off;
    batches.offsets(b, s_off, d_off);
    for (uint64_t i = 0; i < d.ni; ++i)
      for (uint64_t j = 0; j < d.nj; ++j) {
        const uint64_t del = d_off + j * d.dj + i;
        uint8_t* dp = dst + del * (uint64_t)eo;
        convert_element(src + (s_off + i * d.si + j) * (uint64_t)es, dp, es, op, nan_bits);
        if (sum_out) {
          const uint32_t pos0 = (uint32_t)(del * (uint64_t)eo) + d.csum_bias;
          for (int e = 0; e < eo; ++e) sum += dp[e] * ((pos0 + (uint32_t)e) * kKnuth + 1u);
        }
      }
  }
  if (sum_out) __atomic_fetch_add(sum_out, sum, __ATOMIC_RELAXED);
}

}  // namespace

hipError_t launch_transpose(const void* src, void* dst, const TransposeDesc& d, int elem_size, uint32_t op, uint32_t nan_bits,
                            uint32_t* sum_out, Fan, hipStream_t stream) {
  if (d.n_tiles == 0) return hipSuccess;
  if (!transpose_desc_ok(d)) return hipErrorInvalidValue;
  ++launched_forms[form_of(d)];
  const TransposeDesc desc = d;  // a kernel argument: copied when the launch is issued
  const uint32_t lds = d.weave_chunks ? weave_lds((uint32_t)d.ni, d.weave_chunks) : 0;
  cpu_hip::enqueue(stream, [=] { run_transpose(static_cast<const uint8_t*>(src), static_cast<uint8_t*>(dst), desc, elem_size, op, nan_bits, sum_out, lds); });
  return hipSuccess;
}
hipError_t launch_transpose_batch(const TransposeItem* items_dev, uint32_t n_items, uint64_t total_tiles, uint32_t, int elem_size,
                                  uint32_t op, uint32_t nan_bits, hipStream_t stream, uint32_t panel, uint32_t uniform_tiles,
                                  const TransposeDesc* common, const TransposeItem* items_host) {
  if (n_items == 0 || total_tiles == 0) return hipSuccess;
  for (uint32_t k = 0; items_host && k < n_items; ++k) ++launched_forms[form_of(items_host[k].d)];
  const uint32_t lds = panel & kWeaveCode ? panel & ~kWeaveCode : 0;
  if (uniform_tiles && common && items_host) {
    // descriptor and pointers travel as kernel arguments: read now
    std::vector<std::pair<const uint8_t*, uint8_t*>> ptrs;
    for (uint32_t k = 0; k < n_items; ++k) ptrs.emplace_back(items_host[k].src, items_host[k].dst);
    const TransposeDesc desc = *common;
    cpu_hip::enqueue(stream, [=] {
      for (const auto& pr : ptrs) run_transpose(pr.first, pr.second, desc, elem_size, op, nan_bits, nullptr, lds);
    });
    return hipSuccess;
  }
  // the item table is device memory: read when the launch runs
  cpu_hip::enqueue(stream, [=] {
    for (uint32_t k = 0; k < n_items; ++k) run_transpose(items_dev[k].src, items_dev[k].dst, items_dev[k].d, elem_size, op, nan_bits, nullptr, lds);
  });
  return hipSuccess;
}
hipError_t launch_synth(void*, uint64_t, uint32_t, uint32_t, uint64_t, hipStream_t) { return hipErrorNotSupported; }
void synth_host(void*, uint64_t, uint32_t, uint32_t, uint64_t, int) { unsupported("the synthetic-checkpoint generator"); }

}  // namespace mxp
