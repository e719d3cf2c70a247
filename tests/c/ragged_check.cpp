// Host-side check of ragged segments (modelexpress_amd/csrc/mxp_lower.hpp, lower_ragged): random boxes whose
// destination rows abut are lowered twice, with and without ragged segments, both tables are replayed byte by byte
// with the kernel's own addressing, and both must give every destination byte the same source byte.  Of the ragged
// one: stores whole and on their grid, both loads of a unit inside the box, in-tile offsets within 31 bits, tiles
// of at most one batch.
// Usage: ragged_check <first seed> <number of seeds>.  Prints how many of the boxes became ragged.
#include <cinttypes>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <stdexcept>
#include <vector>

#include "mxp_lower.hpp"

using namespace mxp;

namespace {

void require(bool ok, const char* what) {
  if (!ok) throw std::runtime_error(what);
}
uint32_t dst_elem(uint32_t op) { return op == kOpCopy ? 1 : op_dst_elem(op); }
uint64_t src_of(uint32_t op, uint64_t d) { return op_src_bytes(op, d); }

// destination byte -> source byte of the element it comes from, relative to the box; -1 where nothing is stored
std::vector<int64_t> replay(const BoxCopy& b, const LowerOptions& lo, bool& ragged) {
  std::vector<Seg> segs;
  std::vector<WorkItem> work;
  lower_box(b, lo, segs, work);
  const uint64_t total = b.rows * b.row_bytes, es = dst_elem(b.op), src_end = (b.rows - 1) * b.src_pitch + src_of(b.op, b.row_bytes);
  std::vector<int64_t> out(total, -1);
  auto store = [&](uint64_t dst_abs, uint64_t n, uint64_t src_abs) {
    require(dst_abs >= b.dst_off && dst_abs + n <= b.dst_off + total, "store outside the box");
    require(src_abs >= b.src_off && src_abs + src_of(b.op, n) <= b.src_off + src_end, "load outside the box");
    for (uint64_t k = 0; k < n; ++k) {
      int64_t& o = out[dst_abs - b.dst_off + k];
      require(o == -1, "a byte stored twice");
      o = (int64_t)(src_abs - b.src_off + src_of(b.op, k / es * es));
    }
  };
  for (const WorkItem& w : work) {
    const Seg& s = segs[w.seg];
    const uint32_t r0 = w.tile * s.rows_per_tile, nrows = std::min(s.rows - r0, s.rows_per_tile);
    if (!s.ragged) {
      for (uint64_t r = r0; r < r0 + nrows; ++r) store(s.dst_off + r * s.dst_pitch, s.row_bytes, s.src_off + r * s.src_pitch);
      continue;
    }
    ragged = true;
    const uint32_t unit = s.unit, src_unit = (uint32_t)src_of(s.op, unit), sp = (uint32_t)s.src_pitch;
    require(unit == (op_narrows(s.op) ? 8u : 16u) && s.dst_pitch == unit && s.units_per_row == 1 && s.dst_off % unit == 0, "segment shape");
    require(nrows <= (uint32_t)(kPlaceThreads * kPlaceBatch), "tile larger than one batch");
    const uint64_t at0 = s.ragged - 1u + (uint64_t)r0 * unit, row0 = at0 / s.row_bytes;
    const uint32_t col0 = (uint32_t)(at0 - row0 * s.row_bytes);
    for (uint32_t v = 0; v < nrows; ++v) {
      const uint32_t at = col0 + v * unit;
      uint32_t row = (uint32_t)(((uint64_t)at * s.div_magic) >> 32);
      if (row * s.row_bytes > at) --row;
      require(row == at / s.row_bytes, "reciprocal division");
      const uint32_t col = at - row * s.row_bytes, so = row * sp + (uint32_t)src_of(s.op, col), room = s.row_bytes - col;
      require((uint64_t)row * sp + src_of(s.op, col) + sp < (1ull << 31), "in-tile offset");
      const uint64_t base = s.src_off + row0 * s.src_pitch, dst_abs = s.dst_off + ((uint64_t)r0 + v) * unit;
      require(base + so + src_unit <= b.src_off + src_end, "first load of a unit leaves the box");
      if (room >= unit) {
        store(dst_abs, unit, base + so);
        continue;
      }
      const uint32_t taken = (uint32_t)src_of(s.op, room), second = so + sp - (uint32_t)src_of(s.op, s.row_bytes);
      require(base + second >= b.src_off && base + second + src_unit <= b.src_off + src_end, "second load of a unit leaves the box");
      store(dst_abs, room, base + so);
      store(dst_abs + room, unit - room, base + second + taken);
    }
  }
  return out;
}

BoxCopy random_box(std::mt19937_64& g) {
  auto pick = [&](uint64_t lo, uint64_t hi) { return lo + g() % (hi - lo + 1); };
  static const uint32_t ops[] = {kOpCopy, kOpCopy, kOpCopy, kOpCastF32Bf16, kOpCastBf16F32, kOpCastF16F32, kOpCastF32F16,
                                 kOpCastF8E4M3Bf16, kOpCastF16Bf16, kOpCastBf16F16};
  BoxCopy b;
  b.op = ops[g() % (sizeof ops / sizeof ops[0])];
  const uint64_t de = dst_elem(b.op), se = b.op == kOpCopy ? 1 : src_of(b.op, de);
  static const uint64_t longest[] = {12, 40, 700, 20000, 70000};
  b.row_bytes = de * pick(1, longest[g() % 5]);
  b.rows = pick(2, std::max<uint64_t>(3, 400000 / b.row_bytes));
  const uint64_t src_row = src_of(b.op, b.row_bytes);
  b.src_pitch = src_row + se * (g() % 3 ? pick(0, 2000) : 0);
  if (g() % 16 == 0 && b.rows < 40) b.src_pitch = se * pick((1ull << 28) / se, (3ull << 28) / se);  // far apart: the table alone is checked
  b.dst_pitch = b.row_bytes;
  b.dst_off = de * pick(0, 40);
  b.src_off = se * pick(0, 40);
  return b;
}

}  // namespace

int main(int argc, char** argv) {
  const uint64_t first = argc > 1 ? std::strtoull(argv[1], nullptr, 10) : 0, count = argc > 2 ? std::strtoull(argv[2], nullptr, 10) : 200;
  uint64_t n_ragged = 0;
  for (uint64_t seed = first; seed < first + count; ++seed) {
    std::mt19937_64 g(seed * 104729 + 7);
    const BoxCopy b = random_box(g);
    LowerOptions with, without;
    with.ragged = true;
    with.tile_bytes = 1024u << (g() % 8);
    bool ragged = false, none = false;
    try {
      const auto got = replay(b, with, ragged), want = replay(b, without, none);
      require(!none, "ragged without the option");
      for (size_t i = 0; i < want.size(); ++i) require(want[i] >= 0 && got[i] == want[i], "a byte from another place than the plain form takes it");
      n_ragged += ragged;
    } catch (const std::exception& e) {
      std::fprintf(stderr, "seed %" PRIu64 ": op %u rows %" PRIu64 " row_bytes %" PRIu64 " src_off %" PRIu64 " dst_off %" PRIu64
                   " src_pitch %" PRIu64 " tile %u: %s\n", seed, b.op, b.rows, b.row_bytes, b.src_off, b.dst_off, b.src_pitch,
                   with.tile_bytes, e.what());
      return 1;
    }
  }
  std::printf("%" PRIu64 " of %" PRIu64 " boxes ragged\n", n_ragged, count);
  return 0;
}
