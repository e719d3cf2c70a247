// Host-side lowering of logical pitched box copies into the device descriptor tables
// (segments + work items) that place_kernel executes.
#pragma once
#include <algorithm>
#include <cstdint>
#include <stdexcept>
#include <string>
#include <vector>

#include "mxp_device.h"

namespace mxp {

// One logical box of any size: `rows` rows of `row_bytes` DESTINATION bytes each.
// The source row is op_src_bytes(op, row_bytes) long (twice as long for a narrowing cast,
// half as long for a widening one).
struct BoxCopy {
  uint32_t src_buf = 0, dst_buf = 0;
  uint64_t src_off = 0, dst_off = 0;
  uint64_t src_pitch = 0, dst_pitch = 0;
  uint64_t rows = 1, row_bytes = 0;
  uint32_t op = kOpCopy;
  uint32_t csum_slot = 0xFFFFFFFFu;
  uint64_t csum_bias = 0;  // checksum position = destination offset + bias (mod 2^32)
};

struct LowerOptions {
  uint32_t tile_bytes = 128 * 1024;  // SOURCE bytes one workgroup handles (one batch of loads)
  uint32_t max_row_bytes = 32768;   // wider pitched rows are split by columns
  bool ragged = false;              // boxes whose destination rows abut off the 16-byte grid become ragged segments
                                    // (not in the ingest: its readers pack such rows, which then abut on both sides)
};

// Tile size of a launch that moves `bytes` in all (the larger side of every box).  A full tile is one burst of
// reads and one of writes by one workgroup, and a compute unit runs one at a time, so a launch that leaves compute
// units without a tile is cut into smaller ones, as long as they still all run at once and are of 32 KiB or more.
// A copy of 8, 16 and 32 MB in tiles of 16 / 32 / 64 / 128 KiB: 11.5 / 9.0 / 9.4 / 11.1, 18.2 / 13.2 / 11.6 / 12.9,
// 31 / 21 / 19 / 16.6 us; 2 MB: 7.0 / 6.8 / 7.4 / 8.5.
inline uint32_t tile_bytes_for(uint64_t bytes, uint32_t tile_bytes) {
  uint64_t t = tile_bytes;
  while (t >= 64 * 1024 && bytes / (t / 2) <= kChipCus) t /= 2;
  return (uint32_t)t;
}
// Whether a launch over these segments needs a kernel that knows the ragged form.
inline bool any_ragged(const std::vector<Seg>& segs) {
  return std::any_of(segs.begin(), segs.end(), [](const Seg& s) { return s.ragged != 0; });
}
inline uint64_t box_bytes(const BoxCopy& b) { return b.rows * std::max(b.row_bytes, op_src_bytes(b.op, b.row_bytes)); }

// `SegTable` / `WorkTable` are anything with push_back and size: std::vector, or a fixed-capacity
// view over memory the caller already owns.
template <class SegTable, class WorkTable>
inline void emit_seg(const BoxCopy& b, const LowerOptions& o, SegTable& segs, WorkTable& work) {
  if (b.rows == 0 || b.row_bytes == 0) return;
  if (b.rows > 0xFFFFFFFFull || b.row_bytes > o.max_row_bytes)
    throw std::logic_error("emit_seg: box not normalised");
  const uint64_t src_row = op_src_bytes(b.op, b.row_bytes);
  const bool pitched = b.rows > 1;
  auto all_mult = [&](uint64_t m_dst, uint64_t m_src) {
    if (b.dst_off % m_dst || b.row_bytes % m_dst) return false;
    if (b.src_off % m_src) return false;
    if (pitched && (b.dst_pitch % m_dst || b.src_pitch % m_src)) return false;
    return true;
  };
  // The unit is set by the destination side (whole, aligned stores); the source only has to be
  // element aligned, the device reads it with loads that carry no alignment promise.
  uint32_t unit;
  if (op_narrows(b.op)) {
    if (all_mult(8, 4)) unit = 8;
    else if (all_mult(2, 4)) unit = 2;
    else throw std::invalid_argument("cast box is not element aligned");
  } else if (op_widens(b.op)) {
    const uint64_t se = op_dst_elem(b.op) / 2;  // source element
    if (all_mult(16, se)) unit = 16;
    else if (all_mult(4, se)) unit = 4;
    else if (op_dst_elem(b.op) == 2 && all_mult(2, 1)) unit = 2;
    else throw std::invalid_argument("cast box is not element aligned");
  } else if (op_recodes16(b.op)) {
    if (all_mult(16, 2)) unit = 16;
    else if (all_mult(4, 2)) unit = 4;
    else if (all_mult(2, 2)) unit = 2;
    else throw std::invalid_argument("cast box is not element aligned");
  } else {
    unit = all_mult(16, 1) ? 16 : all_mult(4, 1) ? 4 : all_mult(2, 1) ? 2 : 1;
  }
  const uint64_t max_pitch = pitched ? std::max(b.src_pitch, b.dst_pitch) : std::max(b.row_bytes, src_row);
  if (max_pitch >= (1ull << 31)) throw std::invalid_argument("row pitch of 2 GiB or more is not supported");

  Seg s{};
  s.src_off = b.src_off;
  s.dst_off = b.dst_off;
  s.src_pitch = pitched ? b.src_pitch : src_row;
  s.dst_pitch = pitched ? b.dst_pitch : b.row_bytes;
  s.rows = (uint32_t)b.rows;
  s.row_bytes = (uint32_t)b.row_bytes;
  s.src_buf = b.src_buf;
  s.dst_buf = b.dst_buf;
  s.op = b.op;
  s.unit = unit;
  s.csum_slot = b.csum_slot;
  s.csum_bias = (uint32_t)b.csum_bias;
  s.units_per_row = s.row_bytes / unit;
  s.div_magic = s.units_per_row > 1 ? (uint32_t)((1ull << 32) / s.units_per_row) + 1u : 0u;
  uint64_t rpt = std::max<uint64_t>(1, o.tile_bytes / std::max(b.row_bytes, src_row));
  rpt = std::min<uint64_t>(rpt, b.rows);
  // In-tile byte offsets are 32-bit on the device, and the reciprocal division is exact
  // only while (units in tile) * (units per row) < 2^32.
  while (rpt > 1 && (rpt * max_pitch >= (1ull << 31) ||
                     rpt * s.units_per_row * (uint64_t)s.units_per_row >= (1ull << 32)))
    rpt = (rpt + 1) / 2;
  if ((uint64_t)s.units_per_row * s.units_per_row >= (1ull << 32))
    throw std::logic_error("emit_seg: row too wide for its unit");
  // The 16-byte (8-byte for narrowing casts) paths of place_kernel run one batch per tile.
  if ((unit == 16 || unit == 8) && rpt * s.units_per_row > (uint64_t)kPlaceThreads * kPlaceBatch)
    throw std::logic_error("emit_seg: tile larger than one batch");
  s.rows_per_tile = (uint32_t)rpt;
  const uint32_t seg_idx = (uint32_t)segs.size();
  segs.push_back(s);
  const uint64_t tiles = (b.rows + rpt - 1) / rpt;
  for (uint64_t t = 0; t < tiles; ++t) work.push_back(WorkItem{seg_idx, (uint32_t)t});
}

// The contiguous destination of a pitched box whose rows abut off the store grid (a row-parallel slice of odd
// width): a lane stores whole aligned units, and where a unit spans the end of a row it takes its bytes from both
// rows.  Cut into rows instead, such a box moves in 2- or 4-byte units: 46 us for the 2.5 MB share of a two-layer
// model with 357-column slices, against 17 us this way.  Returns false for boxes the form does not fit: rows
// shorter than a unit, rows that overlap in the source, a pitch whose in-tile offsets would not fit 31 bits.
template <class SegTable, class WorkTable>
inline bool lower_ragged(const BoxCopy& b, const LowerOptions& o, SegTable& segs, WorkTable& work) {
  const uint32_t op = b.op;
  const uint64_t unit = op_narrows(op) ? 8 : 16, src_unit = op_src_bytes(op, unit);
  const uint64_t src_row = op_src_bytes(op, b.row_bytes);
  if (op == kOpChecksumOnly || b.dst_pitch != b.row_bytes || b.src_pitch < src_row || b.row_bytes < unit) return false;
  if (b.dst_off % unit == 0 && b.row_bytes % unit == 0) return false;  // whole units per row: the plain form
  if (b.src_pitch >= (1ull << 29) || b.row_bytes >= (1ull << 29)) return false;
  if (op != kOpCopy) {
    const uint64_t de = op_dst_elem(op), se = op_src_bytes(op, de);
    if (b.dst_off % de || b.row_bytes % de || b.src_off % se || b.src_pitch % se) return false;
  }
  const uint64_t total = b.rows * b.row_bytes, head = (unit - b.dst_off % unit) % unit;
  if (total < head + unit) return false;
  uint64_t per_tile = std::min<uint64_t>(o.tile_bytes / std::max(unit, src_unit), (uint64_t)kPlaceThreads * kPlaceBatch);
  while (per_tile > 1 && (per_tile * unit / b.row_bytes + 2) * b.src_pitch >= (1ull << 31)) per_tile /= 2;
  auto piece = [&](uint64_t at, uint64_t n) {  // n contiguous bytes inside one row
    if (!n) return;
    BoxCopy m = b;
    m.src_off = b.src_off + at / b.row_bytes * b.src_pitch + op_src_bytes(op, at % b.row_bytes);
    m.dst_off = b.dst_off + at;
    m.rows = 1;
    m.row_bytes = n;
    m.src_pitch = op_src_bytes(op, n);
    m.dst_pitch = n;
    emit_seg(m, o, segs, work);
  };
  piece(0, head);
  const uint64_t units = (total - head) / unit;
  for (uint64_t done = 0; done < units;) {
    const uint64_t n = std::min<uint64_t>(units - done, 0x40000000ull), at = head + done * unit;
    Seg s{};
    s.src_off = b.src_off + at / b.row_bytes * b.src_pitch;
    s.dst_off = b.dst_off + at;
    s.src_pitch = b.src_pitch;
    s.dst_pitch = unit;
    s.rows = (uint32_t)n;
    s.row_bytes = (uint32_t)b.row_bytes;
    s.src_buf = b.src_buf;
    s.dst_buf = b.dst_buf;
    s.op = op;
    s.unit = (uint32_t)unit;
    s.csum_slot = b.csum_slot;
    s.csum_bias = (uint32_t)b.csum_bias;
    s.units_per_row = 1;
    s.div_magic = (uint32_t)((1ull << 32) / b.row_bytes) + 1u;
    s.rows_per_tile = (uint32_t)std::min<uint64_t>(per_tile, n);
    s.ragged = 1u + (uint32_t)(at % b.row_bytes);
    const uint32_t seg_idx = (uint32_t)segs.size();
    segs.push_back(s);
    const uint64_t tiles = (n + s.rows_per_tile - 1) / s.rows_per_tile;
    for (uint64_t t = 0; t < tiles; ++t) work.push_back(WorkItem{seg_idx, (uint32_t)t});
    done += n;
  }
  const uint64_t tail_at = head + units * unit;
  piece(tail_at, total - tail_at);
  return true;
}

// What a tile of a contiguous run stores at least.
constexpr uint64_t kFlatTileBytes = 8192;

// Split one logical box into device segments.
template <class SegTable, class WorkTable>
inline void lower_box(const BoxCopy& in, const LowerOptions& o, SegTable& segs, WorkTable& work) {
  if (in.rows == 0 || in.row_bytes == 0) return;
  const uint32_t op = in.op;
  BoxCopy b = in;
  // Rows that abut in both layouts are one contiguous run.
  if (b.rows > 1 && b.src_pitch == op_src_bytes(op, b.row_bytes) && b.dst_pitch == b.row_bytes) {
    b.row_bytes *= b.rows;
    b.rows = 1;
  }
  if (b.rows == 1) {
    // Contiguous run: a head up to the destination's next 16-byte boundary (so that the rest moves in whole aligned
    // stores whatever the source's alignment), a body of rows of one unit, a tail.  Where the body's last tile would be
    // of a wavefront's size it is a segment of its own, which bundle_tiny can take.
    // A tile of it stores 8 KiB or more, however small the tile a caller sets: the fixed tables of mxp_checksum32_static hold
    // 98,304 tiles.
    const uint64_t unit = op_narrows(op) ? 8 : 16, src_unit = std::max(unit, op_src_bytes(op, unit));
    LowerOptions flat = o;
    flat.tile_bytes = (uint32_t)std::max<uint64_t>(o.tile_bytes, kFlatTileBytes / unit * src_unit);
    uint64_t done = 0;
    auto piece = [&](uint64_t n, uint64_t row) {  // the next n bytes, in rows of `row`
      BoxCopy m = b;
      m.src_off = b.src_off + op_src_bytes(op, done);
      m.dst_off = b.dst_off + done;
      m.rows = n / row;
      m.row_bytes = row;
      m.src_pitch = op_src_bytes(op, row);
      m.dst_pitch = row;
      emit_seg(m, flat, segs, work);
      done += n;
    };
    if (b.dst_off % 16 && op != kOpChecksumOnly) {
      const uint64_t head = std::min<uint64_t>(16 - b.dst_off % 16, b.row_bytes);
      piece(head, head);
    }
    uint64_t units = (b.row_bytes - done) / unit;
    const uint64_t per_tile = flat.tile_bytes / src_unit, last = units % per_tile;
    const uint64_t apart = units > last && last <= kBundleUnits ? last : 0;
    for (units -= apart; units;) {
      const uint64_t n = std::min<uint64_t>(units, 0x40000000ull / per_tile * per_tile);
      piece(n * unit, unit);
      units -= n;
    }
    if (apart) piece(apart * unit, unit);
    if (const uint64_t rest = b.row_bytes - done) piece(rest, rest);
    return;
  }
  if (o.ragged && lower_ragged(b, o, segs, work)) return;
  // Pitched box whose rows all start at the same distance from a 16-byte boundary of the
  // destination, but not on one (or do not end on one): a column of head bytes, a body that is
  // stored whole and aligned, a column of tail bytes.
  if (op != kOpChecksumOnly && b.dst_pitch % 16 == 0 && (b.dst_off % 16 || b.row_bytes % 16) && b.row_bytes >= 64) {
    const uint64_t head = (16 - b.dst_off % 16) % 16;
    const uint64_t body = (b.row_bytes - head) / 16 * 16;
    const uint64_t cuts[4] = {0, head, head + body, b.row_bytes};
    for (int k = 0; k < 3; ++k) {
      if (cuts[k + 1] == cuts[k]) continue;
      BoxCopy m = b;
      m.src_off = b.src_off + op_src_bytes(op, cuts[k]);
      m.dst_off = b.dst_off + cuts[k];
      m.row_bytes = cuts[k + 1] - cuts[k];
      lower_box(m, o, segs, work);  // the body is aligned now, the edge columns are narrower than 64 bytes
    }
    return;
  }
  // Pitched box: split columns so a row fits max_row_bytes, rows so the count fits 32 bits.
  for (uint64_t c = 0; c < b.row_bytes; c += o.max_row_bytes) {
    const uint64_t cw = std::min<uint64_t>(o.max_row_bytes, b.row_bytes - c);
    for (uint64_t r = 0; r < b.rows; r += 0x80000000ull) {
      BoxCopy m = b;
      m.src_off = b.src_off + r * b.src_pitch + op_src_bytes(op, c);
      m.dst_off = b.dst_off + r * b.dst_pitch + c;
      m.rows = std::min<uint64_t>(0x80000000ull, b.rows - r);
      m.row_bytes = cw;
      emit_seg(m, o, segs, work);
    }
  }
}

// Segments of at most one unit a lane of a wavefront (the edges of contiguous runs, small biases and norms, the last KiB of
// a run) go out sixteen to a workgroup.  Alone in a workgroup of sixteen wavefronts, with a compute unit to itself for the
// two or three microseconds of its loads and stores, each costs as much as a full tile.  888 copies of 74 KB off the
// 16-byte grid take 41.4 us with a workgroup for each of their pieces and 29.9 with the edges in bundles; a 76-buffer
// model of 7 MB with digests 13.2 and 9.8.  One unit a lane at most, which is also what the kernel's stride assumes: with up to
// 512 units in a segment of a bundle (and strides of a wavefront) a snapshot of 36 small tensors took 11.4 us, not 9.6.
inline void bundle_tiny(std::vector<Seg>& segs, std::vector<WorkItem>& work) {
  constexpr uint32_t kWaves = kPlaceThreads / 64;
  auto tiny = [](const Seg& s) { return s.rows <= s.rows_per_tile && (uint64_t)s.rows * s.units_per_row <= kBundleUnits; };
  const size_t n = (size_t)std::count_if(segs.begin(), segs.end(), tiny);
  if (n < 2) return;
  std::vector<Seg> order;
  std::vector<uint32_t> index(segs.size());
  order.reserve(segs.size());
  for (int pass = 0; pass < 2; ++pass)
    for (size_t k = 0; k < segs.size(); ++k)
      if (tiny(segs[k]) == (pass == 1)) {
        index[k] = (uint32_t)order.size();
        order.push_back(segs[k]);
      }
  std::vector<WorkItem> items;
  items.reserve(work.size());
  for (const WorkItem& w : work)
    if (!tiny(segs[w.seg])) items.push_back(WorkItem{index[w.seg], w.tile});
  for (size_t k = 0; k < n; k += kWaves)
    items.push_back(WorkItem{(uint32_t)(segs.size() - n + k), kBundle | (uint32_t)std::min<size_t>(kWaves, n - k)});
  segs.swap(order);
  work.swap(items);
}

}  // namespace mxp
