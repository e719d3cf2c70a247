// Drives the stand-alone operators of the host engine (modelexpress_amd/csrc/mxp_engine.cpp) on the CPU, built against the
// HIP stand-in under tests/c/cpu_hip with -fsanitize=address,undefined (tests/test_host_operators.py builds and runs it).
//
// usage: operators_hosttest <scenario> <empty working directory>      prints "ok" and exits 0 on success
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <memory>
#include <string>
#include <utility>
#include <vector>

#include "mxp.h"
#include "mxp_bench.h"

namespace mxp {
extern int launched_forms[3];  // cpu_hip/cpu_kernels.cpp
}

namespace {

std::string g_dir;

[[noreturn]] void die(const std::string& what) {
  std::fprintf(stderr, "operators_hosttest: %s (last error: %s)\n", what.c_str(), mxp_last_error());
  std::exit(1);
}
#define OK(call)                                                  \
  do {                                                            \
    const int rc_ = (call);                                       \
    if (rc_ != MXP_OK) die(std::string(#call) + " returned " + std::to_string(rc_)); \
  } while (0)

mxp_engine* make_engine(uint32_t tile = 0) {
  mxp_engine_options o{};
  o.tile_bytes = tile;
  o.ring_slots = 2;
  o.slot_bytes = 1 << 16;
  o.reader_threads = 1;
  o.streams = 1;
  mxp_engine* e = nullptr;
  OK(mxp_engine_create(&o, &e));
  return e;
}

uint8_t* device_block(size_t n, uint32_t seed) {
  uint8_t* p = nullptr;
  if (hipMalloc(reinterpret_cast<void**>(&p), n) != hipSuccess) die("hipMalloc");
  for (size_t i = 0; i < n; ++i) p[i] = (uint8_t)((i + seed) * 2654435761u >> 24);
  return p;
}
void sync() {
  if (hipDeviceSynchronize() != hipSuccess) die("sync");
}

// Copies whose tables all but fill the arena's first block, and nobody asks for their checksums: nothing may be added
// behind the tables.
void copies_without_checksums() {
  mxp_engine* eng = make_engine();
  for (const int64_t n : {1, 10400, 10800, 10860}) {
    const uint64_t size = 32;
    uint8_t *src = device_block((size_t)n * size, 1), *dst = device_block((size_t)n * size, 2);
    std::vector<const void*> srcs;
    std::vector<void*> dsts;
    for (int64_t k = 0; k < n; ++k) {
      srcs.push_back(src + k * size);
      dsts.push_back(dst + k * size);
    }
    const std::vector<uint64_t> sizes((size_t)n, size);
    for (int rep = 0; rep < 2; ++rep) OK(mxp_copy_batch(eng, srcs.data(), dsts.data(), sizes.data(), n, nullptr, nullptr));
    sync();
    if (std::memcmp(src, dst, (size_t)n * size) != 0) die("copies");
    (void)hipFree(src);
    (void)hipFree(dst);
  }
  mxp_engine_destroy(eng);
}

struct Transposed {  // a row-major [n, m] of 2-byte elements out of a row-major [m, n]
  int64_t n, m;
  uint8_t *src, *dst;
  mxp_view_copy view() const {
    mxp_view_copy v{};
    v.src = src;
    v.dst = dst;
    v.ndim = 2;
    v.elem_size = 2;
    v.shape[0] = n;
    v.shape[1] = m;
    v.src_strides[0] = 1;
    v.src_strides[1] = n;
    v.contiguous_dst = 1;
    return v;
  }
  void check(const char* what) const {
    for (int64_t i = 0; i < n; ++i)
      for (int64_t j = 0; j < m; ++j)
        if (std::memcmp(dst + 2 * (i * m + j), src + 2 * (j * n + i), 2) != 0) die(what);
  }
};
std::vector<Transposed> transposes(const std::vector<std::pair<int64_t, int64_t>>& shapes) {
  std::vector<Transposed> out;
  for (const auto& [n, m] : shapes) out.push_back({n, m, device_block((size_t)(n * m) * 2, 3), device_block((size_t)(n * m) * 2, 4)});
  return out;
}

// Transposed views recorded on a stream under capture: the replays neither read nor write what later calls of the engine
// use, and the engine's other calls go on working.
void captured_transposes() {
  mxp_engine* eng = make_engine();
  hipStream_t stream;
  if (hipStreamCreateWithFlags(&stream, hipStreamNonBlocking) != hipSuccess) die("stream");
  // of several shapes, of one shape in the staged form, and one alone
  for (const auto& shapes : std::vector<std::vector<std::pair<int64_t, int64_t>>>{
           {{40, 70}, {300, 65}, {7, 9}}, {{128, 256}, {128, 256}, {128, 256}}, {{512, 700}, {30000, 40}, {30000, 40}}, {{33, 44}}}) {
    std::vector<Transposed> ours = transposes(shapes), theirs = transposes({{50, 60}, {70, 80}, {90, 20}, {60, 60}});
    std::vector<mxp_view_copy> a, b;
    for (const auto& t : ours) a.push_back(t.view());
    for (const auto& t : theirs) b.push_back(t.view());
    cpu_hip::begin_capture(stream);
    OK(mxp_copy_views(eng, a.data(), (int64_t)a.size(), stream));
    const auto graph = cpu_hip::end_capture(stream);
    for (int replay = 0; replay < 3; ++replay) {
      for (int call = 0; call < 3; ++call) {  // both arenas are used anew, by operators of two kinds
        OK(mxp_copy_views(eng, b.data(), (int64_t)b.size(), nullptr));
        const void* src = theirs[0].src;
        const uint64_t size = 100;
        uint32_t sum;
        OK(mxp_checksum32(eng, &src, &size, 1, &sum, nullptr));
      }
      sync();
      for (const auto& t : ours) std::memset(t.dst, 0xEE, (size_t)(t.n * t.m) * 2);
      for (const auto& t : theirs) std::memset(t.dst, 0xEE, (size_t)(t.n * t.m) * 2);
      for (const auto& work : graph) cpu_hip::enqueue(stream, work);
      sync();
      for (const auto& t : ours) t.check("a captured transpose");
      for (const auto& t : theirs)
        for (int64_t i = 0; i < t.n * t.m * 2; ++i)
          if (t.dst[i] != 0xEE) die("a replay wrote to another call's destination");
    }
    for (const auto* group : {&ours, &theirs})
      for (const auto& t : *group) {
        (void)hipFree(t.src);
        (void)hipFree(t.dst);
      }
  }
  (void)hipStreamDestroy(stream);
  mxp_engine_destroy(eng);
}

// A small checkpoint of two fp32 tensors, its plan and the buffers a resident placement takes.
struct Placement {
  mxp_ckpt* ck = nullptr;
  mxp_plan* plan = nullptr;
  std::vector<void*> files, dst;
  Placement() {
    const std::string data(4 * (64 * 32 + 100), 'x');
    std::string json = R"({"a":{"dtype":"F32","shape":[64,32],"data_offsets":[0,8192]},"b":{"dtype":"F32","shape":[100],"data_offsets":[8192,8592]}})";
    while (json.size() % 8) json += " ";
    const std::string path = g_dir + "/model.safetensors";
    FILE* fp = std::fopen(path.c_str(), "wb");
    const uint64_t n = json.size();
    if (!fp || std::fwrite(&n, 8, 1, fp) != 1 || std::fwrite(json.data(), 1, json.size(), fp) != json.size() ||
        std::fwrite(data.data(), 1, data.size(), fp) != data.size() || std::fclose(fp) != 0)
      die("cannot write " + path);
    OK(mxp_ckpt_open(path.c_str(), &ck));
    OK(mxp_plan_create(ck, 1, 0, 0, &plan));
    const int64_t a[2] = {64, 32}, b[1] = {100};
    if (mxp_plan_add_param(plan, "a", MXP_DTYPE_F32, 2, a) != 0 || mxp_plan_add_param(plan, "b", MXP_DTYPE_F32, 1, b) != 1) die("mxp_plan_add_param");
    OK(mxp_plan_build(plan));
    files.push_back(device_block(8 + json.size() + data.size(), 1));
    dst.push_back(device_block(8192, 2));
    dst.push_back(device_block(400, 2));
  }
  ~Placement() {
    if (plan) mxp_plan_destroy(plan);
    mxp_ckpt_close(ck);
    for (void* p : files) (void)hipFree(p);
    for (void* p : dst) (void)hipFree(p);
  }
};

// A resident placement that reports its time has run when the call returns, its results delivered.
void timed_placements_with_digests() {
  mxp_engine* eng = make_engine();
  OK(mxp_engine_set_fused_digests(eng, 1));
  {
    Placement p;
    OK(mxp_prepare(eng, p.plan));
    cpu_hip::set_finish_delay_us(30000);
    for (int rep = 0; rep < 2; ++rep) {
      mxp_exec_stats st{};
      OK(mxp_execute_resident(eng, p.plan, p.files.data(), p.dst.data(), nullptr, &st));
      if (cpu_hip::finishes_waiting()) die("the call returned with work of its own still queued");
    }
    cpu_hip::set_finish_delay_us(0);
  }
  mxp_engine_destroy(eng);
}

// mxp_describe_views tells how the views of one call run, as they are shaped together.
void described_views() {
  mxp_engine* eng = make_engine();
  struct Call {
    std::vector<std::pair<int64_t, int64_t>> shapes;  // of the destination
    std::vector<int> kinds;
  };
  const std::vector<Call> calls = {
      {{{100000, 12}}, {2}},                          // 2.4 MB in rows of 12
      {{{20000, 12}}, {1}},                           // less than 2 MB in all
      {{{20000, 12}, {1100, 1100}}, {1, 1}},          // less than 2 MB woven beside others: no launch of its own
      {{{1100, 1100}, {20000, 12}, {9000, 24}}, {1, 1, 1}},
      {{{90000, 12}, {1100, 1100}}, {2, 1}},          // 2.2 MB woven beside others
      {{{60000, 12}, {1100, 1100}, {30000, 12}}, {2, 1, 2}},
      {{{30000, 12}, {70000, 12}}, {2, 2}},
  };
  for (const Call& c : calls) {
    const std::vector<Transposed> views = transposes(c.shapes);
    std::vector<mxp_view_copy> abi;
    for (const auto& t : views) abi.push_back(t.view());
    const int64_t n = (int64_t)abi.size();
    std::vector<int32_t> kinds((size_t)n), rows((size_t)n), row_bytes((size_t)n);
    OK(mxp_describe_views(eng, abi.data(), n, kinds.data(), rows.data(), row_bytes.data()));
    int want[2] = {0, 0};
    for (int64_t k = 0; k < n; ++k) {
      if (kinds[(size_t)k] != c.kinds[(size_t)k]) die("kind of view " + std::to_string(k) + " of " + std::to_string(n));
      const bool staged = kinds[(size_t)k] == 2;
      if (rows[(size_t)k] != (staged ? views[(size_t)k].m : 0) || (row_bytes[(size_t)k] != 0) != staged) die("tile of a described view");
      ++want[staged];
    }
    std::fill_n(mxp::launched_forms, 3, 0);
    OK(mxp_copy_views(eng, abi.data(), n, nullptr));
    if (mxp::launched_forms[0] != want[0] || mxp::launched_forms[1] + mxp::launched_forms[2] != want[1]) die("the views ran in other forms than described");
    sync();
    for (const auto& t : views) {
      t.check("a described transpose");
      (void)hipFree(t.src);
      (void)hipFree(t.dst);
    }
  }
  mxp_engine_destroy(eng);
}

// Transposes into short abutting rows: every row length of the woven form, each geometry of element sizes, source rows from
// 16 bytes to two tiles and what is left of one, pitches and destinations off the grid, batches, tiles of both sizes, and
// several shapes in one launch.  Sources and destinations are blocks of just their size.
void woven_transposes() {
  mxp_engine* eng = make_engine();
  struct Type { int es, eo, cast; };
  const Type types[] = {{1, 1, MXP_CAST_NONE}, {2, 2, MXP_CAST_NONE}, {4, 4, MXP_CAST_NONE}, {4, 2, MXP_CAST_F32_BF16}, {2, 4, MXP_CAST_BF16_F32},
                        {1, 2, MXP_CAST_F8E4M3_BF16}};
  // A contiguous copy in the same call makes it large: of 2 MB for the smallest tiles, of 24 MB for whole ones.
  std::vector<uint8_t> large(24 << 20), copy(24 << 20);
  long checked = 0, woven = 0;
  for (const Type& t : types)
    for (int64_t ni = 2; ni <= 90; ++ni) {
      struct Block { std::unique_ptr<uint8_t[]> src, dst; int64_t ni, nj, pitch, batches, src_first, dst_first, dst_bytes; };
      std::vector<Block> blocks;
      std::vector<mxp_view_copy> views;
      const int64_t big = ni % 4 == 0 ? 24 << 20 : 2 << 20, least = 16 / t.es;
      mxp_view_copy bulk{};
      bulk.src = large.data();
      bulk.dst = copy.data();
      bulk.ndim = 1;
      bulk.elem_size = 1;
      bulk.shape[0] = big;
      bulk.contiguous_src = bulk.contiguous_dst = 1;
      views.push_back(bulk);
      int64_t chunks = 8;
      while (chunks * 2 * ni <= 1024) chunks *= 2;
      const int64_t tile = (big > (2 << 20) ? chunks : 8) * 16 / t.es;
      int64_t k = 0;
      for (const int64_t nj : {least, least + 1, 2 * least - 1, tile - 1, tile, tile + 1, tile + least - 1, 2 * tile + 3}) {
        Block b{nullptr, nullptr, ni, nj, nj + k % 3, 1 + (k & 1), k % 2, k % 5, 0};
        ++k;
        const int64_t src_elems = b.src_first + (b.batches * ni - 1) * b.pitch + nj;
        b.dst_bytes = (b.dst_first + b.batches * ni * nj) * t.eo;
        b.src.reset(new uint8_t[(size_t)(src_elems * t.es)]);
        b.dst.reset(new uint8_t[(size_t)b.dst_bytes]);
        for (int64_t i = 0; i < src_elems * t.es; ++i) {
          b.src[(size_t)i] = (uint8_t)((uint32_t)(i + ni) * 2654435761u >> 24);
          if (t.cast == MXP_CAST_F8E4M3_BF16 || (t.cast == MXP_CAST_F32_BF16 && i % 4 == 3)) b.src[(size_t)i] &= 0x3F;  // no NaN
        }
        mxp_view_copy v{};
        v.src = b.src.get() + b.src_first * t.es;
        v.dst = b.dst.get() + b.dst_first * t.eo;
        v.ndim = 3;
        v.elem_size = t.eo;
        v.cast = t.cast;
        const int64_t shape[3] = {b.batches, nj, ni}, ss[3] = {ni * b.pitch, 1, b.pitch}, ds[3] = {nj * ni, ni, 1};
        std::copy(shape, shape + 3, v.shape);
        std::copy(ss, ss + 3, v.src_strides);
        std::copy(ds, ds + 3, v.dst_strides);
        views.push_back(v);
        blocks.push_back(std::move(b));
      }
      std::vector<int32_t> kinds(views.size()), rows(views.size()), row_bytes(views.size());
      OK(mxp_describe_views(eng, views.data(), (int64_t)views.size(), kinds.data(), rows.data(), row_bytes.data()));
      for (size_t i = 1; i < views.size(); ++i) woven += kinds[i] == 2 && rows[i] == (int32_t)ni;
      OK(mxp_copy_views(eng, views.data(), (int64_t)views.size(), nullptr));
      sync();
      for (const Block& b : blocks) {
        for (int64_t n = 0; n < b.batches; ++n)
          for (int64_t j = 0; j < b.nj; ++j)
            for (int64_t i = 0; i < ni; ++i) {
              const uint8_t* sp = b.src.get() + (b.src_first + (n * ni + i) * b.pitch + j) * t.es;
              const uint8_t* dp = b.dst.get() + (b.dst_first + (n * b.nj + j) * ni + i) * t.eo;
              uint32_t want = 0, got = 0, u = 0;
              std::memcpy(&got, dp, (size_t)t.eo);
              std::memcpy(&u, sp, (size_t)t.es);
              if (t.cast == MXP_CAST_NONE) want = u;
              else if (t.cast == MXP_CAST_BF16_F32) want = u << 16;
              else if (t.cast == MXP_CAST_F32_BF16) want = (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
              else {
                const float f = std::ldexp((float)((u & 7) + (u >> 3 ? 8 : 0)), (int)std::max(1u, u >> 3) - 10);
                std::memcpy(&want, &f, 4);
                want >>= 16;
              }
              if (got != want) die("a woven element");
            }
        ++checked;
      }
    }
  // rows that qualify are woven: all up to 88 elements (80 of one byte), but for the panels' powers of two
  if (checked != 6 * 89 * 8 || woven < 6 * 70 * 8) die("too few views were woven: " + std::to_string(woven) + " of " + std::to_string(checked));
  // one alone, with its checksum: 2.4 MB in rows of 12
  const Transposed one = transposes({{100001, 12}})[0];
  const mxp_view_copy v = one.view();
  uint32_t got = 0, want = 0;
  const int64_t ds[2] = {12, 1};
  OK(mxp_copy_view(eng, v.src, v.dst, 2, v.shape, v.src_strides, ds, 2, MXP_CAST_NONE, &got, nullptr));
  one.check("a woven view by itself");
  for (uint32_t i = 0; i < 100001 * 12 * 2; ++i) want += one.dst[i] * (i * 2654435761u + 1u);
  if (got != want) die("checksum of a woven view");
  (void)hipFree(one.src);
  (void)hipFree(one.dst);
  mxp_engine_destroy(eng);
}

// The fixed tables of the static checksum hold a large buffer also where the engine's tiles are small.
void static_checksum_in_small_tiles() {
  for (const uint32_t tile : {0u, 1024u, 12000u}) {
    mxp_engine* eng = make_engine(tile);
    const uint64_t n = (112 << 20) + 5;
    uint8_t* p = device_block(n, 9);
    uint32_t want = 0, got = 0;
    for (uint64_t i = 0; i < n; ++i) want += p[i] * ((uint32_t)i * 2654435761u + 1u);
    const void* ptr = p;
    OK(mxp_checksum32_static(eng, &ptr, &n, 1, &got, nullptr));
    if (got != want) die("static checksum");
    OK(mxp_checksum32(eng, &ptr, &n, 1, &got, nullptr));
    if (got != want) die("checksum");
    (void)hipFree(p);
    mxp_engine_destroy(eng);
  }
}

// Rows of half a line stay panels in calls that the caches hold, by what the call reads.
void half_line_rows() {
  mxp_engine* eng = make_engine();
  struct Case { int es, eo, cast, rows, mb; bool panel; };
  for (const Case& c : {Case{2, 2, MXP_CAST_NONE, 32, 8, true}, Case{2, 2, MXP_CAST_NONE, 32, 24, true}, Case{2, 2, MXP_CAST_NONE, 32, 40, false},
                        Case{1, 1, MXP_CAST_NONE, 64, 24, true}, Case{1, 1, MXP_CAST_NONE, 64, 40, false}, Case{1, 2, MXP_CAST_F8E4M3_BF16, 32, 24, true},
                        Case{1, 2, MXP_CAST_F8E4M3_BF16, 32, 48, true}, Case{1, 2, MXP_CAST_F8E4M3_BF16, 32, 72, false}}) {
    const int64_t nj = 4096, n = (int64_t)c.mb * 1000000 / (c.rows * nj * c.eo), elems = n * c.rows * nj;
    uint8_t* src = nullptr;
    if (hipMalloc(reinterpret_cast<void**>(&src), (size_t)(elems * c.es)) != hipSuccess) die("hipMalloc");
    std::memset(src, 0x31, (size_t)(elems * c.es));
    uint8_t* dst = device_block((size_t)(elems * c.eo), 0);
    mxp_view_copy v{};
    v.src = src;
    v.dst = dst;
    v.ndim = 3;
    v.elem_size = c.eo;
    v.cast = c.cast;
    v.contiguous_dst = 1;
    const int64_t shape[3] = {n, nj, c.rows}, ss[3] = {c.rows * nj, 1, nj};
    std::copy(shape, shape + 3, v.shape);
    std::copy(ss, ss + 3, v.src_strides);
    std::fill_n(mxp::launched_forms, 3, 0);
    OK(mxp_copy_views(eng, &v, 1, nullptr));
    sync();
    if (mxp::launched_forms[1] != c.panel || mxp::launched_forms[2] == c.panel) die("form of " + std::to_string(c.mb) + " MB in rows of " + std::to_string(c.rows));
    (void)hipFree(src);
    (void)hipFree(dst);
  }
  mxp_engine_destroy(eng);
}

// A plan that goes away before its results are there leaves the thread on the device it was using.
void plan_destroyed_from_another_device() {
  mxp_engine* eng = make_engine();
  OK(mxp_engine_set_fused_digests(eng, 1));
  for (const unsigned delay : {0u, 30000u}) {
    Placement p;
    OK(mxp_prepare(eng, p.plan));
    cpu_hip::set_finish_delay_us(delay);
    OK(mxp_execute_resident(eng, p.plan, p.files.data(), p.dst.data(), nullptr, nullptr));
    if (hipSetDevice(1) != hipSuccess) die("hipSetDevice");
    mxp_plan_destroy(p.plan);
    p.plan = nullptr;
    cpu_hip::set_finish_delay_us(0);
    int device = -1;
    if (hipGetDevice(&device) != hipSuccess || device != 1) die("the thread's device changed");
    if (cpu_hip::finishes_waiting()) die("the plan went away under a launch that stores to it");
  }
  mxp_engine_destroy(eng);
}

}  // namespace

int main(int argc, char** argv) {
  const std::map<std::string, std::function<void()>> scenarios = {{"copies_without_checksums", copies_without_checksums},
                                                                  {"captured_transposes", captured_transposes},
                                                                  {"timed_placements_with_digests", timed_placements_with_digests},
                                                                  {"plan_destroyed_from_another_device", plan_destroyed_from_another_device},
                                                                  {"described_views", described_views},
                                                                  {"woven_transposes", woven_transposes},
                                                                  {"static_checksum_in_small_tiles", static_checksum_in_small_tiles},
                                                                  {"half_line_rows", half_line_rows}};
  const auto it = argc == 3 ? scenarios.find(argv[1]) : scenarios.end();
  if (it == scenarios.end()) {
    std::fprintf(stderr, "usage: operators_hosttest <scenario> <empty working directory>\n");
    return 2;
  }
  g_dir = argv[2];
  it->second();
  std::printf("ok\n");
  return 0;
}
