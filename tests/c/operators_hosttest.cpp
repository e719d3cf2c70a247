// Drives the stand-alone operators of the host engine (modelexpress_amd/csrc/mxp_engine.cpp) on the CPU, built against the
// HIP stand-in under tests/c/cpu_hip with -fsanitize=address,undefined (tests/test_host_operators.py builds and runs it).
//
// usage: operators_hosttest <scenario>      prints "ok" and exits 0 on success
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include <vector>

#include "mxp.h"
#include "mxp_bench.h"

namespace {

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

}  // namespace

int main(int argc, char** argv) {
  const std::map<std::string, std::function<void()>> scenarios = {{"copies_without_checksums", copies_without_checksums}};
  const auto it = argc == 2 ? scenarios.find(argv[1]) : scenarios.end();
  if (it == scenarios.end()) {
    std::fprintf(stderr, "usage: operators_hosttest <scenario>\n");
    return 2;
  }
  it->second();
  std::printf("ok\n");
  return 0;
}
