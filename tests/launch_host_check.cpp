// What the library asks the HIP runtime for, checked on the CPU (fake_hip.h).
#include "fake_hip.h"

#include <stdio.h>

#include "../include/cuot_amd.h"

#define REQUIRE(c)                                                  \
  do {                                                              \
    if (!(c)) {                                                     \
      printf("FAILED %s:%d: %s\n", __FILE__, __LINE__, #c);         \
      return 1;                                                     \
    }                                                               \
  } while (0)

static char buf[1 << 16];  // operands: the stand-in runtime reads none of them

// Both devices of a process get what their launches need: the dynamic LDS above
// 64 KB is allowed on the launch's own device, and no table is uploaded to one
// device only.
static int check_devices() {
  const int64_t lengths[] = {1000, 5000, 40000, (int64_t)1 << 20, 2500001, (int64_t)1 << 24, ((int64_t)1 << 24) + 1};
  for (int dev = 0; dev < 2; dev++) {
    cuot_ctx* ctx = nullptr;
    REQUIRE(cuot_init(dev, &ctx) == CUOT_OK);
    g_launches.clear();
    const cuot_knob_values transform = {0, 0, 0, 0, -1, 0};
    REQUIRE(cuot_set_knobs(&transform) == CUOT_OK);
    for (int64_t n : lengths) {
      REQUIRE(cuot_qc_prepare(ctx, n, (uint8_t*)buf, (uint32_t*)buf, buf, nullptr) == CUOT_OK);
      REQUIRE(cuot_qc_encode(ctx, n, (uint32_t*)buf, (cuot_block*)buf, (cuot_block*)buf, buf, nullptr) == CUOT_OK);
    }
    size_t big = 0;
    for (const Launch& l : g_launches) {
      REQUIRE(l.device == dev);
      if (l.lds <= 64 * 1024) continue;
      big++;
      const auto it = g_lds_limit.find({dev, l.kernel});
      if (it == g_lds_limit.end()) printf("device %d: %s takes %zu bytes of LDS\n", dev, l.kernel.c_str(), l.lds);
      REQUIRE(it != g_lds_limit.end() && (size_t)it->second >= l.lds);
    }
    REQUIRE(big > 0);
    REQUIRE(cuot_destroy(ctx) == CUOT_OK);
  }
  for (const auto& u : g_symbol_uploads) {
    REQUIRE(g_symbol_uploads.count({0, u.first.second}) == 1);
    REQUIRE(g_symbol_uploads.count({1, u.first.second}) == 1);
  }
  return 0;
}

static std::string shapes() {
  std::string s;
  for (const Launch& l : g_launches) s += l.kernel + " " + std::to_string(l.grid.x) + "; ";
  return s;
}

// A split that the knob has none of for a depth is the built-in rule, which gives a
// few deep trees several workgroups each; a valid one means one workgroup per tree.
static int check_ggm_dfs() {
  cuot_ctx* ctx = nullptr;
  REQUIRE(cuot_init(0, &ctx) == CUOT_OK);
  for (int h = 9; h <= 16; h++) {
    std::string rule;
    for (int dfs = 0; dfs <= 6; dfs++) {
      const cuot_knob_values k = {0, 0, dfs, 0, 0, 0};
      REQUIRE(cuot_set_knobs(&k) == CUOT_OK);
      cuot_ggm_params p;
      memset(&p, 0, sizeof(p));
      p.t = 3;
      p.h = h;
      p.mode = CUOT_MODE_SOT;
      p.n_out = p.t << h;
      g_launches.clear();
      REQUIRE(cuot_ggm_sender(ctx, &p, (cuot_block*)buf, (cuot_block*)buf, (cuot_block*)buf, nullptr) == CUOT_OK);
      const bool valid = dfs >= 1 && dfs >= h - 10 && dfs <= h - 8;
      if (dfs == 0) {
        rule = shapes();
        REQUIRE(h < 12 || g_launches.back().grid.x > 3);
      } else if (valid) {
        REQUIRE(g_launches.size() == 1 && g_launches[0].grid.x == 3);
      } else {
        if (shapes() != rule) printf("h = %d, ggm_dfs = %d: %s not %s\n", h, dfs, shapes().c_str(), rule.c_str());
        REQUIRE(shapes() == rule);
      }
    }
  }
  REQUIRE(cuot_destroy(ctx) == CUOT_OK);
  return 0;
}

// A table above 11 MB takes two launches only where the rows pay for the second.
static int check_lpn_slices() {
  cuot_ctx* ctx = nullptr;
  REQUIRE(cuot_init(0, &ctx) == CUOT_OK);
  const struct {
    int64_t n, k;
    size_t launches;
  } rows[] = {{4000000, 720896, 1}, {65536, 720897, 1}, {2 * 720897 - 1, 720897, 1}, {2 * 720897, 720897, 2}};
  for (const auto& r : rows) {
    cuot_lpn_params p;
    memset(&p, 0, sizeof(p));
    p.n = r.n;
    p.k = r.k;
    p.d = 10;
    p.ntasks = 1;
    g_launches.clear();
    REQUIRE(cuot_lpn(ctx, &p, (cuot_block*)buf, (cuot_block*)buf, (cuot_block*)buf, nullptr) == CUOT_OK);
    if (g_launches.size() != r.launches) printf("n = %ld, k = %ld: %zu launches\n", r.n, r.k, g_launches.size());
    REQUIRE(g_launches.size() == r.launches);
  }
  REQUIRE(cuot_destroy(ctx) == CUOT_OK);
  return 0;
}

// Whole words of 2^25 bits and more fill the chip with a lane per two words.
static int check_sparse() {
  cuot_ctx* ctx = nullptr;
  REQUIRE(cuot_init(0, &ctx) == CUOT_OK);
  const int64_t m = (int64_t)1 << 25;
  for (int64_t n : {m - 32, m - 1, m, m + 1, m + 32, 2 * m}) {
    g_launches.clear();
    REQUIRE(cuot_qc_sparse(ctx, n, (uint8_t*)buf, (int64_t*)buf, 16, (uint8_t*)buf, nullptr) == CUOT_OK);
    REQUIRE(g_launches.size() == 1);
    const bool wide = g_launches[0].kernel.find("sparse_encode_wide") != std::string::npos;
    REQUIRE(wide == (n >= m && n % 32 == 0));
  }
  REQUIRE(cuot_destroy(ctx) == CUOT_OK);
  return 0;
}

// upper passes of an encode, there and back, and the one that joins them
static int print_passes(int64_t n, int radix) {
  cuot_ctx* ctx = nullptr;
  REQUIRE(cuot_init(0, &ctx) == CUOT_OK);
  const cuot_knob_values k = {radix, 0, 0, 0, -1, 0};
  REQUIRE(cuot_set_knobs(&k) == CUOT_OK);
  REQUIRE(cuot_qc_encode(ctx, n, (uint32_t*)buf, (cuot_block*)buf, (cuot_block*)buf, buf, nullptr) == CUOT_OK);
  int passes = 0;
  for (const Launch& l : g_launches) passes += l.kernel.find("fa_pass32") != std::string::npos;
  printf("passes %d\n", passes);
  REQUIRE(cuot_destroy(ctx) == CUOT_OK);
  return 0;
}

int main(int argc, char** argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  int rc = 2;
  if (what == "devices") rc = check_devices();
  if (what == "ggm_dfs") rc = check_ggm_dfs();
  if (what == "lpn_slices") rc = check_lpn_slices();
  if (what == "sparse") rc = check_sparse();
  if (what == "passes" && argc > 3) rc = print_passes(atoll(argv[2]), atoi(argv[3]));
  if (!rc) printf("%s ok\n", what.c_str());
  return rc;
}
