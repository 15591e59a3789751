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

int main(int argc, char** argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  int rc = 2;
  if (what == "devices") rc = check_devices();
  if (!rc) printf("%s ok\n", what.c_str());
  return rc;
}
