// The splits that the GEMM launches choose, over every kind of shape: their
// workspace stays within its limit and each workgroup has k to work on.

#include "../../vx_amd/csrc/kernels/gemm_direct.h"
#include "../../vx_amd/csrc/kernels/gemm_f32.h"
#include "../../vx_amd/csrc/kernels/gemm_ring.h"

#include <cmath>
#include <cstdio>
#include <random>

static int failures = 0;

static void expect(bool ok, const char *what, int64_t m, int64_t n, int64_t k) {
  if (!ok) {
    fprintf(stderr, "%s: %lld x %lld x %lld\n", what, (long long)m, (long long)n, (long long)k);
    ++failures;
  }
}

static void check(int64_t m, int64_t n, int64_t k) {
  using namespace vxk;
  for (int cus : {64, 256, 304}) {
    const int f = f32::splits(m, n, k, cus, true);
    expect(f >= 1 && (f == 1 || (k + 31) / 32 / f >= 4), "f32 splits", m, n, k);
    if (f > 1) {
      expect(f32::tiles(m, n) <= split::kMaxTiles, "f32 tickets", m, n, k);
      expect(f32::ws_bytes(m, n, f) <= split::kMaxBytes, "f32 workspace", m, n, k);
    }
    const int r = ring::splits(m, n, k, cus, true);
    expect(r >= 1 && (r == 1 || k / 32 / r >= 8), "ring splits", m, n, k);
    if (r > 1) {
      expect(ring::tiles(m, n) <= split::kMaxTiles, "ring tickets", m, n, k);
      expect(ring::ws_bytes(m, n, r) <= split::kMaxBytes, "ring workspace", m, n, k);
    }
    if (direct::shape_ok(m, n, k, k, n, n)) {
      double us;
      const direct::Plan d = direct::plan(m, n, k, false, cus, true, &us);
      expect(d.splits == 1 || (int64_t)d.tiles_m * d.tiles_n <= split::kMaxTiles, "direct tickets", m, n, k);
      expect(d.ws_bytes <= split::kMaxBytes, "direct workspace", m, n, k);
    }
    expect(f32::splits(m, n, k, cus, false) == 1 && ring::splits(m, n, k, cus, false) == 1,
           "undivided", m, n, k);
  }
}

// Few k over many rounds: 64-row tiles, one to a CU, take twice the time.
static void check_short(int64_t m, int64_t n, int64_t k) {
  double us;
  const vxk::direct::Plan d = vxk::direct::plan(m, n, k, k % 2 != 0, 256, true, &us);
  expect(!(d.along_k && d.mt == 4), "64-row tiles", m, n, k);
}

int main() {
  check_short(146800, 40, 16);
  check_short(15296, 832, 9);
  check_short(1390, 41136, 5);
  check(2176, 7552, 262144);
  check(1920, 8192, 262144);
  check(128 * 1024, 128, 1 << 20); // as many tiles as tickets
  std::mt19937 rng(1);
  std::uniform_real_distribution<double> mn(0, std::log(65536.0)), ks(0, std::log(4194304.0));
  for (int i = 0; i < 20000; ++i) {
    const int64_t m = (int64_t)std::exp(mn(rng)), n = (int64_t)std::exp(mn(rng)), k = (int64_t)std::exp(ks(rng));
    check(m, n, i % 2 ? k : (k + 31) / 32 * 32);
  }
  if (failures) {
    return 1;
  }
  puts("ok");
  return 0;
}
