// planner_check.cpp -- host-only checks of the planner's inner rules (no GPU): the library's host source is compiled into this
// program, with the device queries answered here.  Built and run by tests/test_planner.py; exits non-zero on a failure.
#include <hip/hip_runtime.h>

#include <chrono>
#include <cstdio>
#include <cstring>
#include <random>

// The device queries of the library's host source, answered here.
static int props_calls = 0, props_failing = 0;
static hipError_t fake_count(int* n) {
  *n = 1;
  return hipSuccess;
}
static hipError_t fake_set(int) { return hipSuccess; }
static hipError_t fake_props(hipDeviceProp_t* prop, int) {
  props_calls++;
  if (props_failing > 0) {
    props_failing--;
    return hipErrorNotReady;
  }
  std::memset(prop, 0, sizeof *prop);
  std::strcpy(prop->gcnArchName, "gfx950:sramecc+:xnack-");
  prop->multiProcessorCount = 256;
  return hipSuccess;
}
#undef hipGetDeviceProperties
#define hipGetDeviceCount fake_count
#define hipSetDevice fake_set
#define hipGetDeviceProperties fake_props

#include "../../flashfftstencil_amd/csrc/ffs_api.cpp"

static int failures = 0;

#define EXPECT(cond, ...)                                              \
  do {                                                                 \
    if (!(cond)) {                                                     \
      std::fprintf(stderr, "%s:%d: expected %s: ", __FILE__, __LINE__, #cond); \
      std::fprintf(stderr, __VA_ARGS__);                               \
      std::fprintf(stderr, "\n");                                      \
      failures++;                                                      \
    }                                                                  \
  } while (0)

// Every number of segments by turn, the rule direct_segments states.
static int64_t segments_exhaustive(const ffs_problem& p, int num_cus, int64_t t, int64_t strips) {
  const int64_t n0 = p.sizes[0], fill = 2 * (int64_t)p.radius * t + t - 1;
  const int64_t resident = (int64_t)num_cus * (p.dims == 2 ? 2 : 1);
  double best = 1e300;
  int64_t best_seg = n0;
  int64_t most = std::min<int64_t>(n0, std::max<int64_t>(1, 8 * resident / strips + 1));
  const int64_t of16 = (n0 + 15) / 16;
  if (strips * of16 >= num_cus / 2) most = std::min(most, of16);
  for (int64_t nseg = 1; nseg <= most; nseg++) {
    const int64_t seg = (n0 + nseg - 1) / nseg, units = strips * ((n0 + seg - 1) / seg);
    const double rounds = p.dims == 2 && units <= num_cus ? 0.68 : (double)((units + resident - 1) / resident);
    const double cost = rounds * (double)(seg + fill);
    if (cost < best * (1 - 1e-9)) {
      best = cost;
      best_seg = seg;
    }
  }
  return best_seg;
}

static void segments() {
  std::mt19937_64 rng(7);
  std::uniform_real_distribution<double> u(0.0, 1.0);
  for (int i = 0; i < 20000; i++) {
    ffs_problem p{};
    p.dims = 2 + (int)(rng() % 2);
    p.radius = (int)(rng() % 4);
    p.sizes[0] = (int64_t)std::exp(u(rng) * std::log(2e5));
    const int cus = i % 3 ? 256 : 1 + (int)(rng() % 400);
    const int64_t t = 1 + (int64_t)(rng() % 8), strips = (int64_t)std::exp(u(rng) * std::log(5e4));
    const int64_t got = direct_segments(p, cus, t, strips), want = segments_exhaustive(p, cus, t, strips);
    EXPECT(got == want, "%dD r %d n0 %lld cus %d t %lld strips %lld: %lld, exhaustive %lld", p.dims, p.radius,
           (long long)p.sizes[0], cus, (long long)t, (long long)strips, (long long)got, (long long)want);
    if (failures > 10) return;
  }
}

// It runs on every launch, so it has to be cheap: below a microsecond here, where trying every number takes 30 us.
static void segments_cost() {
  ffs_problem p{};
  p.dims = 2;
  p.radius = 1;
  p.sizes[0] = 65536;
  double best = 1e9;
  int64_t sum = 0;
  for (int batch = 0; batch < 20; batch++) {
    const auto t0 = std::chrono::steady_clock::now();
    for (int i = 0; i < 100; i++) sum += direct_segments(p, 256, 1 + i % 8, 1);
    best = std::min(best, std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count() / 100);
  }
  EXPECT(sum > 0 && best < 5e-6, "%g s per call", best);
}

// A device is asked once, but a query that failed is no answer: the next plan asks again.
static void device_query() {
  props_failing = 1;
  ffs_plan pl;
  EXPECT(plan_device(&pl) == FFS_ERR_HIP && props_calls == 1, "%d calls", props_calls);
  EXPECT(plan_device(&pl) == FFS_OK && props_calls == 2 && pl.num_cus == 256, "%s, %d calls", g_err.c_str(), props_calls);
  EXPECT(plan_device(&pl) == FFS_OK && props_calls == 2 && pl.num_cus == 256, "%s, %d calls", g_err.c_str(), props_calls);
}

int main() {
  device_query();
  segments();
  segments_cost();
  if (failures) {
    std::fprintf(stderr, "%d failures\n", failures);
    return 1;
  }
  std::printf("planner checks passed\n");
  return 0;
}
