// brick_check.cpp -- the bound under which a brick's rows keep a layer's columns in LDS
// without counting them (upf_device_row.hpp, brick_columns_fit) against the count, in the
// kernel's float operations: over origins up to where neighbouring nodes coincide, spacings
// and frequencies on both sides of the limit.  tests/test_brick_columns.py runs it.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <random>

#include "../../unnatural_planets_amd/csrc/upf_device_row.hpp"

namespace {
constexpr int kMost = upf::kRowSlice2 / (upf::kBrickRows * upf::kBrickGroups);
int g_accepted = 0, g_refused = 0;

// the columns of rows of 9 nodes from x0 on, or -1 where floor(x f) leaves the integers
int64_t columns(const float* freq, int oct, float x0, float x1) {
  int64_t total = 0;
  for (int k = 0; k < oct; k++) {
    const float a = std::floor(x0 * freq[k]), b = std::floor(x1 * freq[k]);
    if (!(std::fabs(a) < 2147483520.0f && std::fabs(b) < 2147483520.0f)) return -1;
    total += std::llabs((int64_t)b - (int64_t)a) + 2;
  }
  return total;
}

bool check(float origin, float spacing, int node, const float* freq, int oct) {
  const float x0 = std::fmaf((float)node, spacing, origin), x1 = std::fmaf((float)(node + 8), spacing, origin);
  float sum = 0.0f;
  for (int k = 0; k < oct; k++) sum = sum + std::fabs(freq[k]);
  const bool fit = upf::brick_columns_fit(sum, oct, x0, x1, kMost);
  const int64_t n = columns(freq, oct, x0, x1);
  (fit ? g_accepted : g_refused)++;
  if (!fit || n < 0 || n <= kMost) return true;
  std::printf("origin %.9g spacing %.9g node %d, %d octaves from %.9g: %lld columns accepted, room for %d\n", origin, spacing,
              node, oct, freq[0], (long long)n, kMost);
  return false;
}
}  // namespace

int main() {
  bool ok = true;
  std::mt19937 rng(7);
  std::uniform_real_distribution<double> u(0.0, 1.0);
  for (int i = 0; i < 3000000 && ok; i++) {
    const int oct = 1 + (int)(u(rng) * 8.0);
    const double spacing = std::exp2(12.0 * u(rng) - 8.0);
    const double cells = std::exp2(10.0 * u(rng) - 7.0) / 8.0;  // cells a node, the first octave
    const double lac = 0.5 + 1.7 * u(rng);
    float freq[8];
    double f = cells / spacing;
    for (int k = 0; k < oct; k++, f *= lac) freq[k] = (float)(u(rng) < 0.2 ? -f : f);
    const double origin = spacing * std::exp2(32.0 * u(rng)) * (u(rng) < 0.5 ? -1.0 : 1.0);
    ok = check((float)origin, (float)spacing, 8 * (int)(u(rng) * 8191.0), freq, oct);
  }
  const float inf[1] = {3e38f}, zero[1] = {0.0f};
  ok = ok && check(1e20f, 1e19f, 8, inf, 1) && check(3e38f, 3e37f, 80, zero, 1) && check(0.0f, 1.0f, 0, zero, 1);
  ok = ok && g_accepted > 100000 && g_refused > 100000;
  if (ok) std::printf("brick_check: ok\n");
  return ok ? 0 : 1;
}
