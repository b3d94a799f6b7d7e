// The stage kernels' reciprocal, square root and division by 3 (euler.hpp) on
// the device against IEEE arithmetic on the host: at the special values the same
// result, elsewhere within the bounds that they state.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <limits>
#include <random>
#include <vector>

#include "../../pvcriemannsolvers_amd/csrc/kernels/euler.hpp"

__global__ void Evaluate(const double *x, double *rcp, double *root, double *third, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  rcp[i] = mcfd::FastRcp(x[i]);
  root[i] = mcfd::FastSqrt(x[i]);
  third[i] = mcfd::ThirdOf(x[i]);
}

namespace {

int failures = 0;

int64_t Ordered(double v) {  // neighbours differ by 1
  int64_t b;
  std::memcpy(&b, &v, sizeof(b));
  return b < 0 ? INT64_MIN - b : b;
}

// got is want to the last `ulps` bits; with 0 also the sign of a zero
void Expect(const char *name, double x, double got, double want, int64_t ulps) {
  bool ok;
  if (std::isnan(want) || std::isnan(got)) ok = std::isnan(want) && std::isnan(got);
  else if (ulps == 0) ok = std::memcmp(&got, &want, sizeof(got)) == 0;
  else ok = std::llabs(Ordered(got) - Ordered(want)) <= ulps;
  if (ok) return;
  if (++failures < 20) std::printf("FAIL %s(%a) = %a, expected %a\n", name, x, got, want);
}

#define HIP(call)                                                                \
  do {                                                                           \
    const hipError_t e = (call);                                                 \
    if (e != hipSuccess) {                                                       \
      std::printf("FAIL %s: %s\n", #call, hipGetErrorString(e));                 \
      return 1;                                                                  \
    }                                                                            \
  } while (0)

}  // namespace

int main() {
  const double inf = std::numeric_limits<double>::infinity(), tiny = std::numeric_limits<double>::denorm_min();
  std::vector<double> x{ 0.0, -0.0, inf, -inf, std::nan(""), 1.0, -1.0, 3.0, -3.0 };
  const size_t specials = x.size();
  for (int k = 1; k <= 64; ++k) {  // subnormals and the largest values, for the division alone
    x.push_back(k * tiny);
    x.push_back(-k * tiny);
    x.push_back(std::numeric_limits<double>::max() * (1 - k * 0x1p-53));
    x.push_back(std::numeric_limits<double>::min() * (1 + (k - 32) * 0x1p-52));
  }
  const size_t normals = x.size();  // from here on arguments and results are normal
  std::mt19937_64 rng(5);
  std::uniform_real_distribution<double> mantissa(1, 2), exponent(-1000, 1000);
  for (int i = 0; i < 200000; ++i) x.push_back(std::ldexp(mantissa(rng), (int)exponent(rng)) * (i % 4 ? 1 : -1));
  const int n = (int)x.size();
  double *dx, *out;
  HIP(hipMalloc(&dx, n * sizeof(double)));
  HIP(hipMalloc(&out, 3 * n * sizeof(double)));
  HIP(hipMemcpy(dx, x.data(), n * sizeof(double), hipMemcpyHostToDevice));
  Evaluate<<<(n + 255) / 256, 256>>>(dx, out, out + n, out + 2 * n, n);
  HIP(hipGetLastError());
  std::vector<double> r(3 * n);
  HIP(hipMemcpy(r.data(), out, 3 * n * sizeof(double), hipMemcpyDeviceToHost));
  HIP(hipFree(dx));
  HIP(hipFree(out));
  for (int i = 0; i < n; ++i) {
    Expect("ThirdOf", x[i], r[2 * n + i], x[i] / 3.0, 0);
    if (i >= (int)specials && i < (int)normals) continue;
    const int64_t ulps = i < (int)specials ? 0 : 1;
    Expect("FastRcp", x[i], r[i], 1.0 / x[i], ulps);
    Expect("FastSqrt", x[i], r[n + i], std::sqrt(x[i]), ulps);
  }
  std::printf("%s: %d values, %d failures\n", failures ? "FAIL" : "PASS", n, failures);
  return failures ? 1 : 0;
}
