// The stage kernels' division by 3 (euler.hpp) on the device against IEEE
// arithmetic on the host: the same bits, at the special values too.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <limits>
#include <random>
#include <vector>

#include "../../pvcriemannsolvers_amd/csrc/kernels/euler.hpp"

__global__ void Evaluate(const double *x, double *third, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  third[i] = mcfd::ThirdOf(x[i]);
}

namespace {

int failures = 0;

// got is want to the last bit, the sign of a zero included
void Expect(const char *name, double x, double got, double want) {
  const bool ok = std::isnan(want) ? std::isnan(got) : std::memcmp(&got, &want, sizeof(got)) == 0;
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
  for (int k = 1; k <= 64; ++k) {  // subnormals, the smallest normal values, the largest
    x.push_back(k * tiny);
    x.push_back(-k * tiny);
    x.push_back(std::numeric_limits<double>::max() * (1 - k * 0x1p-53));
    x.push_back(std::numeric_limits<double>::min() * (1 + (k - 32) * 0x1p-52));
  }
  std::mt19937_64 rng(5);
  std::uniform_real_distribution<double> mantissa(1, 2), exponent(-1000, 1000);
  for (int i = 0; i < 200000; ++i) x.push_back(std::ldexp(mantissa(rng), (int)exponent(rng)) * (i % 4 ? 1 : -1));
  const int n = (int)x.size();
  double *dx, *out;
  HIP(hipMalloc(&dx, n * sizeof(double)));
  HIP(hipMalloc(&out, n * sizeof(double)));
  HIP(hipMemcpy(dx, x.data(), n * sizeof(double), hipMemcpyHostToDevice));
  Evaluate<<<(n + 255) / 256, 256>>>(dx, out, n);
  HIP(hipGetLastError());
  std::vector<double> r(n);
  HIP(hipMemcpy(r.data(), out, n * sizeof(double), hipMemcpyDeviceToHost));
  HIP(hipFree(dx));
  HIP(hipFree(out));
  for (int i = 0; i < n; ++i) Expect("ThirdOf", x[i], r[i], x[i] / 3.0);
  std::printf("%s: %d values, %d failures\n", failures ? "FAIL" : "PASS", n, failures);
  return failures ? 1 : 0;
}
