// Device helpers of the FR stage kernels: the XCD-aware block order and the
// RK stage combination.
#ifndef MINICFD_KERNELS_FR_COMMON_HPP_
#define MINICFD_KERNELS_FR_COMMON_HPP_

#include <hip/hip_runtime.h>

#include <cstdint>

#include "euler.hpp"
#include "fr_hex.hpp"

namespace mcfd {
namespace fr {

__device__ __forceinline__ int64_t LogicalBlock(int32_t remap) {
  int64_t b = blockIdx.x;
  if (!remap) return b;
  // Blocks are dispatched round-robin over the 8 XCDs; give each XCD one
  // contiguous range of cells so neighbour traces hit its own L2.
  int64_t n = gridDim.x, per = n / 8, rem = n % 8;
  int64_t xcd = b % 8, idx = b / 8;
  return xcd < rem ? xcd * (per + 1) + idx : rem * (per + 1) + (xcd - rem) * per + idx;
}

// Residual -> RK stage output (temporal/rk.hpp:31-49 with ode.hpp:121-128):
// stage 0 returns the residual; 1: us + dt r; 2: (3 u0 + (us + dt r)) / 4;
// 3: (2 (us + dt r) + u0) / 3, each operation rounded on its own.
__device__ __forceinline__ double RkOutput(int stage, double res, double us, double u0, double dt) {
  if (stage == 0) return res;
  const double next = AddRn(us, MulRn(res, dt));
  if (stage == 1) return next;
  if (stage == 2) return AddRn(MulRn(u0, 3.0), next) / 4.0;
  return ThirdOf(AddRn(MulRn(next, 2.0), u0));
}

}  // namespace fr
}  // namespace mcfd

#endif  // MINICFD_KERNELS_FR_COMMON_HPP_
