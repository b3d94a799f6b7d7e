// Launch interface of the mixed-precision form of nodal FR (fr_mixed.hip); the
// arguments are FrHexArgs with its mixed part set, states as columns.
#ifndef MINICFD_KERNELS_FR_MIXED_HPP_
#define MINICFD_KERNELS_FR_MIXED_HPP_

#include "fr_hex.hpp"

namespace mcfd {

// Per-cell affine geometry record (20 doubles):
//   [0..8]  J* = det(J) J^{-1} (row-major, F~ = F J*)
//   [9]     1 / det(J)
//   [10..15] signed face scale +-|J*.col(normal dir)| of local faces 0..5
//   [16]    length = cbrt(volume) / 2
constexpr int kMixedGeoStride = 20;
constexpr int kFrameStride = 6;  // n, t

hipError_t LaunchFrMixedStage(int q, int riemann, const FrHexArgs &args, const MixedTables &lt, hipStream_t stream);
int FrMixedStageTileCells(int q);
int FrMixedTileCells(int q, int tile);
int FrMixedTileLdsBytes(int q, int tile);
hipError_t LaunchFrMixedBatch(int riemann, const FrHexBatchArgs &args, int n_workgroups, hipStream_t stream);
hipError_t FrMixedBatchResident(int riemann, int lds_bytes, int *per_cu);
hipError_t LaunchFrMixedTimeStep(int q, const double *u, const int32_t *geo_id, const double *geo, int64_t n_cells,
                                 unsigned long long *dt_min_bits, hipStream_t stream);

}  // namespace mcfd

#endif  // MINICFD_KERNELS_FR_MIXED_HPP_
