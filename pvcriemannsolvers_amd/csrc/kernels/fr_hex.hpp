// Launch interface of the nodal FR kernels on hexahedra (affine or trilinear).
#ifndef MINICFD_KERNELS_FR_HEX_HPP_
#define MINICFD_KERNELS_FR_HEX_HPP_

#include <hip/hip_runtime.h>

#include <cstdint>

namespace mcfd {

constexpr int kMaxQ = 6;
constexpr int kMaxBatchGroups = 4;

// 1-D tables of the solution-point line (Q points):
//   dg[i][m]  = l_m'(x_i) - g_L'(x_i) l_m(-1) - g_R'(x_i) l_m(+1): the derivative
//               of the line's flux with the line ends' own flux values already
//               lifted out, so that only the upwind fluxes are left to lift
//   end[m]    = l_m(-1), the extrapolation to a line end from the node next to it
//               inwards (the points are symmetric: l_{Q-1-m}(+1) = l_m(-1))
//   gp[e][i]  = g_L'(x_i), g_R'(x_i) (Vincent correction derivatives)
struct LineTables {
  double dg[kMaxQ][kMaxQ];
  double end[kMaxQ];
  double gp[2][kMaxQ];
};
// The mixed form's tables: d[i][m] = l_m'(x_i), lend[e][m] = l_m(-1), l_m(+1), gp as above.
struct MixedTables {
  double d[kMaxQ][kMaxQ];
  double lend[2][kMaxQ];
  double gp[2][kMaxQ];
};

// Per-cell affine geometry record (16 doubles):
//   [4 r + e]  e = 0..2: J*.col(r), J* = det(J) J^{-1} (F~_r = sum_e F_e [4 r + e]);
//              e = 3: its length, the face scale of the two faces normal to r
//   [12]       1 / det(J)
//   [13]       length = cbrt(volume) / 2
constexpr int kGeoStride = 16;
constexpr int kGeoInvDet = 12, kGeoLength = 13;
constexpr int kNormalStride = 4;  // unit normal, pad

// Per cell face: the neighbour (or -(1 + boundary tag)); the neighbour's node
// behind in-face point (a, b), m nodes in from the face, as
// first + sa a + sb b + sm m, packed first | sa << 8 | sb << 16 | sm << 24
// (bytes, the strides signed); the unit normal's index, pointing from the
// pair's left to its right state, << 1 | swap; the boundary face index (-1
// for interior faces).  The left state is that of the cell whose upper (+1)
// end the face is; where the two cells do not agree on that (neighbours turned
// against each other), and always for the exact solver, whose state has a
// sign, it is the holder's, and `swap` marks the cell whose place that changes.
struct alignas(16) FrFace {
  int32_t nbr, gather, normal, bface;
};

// Lane operators of the one-wavefront-per-cell kernel (Q = 4), lane = 16 h + 4 m + l:
struct CellOps {
  double dg[64];   // dg[l][h]
  double end[64];  // extrapolation to the lower (l even) and upper (l odd) line end from node h
  double gp[64];   // g_L'(x_l) (h even) and g_R'(x_l) (h odd)
};

// States live in planes, [cell][5][node]: a wavefront's lines are then read
// 8 bytes per lane from consecutive addresses, where the column layout
// [cell][node][5] of the interface spreads them over 40 (LaunchFrLayout
// converts).  The residual is written as a column.
struct FrHexArgs {
  const CellOps *cell_ops;  // lane operators of the one-wavefront-per-cell kernel (Q = 4)
  const double *us;      // state of this stage, also read for neighbour traces
  const double *u0;      // U0 for RK stages 2 and 3
  double *out;           // residual (stage 0, a column) or next state
  const FrFace *faces;   // [cell][6]
  const int32_t *geo_id; // [cell]
  const double *geo;     // [geo][kGeoStride]; curved: [cell], the length only
  const double *normals; // [normal][kNormalStride] (affine cells)
  // curved (trilinear) meshes: J*.col(r) of every node [cell][r][node][3],
  // 1 / det(J) [cell][node], and per cell flux point its unit normal (left to
  // right) and face scale [cell][local face][a * Q + b][4]; null otherwise
  const double *col_node;
  const double *inv_det_node;
  const double *face_point;
  const int32_t *bc_kind;   // [tag]: BcKind (euler.hpp)
  const double *bc_state;   // [tag][5] given state (conservative, or the subsonic parameters)
  // If set, the given state of every boundary flux point instead:
  // [boundary face][a * Q + b][5] (the tag's boundary function at the stage time)
  const double *bc_point_state;
  const int32_t *cell_case; // [cell] case index, or null (one time step for all cells)
  const double *case_dt;    // [case] time step when cell_case is set
  int64_t n_cells;
  double dt;
  int32_t stage;         // 0 residual, 1..3 SSP-RK3 stage
  int32_t xcd_remap;     // remap block ids so each XCD sweeps a contiguous range
  int32_t any_swap;      // some FrFace has its swap bit set
  int32_t mixed;         // FP32 flux-column contractions (mixed-precision form, fr_mixed.hip)
  int32_t curved;        // per-node metrics and per-point normals and scales
  const int32_t *tile_order;  // [tile]: tile swept by logical block b (spatial locality), or null
  // If set, the time-step reduction of LaunchFrHexTimeStep over the state this
  // pass writes is folded into *dt_min_bits (same arithmetic, no extra pass).
  unsigned long long *dt_min_bits;
  // mixed form only, whose states are columns [cell][node][5] and whose geo has
  // records of kMixedGeoStride:
  const int32_t *nbr;       // [cell][6]: neighbour cell, or -(1 + boundary tag)
  const int32_t *finfo;     // [cell][6]: frame id << 7 | holder << 6 | orient << 3 | neighbour face
  const double *frames;     // [frame][kFrameStride]
  const int32_t *bface_of;  // [cell][6] boundary face index, -1 elsewhere
  int32_t diag_metric;      // every J* is diagonal (axis-aligned cells)
  // exact solver only: [cell][local face][point] sign of each flux point's
  // last star velocity (ExactFlux), zero-initialised at creation
  uint8_t *exact_star;
};

// Launches one residual / RK-stage pass for Q points per direction and the
// given Riemann solver on `stream`.  Returns hipSuccess or the launch error.
hipError_t LaunchFrHexStage(int q, int riemann, const FrHexArgs &args, const LineTables &lt, const MixedTables &mt,
                            hipStream_t stream);
// Cells per workgroup (one tile) of LaunchFrHexStage for Q points per direction.
int FrHexStageTileCells(int q, bool mixed);

// One degree group of a batched launch: its own arrays, line tables and tile
// variant (cells per workgroup, see FrHexTileCells).
struct FrHexBatchGroup {
  FrHexArgs args;
  LineTables lt;
  MixedTables mt;
  int32_t q;
  int32_t tile;
  int64_t first_item;   // first work item of this group
};
struct FrHexBatchArgs {
  const FrHexBatchGroup *group;  // device array of n_groups entries (one stage)
  int32_t n_groups;
  int32_t max_tile_lds;          // LDS bytes of the largest tile in use
  int64_t n_items;
};

// Cells per workgroup and LDS bytes of tile variant `tile` (0..2) for q
// points (2..4); 0 if invalid.
int FrHexTileCells(int q, int tile, bool mixed);
int FrHexTileLdsBytes(int q, int tile, bool mixed);

// Persistent batched stage over all groups with n_workgroups workgroups.
hipError_t LaunchFrHexBatch(int riemann, bool mixed, const FrHexBatchArgs &args, int n_workgroups,
                            hipStream_t stream);
// Workgroups of the batched kernel resident on the whole device with the
// given dynamic LDS (0 on failure).
int FrHexBatchResidentWorkgroups(int riemann, bool mixed, int lds_bytes);

// Column layout [cell][node][5] -> planes [cell][5][node] (to_planes), or back.
hipError_t LaunchFrLayout(bool to_planes, const double *in, double *out, int np, int64_t n_cells, hipStream_t stream);
// Per-cell minimum of length / max wave speed over the solution points
// (spatial/fem.hpp:417-435), reduced to one double in *dt_min (device).
// *bits = the ordered bits of 1e300, the start of a time-step reduction.
hipError_t LaunchResetTimeStepBits(unsigned long long *bits, hipStream_t stream);
hipError_t LaunchFrHexTimeStep(int q, bool mixed, const double *u, const int32_t *geo_id, const double *geo,
                               int64_t n_cells, unsigned long long *dt_min_bits, hipStream_t stream);

}  // namespace mcfd

#endif  // MINICFD_KERNELS_FR_HEX_HPP_
