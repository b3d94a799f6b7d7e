// Nodal flux reconstruction on hexahedra for CDNA4 (gfx950).
//
// One pass = residual of spatial/fr/general.hpp (volume term :271-288, face
// correction :296-315,409-434, boundary corrections :435-640, det(J) scaling
// :249-268) fused with one SSP-RK3 stage of temporal/rk.hpp:31-49.
//
// Two kernels.  FP64 at Q = 4 points: one wavefront per cell or per two cells
// on v_mfma_f64_4x4x4 (below).  All else: lanes that own a line of solution
// points.  A workgroup owns C cells (16, 7, 3, 1 for Q = 2, 3, 5, 6), and each lane
//   1. gathers, for the flux points at its line's ends, the neighbours' lines
//      behind them (through L1 and L2); the cells' own states go to LDS once;
//   2. extrapolates both traces of each end and solves the upwind flux there;
//   3. forms F~_r = F J*.col(r) at its nodes and contracts it in registers with
//      the tables in scalar registers, the ends' own fluxes lifted out of the
//      derivative table, and lifts the upwind fluxes;
//   4. writes the line's part of the divergence to LDS.
// Then the threads, one per value, sum the three directions' parts and do the
// RK stage in the reference's operation order.  Each interior face is solved by
// both of its cells with bit-identical inputs, so the scheme stays conservative
// without atomics or a separate face pass.  The bodies serve the single-mesh
// launch and the persistent batched launch that walks a work list spanning several
// polynomial degrees.
//
// What bounds both: a pass must move U, U0 and the new U, 120 B per node (HBM at
// about half its copy rate), and issues its FP64 instructions in about half the
// pass's cycles; the vector memory unit, four lanes per clock whatever the width,
// takes a third to a half.  No one unit is full, so the number of wavefronts
// in flight decides, and with it the registers: hence lines taken one end at a
// time and contracted node by node, and states in planes, where a line gather
// costs four lanes one cache line.  Per pass, against one thread per node with
// tasks per flux point, columns and a derivative through LDS: 64^3 p3 900 -> 595
// us, 30 x 28 x 26 curved p3 113 -> 73, 35 x 37 x 33 p4 322 -> 246, 47 x 41 x 43
// p2 180 -> 121, 64^3 p1 147 -> 116, 24 x 25 x 23 p5
// 185 -> 157, 8^3 p3 10.6 -> 9.0 (Roe, p2 HLLC); exact solver 24^3 p3 350 -> 63,
// 32^3 p2 531 -> 88 (most of it the solver itself, FastExactState).
#include "fr_hex.hpp"

#include <algorithm>

#include "euler.hpp"
#include "fr_common.hpp"
#include "fr_mixed.hpp"

namespace mcfd {

namespace {

using fr::LogicalBlock;

template <int Q>
struct Shape {
  static constexpr int kPoints = Q * Q * Q;        // solution points per cell
  static constexpr int kLines = Q * Q;             // lines per cell and direction
  static constexpr int kCells = Q == 6 ? 1 : (Q == 5 ? 3 : 64 / kLines);  // cells per workgroup
  // Q = 6: two lanes per line, each with one end and the half of the nodes next
  // to it; a whole line's registers cost a wavefront per SIMD there
  static constexpr bool kSplit = Q == 6;
  static constexpr int kRows = kSplit ? Q / 2 : Q, kEnds = kSplit ? 1 : 2;  // per lane
  // lanes per direction: one wavefront for Q <= 4; two cells of Q = 5 or one of
  // Q = 6 would leave 22 % and 44 % of its lanes idle, so there the directions
  // follow each other (88 % and 84 % in use)
  static constexpr int kDirLanes = Q <= 4 ? 64 : kCells * kLines * (kSplit ? 2 : 1);
  static constexpr int kThreads = (3 * kDirLanes + 63) / 64 * 64;
  // LDS position of solution point (i, j, k): i * kSI + j * kSJ + k.  The Q x Q
  // points at one depth of any line family must fall in distinct LDS banks: for
  // odd Q they do in the states' own order, for even Q with kSJ = Q + 1 and
  // kSI = Q (Q + 1) (Q = 4: 20 i + 5 j + k).
  static constexpr bool kSkew = Q % 2 == 0;
  static constexpr int kSJ = kSkew ? Q + 1 : Q;
  static constexpr int kSI = Q * kSJ;
  static constexpr int kPad = kSkew ? ((Q - 1) * (kSI + kSJ + 1) + 1) | 1 : Q * Q * Q;  // of a component
  // the cells' states, later the z direction's part of the divergence; the x
  // direction's; and the y direction's
  static constexpr int kShare = kCells * 5 * kPad;
  static constexpr int kCellData = 3 * kShare;  // per cell: 1 / det(J), time step
  static constexpr int kFlux = kCellData + 2 * kCells;  // kSplit: the fluxes, for the line's other lane
  static constexpr int kLdsDoubles = kFlux + (kSplit ? 3 * kDirLanes * 5 : 0);
  static constexpr int kValues = kCells * 5 * kPoints, kLoads = (kValues + kThreads - 1) / kThreads;
  // LDS position of value e of the workgroup's planes [cell][5][node]
  __device__ static int At(int e) {
    if (!kSkew) return e;
    const int plane = e / kPoints, node = e - plane * kPoints;
    return plane * kPad + node / (Q * Q) * kSI + node / Q % Q * kSJ + node % Q;
  }
};

// dg[i][m] and g_R'(x_i) through the symmetry of the points about 0: half of
// the table suffices, and the other half's sign is free in the FMA.
template <int Q>
__device__ __forceinline__ double DerivativeEntry(const LineTables &lt, int i, int m) {
  const bool low = i < Q - 1 - i || (i == Q - 1 - i && m < Q - 1 - m);
  return low ? lt.dg[i][m] : -lt.dg[Q - 1 - i][Q - 1 - m];
}

// Makes the compiler form v here: left to itself it sinks the flux below to its
// use, past the other end's solve, and both ends' traces stay in registers.
template <class T>
__device__ __forceinline__ void Pin(T *v) {
#pragma unroll
  for (int k = 0; k < 5; ++k) asm volatile("" : "+v"(v[k]));
}

// kCurved (trilinear cells): J* and 1/det(J) are read per solution point, the
// normal and the scale per cell flux point instead of per cell and per face.
template <int Q, int kRiemann, bool kCurved>
__device__ __forceinline__ void FrLineBody(const FrHexArgs &a, const LineTables &lt, int64_t block, double *lds) {
  using S = Shape<Q>;
  constexpr int NP = S::kPoints, NL = S::kLines, C = S::kCells, PAD = S::kPad, DL = S::kDirLanes;
  const int64_t c0 = block * C;
  if (c0 >= a.n_cells) return;
  const int64_t left_over = a.n_cells - c0;
  const int nc = left_over < C ? (int)left_over : C;

  const int tid = threadIdx.x;
  const int dir = DL == 64 ? __builtin_amdgcn_readfirstlane(tid >> 6) : min(tid / DL, 2);
  const int half = S::kSplit ? (tid - dir * DL) / (C * NL) : 0;  // of a split line: its end
  const int lane = tid - dir * DL - half * (C * NL);
  const int cell = lane / NL, line = lane - (lane / NL) * NL;
  const int la = line / Q, lb = line - (line / Q) * Q;  // in-face indices of the line's two ends
  const bool active = half < 2 && cell < nc;
  const int64_t c = c0 + (active ? cell : 0);
  const int stride = dir == 0 ? Q * Q : (dir == 1 ? Q : 1);
  const int node0 = la * (dir == 0 ? Q : Q * Q) + lb * (dir == 2 ? Q : 1);
  // local faces at the line's lower and upper end: x {4, 2}, y {1, 3}, z {0, 5}
  const int f_lo = dir == 0 ? 4 : (dir == 1 ? 1 : 0), f_hi = dir == 0 ? 2 : (dir == 1 ? 3 : 5);
  // Loads are waited for in the order of their issue: what is needed first, or
  // needed to form an address, goes first.
  const int f_first = half == 1 ? f_hi : f_lo;
  const FrFace lower = a.faces[c * 6 + f_first], upper = S::kSplit ? lower : a.faces[c * 6 + f_hi];
  const int geo_id = kCurved ? 0 : a.geo_id[c];
  double v[S::kLoads];  // the cells' states, one load per value for all three directions
  const int values = nc * 5 * NP;
  auto value = [&](int it) {  // threads past the end repeat the last value
    const int e = tid + it * S::kThreads;
    return e < values ? e : values - 1;
  };
#pragma unroll
  for (int it = 0; it < S::kLoads; ++it) v[it] = a.us[c0 * (5 * NP) + value(it)];
  // unit normal (left to right) and face scale of end s
  double n[3], scale = 0;
  auto geometry = [&](FrFace const &face, int s) {
    if constexpr (kCurved) {
      const double *fp = a.face_point + ((c * 6 + (s ? f_hi : f_first)) * NL + line) * 4;
#pragma unroll
      for (int d = 0; d < 3; ++d) n[d] = fp[d];
      scale = fp[3];
    } else {
      const double *fp = a.normals + (int64_t)(face.normal >> 1) * kNormalStride;
#pragma unroll
      for (int d = 0; d < 3; ++d) n[d] = fp[d];
    }
  };
  // the neighbour's line behind end s, from its lower end upwards
  struct Line { double v[Q][5]; };
  auto gather = [&](FrFace const &face) {
    Line nb;  // left undefined without a neighbour
    if (!active || face.nbr < 0) return nb;
    const int g = face.gather, step = g >> 24;
    const int first = (g & 255) + (int)(int8_t)(g >> 8) * la + (int)(int8_t)(g >> 16) * lb + (step < 0 ? (Q - 1) * step : 0);
    const int up = step < 0 ? -step : step;
    const double *src = a.us + (int64_t)face.nbr * (5 * NP) + first;
    if (__all(up == 1)) {  // along consecutive nodes
      typedef double Two __attribute__((ext_vector_type(2), aligned(8)));
#pragma unroll
      for (int k = 0; k < 5; ++k) {
#pragma unroll
        for (int q = 0; q + 1 < Q; q += 2) {
          const Two w = *reinterpret_cast<const Two *>(src + k * NP + q);
          nb.v[q][k] = w.x;
          nb.v[q + 1][k] = w.y;
        }
        if (Q & 1) nb.v[Q - 1][k] = src[k * NP + Q - 1];
      }
      asm volatile("; 16-byte loads" ::: "memory");  // keeps the compiler from merging the two branches' loads
    } else {
#pragma unroll
      for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int k = 0; k < 5; ++k) nb.v[q][k] = src[k * NP + q * up];
    }
    return nb;
  };
  geometry(lower, 0);
  if (tid < nc) {
    lds[S::kCellData + tid] = kCurved ? 0.0 : a.geo[(int64_t)a.geo_id[c0 + tid] * kGeoStride + kGeoInvDet];
    lds[S::kCellData + C + tid] = a.case_dt ? a.case_dt[a.cell_case[c0 + tid]] : a.dt;
  }
  double dir_col[3] = { 0, 0, 0 };
  if constexpr (!kCurved) {
    const double *src = a.geo + (int64_t)geo_id * kGeoStride + 4 * dir;
#pragma unroll
    for (int e = 0; e < 3; ++e) dir_col[e] = src[e];
    scale = src[3];
  }
  Line nb = gather(lower);
#pragma unroll
  for (int it = 0; it < S::kLoads; ++it) lds[S::At(value(it))] = v[it];
  __syncthreads();

  const int pos0 = cell * 5 * PAD + la * (dir == 0 ? S::kSJ : S::kSI) + lb * (dir == 2 ? S::kSJ : 1);
  const int pos_step = dir == 0 ? S::kSI : (dir == 1 ? S::kSJ : 1);
  double flux[S::kEnds][5];  // upwind fluxes at the line's ends times the face scale, along +r
  if (active) {
#pragma unroll
    for (int s = 0; s < S::kEnds; ++s) {
      const bool at_upper = S::kSplit ? half == 1 : s == 1;
      const FrFace face = s ? upper : lower;
      const int64_t point = (c * 6 + (s ? f_hi : f_first)) * NL + line;  // this cell's flux point
      const bool swap = (kRiemann == kExact || a.any_swap) ? (face.normal & 1) != 0 : false;
      State other;
      int kind = kBcSmart;
      if (face.nbr >= 0) {
        // the neighbour's trace at the end it has here, in that same order
        const bool lower_end = (face.gather >> 24) > 0;
        double end[Q];
#pragma unroll
        for (int m = 0; m < Q; ++m) end[m] = lower_end ? lt.end[m] : lt.end[Q - 1 - m];
#pragma unroll
        for (int k = 0; k < 5; ++k) {
          double acc = end[0] * nb.v[0][k];
#pragma unroll
          for (int m = 1; m < Q; ++m) acc = __fma_rn(end[m], nb.v[m][k], acc);
          other.v[k] = acc;
        }
      } else {
        const int tag = -face.nbr - 1;
        kind = a.bc_kind[tag];
        // the tag's constant state, or this point's value of the tag's
        // boundary function at the stage time
        const double *gs = a.bc_point_state ? a.bc_point_state + ((int64_t)face.bface * NL + line) * 5
                                            : a.bc_state + tag * 5;
#pragma unroll
        for (int k = 0; k < 5; ++k) other.v[k] = gs[k];
      }
      Pin(other.v);
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      // the own trace: a fused chain from the line's lower node upwards, the
      // order in which the cell behind the face forms it too
      State own;
      double own_end[Q];
#pragma unroll
      for (int m = 0; m < Q; ++m) own_end[m] = at_upper ? lt.end[Q - 1 - m] : lt.end[m];
#pragma unroll
      for (int k = 0; k < 5; ++k) {
        double acc = own_end[0] * lds[pos0 + k * PAD];
#pragma unroll
        for (int m = 1; m < Q; ++m) acc = __fma_rn(own_end[m], lds[pos0 + k * PAD + m * pos_step], acc);
        own.v[k] = acc;
      }
      Pin(own.v);
      // the exact solver's state of this flux point, one copy per side: both
      // sides solve the same problem with the same inputs every pass, so the
      // two copies stay equal
      bool star = kRiemann == kExact ? a.exact_star[point] != 0 : false;
      State l, r;
#pragma unroll
      for (int k = 0; k < 5; ++k) {
        l.v[k] = at_upper ? own.v[k] : other.v[k];
        r.v[k] = at_upper ? other.v[k] : own.v[k];
      }
      if (kRiemann == kExact || a.any_swap) {
#pragma unroll
        for (int k = 0; k < 5; ++k) {
          const double x = l.v[k], y = r.v[k];
          l.v[k] = swap ? y : x;
          r.v[k] = swap ? x : y;
        }
      }
      State fu;
      if (kind == kBcSmart) {
        fu = FaceFlux<kRiemann>(n, l, r, star);
      } else {  // the flux through the left-to-right normal, as the upwind one
        const bool left = at_upper != swap;
        fu = BoundaryFlux(kind, left, n, left ? l : r, left ? r : l);
      }
      if constexpr (kRiemann == kExact) a.exact_star[point] = star ? 1 : 0;
      // left-to-right is the +r direction of this cell unless the roles are swapped
      const double along = swap ? -scale : scale;
#pragma unroll
      for (int k = 0; k < 5; ++k) flux[s][k] = fu.v[k] * along;
      Pin(flux[s]);
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      if (s + 1 < S::kEnds) {  // not in flight during the solve: that would cost a wavefront per SIMD
        geometry(upper, 1);
        nb = gather(upper);
      }
    }
  }

  double *const my_flux = lds + S::kFlux + 5 * tid, *const far_flux = my_flux + (half ? -5 : 5) * (C * NL);
  if (S::kSplit && active) {
#pragma unroll
    for (int k = 0; k < 5; ++k) my_flux[k] = flux[0][k];
  }

  // ---- each thread's values of U, and U0, for the RK stage
  double u0[S::kLoads];
  if (a.stage >= 2) {
#pragma unroll
    for (int it = 0; it < S::kLoads; ++it) u0[it] = __builtin_nontemporal_load(a.u0 + c0 * (5 * NP) + value(it));
  }
#pragma unroll
  for (int it = 0; it < S::kLoads; ++it) v[it] = lds[S::At(value(it))];

  // ---- F~_r along the line, contracted node by node, so that only the Q x 5
  // sums stay in registers; then the fluxes lifted
  double d[S::kRows][5];
  // Nodes are taken upwards, and mirror from the lane's end of a split line:
  // the tables' symmetry leaves the sums there with the opposite sign.
  const bool mirror = S::kSplit && half == 1;
  const int first_pos = pos0 + (mirror ? (Q - 1) * pos_step : 0), node_step = mirror ? -pos_step : pos_step;
  if (active) {
    const double *col_src = kCurved ? a.col_node + ((c * 3 + dir) * NP + node0 + (mirror ? (Q - 1) * stride : 0)) * 3 : nullptr;
    const int col_step = mirror ? -3 * stride : 3 * stride;
    double col[3], next[3] = { dir_col[0], dir_col[1], dir_col[2] };
    if constexpr (kCurved) {
#pragma unroll
      for (int e = 0; e < 3; ++e) next[e] = col_src[e];
    }
#pragma unroll
    for (int m = 0; m < Q; ++m) {
      double w[5];
#pragma unroll
      for (int k = 0; k < 5; ++k) w[k] = lds[first_pos + k * PAD + m * node_step];
#pragma unroll
      for (int e = 0; e < 3; ++e) col[e] = next[e];
      if (kCurved && m + 1 < Q) {
#pragma unroll
        for (int e = 0; e < 3; ++e) next[e] = col_src[(m + 1) * col_step + e];
      }
      // contravariant momentum and velocity, and pressure; the zeroing rule of
      // types.hpp:195-202,289-301 only where some lane of the wavefront needs it
      const double inv = FiniteRcp(w[0]);
      const double mom = w[1] * col[0] + w[2] * col[1] + w[3] * col[2];
      double vel = mom * inv;
      double p = (w[4] - 0.5 * (w[1] * w[1] + w[2] * w[2] + w[3] * w[3]) * inv) * kGm1;
      if (!__all(w[0] > 0 && w[4] >= 0 && p >= 0)) {
        const bool bad = w[0] < 0 || w[4] < 0;
        const bool vacuum = !bad && w[0] == 0;
        const bool zero = bad || (!vacuum && p < 0);
        vel = zero ? 0.0 : (vacuum ? mom : vel);
        p = zero ? 0.0 : (vacuum ? w[4] : p);
      }
#pragma unroll
      for (int k = 0; k < 5; ++k) {
        const double f = k == 0 ? mom : (k == 4 ? (w[4] + p) * vel : w[k] * vel + p * col[k == 0 ? 0 : k - 1]);
        #pragma unroll
        for (int i = 0; i < S::kRows; ++i)
          d[i][k] = m ? __fma_rn(DerivativeEntry<Q>(lt, i, m), f, d[i][k]) : DerivativeEntry<Q>(lt, i, 0) * f;
      }
#pragma unroll
      for (int i = 0; i < S::kRows; ++i) Pin(d[i]);  // else the sums are put off and all nodes' fluxes stay in registers
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  __syncthreads();  // from here on the z lines' parts replace the states
  double *const part = lds + (dir == 2 ? 0 : (dir == 1 ? 2 : 1) * S::kShare) + pos0;
  if (active) {
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      // the lower and the upper end's gap; of a split line the near and the far end's
      double gap[2] = { flux[0][k], S::kSplit ? far_flux[k] : flux[S::kEnds - 1][k] };
#pragma unroll
      for (int i = 0; i < S::kRows; ++i) {
        double sum = __fma_rn(lt.gp[0][i], gap[0], d[i][k]);
        sum = __fma_rn(-lt.gp[0][Q - 1 - i], gap[1], sum);
        if (mirror) sum = -sum;
        const int at = k * PAD + (mirror ? Q - 1 - i : i) * pos_step;
        part[at] = sum;
      }
    }
  }
  __syncthreads();

  // ---- per value: the three directions' sum, 1/det(J), RK stage, store
#pragma unroll
  for (int it = 0; it < S::kLoads; ++it) {
    const int e = tid + it * S::kThreads;
    if (e >= values) continue;
    const int at = S::At(e), cl = C == 1 ? 0 : e / (5 * NP), k = (e - cl * (5 * NP)) / NP, node = e - (cl * 5 + k) * NP;
    const double inv_det = kCurved ? a.inv_det_node[(c0 + cl) * NP + node] : lds[S::kCellData + cl];
    const double sum = lds[S::kShare + at] + lds[2 * S::kShare + at] + lds[at];
    const double out = fr::RkOutput(a.stage, -sum * inv_det, v[it], u0[it], lds[S::kCellData + C + cl]);
    // the residual is handed out as a column, states stay in planes; streamed,
    // so that the states which neighbours still gather keep the L2
    __builtin_nontemporal_store(out, a.out + (a.stage == 0 ? ((c0 + cl) * NP + node) * 5 + k : c0 * (5 * NP) + e));
    if (a.dt_min_bits) lds[at] = out;
  }
  if (a.dt_min_bits) {
    // fem.hpp:412-435 on the state just written, as FrHexTimeStepKernel: min
    // over cells of length / max(1e-5, max over nodes of |u| + c), which is the
    // min over nodes of length / max(1e-5, |u| + c); the bits of positive
    // doubles order as the doubles do
    __syncthreads();
    double local = 1e300;
    for (int w = tid; w < nc * NP; w += S::kThreads) {
      const int cl = w / NP, at = S::At(cl * 5 * NP + w - cl * NP);
      State out;
#pragma unroll
      for (int k = 0; k < 5; ++k) out.v[k] = lds[at + k * PAD];
      local = fmin(local, a.geo[(int64_t)(kCurved ? c0 + cl : a.geo_id[c0 + cl]) * kGeoStride + kGeoLength] /
                              fmax(1e-5, MaxSpeed(out)));
    }
#pragma unroll
    for (int o = 32; o >= 1; o /= 2) local = fmin(local, __shfl_xor(local, o));
    if ((tid & 63) == 0) FoldMin(a.dt_min_bits, local);
  }
}

// Wavefronts per SIMD to leave room for: what the registers allow without
// spills (whose traffic has cost more than a wavefront every time).
template <int Q>
constexpr int LineWaves() {
  return Q <= 3 || Q == 6 ? 4 : 3;
}

template <int Q, int kRiemann, bool kCurved>
__global__ __launch_bounds__(Shape<Q>::kThreads) __attribute__((amdgpu_waves_per_eu(LineWaves<Q>())))
void FrHexStageKernel(FrHexArgs a, LineTables lt) {
  __shared__ double lds[Shape<Q>::kLdsDoubles];
  int64_t block = LogicalBlock(a.xcd_remap);
  if (a.tile_order) block = a.tile_order[block];
  FrLineBody<Q, kRiemann, kCurved>(a, lt, block, lds);
}

// ------------------------------------------------------------ Q = 4, FP64
// One wavefront per cell: its 64 lanes are the cell's 4^3 nodes, and the 4 x 4
// line operators are v_mfma_f64_4x4x4 (four independent 4 x 4 products): with
// lane = 16 h + 4 m + l,
//   D(h, m, l) = C(h, m, l) + sum_k A(k, m, h) B(k, m, l),
// a fused chain over k = 0..3, where X(k, m, l) is X's value in lane
// 16 k + 4 m + l.  A field F given with the contracted index in h is
// multiplied by a table T as mfma(T^, F), T^(k, m, r) = T[r][k].
__device__ __forceinline__ double Mfma(double a, double b, double c) {
  return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}

constexpr int kCellTile = 4;  // cells of one tile of tile_order
// LDS of the kernel below, in doubles: the cells' states (skewed as Shape<Q>'s)
// and the records of the flux points to come.
template <int kCells>
struct CellShape {
  static constexpr int kState = 5 * 79, kLater = kCells * kState + (kCells & 1);
  static constexpr int kLdsDoubles = kLater + kCells * 2 * 64;
};

// kCells = 1 or 2 cells, c0 and c0 + 1, on one wavefront.  The 32 z flux points
// of a cell fill half a wavefront: two cells share one pass over theirs.
// Against one line per lane at the same size (64^3, Roe): 862 -> 638 us with one
// cell per wavefront.  4 wavefronts per SIMD; 5 gave nothing.
template <int kCells, int kRiemann, bool kCurved>
__device__ __forceinline__ void FrCellBody(const FrHexArgs &a, const LineTables &lt, int64_t c0, double *lds) {
  using S = CellShape<kCells>;
  constexpr int NP = 64, Z = kCells;  // slots 0 .. Z - 1: the cells' x and y faces; slot Z: the z faces
  const int lane = threadIdx.x & 63;
  const int h = lane >> 4, m = (lane >> 2) & 3, l = lane & 3;
  // This lane's flux points.  Slots below Z: x-, x+, y-, y+ in h = 0..3 at in-face
  // (m, l).  Slot Z: z-, z+ of the first cell in h = 0, 1 and of the second in
  // h = 2, 3 (or of the first again), at (l, m).
  const int f_xy = (0x3124 >> (4 * h)) & 7, f_z = (h & 1) ? 5 : 0;
  const int64_t c1 = kCells == 2 && c0 + 1 < a.n_cells ? c0 + 1 : c0;  // an odd last cell is done twice
  // Loads are waited for in the order of their issue: what is needed first, or
  // needed to form an address, goes first.  The cells' geometry is uniform and
  // comes through scalar loads, as long as no store precedes them.
  double geo[kCells][14], dt[kCells];
#pragma unroll
  for (int g = 0; g < kCells; ++g) {
    const int64_t c = g ? c1 : c0;
    const double *src = a.geo + (int64_t)a.geo_id[c] * kGeoStride;
#pragma unroll
    for (int e = 0; e < 14; ++e) geo[g][e] = src[e];
    dt[g] = a.case_dt ? a.case_dt[a.cell_case[c]] : a.dt;
  }
  auto cell_at = [&](int s) -> int64_t { return s == Z ? (h < 2 ? c0 : c1) : (s ? c1 : c0); };
  FrFace face = a.faces[cell_at(Z) * 6 + f_z];
  double u[kCells][5];
  FrFace *const later = reinterpret_cast<FrFace *>(lds + S::kLater);  // the later slots' records wait in LDS
#pragma unroll
  for (int s = 0; s < Z; ++s) later[s * 64 + lane] = a.faces[cell_at(s) * 6 + f_xy];
#pragma unroll
  for (int g = 0; g < kCells; ++g)
#pragma unroll
    for (int k = 0; k < 5; ++k) u[g][k] = a.us[(g ? c1 : c0) * (5 * NP) + k * NP + lane];
  const CellOps *ops = a.cell_ops;

  // the neighbour's line behind flux point s, from its lower end upwards
  struct Line { double v[4][5]; };
  auto gather = [&](int s) {
    Line nb;  // left undefined without a neighbour
    if (face.nbr < 0) return nb;
    const int g = face.gather, step = g >> 24;
    const int first = (g & 255) + (int)(int8_t)(g >> 8) * m + (int)(int8_t)(g >> 16) * l + (step < 0 ? 3 * step : 0);
    const int up = step < 0 ? -step : step;
    const double *src = a.us + (int64_t)face.nbr * (5 * NP) + first;
    if (s == Z && __all(up == 1)) {
#pragma unroll
      for (int k = 0; k < 5; ++k) {
        const double2 lo = *reinterpret_cast<const double2 *>(src + k * NP);
        const double2 hi = *reinterpret_cast<const double2 *>(src + k * NP + 2);
        nb.v[0][k] = lo.x;
        nb.v[1][k] = lo.y;
        nb.v[2][k] = hi.x;
        nb.v[3][k] = hi.y;
      }
      asm volatile("; 16-byte loads" ::: "memory");  // keeps the compiler from merging the two branches' loads
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int k = 0; k < 5; ++k) nb.v[q][k] = src[k * NP + q * up];
    }
    return nb;
  };
  // unit normal (left to right) and face scale of flux point s
  double n[3], scale;
  auto point_of = [&](int s) { return (cell_at(s) * 6 + (s == Z ? f_z : f_xy)) * 16 + (s == Z ? l * 4 + m : m * 4 + l); };
  auto geometry = [&](int s) {
    if constexpr (kCurved) {
      const double *fp = a.face_point + point_of(s) * 4;
#pragma unroll
      for (int d = 0; d < 3; ++d) n[d] = fp[d];
      scale = fp[3];
    } else {
      const double *fp = a.normals + (int64_t)(face.normal >> 1) * kNormalStride;
#pragma unroll
      for (int d = 0; d < 3; ++d) n[d] = fp[d];
      scale = s == Z ? (h < 2 ? geo[0][11] : geo[kCells - 1][11]) : (h < 2 ? geo[s % kCells][3] : geo[s % kCells][7]);
    }
  };
  geometry(Z);
  Line nb = gather(Z);
  // states with j, and with k, in h: (i, k) and (j, i) in (m, l)
  const int at_x = h * 20 + m * 5 + l, at_y = m * 20 + h * 5 + l, at_z = l * 20 + m * 5 + h;
#pragma unroll
  for (int g = 0; g < kCells; ++g)
#pragma unroll
    for (int k = 0; k < 5; ++k) lds[g * S::kState + k * 79 + at_x] = u[g][k];
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  const double end = ops->end[lane];
  // the cell's own traces at its ends
  auto own_trace = [&](int s) {
    State own;
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      const double *const su = lds + (s == Z ? 0 : s) * S::kState + k * 79;
      // selected, not added to the other half's zeros: 0 times a NaN or an infinity
      // there, of another line or even of the other cell, is a NaN
      if (s < Z) {
        const double x = Mfma(end, su[at_x], 0.0), y = Mfma(end, su[at_y], 0.0);
        own.v[k] = h < 2 ? x : y;
      } else if (kCells == 1) {
        own.v[k] = Mfma(end, su[at_z], 0.0);
      } else {
        const double first = Mfma(end, su[at_z], 0.0), second = Mfma(end, su[S::kState + at_z], 0.0);
        own.v[k] = h < 2 ? first : second;
      }
    }
    return own;
  };
  double flux_z[5];
#pragma unroll
  for (int turn = 0; turn <= Z; ++turn) {
    const int s = turn == 0 ? Z : turn - 1;
    State own = own_trace(s);
    Pin(own.v);
    double flux[5];

    // ---- flux points
    const bool upper = (h & 1) != 0;
    const bool swap = (face.normal & 1) != 0, left = upper != swap;
    State other;
    int kind = kBcSmart;
    if (face.nbr >= 0) {
      // the neighbour's trace at the end it has here, in its own order
      const bool lower_end = (face.gather >> 24) > 0;
#pragma unroll
      for (int k = 0; k < 5; ++k) {
        double acc = (lower_end ? lt.end[0] : lt.end[3]) * nb.v[0][k];
#pragma unroll
        for (int q = 1; q < 4; ++q) acc = __fma_rn(lower_end ? lt.end[q] : lt.end[3 - q], nb.v[q][k], acc);
        other.v[k] = acc;
      }
    } else {
      const int tag = -face.nbr - 1;
      kind = a.bc_kind[tag];
      // the tag's constant state, or this point's value of the tag's boundary
      // function at the stage time
      const double *gs = a.bc_point_state
          ? a.bc_point_state + ((int64_t)face.bface * 16 + m * 4 + l) * 5 : a.bc_state + tag * 5;
#pragma unroll
      for (int k = 0; k < 5; ++k) other.v[k] = gs[k];
    }
    if (s == Z) {  // gathered at (m, l), where four lanes share a cache line; wanted at (l, m)
      kind = __shfl(kind, 16 * h + 4 * l + m);
#pragma unroll
      for (int k = 0; k < 5; ++k) other.v[k] = __shfl(other.v[k], 16 * h + 4 * l + m);
    }
    Pin(other.v);
    asm volatile("" ::: "memory");
    const double along = swap ? -scale : scale;
    __builtin_amdgcn_sched_barrier(0);
    // the exact solver's state of this flux point, one copy per side: both
    // sides solve the same problem with the same inputs every pass, so the
    // two copies stay equal
    bool star = kRiemann == kExact ? a.exact_star[point_of(s)] != 0 : false;
    State ls, rs;
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      ls.v[k] = left ? own.v[k] : other.v[k];
      rs.v[k] = left ? other.v[k] : own.v[k];
    }
    State fu;
    if (kind == kBcSmart) fu = FaceFlux<kRiemann>(n, ls, rs, star);
    else fu = BoundaryFlux(kind, left, n, left ? ls : rs, left ? rs : ls);
    if constexpr (kRiemann == kExact) a.exact_star[point_of(s)] = star ? 1 : 0;
    // left-to-right is the +r direction of this cell unless the roles are swapped
#pragma unroll
    for (int k = 0; k < 5; ++k) flux[k] = fu.v[k] * along;
    Pin(flux);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    if (s == Z) {
#pragma unroll
      for (int k = 0; k < 5; ++k) flux_z[k] = flux[k];
      face = later[lane];
      geometry(0);
      nb = gather(0);
      continue;
    }

  // ---- F~_r = F J*.col(r) at the nodes, contracted: x and z into div in the
  // node order, y into divy with j in h; and the fluxes lifted
    const double dg = ops->dg[lane], gp = ops->gp[lane];
    const int g = s;
    const int64_t c = g ? c1 : c0;
    double *const su = lds + g * S::kState;
    double u0[5] = { 0, 0, 0, 0, 0 };
    const double inv_det = kCurved ? a.inv_det_node[c * NP + lane] : geo[g][kGeoInvDet];
    if (a.stage >= 2) {
#pragma unroll
      for (int k = 0; k < 5; ++k) u0[k] = __builtin_nontemporal_load(a.u0 + c * (5 * NP) + k * NP + lane);
    }
    double col[3][3];
    if constexpr (kCurved) {
      const int node[3] = { lane, 16 * m + 4 * h + l, 16 * l + 4 * m + h };
#pragma unroll
      for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int e = 0; e < 3; ++e) col[r][e] = a.col_node[((c * 3 + r) * NP + node[r]) * 3 + e];
    } else {
#pragma unroll
      for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int e = 0; e < 3; ++e) col[r][e] = geo[g][4 * r + e];
    }
    double div[5], divy[5];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      double v[5];
#pragma unroll
      for (int k = 0; k < 5; ++k) v[k] = su[k * 79 + (r == 0 ? at_x : (r == 1 ? at_y : at_z))];
      // contravariant momentum and velocity, and pressure
      const double inv = FiniteRcp(v[0]);
      const double mom = v[1] * col[r][0] + v[2] * col[r][1] + v[3] * col[r][2];
      double vel = mom * inv;
      double p = (v[4] - 0.5 * (v[1] * v[1] + v[2] * v[2] + v[3] * v[3]) * inv) * kGm1;
      if (!__all(v[0] > 0 && v[4] >= 0 && p >= 0)) {  // the zeroing rule of types.hpp:195-202,289-301
        const bool bad = v[0] < 0 || v[4] < 0;
        const bool vacuum = !bad && v[0] == 0;
        const bool zero = bad || (!vacuum && p < 0);
        vel = zero ? 0.0 : (vacuum ? mom : vel);
        p = zero ? 0.0 : (vacuum ? v[4] : p);
      }
#pragma unroll
      for (int k = 0; k < 5; ++k) {
        const double fk = k == 0 ? mom : (k == 4 ? (v[4] + p) * vel : v[k] * vel + p * col[r][k == 0 ? 0 : k - 1]);
        // the fluxes of this direction, or in z of this cell: see own_trace
        if (r == 0) div[k] = Mfma(gp, h < 2 ? flux[k] : 0.0, Mfma(dg, fk, 0.0));
        else if (r == 1) divy[k] = Mfma(gp, h < 2 ? 0.0 : flux[k], Mfma(dg, fk, 0.0));
        else div[k] = Mfma((h < 2) == (g == 0) ? flux_z[k] : 0.0, gp, Mfma(fk, dg, div[k]));
      }
    }

    double uc[5];
    // y's part to the node order; 1/det(J), RK stage, store
#pragma unroll
    for (int k = 0; k < 5; ++k) uc[k] = su[k * 79 + at_x];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int k = 0; k < 5; ++k) su[k * 79 + at_y] = divy[k];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    State out;
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      const double sum = div[k] + su[k * 79 + at_x];
      out.v[k] = fr::RkOutput(a.stage, -sum * inv_det, uc[k], u0[k], dt[g]);
    }
    // An odd last cell's second turn is worth nothing: stage 3 has written over its
    // U0.  (Left out by a branch ahead of it, the solvers' other kernels spill.)
    const bool real = g == 0 || c1 != c0;
    if (real) {
      // the residual is handed out as a column, states stay in planes; streamed,
      // so that the states which neighbours still gather keep the L2
      const int64_t to = a.stage == 0 ? (c * NP + lane) * 5 : c * (5 * NP) + lane;
      const int step = a.stage == 0 ? 1 : NP;
#pragma unroll
      for (int k = 0; k < 5; ++k) __builtin_nontemporal_store(out.v[k], a.out + to + k * step);
    }
    if (a.dt_min_bits && real) {
      // fem.hpp:412-435 on the state just written, as FrHexTimeStepKernel: min
      // over cells of length / max(1e-5, max over nodes of |u| + c); the bits of
      // positive doubles order as the doubles do
      double v = fmax(1e-5, MaxSpeed(out));
#pragma unroll
      for (int o = 32; o >= 1; o /= 2) v = fmax(v, __shfl_xor(v, o));
      if (lane == 0) FoldMin(a.dt_min_bits, geo[g][kGeoLength] / v);
    }
    if (turn < Z) {
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      face = later[(s + 1) * 64 + lane];
      geometry(s + 1);
      nb = gather(s + 1);
    }
  }
}

template <int kCells, int kRiemann, bool kCurved>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4)))
void FrHexCellKernel(FrHexArgs a, LineTables lt) {
  __shared__ __attribute__((aligned(16))) double lds[CellShape<kCells>::kLdsDoubles];
  constexpr int kPerTile = kCellTile / kCells;
  const int64_t block = LogicalBlock(a.xcd_remap);
  const int64_t tile = a.tile_order ? a.tile_order[block / kPerTile] : block / kPerTile;
  const int64_t c = tile * kCellTile + block % kPerTile * kCells;
  if (c >= a.n_cells) return;
  FrCellBody<kCells, kRiemann, kCurved>(a, lt, c, lds);
}

// Tile variants of the persistent batched launch: a work item is 1, 2 or 4
// consecutive blocks of BatchCells(q) cells.
constexpr int TileBlocks(int tile) { return 1 << tile; }
constexpr int kBatchThreads = Shape<3>::kThreads, kBatchWaves = kBatchThreads / 64;
static_assert(Shape<2>::kThreads == kBatchThreads, "one workgroup size for all degrees");
constexpr int BatchCells(int q) { return q == 2 ? Shape<2>::kCells : (q == 3 ? Shape<3>::kCells : kBatchWaves); }

// One out-of-line body per Q: each is register-allocated on its own within the
// kernel's budget, where the inlined bodies would share one allocation.  The same
// bodies as in the launches per degree group, so that both forms give the same
// bits: at Q = 4 a cell to each wavefront.  256 tubes, ms per step: 11.2 (11.5 with
// lines at Q = 4 too), 3.9 per degree group, as calls spill their callee's registers.
template <int Q, int kRiemann>
__device__ __noinline__ void BatchBody(const FrHexBatchGroup *g, int64_t block, double *lds) {
  if constexpr (Q == 4) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t c = block * kBatchWaves + wave;
    if (c < g->args.n_cells)
      FrCellBody<1, kRiemann, false>(g->args, g->lt, c, lds + wave * CellShape<1>::kLdsDoubles);
  } else {
    FrLineBody<Q, kRiemann, false>(g->args, g->lt, block, lds);
  }
}

// Persistent batched pass: workgroup w processes the contiguous item range
// [w * n_items / W, (w + 1) * n_items / W) of the work list (blocks of all
// degree groups in order), so consecutive blocks -- and their neighbour
// cells -- stay in one XCD's L2.  LDS is sized at launch for the largest block
// in use.
template <int kRiemann>
__global__ __launch_bounds__(kBatchThreads) __attribute__((amdgpu_waves_per_eu(3))) void FrHexBatchKernel(FrHexBatchArgs b) {
  extern __shared__ __attribute__((aligned(16))) double lds[];
  const int64_t w = blockIdx.x, nw = gridDim.x;
  const int64_t begin = w * b.n_items / nw, end = (w + 1) * b.n_items / nw;
  int gi = 0;
  for (int64_t item = begin; item < end; ++item) {
    // the group table lives in device memory and gi is uniform, so every
    // field is fetched with scalar loads
    while (gi + 1 < b.n_groups && item >= b.group[gi + 1].first_item) ++gi;
    const FrHexBatchGroup &g = b.group[gi];
    const int blocks = TileBlocks(g.tile);
    for (int v = 0; v < blocks; ++v) {
      const int64_t block = (item - g.first_item) * blocks + v;
      switch (g.q) {
      case 2: BatchBody<2, kRiemann>(&g, block, lds); break;
      case 3: BatchBody<3, kRiemann>(&g, block, lds); break;
      default: BatchBody<4, kRiemann>(&g, block, lds); break;
      }
      __syncthreads();  // the next block reuses the LDS buffers
    }
  }
}

// Column layout [cell][node][5] <-> the kernels' planes [cell][5][node], one
// thread per value of the planes (several above 2^30 values: a launch holds 2^32
// threads at most).
template <bool kToPlanes>
__global__ __launch_bounds__(256) void FrLayoutKernel(const double *in, double *out, int np, int64_t n) {
  for (int64_t w = (int64_t)blockIdx.x * 256 + threadIdx.x; w < n; w += (int64_t)gridDim.x * 256) {
    const int64_t c = w / (5 * np);
    const int r = (int)(w - c * (5 * np)), k = r / np, node = r - k * np;
    const int64_t col = (c * np + node) * 5 + k;
    if constexpr (kToPlanes) out[w] = in[col];
    else out[col] = in[w];
  }
}

__global__ void ResetTimeStepBitsKernel(unsigned long long *bits) {
  *bits = (unsigned long long)__double_as_longlong(1e300);
}

// fem.hpp:412-435: min over cells of length / max(1e-5, max over nodes of |u| + c),
// which is the min over nodes of length / max(1e-5, |u| + c).  Bound by the read of
// the states: consecutive lanes take consecutive nodes of the planes (a cell per
// lane, as for columns, reads lines 5 Q^3 doubles apart: 64^3 p3 1480 us, traced).  The
// call, us: 64^3 p3 180, 32^3 p4 100, 8^3 p3 27.
template <int Q>
__global__ __launch_bounds__(256) void FrHexTimeStepKernel(const double *u, const int32_t *geo_id,
    const double *geo, int64_t n_cells, unsigned long long *dt_min_bits) {
  constexpr int NP = Q * Q * Q;
  double local = 1e300;
  for (int64_t w = (int64_t)blockIdx.x * 256 + threadIdx.x; w < n_cells * NP; w += (int64_t)gridDim.x * 256) {
    const int64_t c = w / NP;
    const double *uc = u + c * (4 * NP) + w;
    State s;
#pragma unroll
    for (int k = 0; k < 5; ++k) s.v[k] = uc[k * NP];
    local = fmin(local, geo[(int64_t)geo_id[c] * kGeoStride + kGeoLength] / fmax(1e-5, MaxSpeed(s)));
  }
#pragma unroll
  for (int o = 32; o >= 1; o /= 2) local = fmin(local, __shfl_xor(local, o));
  if ((threadIdx.x & 63) == 0) FoldMin(dt_min_bits, local);
}

// Q = 4: two cells per wavefront save a quarter of the flux points' lanes but
// halve the wavefronts, so a mesh that does not fill the chip with one cell per
// wavefront (256 CUs, 16 wavefronts each) is better served that way.  Measured,
// one against two cells, us per pass: 12^3 11.1 / 12.6, 16^3 16.4 / 16.7, 18^3
// 21.5 / 21.0, 20^3 26.9 / 25.5, 32^3 90.5 / 84.5, 64^3 638 / 595.
constexpr int64_t kPairCells = 4096;

template <int Q, int R>
hipError_t Launch(const FrHexArgs &args, const LineTables &lt, hipStream_t stream) {
  constexpr int C = Q == 4 ? kCellTile : Shape<Q>::kCells;
  const int64_t blocks = (args.n_cells + C - 1) / C;
  if (blocks > 0x7fffffff) return hipErrorInvalidValue;
  if constexpr (Q == 4) {
    if (blocks * C > 0x7fffffff || !args.cell_ops) return hipErrorInvalidValue;
    const bool pair = args.n_cells > kPairCells;
    const dim3 cells((unsigned)(blocks * (pair ? C / 2 : C))), wave(64);
    if (pair) {
      if (args.curved) hipLaunchKernelGGL((FrHexCellKernel<2, R, true>), cells, wave, 0, stream, args, lt);
      else hipLaunchKernelGGL((FrHexCellKernel<2, R, false>), cells, wave, 0, stream, args, lt);
    } else {
      if (args.curved) hipLaunchKernelGGL((FrHexCellKernel<1, R, true>), cells, wave, 0, stream, args, lt);
      else hipLaunchKernelGGL((FrHexCellKernel<1, R, false>), cells, wave, 0, stream, args, lt);
    }
  } else {
    const dim3 grid((unsigned)blocks), block(Shape<Q>::kThreads);
    if (args.curved) hipLaunchKernelGGL((FrHexStageKernel<Q, R, true>), grid, block, 0, stream, args, lt);
    else hipLaunchKernelGGL((FrHexStageKernel<Q, R, false>), grid, block, 0, stream, args, lt);
  }
  return hipGetLastError();
}

template <int Q>
hipError_t LaunchQ(int riemann, const FrHexArgs &args, const LineTables &lt, hipStream_t stream) {
  switch (riemann) {
  case kExact: return Launch<Q, kExact>(args, lt, stream);
  case kHllc: return Launch<Q, kHllc>(args, lt, stream);
  case kRoe: return Launch<Q, kRoe>(args, lt, stream);
  default: return hipErrorInvalidValue;
  }
}

}  // namespace

hipError_t LaunchFrHexStage(int q, int riemann, const FrHexArgs &args, const LineTables &lt, const MixedTables &mt,
                            hipStream_t stream) {
  if (args.curved && args.mixed) return hipErrorInvalidValue;
  if (args.mixed) return LaunchFrMixedStage(q, riemann, args, mt, stream);
  switch (q) {
  case 2: return LaunchQ<2>(riemann, args, lt, stream);
  case 3: return LaunchQ<3>(riemann, args, lt, stream);
  case 4: return LaunchQ<4>(riemann, args, lt, stream);
  case 5: return LaunchQ<5>(riemann, args, lt, stream);
  case 6: return LaunchQ<6>(riemann, args, lt, stream);
  default: return hipErrorInvalidValue;
  }
}

int FrHexStageTileCells(int q, bool mixed) {
  if (mixed) return FrMixedStageTileCells(q);
  switch (q) {
  case 2: return Shape<2>::kCells;
  case 3: return Shape<3>::kCells;
  case 4: return kCellTile;
  case 5: return Shape<5>::kCells;
  case 6: return Shape<6>::kCells;
  default: return 0;
  }
}

int FrHexTileLdsBytes(int q, int tile, bool mixed) {
  if (mixed) return FrMixedTileLdsBytes(q, tile);
  if (q < 2 || q > 4 || tile < 0 || tile > 2) return 0;
  return (int)sizeof(double) * (q == 2 ? Shape<2>::kLdsDoubles
                                       : (q == 3 ? Shape<3>::kLdsDoubles : kBatchWaves * CellShape<1>::kLdsDoubles));
}

int FrHexTileCells(int q, int tile, bool mixed) {
  if (mixed) return FrMixedTileCells(q, tile);
  if (q < 2 || q > 4 || tile < 0 || tile > 2) return 0;
  return BatchCells(q) * TileBlocks(tile);
}

hipError_t LaunchFrHexBatch(int riemann, bool mixed, const FrHexBatchArgs &args, int n_workgroups,
                            hipStream_t stream) {
  if (mixed) return LaunchFrMixedBatch(riemann, args, n_workgroups, stream);
  if (args.n_groups < 1 || args.n_groups > kMaxBatchGroups || n_workgroups < 1) return hipErrorInvalidValue;
  const dim3 grid((unsigned)n_workgroups), block(kBatchThreads);
  const size_t lds = (size_t)args.max_tile_lds;
  switch (riemann) {
  case kExact: hipLaunchKernelGGL(FrHexBatchKernel<kExact>, grid, block, lds, stream, args); break;
  case kHllc: hipLaunchKernelGGL(FrHexBatchKernel<kHllc>, grid, block, lds, stream, args); break;
  case kRoe: hipLaunchKernelGGL(FrHexBatchKernel<kRoe>, grid, block, lds, stream, args); break;
  default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

int FrHexBatchResidentWorkgroups(int riemann, bool mixed, int lds_bytes) {
  int per_cu = 0;
  hipError_t e = hipErrorInvalidValue;
  if (mixed) e = FrMixedBatchResident(riemann, lds_bytes, &per_cu);
  else if (riemann == kExact) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, FrHexBatchKernel<kExact>, kBatchThreads, lds_bytes);
  else if (riemann == kHllc) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, FrHexBatchKernel<kHllc>, kBatchThreads, lds_bytes);
  else if (riemann == kRoe) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, FrHexBatchKernel<kRoe>, kBatchThreads, lds_bytes);
  int dev = 0, cus = 0;
  if (e != hipSuccess || hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return 0;
  return std::max(1, per_cu) * cus;
}

hipError_t LaunchFrLayout(bool to_planes, const double *in, double *out, int np, int64_t n_cells, hipStream_t stream) {
  const int64_t n = n_cells * np * 5, blocks = std::min<int64_t>((n + 255) / 256, int64_t(1) << 22);
  if (blocks < 1) return hipSuccess;
  if (to_planes) {
    hipLaunchKernelGGL(FrLayoutKernel<true>, dim3((unsigned)blocks), dim3(256), 0, stream, in, out, np, n);
  } else {
    hipLaunchKernelGGL(FrLayoutKernel<false>, dim3((unsigned)blocks), dim3(256), 0, stream, in, out, np, n);
  }
  return hipGetLastError();
}

hipError_t LaunchResetTimeStepBits(unsigned long long *bits, hipStream_t stream) {
  hipLaunchKernelGGL(ResetTimeStepBitsKernel, dim3(1), dim3(1), 0, stream, bits);
  return hipGetLastError();
}

hipError_t LaunchFrHexTimeStep(int q, bool mixed, const double *u, const int32_t *geo_id, const double *geo,
                               int64_t n_cells, unsigned long long *dt_min_bits, hipStream_t stream) {
  if (mixed) return LaunchFrMixedTimeStep(q, u, geo_id, geo, n_cells, dt_min_bits, stream);
  // four nodes per thread, up to two rounds of wavefronts
  int64_t blocks = std::min<int64_t>((n_cells * q * q * q + 1023) / 1024, 4096);
  if (blocks < 1) blocks = 1;
  switch (q) {
#define MCFD_TS_CASE(QQ) \
  case QQ: hipLaunchKernelGGL((FrHexTimeStepKernel<QQ>), dim3((unsigned)blocks), dim3(256), 0, stream, \
                              u, geo_id, geo, n_cells, dt_min_bits); break;
  MCFD_TS_CASE(2) MCFD_TS_CASE(3) MCFD_TS_CASE(4) MCFD_TS_CASE(5) MCFD_TS_CASE(6)
#undef MCFD_TS_CASE
  default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace mcfd
