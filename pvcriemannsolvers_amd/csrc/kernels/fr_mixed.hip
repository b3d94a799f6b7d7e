// The mixed-precision form of nodal flux reconstruction on affine hexahedra
// (gfx950), on columns [cell][node][5].
//
// The FP32 deviations of this form amplify a last-bit difference anywhere in the
// FP64 arithmetic: one rounding that falls the other way moves its neighbours'
// roundings, and within some tens of steps the whole field differs by the form's
// own error, 1e-9 to 1e-8 (5 x 7 x 5 cells p = 3, 36 steps: 2.9e-9 between this
// kernel and the line kernel of fr_hex.hip contracting in FP32, each 1.1e-8 from
// 64 bits).  Results are kept by keeping the operations: frames, traces, gaps
// and sums are formed here in one order, apart from the FP64 kernels.  The line
// kernel with FP32 sums was faster (us per stage, here / there: 48^3 p = 3 402 / 314,
// 36^3 p = 4 368 / 296) and is left out for that difference.
//
// One pass = residual of spatial/fr/general.hpp (volume term :271-288, face
// correction :296-315,409-434, boundary corrections :435-640, det(J) scaling
// :249-268) fused with one SSP-RK3 stage of temporal/rk.hpp:31-49.
//
// Work decomposition: a 256-thread workgroup owns C consecutive cells.  Each
// pass
//   0. loads the cells' states (one thread per solution point) and keeps a
//      skewed structure-of-arrays copy in LDS;
//   1. the three columns of F~ = F J* go through LDS (Q >= 3: all three in
//      one round behind one barrier, while the first face task's neighbour
//      line is already in flight; Q = 2: one column per round), every
//      solution point accumulates its sum-factorised Q-point derivatives
//      and every flux point extrapolates its direction's column to the face;
//   2. per flux point of the cells' 6 faces: own trace (LDS), neighbour trace
//      (the neighbour's line of Q points, gathered through L2), upwind flux
//      and flux gap.  Each interior face is solved by both of its cells with
//      bit-identical inputs, so the scheme stays conservative without
//      atomics or a separate face pass;
//   3. per solution point: lifted gaps, 1/det(J), RK stage in the
//      reference's operation order, store.
// The same body serves the single-mesh launch and the persistent batched
// launch that walks a work list spanning several polynomial degrees.
#include "fr_mixed.hpp"

#include <algorithm>

#include "euler.hpp"
#include "fr_common.hpp"

namespace mcfd {

namespace {

using fr::LogicalBlock;

// Line of solution points through in-face point (a, b) of local face f:
// node(m) = a * A + b * B + m * S.  Branch-free for lane-varying f.
struct LineIndex { int a_mul, b_mul, stride, side, dir; };
__device__ __forceinline__ LineIndex FaceLineIndex(int q, int f) {
  const int dir = (2118 >> (2 * f)) & 3;  // {2, 1, 0, 1, 0, 2}
  const int side = (0x2C >> f) & 1;       // {0, 0, 1, 1, 0, 1}
  LineIndex li;
  li.dir = dir;
  li.side = side;
  li.a_mul = dir == 0 ? q : q * q;
  li.b_mul = dir == 2 ? q : 1;
  li.stride = dir == 0 ? q * q : (dir == 1 ? q : 1);
  return li;
}
// The same line in the skewed LDS layout of Shape<Q>.
template <int Q>
__device__ __forceinline__ LineIndex SkewedLineIndex(int f) {
  constexpr int SI = Q * (Q + 1), SJ = Q + 1;
  const int dir = (2118 >> (2 * f)) & 3;
  LineIndex li;
  li.dir = dir;
  li.side = (0x2C >> f) & 1;
  li.a_mul = dir == 0 ? SJ : SI;
  li.b_mul = dir == 2 ? SJ : 1;
  li.stride = dir == 0 ? SI : (dir == 1 ? SJ : 1);
  return li;
}

// Extrapolation to a line end: a fixed-order fused chain so that both cells of
// a face evaluate a given trace with identical rounding.
template <int Q>
__device__ __forceinline__ double Extrapolate(const double *w, const double *v) {
  double acc = w[0] * v[0];
#pragma unroll
  for (int m = 1; m < Q; ++m) acc = __fma_rn(w[m], v[m], acc);
  return acc;
}

// Column d of the local flux F~ = F J* at one solution point.
template <bool kDiag>
__device__ __forceinline__ void LocalFluxColumn(State const &c, State const &p, const double *js, int d,
                                                double *out) {
  const double rh = c.v[4] + p.v[4];
  if constexpr (kDiag) {
    const double vel = p.v[1 + d], s = js[4 * d];
    out[0] = c.v[1 + d] * s;
    out[1] = (c.v[1] * vel + (d == 0 ? p.v[4] : 0.0)) * s;
    out[2] = (c.v[2] * vel + (d == 1 ? p.v[4] : 0.0)) * s;
    out[3] = (c.v[3] * vel + (d == 2 ? p.v[4] : 0.0)) * s;
    out[4] = rh * vel * s;
  } else {
#pragma unroll
    for (int k = 0; k < 5; ++k) out[k] = 0;
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      const double vel = p.v[1 + e], s = js[3 * e + d];
      out[0] += c.v[1 + e] * s;
      out[1] += (c.v[1] * vel + (e == 0 ? p.v[4] : 0.0)) * s;
      out[2] += (c.v[2] * vel + (e == 1 ? p.v[4] : 0.0)) * s;
      out[3] += (c.v[3] * vel + (e == 2 ? p.v[4] : 0.0)) * s;
      out[4] += rh * vel * s;
    }
  }
}

// Lifted flux gaps at solution point (ni, nj, nk) (fr/general.hpp:409-434):
// the six faces' gaps times the Vincent derivatives g', summed in a fixed
// order.  g holds one component's gaps face-major, g[f * Q^2 + a * Q + b].
template <int Q>
__device__ __forceinline__ double LiftedGaps(const double *g, const MixedTables &lt, int ni, int nj, int nk) {
  constexpr int NFP = Q * Q;
  double c = g[5 * NFP + ni * Q + nj] * lt.gp[1][nk];
  c = __fma_rn(g[0 * NFP + ni * Q + nj], lt.gp[0][nk], c);
  c = __fma_rn(g[1 * NFP + ni * Q + nk], lt.gp[0][nj], c);
  c = __fma_rn(g[3 * NFP + ni * Q + nk], lt.gp[1][nj], c);
  c = __fma_rn(g[4 * NFP + nj * Q + nk], lt.gp[0][ni], c);
  return __fma_rn(g[2 * NFP + nj * Q + nk], lt.gp[1][ni], c);
}

// Conservative -> primitive with the reference's zeroing rule
// (types.hpp:195-202,289-301) via one reciprocal of rho.  The plain
// arithmetic is done first; the rule only selects among its results, so
// a wavefront where no lane needs the rule (rho > 0, E >= 0, p >= 0 on every
// lane) skips the selects and gets bitwise the same values as one that
// applies them.  *inv_rho receives FiniteRcp of the returned density.
__device__ __forceinline__ State FastPrimitive(State const &c, double *inv_rho) {
  const double rho = c.v[0];
  const double inv = FiniteRcp(rho);
  State p;
  p.v[0] = rho;
  p.v[1] = c.v[1] * inv;
  p.v[2] = c.v[2] * inv;
  p.v[3] = c.v[3] * inv;
  const double ke = 0.5 * (p.v[1] * p.v[1] + p.v[2] * p.v[2] + p.v[3] * p.v[3]);
  p.v[4] = (c.v[4] - rho * ke) * kGm1;
  *inv_rho = inv;
  if (__all(rho > 0 && c.v[4] >= 0 && p.v[4] >= 0)) return p;
  // rho < 0 or E < 0: all zero; rho == 0: momenta and E kept as they are;
  // otherwise p < 0: all zero
  const bool bad = c.v[0] < 0 || c.v[4] < 0;
  const bool vacuum = !bad && c.v[0] == 0;
  const bool zero = bad || (!vacuum && p.v[4] < 0);
#pragma unroll
  for (int k = 1; k < 5; ++k) p.v[k] = zero ? 0.0 : (vacuum ? c.v[k] : p.v[k]);
  p.v[0] = zero ? 0.0 : rho;  // a vacuum keeps its signed zero
  if (zero || vacuum) *inv_rho = FiniteRcp(p.v[0]);
  return p;
}
__device__ __forceinline__ State FastPrimitive(State const &c) {
  double inv;
  return FastPrimitive(c, &inv);
}

// Roe flux of normal-frame primitives (same waves as RoeFlux) with
// reciprocals instead of divisions; inv_l, inv_r = FiniteRcp of the densities.
__device__ __forceinline__ State FastRoeFlux(State const &l, State const &r, double inv_l, double inv_r) {
  constexpr double kGoGm1 = kGamma / kGm1;
  double kel = 0.5 * (l.v[1] * l.v[1] + l.v[2] * l.v[2] + l.v[3] * l.v[3]);
  double ker = 0.5 * (r.v[1] * r.v[1] + r.v[2] * r.v[2] + r.v[3] * r.v[3]);
  double el = l.v[4] * (1 / kGm1) + l.v[0] * kel;  // total energy per volume
  double er = r.v[4] * (1 / kGm1) + r.v[0] * ker;
  State flux;
  flux.v[0] = 0.5 * (l.v[0] * l.v[1] + r.v[0] * r.v[1]);
  flux.v[1] = 0.5 * ((l.v[0] * l.v[1]) * l.v[1] + l.v[4] + (r.v[0] * r.v[1]) * r.v[1] + r.v[4]);
  flux.v[2] = 0.5 * ((l.v[0] * l.v[2]) * l.v[1] + (r.v[0] * r.v[2]) * r.v[1]);
  flux.v[3] = 0.5 * ((l.v[0] * l.v[3]) * l.v[1] + (r.v[0] * r.v[3]) * r.v[1]);
  flux.v[4] = 0.5 * ((el + l.v[4]) * l.v[1] + (er + r.v[4]) * r.v[1]);
  double sl = sqrt(l.v[0]), sr = sqrt(r.v[0]);
  double inv = FiniteRcp(sl + sr);
  double h0l = l.v[4] * inv_l * kGoGm1 + kel;
  double h0r = r.v[4] * inv_r * kGoGm1 + ker;
  double rho = sl * sr;
  double u = (sl * l.v[1] + sr * r.v[1]) * inv;
  double v = (sl * l.v[2] + sr * r.v[2]) * inv;
  double w = (sl * l.v[3] + sr * r.v[3]) * inv;
  double h = (sl * h0l + sr * h0r) * inv;
  double ke = (u * u + v * v + w * w) * 0.5;
  double aa = kGm1 * (h - ke);
  double a = sqrt(aa), ua = u * a, inv_aa = FiniteRcp(aa);
  double dp = r.v[4] - l.v[4], du = r.v[1] - l.v[1];
  double s1 = 0.25 * (dp - rho * a * du) * inv_aa * fabs(u - a);
  double s2 = 0.5 * ((r.v[0] - l.v[0]) - dp * inv_aa) * fabs(u);
  double s3 = 0.5 * (rho * (r.v[2] - l.v[2])) * fabs(u);
  double s4 = 0.5 * (rho * (r.v[3] - l.v[3])) * fabs(u);
  double s5 = 0.25 * (dp + rho * a * du) * inv_aa * fabs(u + a);
  flux.v[0] -= s1 + s2 + s5;
  flux.v[1] -= s1 * (u - a) + s2 * u + s5 * (u + a);
  flux.v[2] -= (s1 + s2 + s5) * v + s3;
  flux.v[3] -= (s1 + s2 + s5) * w + s4;
  flux.v[4] -= s1 * (h - ua) + s2 * ke + s3 * v + s4 * w + s5 * (h + ua);
  return flux;
}

// The upwind flux, in the rotated frame: Roe on primitives
// recovered with one reciprocal of rho per side (FastPrimitive, FastRoeFlux),
// the other solvers as UpwindFlux.
template <int kRiemann>
__device__ __forceinline__ State FrameFlux(FaceFrame const &f, State const &cl, State const &cr, bool &star) {
  if constexpr (kRiemann == kRoe) {
    double inv_l, inv_r;
    State l = FastPrimitive(cl, &inv_l), r = FastPrimitive(cr, &inv_r);
    GlobalToNormal(f, &l);
    GlobalToNormal(f, &r);
    State flux = FastRoeFlux(l, r, inv_l, inv_r);
    NormalToGlobal(f, &flux);
    return flux;
  } else {
    return UpwindFlux<kRiemann>(f, cl, cr, star);
  }
}

template <int Q, int Cells = 256 / (Q * Q * Q), int Threads = 256, bool OneRound = false>
struct Shape {
  static constexpr int kPoints = Q * Q * Q;        // solution points per cell
  static constexpr int kFacePoints = Q * Q;        // flux points per face
  static constexpr int kFaceTasks = 6 * Q * Q;     // flux points per cell
  static constexpr int kCells = Cells;             // cells per workgroup
  static constexpr int kThreads = Threads;         // workgroup size
  static_assert(Cells * Q * Q * Q <= Threads, "one thread per solution point");
  static_assert(Threads % 64 == 0 && Threads <= 1024, "whole wavefronts");
  // Skewed LDS position of solution point (i, j, k): i * kSI + j * kSJ + k.
  // With kSJ = Q + 1 and kSI = Q (Q + 1) the Q x Q points of any line family
  // read by one wavefront fall in distinct LDS banks (Q = 4: 20 i + 5 j + k).
  static constexpr int kSJ = Q + 1;
  static constexpr int kSI = Q * (Q + 1);
  static constexpr int kSpan = (Q - 1) * (kSI + kSJ + 1) + 1;
  static constexpr int kPad = kSpan | 1;           // odd row stride per component
  static constexpr int kFacePad = kFaceTasks + 1;
  // per cell: the F~ column(s) in flight (one direction, or all three with
  // OneRound), later the flux gaps
  static constexpr int kColumns = (OneRound ? 15 : 5) * kPad;
  static constexpr int kScratch = kColumns > 5 * kFacePad ? kColumns : 5 * kFacePad;
  static constexpr int kTasks = (kCells * kFaceTasks + Threads - 1) / Threads;  // per thread
  static_assert(kCells >= 1, "at most one workgroup of solution points per cell");
  // states, F~ columns / flux gaps, mixed reference values, face area scales
  static constexpr int kLdsDoubles = kCells * 5 * kPad + kCells * kScratch + kCells * 15 + kCells * 6;
};

// The F~ columns cross LDS as FP32 deviations from the cell's first
// solution point and are contracted with FP32 FMAs (each row of the
// derivative matrix sums to zero, so the FP64 reference value drops out of
// the divergence); each direction's FP32 partial is accumulated in FP64.
// States, pressure recovery, traces, the Riemann solve, the flux gaps and
// the RK combination stay FP64.
//
// kOneRound: all three F~ columns cross LDS in one round (three times the
// column space; one barrier instead of six, two in the mixed form); the
// arithmetic and its order are those of the three-round form, so both give
// bitwise the same results.  kPrefetch (with kOneRound): the neighbour lines
// of that many face-task slots are loaded before the passes.
template <int Q, int Cells, int Threads, int kRiemann, bool kDiag, bool kOneRound = false,
          int kPrefetch = 0>
__device__ __forceinline__ void FrMixedStageBody(const FrHexArgs &a, const MixedTables &lt, int64_t block,
                                               double *lds) {
  using S = Shape<Q, Cells, Threads, kOneRound>;
  constexpr int NP = S::kPoints, NFP = S::kFacePoints, C = S::kCells;
  constexpr int PAD = S::kPad, FPAD = S::kFacePad, T = S::kTasks;
  double *s_u = lds;                          // states, SoA per cell
  double *s_x = lds + C * 5 * PAD;            // F~ column per pass, then flux gaps
  double *s_ref = s_x + C * S::kScratch;      // mixed: FP64 column values at node 0, [d][cell][5]
  double *s_scale = s_ref + C * 15;           // signed face area scales of each cell
  float *s_x32 = reinterpret_cast<float *>(s_x);

  const int tid = threadIdx.x;
  const int64_t c0 = block * C;
  if (c0 >= a.n_cells) return;
  const int nc = (int)min<int64_t>(C, a.n_cells - c0);
  const int64_t base = c0 * NP * 5;

  // ---- node phase: load, primitive, SoA copy of the state
  const bool node_active = tid < nc * NP;
  const int ncell = tid / NP, node = tid - (tid / NP) * NP;
  const int ni = node / (Q * Q), nj = (node / Q) % Q, nk = node % Q;
  const int spos = ni * S::kSI + nj * S::kSJ + nk;  // skewed LDS position
  State cu, pu;
  double u0v[5] = { 0, 0, 0, 0, 0 };
  const double *js = nullptr;
  double inv_det = 0;
  if (node_active) {
#pragma unroll
    for (int k = 0; k < 5; ++k) cu.v[k] = a.us[base + tid * 5 + k];
    pu = FastPrimitive(cu);
    if (a.stage >= 2) {  // U0 of the RK combination, fetched early
#pragma unroll
      for (int k = 0; k < 5; ++k) u0v[k] = a.u0[base + tid * 5 + k];
    }
    js = a.geo + (int64_t)a.geo_id[c0 + ncell] * kMixedGeoStride;
    if (node < 6) s_scale[ncell * 6 + node] = js[10 + node];
    inv_det = js[9];
#pragma unroll
    for (int k = 0; k < 5; ++k) s_u[(ncell * 5 + k) * PAD + spos] = cu.v[k];
  }

  // ---- face task bookkeeping (flux points of the workgroup's cells)
  // Tasks are numbered direction-major: w = ((d * C + cell) * 2 + side) * Q^2
  // + a * Q + b covers the two faces normal to reference direction d.  A
  // wavefront then holds flux points of one direction (of at most two where
  // C * 2 Q^2 is not a multiple of 64), so the extrapolation of pass d runs
  // only in the wavefronts that own direction d instead of in all of them.
  constexpr int PER_DIR = C * 2 * NFP;
  int t_cell[T], t_f[T], t_a[T], t_b[T];
  bool t_on[T];
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const int w = tid + Threads * t;
    const int d = w / PER_DIR, rd = w - d * PER_DIR;
    const int cell = rd / (2 * NFP), rc = rd - cell * (2 * NFP);
    const int side = rc / NFP, fp = rc - side * NFP;
    t_on[t] = d < 3 && cell < nc;
    t_cell[t] = cell;
    // local face of (direction, side): x {4, 2}, y {1, 3}, z {0, 5}
    t_f[t] = d == 0 ? (side ? 2 : 4) : (d == 1 ? (side ? 3 : 1) : (side ? 5 : 0));
    t_a[t] = fp / Q;
    t_b[t] = fp - (fp / Q) * Q;
  }
  // neighbour and face-info words of the face tasks, fetched before the
  // volume passes so that the face phase starts its gathers at once
  int32_t t_nb[T], t_info[T];
#pragma unroll
  for (int t = 0; t < T; ++t) {
    t_nb[t] = t_on[t] ? a.nbr[(c0 + t_cell[t]) * 6 + t_f[t]] : 0;
    t_info[t] = t_on[t] ? a.finfo[(c0 + t_cell[t]) * 6 + t_f[t]] : 0;
  }
  double fn[T][5];

  // mixed: node 0 of each cell publishes its three F~ columns, the FP64
  // references of the FP32 deviations; the first pass's barrier orders them
  {
    if (node_active && node == 0) {
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        double col[5];
        LocalFluxColumn<kDiag>(cu, pu, js, d, col);
#pragma unroll
        for (int k = 0; k < 5; ++k) s_ref[(d * C + ncell) * 5 + k] = col[k];
      }
    }
  }

  // neighbour line of face task t (Q nodes of the neighbour cell along the
  // face normal, in the orientation of this cell's flux point)
  auto gather = [&](int t, double (*raw)[5]) {
    const int32_t nb = t_nb[t], info = t_info[t];
    const int ia = t_a[t], ib = t_b[t];
    const int nf = info & 7, orient = (info >> 3) & 7;
    const int s = (orient & 1) ? ib : ia, tt = (orient & 1) ? ia : ib;
    const int na = (orient & 2) ? Q - 1 - s : s;
    const int nbb = (orient & 4) ? Q - 1 - tt : tt;
    const LineIndex ln = FaceLineIndex(Q, nf);
    const double *src = a.us + ((int64_t)nb * NP + na * ln.a_mul + nbb * ln.b_mul) * 5;
#pragma unroll
    for (int m = 0; m < Q; ++m)
#pragma unroll
      for (int k = 0; k < 5; ++k) raw[m][k] = src[m * ln.stride * 5 + k];
  };
  constexpr int PF = kPrefetch < T ? kPrefetch : T;
  double pre[PF > 0 ? PF : 1][Q][5];

  // ---- three passes: one column of F~ at a time through LDS (or all three
  // written at once with kOneRound)
  double div[5] = { 0, 0, 0, 0, 0 };
  if constexpr (kOneRound) {
    __syncthreads();  // the FP64 references of the deviations
    if (node_active) {
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        double col[5];
        LocalFluxColumn<kDiag>(cu, pu, js, d, col);
        {
#pragma unroll
          for (int k = 0; k < 5; ++k)
            s_x32[ncell * S::kScratch + (5 * d + k) * PAD + spos] = (float)(col[k] - s_ref[(d * C + ncell) * 5 + k]);
        }
      }
    }
    __syncthreads();
    // the first face tasks' neighbour lines, in flight during the passes
#pragma unroll
    for (int t = 0; t < PF; ++t)
      if (t_on[t] && t_nb[t] >= 0) gather(t, pre[t]);
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const int cb = kOneRound ? 5 * d * PAD : 0;  // column d within the cell's scratch
    if constexpr (!kOneRound) {
      __syncthreads();
      double col[5];
      if (node_active) {
        LocalFluxColumn<kDiag>(cu, pu, js, d, col);
        {
#pragma unroll
          for (int k = 0; k < 5; ++k)
            s_x32[ncell * S::kScratch + k * PAD + spos] = (float)(col[k] - s_ref[(d * C + ncell) * 5 + k]);
        }
      }
      __syncthreads();
    }
    if (node_active) {
      const int id = d == 0 ? ni : (d == 1 ? nj : nk);
      const int stride = d == 0 ? S::kSI : (d == 1 ? S::kSJ : 1);
      const int line0 = spos - id * stride;
      {
        const float *sx = s_x32 + ncell * S::kScratch + cb;
#pragma unroll
        for (int k = 0; k < 5; ++k) {
          float acc = 0.0f;
#pragma unroll
          for (int m = 0; m < Q; ++m) acc = __fmaf_rn((float)lt.d[id][m], sx[k * PAD + line0 + m * stride], acc);
          div[k] += (double)acc;
        }
      }
    }
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const LineIndex li = SkewedLineIndex<Q>(t_f[t]);
      if (t_on[t] && li.dir == d) {
        const int l0 = t_a[t] * li.a_mul + t_b[t] * li.b_mul;
        const double *lw = lt.lend[li.side];
        {
          const float *sx = s_x32 + t_cell[t] * S::kScratch + cb;
#pragma unroll
          for (int k = 0; k < 5; ++k) {
            float acc = (float)lw[0] * sx[k * PAD + l0];
#pragma unroll
            for (int m = 1; m < Q; ++m) acc = __fmaf_rn((float)lw[m], sx[k * PAD + l0 + m * li.stride], acc);
            fn[t][k] = s_ref[(d * C + t_cell[t]) * 5 + k] + (double)acc;
          }
        }
      }
    }
  }

  // ---- flux points: traces, upwind flux, flux gap
  double gap[T][5];
#pragma unroll
  for (int t = 0; t < T; ++t) {
    if (!t_on[t]) continue;
    const int f = t_f[t], ia = t_a[t], ib = t_b[t];
    const LineIndex li = SkewedLineIndex<Q>(f);
    const double *lw = lt.lend[li.side];
    State own;
    {
      const int l0 = ia * li.a_mul + ib * li.b_mul;
      const double *su = s_u + t_cell[t] * 5 * PAD;
#pragma unroll
      for (int k = 0; k < 5; ++k) {
        double vals[Q];
#pragma unroll
        for (int m = 0; m < Q; ++m) vals[m] = su[k * PAD + l0 + m * li.stride];
        own.v[k] = Extrapolate<Q>(lw, vals);
      }
    }
    const int32_t nb = t_nb[t];
    const int32_t info = t_info[t];
    const double *fr;
    double scale;
    fr = a.frames + (int64_t)(info >> 7) * kFrameStride;
    scale = s_scale[t_cell[t] * 6 + f];
    FaceFrame frame;
#pragma unroll
    for (int d = 0; d < 3; ++d) { frame.n[d] = fr[d]; frame.t[d] = fr[3 + d]; }
    frame.b[0] = frame.n[1] * frame.t[2] - frame.n[2] * frame.t[1];
    frame.b[1] = frame.n[2] * frame.t[0] - frame.n[0] * frame.t[2];
    frame.b[2] = frame.n[0] * frame.t[1] - frame.n[1] * frame.t[0];
    State fu;
    double sgn = 1.0;
    // the exact solver's state of this flux point, one copy per side: both
    // sides solve the same problem with the same inputs every pass, so the
    // two copies stay equal
    const int64_t star_slot = ((c0 + t_cell[t]) * 6 + f) * NFP + ia * Q + ib;
    bool star = kRiemann == kExact ? a.exact_star[star_slot] != 0 : false;
    if (nb >= 0) {
      const bool holder = (info >> 6) & 1;
      const double *nw = lt.lend[FaceLineIndex(Q, info & 7).side];
      double raw[Q][5];
      if (kOneRound && t < PF) {
#pragma unroll
        for (int m = 0; m < Q; ++m)
#pragma unroll
          for (int k = 0; k < 5; ++k) raw[m][k] = pre[t < PF ? t : 0][m][k];
      } else {
        gather(t, raw);
      }
      State other;
#pragma unroll
      for (int k = 0; k < 5; ++k) {
        double vals[Q];
#pragma unroll
        for (int m = 0; m < Q; ++m) vals[m] = raw[m][k];
        other.v[k] = Extrapolate<Q>(nw, vals);
      }
      fu = FrameFlux<kRiemann>(frame, holder ? own : other, holder ? other : own, star);
      sgn = holder ? 1.0 : -1.0;
    } else {
      const int tag = -nb - 1;
      const int kind = a.bc_kind[tag];
      // the tag's constant state, or this point's value of the tag's
      // boundary function at the stage time
      const double *gs = a.bc_point_state
          ? a.bc_point_state + ((int64_t)a.bface_of[(c0 + t_cell[t]) * 6 + f] * NFP + ia * Q + ib) * 5
          : a.bc_state + tag * 5;
      State given;
#pragma unroll
      for (int k = 0; k < 5; ++k) given.v[k] = gs[k];
      if (kind == kBcInviscidWall) {
        fu = WallFlux(frame, own);
      } else if (kind == kBcSupersonicOutlet) {
        fu = StateFlux(frame, own);
      } else if (kind == kBcSupersonicInlet) {
        fu = StateFlux(frame, given);
      } else if (kind == kBcSubsonicInlet) {
        fu = SubsonicInletFlux(frame, own, given);
      } else if (kind == kBcSubsonicOutlet) {
        fu = SubsonicOutletFlux(frame, own, given);
      } else {
        fu = FrameFlux<kRiemann>(frame, own, given, star);
      }
    }
    if constexpr (kRiemann == kExact) a.exact_star[star_slot] = star ? 1 : 0;
#pragma unroll
    for (int k = 0; k < 5; ++k) gap[t][k] = fu.v[k] * (sgn * scale) - fn[t][k];
  }
  __syncthreads();  // every read of the F~ columns is done
#pragma unroll
  for (int t = 0; t < T; ++t) {
    if (!t_on[t]) continue;
    const int r = t_f[t] * NFP + t_a[t] * Q + t_b[t];  // face-major gap slot of the node phase
#pragma unroll
    for (int k = 0; k < 5; ++k) s_x[t_cell[t] * S::kScratch + k * FPAD + r] = gap[t][k];
  }
  __syncthreads();

  // ---- node phase: lifted gaps, 1/det(J), RK stage, store
  double speed = 0.0;  // |u| + c of the new state, for a fused time step
  if (node_active) {
    const double *sg = s_x + ncell * S::kScratch;
    const double *su = s_u + ncell * 5 * PAD;
    const double dt = a.case_dt ? a.case_dt[a.cell_case[c0 + ncell]] : a.dt;
    double outv[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      const double *g = sg + k * FPAD;
      const double corr = LiftedGaps<Q>(g, lt, ni, nj, nk);
      const double res = (-div[k] - corr) * inv_det;
      outv[k] = fr::RkOutput(a.stage, res, su[k * PAD + spos], u0v[k], dt);
    }
    // one basic block of stores: merged into 16-byte stores of the node record
#pragma unroll
    for (int k = 0; k < 5; ++k) a.out[base + tid * 5 + k] = outv[k];
    if (a.dt_min_bits) {
      State nw;
#pragma unroll
      for (int k = 0; k < 5; ++k) nw.v[k] = outv[k];
      speed = MaxSpeed(nw);
    }
  }
  if (a.dt_min_bits) {
    // fem.hpp:412-435 on the state just written, as FrMixedTimeStepKernel:
    // min over cells of length / max(1e-5, max over nodes of |u| + c)
    __syncthreads();  // every read of the LDS states and gaps is done
    double *s_speed = s_u, *s_cell = s_x;
    if (node_active) s_speed[tid] = speed;
    __syncthreads();
    if (tid < nc) {
      double vmax = 1e-5;
      for (int p = 0; p < NP; ++p) vmax = fmax(vmax, s_speed[tid * NP + p]);
      s_cell[tid] = a.geo[(int64_t)a.geo_id[c0 + tid] * kMixedGeoStride + 16] / vmax;
    }
    __syncthreads();
    if (tid == 0) {
      double local = 1e300;
      for (int c = 0; c < nc; ++c) local = fmin(local, s_cell[c]);
      atomicMin(a.dt_min_bits, (unsigned long long)__double_as_longlong(local));
    }
  }
}

template <int Q, int Cells, int Threads, int kRiemann, bool kDiag, bool kOneRound, int kPrefetch>
__global__ __launch_bounds__(Threads) void FrMixedStageKernel(FrHexArgs a, MixedTables lt) {
  __shared__ double lds[Shape<Q, Cells, Threads, kOneRound>::kLdsDoubles];
  // The line tables are indexed by lane-varying node indices: read from the
  // kernel arguments they would be vector loads on the critical path of every
  // pass, so they are staged in LDS once (the body's first barrier orders it).
  __shared__ MixedTables s_lt;
  constexpr int kTableDoubles = sizeof(MixedTables) / sizeof(double);
  if (threadIdx.x < kTableDoubles)
    reinterpret_cast<double *>(&s_lt)[threadIdx.x] = reinterpret_cast<const double *>(&lt)[threadIdx.x];
  int64_t block = LogicalBlock(a.xcd_remap);
  if (a.tile_order) block = a.tile_order[block];
  FrMixedStageBody<Q, Cells, Threads, kRiemann, kDiag, kOneRound, kPrefetch>(a, s_lt, block, lds);
}

// Single-mesh launch shape per Q: one thread per solution point.  Q = 4 and
// 5 run on 128-thread workgroups (2 cells and 1 cell): the same 3 waves per
// SIMD as 256-thread ones, with each barrier waiting on two wavefronts
// instead of four (Q = 4: 0.93 against 0.96 ms per stage at 64^3; Q = 3 as
// 4 cells on 128 threads leaves 20 threads idle and measured no better).  At Q = 4
// the face tasks (96 per cell) fill two slots in half of the wavefronts; 96
// threads per cell (one task each) measured slower on MI355X, since the extra
// wavefronts idle through the volume passes and occupy wave slots that other
// workgroups would fill.
template <int Q> struct StageTile {
  static constexpr int kCells = Q == 4 ? 2 : (Q == 5 ? 1 : Shape<Q>::kCells);
  static constexpr int kThreads = (Q == 4 || Q == 5) ? 128 : 256;
  static constexpr bool kOneRound = Q >= 3;  // at Q = 2 the column space would cost a workgroup per CU
  // face tasks whose neighbour lines are issued before the passes: one, as
  // the registers of the three-waves-per-SIMD budget allow
  static constexpr int kPrefetch = 1;
};

// Tile variants per Q (cells per workgroup) that the batched launch and its
// autotuner choose from.
template <int Q, int V> struct TileOf;
template <> struct TileOf<2, 0> { static constexpr int kCells = 32; };
template <> struct TileOf<2, 1> { static constexpr int kCells = 16; };
template <> struct TileOf<2, 2> { static constexpr int kCells = 8; };
template <> struct TileOf<3, 0> { static constexpr int kCells = 9; };
template <> struct TileOf<3, 1> { static constexpr int kCells = 4; };
template <> struct TileOf<3, 2> { static constexpr int kCells = 2; };
template <> struct TileOf<4, 0> { static constexpr int kCells = 4; };
template <> struct TileOf<4, 1> { static constexpr int kCells = 2; };
template <> struct TileOf<4, 2> { static constexpr int kCells = 1; };

template <int Q, int V>
constexpr int TileLds() { return Shape<Q, TileOf<Q, V>::kCells, 256, (Q >= 3)>::kLdsDoubles; }

// One out-of-line body per (Q, tile): each is register-allocated on its own
// within the kernel's 3-waves-per-SIMD budget, where nine inlined bodies
// would share one allocation and spill.  Q >= 3 bodies pass all three F~
// columns through LDS in one round, as the single-mesh launch does.
template <int Q, int V, int kRiemann>
__device__ __noinline__ void BatchBody(const FrHexBatchGroup *g, int64_t block, double *lds) {
  FrMixedStageBody<Q, TileOf<Q, V>::kCells, 256, kRiemann, true, (Q >= 3), 1>(g->args, g->mt, block, lds);
}

template <int Q, int kRiemann>
__device__ __forceinline__ void BatchItem(const FrHexBatchGroup &g, int64_t block, double *lds) {
  switch (g.tile) {
  case 0: BatchBody<Q, 0, kRiemann>(&g, block, lds); break;
  case 1: BatchBody<Q, 1, kRiemann>(&g, block, lds); break;
  default: BatchBody<Q, 2, kRiemann>(&g, block, lds); break;
  }
}

// Persistent batched pass: workgroup w processes the contiguous item range
// [w * n_items / W, (w + 1) * n_items / W) of the work list (blocks of all
// degree groups in order), so consecutive blocks -- and their neighbour
// cells -- stay in one XCD's L2.  LDS is sized at launch for the largest tile
// in use.
template <int kRiemann>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void FrMixedBatchKernel(FrHexBatchArgs b) {
  extern __shared__ double lds[];
  const int64_t w = blockIdx.x, nw = gridDim.x;
  const int64_t begin = w * b.n_items / nw, end = (w + 1) * b.n_items / nw;
  int gi = 0;
  for (int64_t item = begin; item < end; ++item) {
    // the group table lives in device memory and gi is uniform, so every
    // field is fetched with scalar loads
    while (gi + 1 < b.n_groups && item >= b.group[gi + 1].first_item) ++gi;
    const FrHexBatchGroup &g = b.group[gi];
    const int64_t block = item - g.first_item;
    switch (g.q) {
    case 2: BatchItem<2, kRiemann>(g, block, lds); break;
    case 3: BatchItem<3, kRiemann>(g, block, lds); break;
    default: BatchItem<4, kRiemann>(g, block, lds); break;
    }
    __syncthreads();  // the next item reuses the LDS buffers
  }
}

template <int Q>
__global__ __launch_bounds__(256) void FrMixedTimeStepKernel(const double *u, const int32_t *geo_id,
    const double *geo, int64_t n_cells, unsigned long long *dt_min_bits) {
  constexpr int NP = Q * Q * Q;
  __shared__ double s_min[256];
  double local = 1e300;
  for (int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x; c < n_cells; c += (int64_t)gridDim.x * 256) {
    double vmax = 1e-5;  // fem.hpp:419, avoids 0 in the divisor
    const double *uc = u + c * NP * 5;
    for (int p = 0; p < NP; ++p) {
      State s;
#pragma unroll
      for (int k = 0; k < 5; ++k) s.v[k] = uc[p * 5 + k];
      vmax = fmax(vmax, MaxSpeed(s));
    }
    local = fmin(local, geo[(int64_t)geo_id[c] * kMixedGeoStride + 16] / vmax);
  }
  s_min[threadIdx.x] = local;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) s_min[threadIdx.x] = fmin(s_min[threadIdx.x], s_min[threadIdx.x + s]);
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicMin(dt_min_bits, (unsigned long long)__double_as_longlong(s_min[0]));
}

template <int Q, int R>
hipError_t Launch(const FrHexArgs &args, const MixedTables &lt, hipStream_t stream) {
  constexpr int C = StageTile<Q>::kCells, W = StageTile<Q>::kThreads;
  constexpr bool O = StageTile<Q>::kOneRound;
  constexpr int PF = StageTile<Q>::kPrefetch;
  int64_t blocks = (args.n_cells + C - 1) / C;
  if (blocks > 0x7fffffff) return hipErrorInvalidValue;
  const dim3 grid((unsigned)blocks), block(W);
  if (args.diag_metric) {
    hipLaunchKernelGGL((FrMixedStageKernel<Q, C, W, R, true, O, PF>), grid, block, 0, stream, args, lt);
  } else {
    hipLaunchKernelGGL((FrMixedStageKernel<Q, C, W, R, false, O, PF>), grid, block, 0, stream, args, lt);
  }
  return hipGetLastError();
}

template <int Q>
hipError_t LaunchQ(int riemann, const FrHexArgs &args, const MixedTables &lt, hipStream_t stream) {
  switch (riemann) {
  case kExact: return Launch<Q, kExact>(args, lt, stream);
  case kHllc: return Launch<Q, kHllc>(args, lt, stream);
  case kRoe: return Launch<Q, kRoe>(args, lt, stream);
  default: return hipErrorInvalidValue;
  }
}

}  // namespace

hipError_t LaunchFrMixedStage(int q, int riemann, const FrHexArgs &args, const MixedTables &lt,
                            hipStream_t stream) {
  switch (q) {
  case 2: return LaunchQ<2>(riemann, args, lt, stream);
  case 3: return LaunchQ<3>(riemann, args, lt, stream);
  case 4: return LaunchQ<4>(riemann, args, lt, stream);
  case 5: return LaunchQ<5>(riemann, args, lt, stream);
  case 6: return LaunchQ<6>(riemann, args, lt, stream);
  default: return hipErrorInvalidValue;
  }
}

int FrMixedTileLdsBytes(int q, int tile) {
  static const int lds[3][3] = { { TileLds<2, 0>(), TileLds<2, 1>(), TileLds<2, 2>() },
                                 { TileLds<3, 0>(), TileLds<3, 1>(), TileLds<3, 2>() },
                                 { TileLds<4, 0>(), TileLds<4, 1>(), TileLds<4, 2>() } };
  if (q < 2 || q > 4 || tile < 0 || tile > 2) return 0;
  return lds[q - 2][tile] * (int)sizeof(double);
}

int FrMixedStageTileCells(int q) {
  switch (q) {
  case 2: return StageTile<2>::kCells;
  case 3: return StageTile<3>::kCells;
  case 4: return StageTile<4>::kCells;
  case 5: return StageTile<5>::kCells;
  case 6: return StageTile<6>::kCells;
  default: return 0;
  }
}

int FrMixedTileCells(int q, int tile) {
  static const int cells[3][3] = { { 32, 16, 8 }, { 9, 4, 2 }, { 4, 2, 1 } };
  if (q < 2 || q > 4 || tile < 0 || tile > 2) return 0;
  return cells[q - 2][tile];
}

hipError_t LaunchFrMixedBatch(int riemann, const FrHexBatchArgs &args, int n_workgroups, hipStream_t stream) {
  if (args.n_groups < 1 || args.n_groups > kMaxBatchGroups || n_workgroups < 1) return hipErrorInvalidValue;
  const dim3 grid((unsigned)n_workgroups), block(256);
  const size_t lds = (size_t)args.max_tile_lds;
  switch (riemann) {
  case kExact: hipLaunchKernelGGL(FrMixedBatchKernel<kExact>, grid, block, lds, stream, args); break;
  case kHllc: hipLaunchKernelGGL(FrMixedBatchKernel<kHllc>, grid, block, lds, stream, args); break;
  case kRoe: hipLaunchKernelGGL(FrMixedBatchKernel<kRoe>, grid, block, lds, stream, args); break;
  default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t FrMixedBatchResident(int riemann, int lds_bytes, int *per_cu) {
  switch (riemann) {
  case kExact: return hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, FrMixedBatchKernel<kExact>, 256, lds_bytes);
  case kHllc: return hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, FrMixedBatchKernel<kHllc>, 256, lds_bytes);
  case kRoe: return hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, FrMixedBatchKernel<kRoe>, 256, lds_bytes);
  default: return hipErrorInvalidValue;
  }
}

hipError_t LaunchFrMixedTimeStep(int q, const double *u, const int32_t *geo_id, const double *geo,
                               int64_t n_cells, unsigned long long *dt_min_bits, hipStream_t stream) {
  int64_t blocks = std::min<int64_t>((n_cells + 255) / 256, 4096);
  if (blocks < 1) blocks = 1;
  switch (q) {
#define MCFD_TS_CASE(QQ) \
  case QQ: hipLaunchKernelGGL((FrMixedTimeStepKernel<QQ>), dim3((unsigned)blocks), dim3(256), 0, stream, \
                              u, geo_id, geo, n_cells, dt_min_bits); break;
  MCFD_TS_CASE(2) MCFD_TS_CASE(3) MCFD_TS_CASE(4) MCFD_TS_CASE(5) MCFD_TS_CASE(6)
#undef MCFD_TS_CASE
  default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace mcfd
