// Device-only Euler helpers of the stage kernels (FP64), on top of the
// portable physics of mini/riemann/euler_core.hpp: refined reciprocals and
// square roots, and the face fluxes in vector form as the FR kernels evaluate
// them.
#ifndef MINICFD_KERNELS_EULER_HPP_
#define MINICFD_KERNELS_EULER_HPP_

#include <hip/hip_runtime.h>

#include "../../../include/mini/riemann/euler_core.hpp"

namespace mcfd {

// ------------------------------------------------- fast FP64 reciprocal
// v_rcp_f64 refined by two Newton steps: within 1 ulp of 1/x for normal x.
// Used by the throughput kernels in place of IEEE division (a ~10
// instruction sequence on CDNA); both cells of a face run the same code, so
// the face flux stays bit-identical on the two sides.  NaN for zeros and
// infinities, of which the steps know nothing: for arguments that are neither, or
// where a NaN, or the zeroing rule's values, come of it either way.
__device__ __forceinline__ double FiniteRcp(double x) {
  double r = __builtin_amdgcn_rcp(x);
  double e = __fma_rn(-x, r, 1.0);
  r = __fma_rn(r, e, r);
  e = __fma_rn(-x, r, 1.0);
  return __fma_rn(r, e, r);
}
// The same with zeros and infinities as the divide has them, one instruction more
// (everywhere, 0.3 to 0.6 % of a pass of 64^3 p3, 1 to 2 % of a small one's chain).
__device__ __forceinline__ double FastRcp(double x) { return __builtin_amdgcn_div_fixup(FiniteRcp(x), x, 1.0); }

// The smallest of the positive `value`s in *bits (the bits of positive doubles
// order as the doubles do).  Atomics on one address pass at about 11 ns each, 3 ms
// for the 262144 of a 64^3 box; what cannot lower the minimum is left out, by a
// read that may be old: the minimum only falls.
__device__ __forceinline__ void FoldMin(unsigned long long *bits, double value) {
  const unsigned long long own = (unsigned long long)__double_as_longlong(value);
  if (own < __hip_atomic_load(bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMin(bits, own);
}

// sqrt by v_rsq_f64 and two fused corrections: within 1 ulp for normal x, x for
// zeros and infinity, NaN for x < 0.  The compiler's correctly rounded sqrt adds range
// scaling and class checks, about twice the instructions.
constexpr int kZerosAndInfinity = 0x20 | 0x40 | 0x200;  // v_cmp_class: -0, +0, +inf
__device__ __forceinline__ double FastSqrt(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double r = __fma_rn(-h, g, 0.5);
  g = __fma_rn(g, r, g);
  h = __fma_rn(h, r, h);
  g = __fma_rn(__fma_rn(-g, g, x), h, g);
  return __builtin_amdgcn_class(x, kZerosAndInfinity) ? x : g;
}

// x / 3, correctly rounded: the quotient by the rounded reciprocal is at most
// one unit off, and the fused remainder, exact also below the normal range, puts
// it right (Markstein's division for a constant divisor); the fixup returns
// infinities and signed zeros as the divide does.  4 instructions instead of 10.
__device__ __forceinline__ double ThirdOf(double x) {
  const double q = x * (1.0 / 3.0);
  return __builtin_amdgcn_div_fixup(__fma_rn(__fma_rn(-3.0, q, x), 1.0 / 3.0, q), 3.0, x);
}

// One trace of a face with what the fluxes need of it: density and its
// reciprocal, velocity, pressure, total energy, and the velocity along the
// unit normal.  The reference rotates both traces into the face
// frame, solves there and rotates the flux back (rotated/euler.hpp:117-159);
// the solvers only need the normal velocity, so the fluxes below keep the
// vectors in global coordinates: no tangents, two dot products instead of
// three rotations.
struct FaceTrace { double rho, inv, v[3], p, e, un; };

// The trace's plain arithmetic (types.hpp:289-301, one reciprocal); *plain is
// cleared where the zeroing rule (ApplyZeroRule) changes the result.
__device__ __forceinline__ FaceTrace PlainTrace(State const &c, const double *n, bool *plain) {
  FaceTrace t;
  t.rho = c.v[0];
  t.inv = FiniteRcp(t.rho);
#pragma unroll
  for (int d = 0; d < 3; ++d) t.v[d] = c.v[1 + d] * t.inv;
  t.e = c.v[4];
  const double rk = c.v[1] * t.v[0] + c.v[2] * t.v[1] + c.v[3] * t.v[2];  // 2 rho k
  t.p = (t.e - 0.5 * rk) * kGm1;
  t.un = t.v[0] * n[0] + t.v[1] * n[1] + t.v[2] * n[2];
  *plain = *plain && t.rho > 0 && t.e >= 0 && t.p >= 0;
  return t;
}
// types.hpp:195-202: all zero where rho < 0, E < 0 or p < 0; momenta and E kept
// as velocity and pressure where rho == 0.  kStill (HLLC): such a state with pressure
// takes 1 / rho = 0, which gives it the wave speed u of a side whose a is 0 and whose
// q is finite.
template <bool kStill = false>
__device__ __forceinline__ void ApplyZeroRule(State const &c, const double *n, FaceTrace *t) {
  const bool bad = c.v[0] < 0 || c.v[4] < 0;
  const bool vacuum = !bad && c.v[0] == 0;
  const bool zero = bad || (!vacuum && t->p < 0);
#pragma unroll
  for (int d = 0; d < 3; ++d) t->v[d] = zero ? 0.0 : (vacuum ? c.v[1 + d] : t->v[d]);
  t->p = zero ? 0.0 : (vacuum ? c.v[4] : t->p);
  t->e = zero ? 0.0 : (vacuum ? c.v[4] * (1 / kGm1) : t->e);
  t->rho = zero ? 0.0 : t->rho;
  if (zero || vacuum) t->inv = kStill && t->p > 0 ? 0.0 : FastRcp(t->rho);
  t->un = t->v[0] * n[0] + t->v[1] * n[1] + t->v[2] * n[2];
}
__device__ __forceinline__ FaceTrace TraceOf(State const &c, const double *n) {
  bool plain = true;
  FaceTrace t = PlainTrace(c, n, &plain);
  if (!__all(plain)) ApplyZeroRule(c, n, &t);
  return t;
}

// types.hpp:313-321: physical flux of one trace through the unit normal n.
__device__ __forceinline__ State TraceFlux(FaceTrace const &t, const double *n) {
  State f;
  f.v[0] = t.rho * t.un;
#pragma unroll
  for (int d = 0; d < 3; ++d) f.v[1 + d] = f.v[0] * t.v[d] + t.p * n[d];
  f.v[4] = (t.e + t.p) * t.un;
  return f;
}

// Roe flux (the waves of RoeFlux in euler_core.hpp): sqrt(rho_r / rho_l) gives
// both the averaging weight and the mean density, one reciprocal square root
// the sound speed and its inverse square.
__device__ __forceinline__ State FastRoe(FaceTrace const &l, FaceTrace const &r, const double *n) {
  const double hl = (l.e + l.p), hr = (r.e + r.p);  // rho times total enthalpy
  const double ratio = FastSqrt(r.rho * l.inv);
  const double wr = ratio * FiniteRcp(1.0 + ratio);
  const double rho = l.rho * ratio;
  double dv[3], v[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    dv[d] = r.v[d] - l.v[d];
    v[d] = l.v[d] + wr * dv[d];
  }
  const double dun = r.un - l.un, un = l.un + wr * dun, dp = r.p - l.p;
  const double h0l = hl * l.inv, h = h0l + wr * (hr * r.inv - h0l);
  const double ke = 0.5 * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
  const double aa = kGm1 * (h - ke);
  const double a = FastSqrt(aa), inv_aa = FiniteRcp(aa);
  const double rad = rho * a * dun;
  const double s1 = 0.25 * (dp - rad) * inv_aa * fabs(un - a);
  const double s5 = 0.25 * (dp + rad) * inv_aa * fabs(un + a);
  const double s2 = 0.5 * ((r.rho - l.rho) - dp * inv_aa) * fabs(un);
  const double t = 0.5 * rho * fabs(un);           // both shear waves
  const double s = s1 + s2 + s5, b = (s5 - s1) * a, bn = b - t * dun;
  State f;
  const double ml = 0.5 * (l.rho * l.un), mr = 0.5 * (r.rho * r.un);
  f.v[0] = ml + mr - s;
  const double pm = 0.5 * (l.p + r.p) - bn;
#pragma unroll
  for (int d = 0; d < 3; ++d) f.v[1 + d] = ml * l.v[d] + mr * r.v[d] + pm * n[d] - s * v[d] - t * dv[d];
  const double vdv = v[0] * dv[0] + v[1] * dv[1] + v[2] * dv[2];
  f.v[4] = 0.5 * (hl * l.un + hr * r.un) - ((s1 + s5) * h + s2 * ke + un * bn + t * vdv);
  return f;
}

// HLLC flux (hllc.hpp:30-109): wave speeds u -+ a q from one square root each
// (a q = sqrt(a^2 + c (p* - p) / rho) needs no division by p; kStill of the zeroing
// rule sees to a side without density), the star state formed once, for the side the
// contact selects.
__device__ __forceinline__ State FastHllc(FaceTrace const &l, FaceTrace const &r, const double *n) {
  const double al = l.rho > 0 && l.p > 0 ? FastSqrt(kGamma * l.p * l.inv) : 0.0;
  const double ar = r.rho > 0 && r.p > 0 ? FastSqrt(kGamma * r.p * r.inv) : 0.0;
  const double p_est = fmax(0.0, 0.5 * (l.p + r.p - (r.un - l.un) * (0.25 * (l.rho + r.rho) * (al + ar))));
  const double aql = p_est > l.p ? FastSqrt((kGamma * l.p + (kGp1 / 2) * (p_est - l.p)) * l.inv) : al;
  const double aqr = p_est > r.p ? FastSqrt((kGamma * r.p + (kGp1 / 2) * (p_est - r.p)) * r.inv) : ar;
  const double wl = l.un - aql, wr = r.un + aqr;
  const double ml = l.rho * (wl - l.un), mr = r.rho * (wr - r.un);
  const double ws = (r.p - l.p + ml * l.un - mr * r.un) * FiniteRcp(ml - mr);
  const bool super_l = 0.0 <= wl, super_r = !super_l && wr <= 0.0;
  const bool left = super_l || (!super_r && 0.0 <= ws);
  FaceTrace k;
  k.rho = left ? l.rho : r.rho;
  k.inv = left ? l.inv : r.inv;
#pragma unroll
  for (int d = 0; d < 3; ++d) k.v[d] = left ? l.v[d] : r.v[d];
  k.p = left ? l.p : r.p;
  k.e = left ? l.e : r.e;
  k.un = left ? l.un : r.un;
  const double wk = left ? wl : wr, mk = left ? ml : mr;
  State f = TraceFlux(k, n);
  if (super_l || super_r) return f;
  const double inv_ws = FastRcp(wk - ws), temp = mk * inv_ws, du = ws - k.un;
  f.v[0] += wk * (temp - k.rho);
#pragma unroll
  for (int d = 0; d < 3; ++d) f.v[1 + d] += wk * (temp * (k.v[d] + du * n[d]) - k.rho * k.v[d]);
  f.v[4] += wk * (temp * (k.e * k.inv) + du * (temp * ws + k.p * inv_ws) - k.e);
  return f;
}

// x^(1/7) of a positive normal or subnormal x, within 0.81 units of 2^-52 (1e6
// arguments from 5e-324 to 64; pow(x, 1 / 7.0), its exponent rounded, up to 25): a single-precision
// estimate of the mantissa's root (the exponent divided by 7 beforehand), then one
// step of Halley's iteration for y^7 = x, which cubes the estimate's 1e-6.
__device__ __forceinline__ double SeventhRoot(double x) {
  const int e = __builtin_amdgcn_frexp_exp(x);
  const int q = (e >= 0 ? e : e - 6) / 7;
  const double m = __builtin_amdgcn_ldexp(__builtin_amdgcn_frexp_mant(x), e - 7 * q);  // in [1/2, 64)
  const double y = (double)__builtin_amdgcn_exp2f(__builtin_amdgcn_logf((float)m) * (1.0f / 7));
  const double y2 = y * y, y3 = y2 * y, y7 = y3 * y3 * y;
  const double root = __fma_rn(y * (m - y7), FiniteRcp(__fma_rn(4.0, y7, 3.0 * m)), y);
  return __builtin_amdgcn_ldexp(root, q);
}

// The exact solver is bound by its serial chain, one flux point to a lane: two
// pressure functions and their slopes per Newton step, at first a pow each.  With
// gamma = 1.4 the rarefaction's powers are z - 1 and z^-6 of the one seventh root z
// of pa / p, function and slope come from one evaluation, and the state inside a
// fan from rho (a / a0)^5.  us per stage: FR 24^3 p3 217 -> 63, 32^3 p2 330 -> 88; DG
// on the 640 hexahedra of a Sod tube 41 -> 14 (face and cell pass -> one, too).
//
// One side's pressure function (exact.hpp:153-200) and its derivative at pa.
struct FastWave {
  double rho, p, a, inv_p;
  __device__ __forceinline__ explicit FastWave(State const &b)
      : rho(b.v[0]), p(b.v[4]), a(FastSqrt(kGamma * b.v[4] * FastRcp(b.v[0]))), inv_p(FastRcp(b.v[4])) {}
  __device__ __forceinline__ double F(double pa, double *slope) const {
    if (pa >= p) {
      const double pp = (kGp1 / 2) * pa + (kGm1 / 2) * p;
      const double inv = 1 / sqrt(rho * pp);
      *slope = __fma_rn((kGp1 / 4) * (p - pa), 1 / pp, 1.0) * inv;
      return (pa - p) * inv;
    }
    const double z = SeventhRoot(pa * inv_p), z2 = z * z;
    *slope = FastRcp(z2 * z2 * z2 * (rho * a));
    return (z - 1) * ((2 / kGm1) * a);
  }
  // F(0): the vacuum's limit
  __device__ __forceinline__ double Vacuum() const { return 0 >= p ? -p / sqrt(rho * ((kGm1 / 2) * p)) : -((2 / kGm1) * a); }
};
// exact.hpp:255-266 through rho (a / a0)^5, a0 the sound speed before the fan:
// the state's isentrope needs no power of the density.
__device__ __forceinline__ State FastInsideFan(double rho0, double a0, double gri_2) {
  const double a = (kGm1 / kGp1) * gri_2, a2 = a * a, ratio = a2 / (a0 * a0);
  State s;
  s.v[0] = rho0 * (ratio * ratio * sqrt(ratio));
  s.v[1] = a; s.v[2] = 0; s.v[3] = 0;
  s.v[4] = a2 * s.v[0] * (1 / kGamma);
  return s;
}
// The state on the face (density, normal velocity, pressure; passive velocities 0),
// by ExactFlux's branches, starting point, iteration and stopping rule
// (euler_core.hpp) on the functions above.
__device__ __forceinline__ State FastExactState(State const &l, State const &r, bool &star_positive) {
  State res;
#pragma unroll
  for (int i = 0; i < 5; ++i) res.v[i] = 0;
  const bool has_l = l.v[0] > 0, has_r = r.v[0] > 0;
  if (!has_l && !has_r) return res;
  const FastWave wl(l), wr(r);
  const double du = r.v[1] - l.v[1];
  // the fans' edges in a vacuum, exact.hpp:62-138,293-320
  const double edge_l = l.v[1] + wl.a * (2 / kGm1), edge_r = r.v[1] - wr.a * (2 / kGm1);
  if (!has_r) {
    if (l.v[1] >= wl.a) res = l;
    else if (edge_l > 0) res = FastInsideFan(l.v[0], wl.a, edge_l);
    return res;
  }
  if (!has_l) {
    if (r.v[1] + wr.a <= 0) res = r;
    else if (edge_r < 0) res = FastInsideFan(r.v[0], wr.a, edge_r);
    return res;
  }
  if (!(wl.Vacuum() + wr.Vacuum() + du < 0)) {
    if (l.v[1] > wl.a) return l;
    if (r.v[1] + wr.a < 0) return r;
    if (edge_l >= 0) return FastInsideFan(l.v[0], wl.a, edge_l);
    if (edge_r < 0) return FastInsideFan(r.v[0], wr.a, edge_r);
    return res;
  }
  // exact.hpp:140-152 FindRoot: halve, then Newton
  double x = l.v[4], fl, fr, sl, sr;
  for (int it = 0; it < 2100; ++it) {
    fl = wl.F(x, &sl);
    fr = wr.F(x, &sr);
    if (!(fl + fr + du > 0)) break;
    x *= 0.5;
  }
  for (int it = 0; it < 200; ++it) {
    const double f = fl + fr + du;
    if (!(f < -1e-8)) break;
    x -= f / (sl + sr);
    fl = wl.F(x, &sl);
    fr = wr.F(x, &sr);
  }
  State star;
  star.v[0] = 0; star.v[2] = 0; star.v[3] = 0; star.v[4] = x;
  star.v[1] = 0.5 * (r.v[1] + fr + l.v[1] - fl);
  star_positive = star.v[1] > 0;
  // toward the t axis through wave 1 (left) or 3 (right)
  const bool left = star_positive;
  const State before = left ? l : r;
  if (x >= before.v[4]) return NearShock(before, star, left);
  const double a_before = left ? wl.a : wr.a;
  const double e = (kGm1 / 2) * (before.v[1] - star.v[1]);
  const double a_after = left ? a_before + e : a_before - e;
  if (left ? star.v[1] - a_after < 0 : star.v[1] + a_after > 0) {
    star.v[0] = kGamma * x / (a_after * a_after);
    return star;
  }
  if (left ? before.v[1] - a_before > 0 : before.v[1] + a_before < 0) return before;
  return FastInsideFan(before.v[0], a_before, left ? edge_l : edge_r);
}

// Exact flux (ExactFlux in euler_core.hpp) with the passive tangential velocity
// as a vector: that of the side the contact moves away from.
__device__ __forceinline__ State VectorExact(FaceTrace const &l, FaceTrace const &r, const double *n, bool &star) {
  const State pl = { { l.rho, l.un, 0.0, 0.0, l.p } }, pr = { { r.rho, r.un, 0.0, 0.0, r.p } };
  const State s = FastExactState(pl, pr, star);
  FaceTrace t;
  t.rho = s.v[0];
  t.un = s.v[1];
  t.p = s.v[4];
  const double du = t.un - (star ? l.un : r.un);
#pragma unroll
  for (int d = 0; d < 3; ++d) t.v[d] = (star ? l.v[d] : r.v[d]) + du * n[d];
  t.e = t.p * (1 / kGm1) + t.rho * (0.5 * (t.v[0] * t.v[0] + t.v[1] * t.v[1] + t.v[2] * t.v[2]));
  return TraceFlux(t, n);
}

template <int kRiemann>
__device__ __forceinline__ State TraceUpwind(FaceTrace const &l, FaceTrace const &r, const double *n, bool &star) {
  if constexpr (kRiemann == kExact) return VectorExact(l, r, n, star);
  else if constexpr (kRiemann == kHllc) return FastHllc(l, r, n);
  else return FastRoe(l, r, n);
}
// The upwind flux through the unit normal n (from left to right) as the FR
// stage kernels evaluate it.  `star` is the exact solver's per-point state.
template <int kRiemann>
__device__ __forceinline__ State FaceFlux(const double *n, State const &cl, State const &cr, bool &star) {
  bool plain = true;
  FaceTrace l = PlainTrace(cl, n, &plain), r = PlainTrace(cr, n, &plain);
  if (!__all(plain)) {
    ApplyZeroRule<kRiemann == kHllc>(cl, n, &l);
    ApplyZeroRule<kRiemann == kHllc>(cr, n, &r);
  }
  return TraceUpwind<kRiemann>(l, r, n, star);
}

// Flux of a boundary point whose condition is not a Riemann problem
// (rotated/euler.hpp:144-174,181-280; the rotated forms are in
// euler_core.hpp), through the unit normal n, which points out of the cell
// (outward) or into it: the physical flux of a boundary state, (0, p n, 0) at
// a wall.  pow(x, gamma / (gamma - 1)) of the subsonic inlet is x^3 sqrt(x).
__device__ __forceinline__ State BoundaryFlux(int kind, bool outward, const double *n, State const &own,
                                              State const &given) {
  const bool inlet = kind == kBcSupersonicInlet;
  State c;
#pragma unroll
  for (int k = 0; k < 5; ++k) c.v[k] = inlet ? given.v[k] : own.v[k];
  FaceTrace t = TraceOf(c, n);
  if (kind == kBcInviscidWall) t.un = 0.0;
  if (kind == kBcSubsonicInlet || kind == kBcSubsonicOutlet) {
    if (kind == kBcSubsonicOutlet) {  // the interior's p / rho and velocity at the given pressure
      t.rho = given.v[4] / (t.p / t.rho);
      t.p = given.v[4];
    } else {
      const double c_in = t.rho > 0 && t.p > 0 ? sqrt(kGamma * t.p / t.rho) : 0.0;
      const double r_in = (outward ? -t.un : t.un) - c_in * (2 / kGm1);
      const double cos_n = n[0] * given.v[1] + n[1] * given.v[2] + n[2] * given.v[3], a2 = cos_n * cos_n;
      const double gamma_r = kGamma * kGasR, t_total = given.v[4];
      // larger root of qa x^2 + 2 r_in x + qc = 0
      const double qa = a2 + 2 / kGm1, qc = (kGm1 / 2) * (r_in * r_in) - a2 * gamma_r * t_total;
      const double c_b = (sqrt(r_in * r_in - qa * qc) - r_in) / qa;
      const double t_b = c_b * c_b / gamma_r;
      const double mach = sqrt((t_total / t_b - 1) / (kGm1 / 2));
      const double x = 1 + (kGm1 / 2) * mach * mach;
      t.p = given.v[0] / (x * x * x * sqrt(x));
      t.rho = t.p / kGasR / t_b;
#pragma unroll
      for (int d = 0; d < 3; ++d) t.v[d] = given.v[1 + d] * (mach * c_b);
      t.un = t.v[0] * n[0] + t.v[1] * n[1] + t.v[2] * n[2];
    }
    t.e = t.p * (1 / kGm1) + t.rho * (0.5 * (t.v[0] * t.v[0] + t.v[1] * t.v[1] + t.v[2] * t.v[2]));
  }
  return TraceFlux(t, n);
}

}  // namespace mcfd

#endif  // MINICFD_KERNELS_EULER_HPP_
