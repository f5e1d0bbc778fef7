// mf_pair.hpp -- per-pair field and force-tensor coefficients for gfx950.
//
// Both pair kernels of the reference reduce to two radial scalars per pair:
//
// Field (fmmtl_minimum/kernel/Dipole_B.kern:46-104, == magnetic_force.cu:63-98)
//   K(d) m = u (u.m)(w_avr - w_dens) - (w_avr/3 - w_dens) m,   u = d/|d|
//          = c [ 3 alpha d (d.m) - beta m ],                    c = 1/(4 pi)
// with (w~ = w / c)
//   far  (q >= 2): alpha = |d|^-5,                 beta = |d|^-3
//   q < 1       : alpha = (0.8 - 0.5 q)/h^5,       beta = (-8/3 + 4.8 q^2 - 2.5 q^3)/h^3
//   1 <= q < 2  : alpha = (g(q)/r^3 - ((2-q)/h)^3)/(3 r^2),
//                 beta  =  g(q)/(3 r^3) - ((2-q)/h)^3,
//                 g(q) = -3 (q^6/6 - 6q^5/5 + 3q^4 - 8q^3/3 + 1/15)
// The q < 1 forms are the reference's w_avr/w_dens polynomials with the
// common factors cancelled exactly (w_avr - w_dens = sigma q^2 (0.6 - 0.375 q)),
// which also removes the 0/0 at r = 0 (self term (2/3) sigma m).
//
// Force tensor (Dipole_hessian.kern:53-238, == magnetic_force.cu:239-427)
//   B(d)[m]_ab = P (d_a m_b + m_a d_b + delta_ab d.m) + R d_a d_b (d.m)
// scaled by s = 3 mu0/(4 pi):
//   far  (q > 4) : P = |d|^-5,            R = -5 |d|^-7
//   0 < q <= 4   : P = C1(q)/(s h^4 r),   R = (C2(q) - 3 C1(q))/(s h^4 r^3)
//   q == 0       : 0
// The rotation-frame product M U M^T of the reference equals this isotropic
// form.  C1, C2 are the reference's fitted quartics.  The kernels read alpha,
// beta, C1 and C2 from tables of local cubics (below), whose FP32 evaluation
// does not cancel as the powers of q do.
#pragma once

#include <hip/hip_runtime.h>

namespace mf {

constexpr double kPi = 3.14159265358979323846;
constexpr double kMu0 = 1.25663706e-6;  // the reference's truncated value

// Field constants passed by value (kernel arguments live in SGPRs).
struct FieldConsts {
  float h;
  float near2;   // (2h)^2
  float tab_scale;  // kFieldTabN / (2h): r -> table coordinate q kFieldTabN / 2
  float tab_high;   // how far tab_scale is rounded up, relative
  float2 tab_a, tab_b;  // h^-5 and h^-3, each as its FP32 value and what that leaves
};

// Near-field coefficient table.  Interval k of
// kFieldTabN covers u = q kFieldTabN / 2 in [k, k + 1) (q = 1 is a boundary,
// so no interval straddles the two forms) and holds two cubics in t = u - k,
// for alpha and for beta, each interpolating the exact FP64 form at the four
// Chebyshev points of the interval: tab[8k + 0..3] = alpha coefficients,
// tab[8k + 4..7] = beta coefficients (ascending powers, h included).  Entry
// kFieldTabN continues the last interval's cubics one interval further, so a
// u that rounds up to kFieldTabN at q -> 2 reads a finite value with no
// clamp.  At FP32 inputs q in [0, 2) the error is at most 1.5e-7 of
// max(|alpha|, (2h)^-5) and of max(|beta|, (2h)^-3); an FP32 evaluation of the
// closed forms stays within 7e-7 and 1.6e-6.  The all-pairs kernels take the
// table at h = 1 (a constant of the code object) times h^-5, h^-3 into LDS; the
// FMM's tables hold h.
//
// Device copies of both tables (split_near_table) hold the first curve's
// cubic of every entry, then the second's: at a 16-byte stride, lanes that
// read neighbouring entries meet in half as many LDS banks as at 32 bytes.
constexpr int kFieldTabN = 64;
constexpr int kFieldTabEntries = kFieldTabN + 1;

// Force-tensor constants.
struct HessConsts {
  float h;
  float near2;       // (4h)^2
  float tab_scale;   // kHessTabN / (4h): r -> table coordinate q kHessTabN / 4
  float tab_high;    // how far tab_scale is rounded up, relative
  float2 tab_a, tab_b;  // h^-4 (both curves), as its FP32 value and what that leaves
};

// Force-curve table: kHessTabN intervals over q in
// (0, 4], 16 per unit, each inside one of the reference's quartic pieces
// (piece p covers (p, p + 1], so an integer q stays with the lower piece).
// Entry e = ceil(u), u = q kHessTabN / 4, covers u in (e - 1, e] and holds two
// cubics in t = u - e, in (-1, 0]: [0..3] C1 / (s h^4), [4..7]
// (C2 - 3 C1) / (s h^4), from which R follows with no further factor.  Entries
// 1 .. kHessTabN interpolate at their interval's four Chebyshev points;
// entry 0 (u = 0, a pair at d = 0) continues entry 1's cubics and entry
// kHessTabN + 1 (u rounded above kHessTabN at q -> 4) entry kHessTabN's, so
// the lookup needs no clamp.  Within 9e-8 of the largest curve value (the
// FP32 rounding of the curves is 6e-8).
constexpr int kHessTabN = 64;
constexpr int kHessTabEntries = kHessTabN + 2;

FieldConsts make_field_consts(double h);
HessConsts make_hess_consts(double h);
void make_field_table(double h, float *tab);  // kFieldTabEntries x 8 floats
void make_hess_table(double h, float *tab);   // kHessTabEntries x 8 floats
// [entries][8] -> [2][entries][4]: the device layout of both tables.
void split_near_table(const float *tab, int entries, float *out);

// ---------------------------------------------------------------------------
// Field pair coefficients from the table (split layout, in LDS), for
// r2 < (2h)^2: alpha, beta such that the pair adds c (3 alpha d (d.m) - beta m);
// `ir` = 1/|d| (may be inf at r2 == 0).  12 VALU operations and two LDS reads,
// where the closed forms of the header take about 30 operations.
__device__ __forceinline__ void field_near_coeffs_tab(const float4 *tab, float tab_scale, float r2,
                                                      float ir, float &alpha, float &beta) {
  // u = q kFieldTabN / 2.  The clamp keeps the pair at d = 0 (ir = inf) at
  // u = 0 instead of 0 x inf; u < kFieldTabN up to rounding at q -> 2, and
  // entry kFieldTabN takes a u rounded up to it.
  const float irc = __builtin_amdgcn_fmed3f(ir, 0.f, 1e30f);
  const float u = r2 * tab_scale * irc;
  const int k = static_cast<int>(u);
  const float t = __builtin_amdgcn_fractf(u);
  const float4 a = tab[k], b = tab[kFieldTabEntries + k];
  alpha = fmaf(fmaf(fmaf(a.w, t, a.z), t, a.y), t, a.x);
  beta = fmaf(fmaf(fmaf(b.w, t, b.z), t, b.y), t, b.x);
}

// The two curves of a force pair within 4h (r2 <= near2) from the table
// (LDS): P = c1 irc and R = dq irc^3.  The caller clamps the inverse
// distance irc to a finite value, so a pair at d = 0 (a particle and itself,
// or two coincident ones) gets finite coefficients, whose terms all vanish
// with d.
__device__ __forceinline__ void hess_near_curves_tab(const float4 *tab, float tab_scale, float r2,
                                                     float irc, float &c1, float &dq) {
  const float u = r2 * irc * tab_scale;  // in [0, kHessTabN], up to rounding
  const float kc = ceilf(u);              // entry 0 .. kHessTabN + 1
  const float t = u - kc;
  const int e = static_cast<int>(kc);
  const float4 a = tab[e], b = tab[kHessTabEntries + e];
  c1 = fmaf(fmaf(fmaf(a.w, t, a.z), t, a.y), t, a.x);
  dq = fmaf(fmaf(fmaf(b.w, t, b.z), t, b.y), t, b.x);
}

}  // namespace mf
