// mf_check64.hip -- FP64 all-pairs field and force on the GPU.
//
// This is the FP64 check path: it evaluates the reference's formulas
// literally (Dipole_B.kern:46-104 for the field, Dipole_hessian.kern:53-238
// with the original Horner curves for the force tensor) in double precision,
// so FP32 and mixed-precision results can be scored at sizes the CPU oracle
// cannot reach.  It is validated against the CPU oracle at small N.
//
// One target per lane, the source index uniform over the wave: source values
// come through scalar loads, with no LDS and no barrier.  The source range is
// split into chunks along grid.y, whose FP64 partial sums a second kernel adds
// in a fixed order: a check on 1,024 samples has 16 waves of targets, which
// alone would leave 252 of the 256 CUs idle for the whole source loop.
// FP64 instructions issue at half the FP32 rate here, so the pair math is what
// bounds these kernels: one v_rsq_f64 with a third-order correction in place
// of a square root and two to five divisions, and the smoothed forms only in
// waves where some pair needs them.  Measured with sources staged in LDS, one target a
// lane and no split / now, 8,192 particles in a cube of 20 at h = 2: field product 3,590 /
// 154 us, force at 1,024 samples 4,170 / 52 us, at all particles 4,190 / 231 us.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "mf_allpairs.hpp"
#include "mf_internal.hpp"

namespace mf {
namespace {

constexpr int kB = 256;

__constant__ double c_C1[4][5] = {
    {9.97813616438174e-09, -2.97897856524718e-08, 2.38918644566813e-09, 4.53199938857366e-08,
     2.44617454752747e-11},
    {-2.76473728643294e-09, 2.86975546540539e-08, -9.94582836806651e-08, 1.25129924573675e-07,
     -2.37010166723652e-08},
    {-1.09679990621465e-09, 9.77055663264614e-09, -2.54781238661150e-08, 2.65020634884934e-09,
     5.00787562417835e-08},
    {3.79927162333632e-10, -6.26368404962679e-09, 3.94760528277489e-08, -1.13580541622200e-07,
     1.27491333574323e-07}};
__constant__ double c_C2[4][5] = {
    {6.69550479838731e-08, -1.61753307173877e-07, 1.68213714992711e-08, 1.34558143036838e-07,
     1.10976027980100e-10},
    {-3.08460139955194e-08, 2.29192245602275e-07, -5.88399621128587e-07, 5.61170054591844e-07,
     -1.14421132829680e-07},
    {3.50477408060213e-09, -5.25956271895141e-08, 2.78876509535747e-07, -6.24199554212217e-07,
     4.91807818904985e-07},
    {7.33485346367840e-10, -9.58855788627803e-09, 4.37085309763591e-08, -7.48004594092261e-08,
     2.34161209605651e-08}};

__device__ inline double horner4(const double *c, double x) {
  return x * (x * (x * (x * c[0] + c[1]) + c[2]) + c[3]) + c[4];
}

// 1/sqrt(r2) to about one unit in the last place: the hardware estimate y times
// 1 + e/2 + 3/8 e^2 + 5/16 e^3, e = 1 - r2 y^2.  Over 6.7e7 inputs |e| was at most 2^-23.1;
// the next term, 35/128 e^4, stays below 2^-53 for any |e| below 2^-12.8.  The clamps keep r2 = 0 and an overflowed
// r2 finite.
__device__ __forceinline__ double rsqrt64(double r2) {
  const double x = fmin(fmax(r2, 1e-290), 1e290);
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-(x * y), y, 1.0);
  return fma(y * e, fma(e, fma(e, 0.3125, 0.375), 0.5), y);
}

// Field pair, Dipole_B.kern:46-104: a1 += alpha (d.m) d, a2 += beta m, for
// out = c (3 a1 - a2), c = 1/(4 pi).
struct FieldConsts64 {
  double near2, inv_h, inv_h3, inv_h5;
};
__device__ __forceinline__ void field_pair64(double dx, double dy, double dz, double mx, double my,
                                             double mz, const FieldConsts64 &fc, double (&a1)[3],
                                             double (&a2)[3]) {
  const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
  const double ir = rsqrt64(r2);
  const double ir2 = ir * ir;
  double beta = ir2 * ir;
  double alpha = beta * ir2;
  if (r2 < fc.near2) {
    const double q = r2 * ir * fc.inv_h;
    const double t = 2.0 - q;
    if (q >= 1.0) {
      const double q3 = q * q * q;
      const double g = -3.0 * (q3 * (((q / 6.0 - 1.2) * q + 3.0) * q - 8.0 / 3.0) + 1.0 / 15.0);
      const double wa = g * beta, wd = t * t * t * fc.inv_h3;
      alpha = (wa - wd) * ir2 * (1.0 / 3.0);
      beta = wa * (1.0 / 3.0) - wd;
    } else {
      alpha = (0.8 - 0.5 * q) * fc.inv_h5;
      beta = (q * q * (4.8 - 2.5 * q) - 8.0 / 3.0) * fc.inv_h3;
    }
  }
  const double s1 = fma(dx, mx, fma(dy, my, dz * mz)) * alpha;
  a1[0] = fma(dx, s1, a1[0]);
  a1[1] = fma(dy, s1, a1[1]);
  a1[2] = fma(dz, s1, a1[2]);
  a2[0] = fma(mx, beta, a2[0]);
  a2[1] = fma(my, beta, a2[1]);
  a2[2] = fma(mz, beta, a2[2]);
}

// Where a chunk's sums go: its slab of the partials, or (one chunk) the outputs.
struct Out64 {
  double *p[3];
  int64_t stride;  // between chunks
  double hc[3];    // added by a single chunk
  __device__ __forceinline__ void put(int64_t i, double a, double b, double c) const {
    const int64_t o = static_cast<int64_t>(blockIdx.y) * stride + i;
    p[0][o] = a + hc[0];
    p[1][o] = b + hc[1];
    p[2][o] = c + hc[2];
  }
};

// Source range [j0, j1) of this block's chunk (grid.y).
__device__ __forceinline__ void chunk_of(int64_t ns, int64_t per, int64_t &j0, int64_t &j1) {
  j0 = static_cast<int64_t>(blockIdx.y) * per;
  j1 = j0 + per < ns ? j0 + per : ns;
}

__global__ __launch_bounds__(kB) void field64_kernel(
    int64_t nt, const double *__restrict__ tx, const double *__restrict__ ty,
    const double *__restrict__ tz, int64_t ns, const double *__restrict__ sx,
    const double *__restrict__ sy, const double *__restrict__ sz, const double *__restrict__ mx,
    const double *__restrict__ my, const double *__restrict__ mz, FieldConsts64 fc, int64_t per,
    Out64 out) {
  int64_t i = static_cast<int64_t>(blockIdx.x) * kB + threadIdx.x;
  const bool valid = i < nt;
  i = valid ? i : nt - 1;
  const double px = tx[i], py = ty[i], pz = tz[i];
  double a1[3] = {0.0, 0.0, 0.0}, a2[3] = {0.0, 0.0, 0.0};
  int64_t j0, j1;
  chunk_of(ns, per, j0, j1);
#pragma unroll 4
  for (int64_t j = j0; j < j1; ++j)
    field_pair64(px - sx[j], py - sy[j], pz - sz[j], mx[j], my[j], mz[j], fc, a1, a2);
  if (!valid) return;
  const double c = 1.0 / (4.0 * kPi);
  out.put(i, c * (3.0 * a1[0] - a2[0]), c * (3.0 * a1[1] - a2[1]), c * (3.0 * a1[2] - a2[2]));
}

// Force: F_i = sum_j B(x_i - x_j)[m_j] m_i with the isotropic closed form of
// Dipole_hessian.kern (far q > 4, near (0, 4] with the original curves):
// F = sum d (P (m.n) + R (d.m)(d.n)) + m P (d.n) + n P (d.m).
__global__ __launch_bounds__(kB) void force64_kernel(
    int64_t n, int64_t nt, const int64_t *__restrict__ idx, const double *__restrict__ x,
    const double *__restrict__ y, const double *__restrict__ z, const double *__restrict__ mx,
    const double *__restrict__ my, const double *__restrict__ mz, double h, int64_t per,
    Out64 out) {
  int64_t i = static_cast<int64_t>(blockIdx.x) * kB + threadIdx.x;
  const bool valid = i < nt;
  i = valid ? i : nt - 1;
  int64_t ii = idx ? idx[i] : i;
  ii = (ii >= 0 && ii < n) ? ii : 0;
  const double px = x[ii], py = y[ii], pz = z[ii];
  const double nx = mx[ii], ny = my[ii], nz = mz[ii];
  const double inv_h = 1.0 / h, inv_h4 = 1.0 / (h * h * h * h), near2 = 16.0 * h * h;
  const double cfar = 3.0 * kMu0 / (4.0 * kPi);
  double ad[3] = {0.0, 0.0, 0.0}, am[3] = {0.0, 0.0, 0.0}, an = 0.0;
  int64_t j0, j1;
  chunk_of(n, per, j0, j1);
#pragma unroll 2
  for (int64_t j = j0; j < j1; ++j) {
    const double dx = px - x[j], dy = py - y[j], dz = pz - z[j];
    const double jx = mx[j], jy = my[j], jz = mz[j];
    const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
    const double ir = rsqrt64(r2);
    const double ir2 = ir * ir;
    double P = cfar * (ir2 * ir2 * ir);
    double R = -5.0 * P * ir2;
    // the margin covers the rounding of r2: q itself decides below
    if (r2 < near2 * (1.0 + 1e-12)) {
      // |d| correctly rounded, as a square root: an integer q (a regular
      // lattice) has to stay with the lower curve
      double r = r2 * ir;
      r = fma(fma(-r, r, r2), 0.5 * ir, r);
      const double q = r * inv_h;
      if (q == 0.0) {
        P = R = 0.0;
      } else if (q <= 4.0) {
        const int kk = (q <= 1.0) ? 0 : (q <= 2.0) ? 1 : (q <= 3.0) ? 2 : 3;
        const double c1 = horner4(c_C1[kk], q), c2 = horner4(c_C2[kk], q);
        P = c1 * inv_h4 * ir;
        R = (c2 - 3.0 * c1) * inv_h4 * (ir2 * ir);
      }
    }
    const double dm = fma(dx, jx, fma(dy, jy, dz * jz));
    const double dn = fma(dx, nx, fma(dy, ny, dz * nz));
    const double mn = fma(jx, nx, fma(jy, ny, jz * nz));
    const double e = fma(R, dm * dn, P * mn);
    const double f = P * dn;
    ad[0] = fma(dx, e, ad[0]);
    ad[1] = fma(dy, e, ad[1]);
    ad[2] = fma(dz, e, ad[2]);
    am[0] = fma(jx, f, am[0]);
    am[1] = fma(jy, f, am[1]);
    am[2] = fma(jz, f, am[2]);
    an = fma(P, dm, an);
  }
  if (!valid) return;
  out.put(i, ad[0] + am[0] + nx * an, ad[1] + am[1] + ny * an, ad[2] + am[2] + nz * an);
}

// out[c][i] = h_c + the chunks' partials in chunk order.  A block takes 64
// targets of one component; its four waves add every fourth chunk each and
// the first wave adds the four sums.
__global__ __launch_bounds__(256) void reduce64_kernel(int64_t nt, int nchunk,
                                                       const double *__restrict__ partial,
                                                       double h0, double h1, double h2,
                                                       double *__restrict__ ox,
                                                       double *__restrict__ oy,
                                                       double *__restrict__ oz) {
  __shared__ double sh[4][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, a = blockIdx.y;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 64 + lane;
  double s = 0.0;
  if (i < nt)
    for (int c = w; c < nchunk; c += 4) s += partial[(static_cast<int64_t>(c) * 3 + a) * nt + i];
  sh[w][lane] = s;
  __syncthreads();
  if (w != 0 || i >= nt) return;
  const double hc = a == 0 ? h0 : a == 1 ? h1 : h2;
  double *out = a == 0 ? ox : a == 1 ? oy : oz;
  out[i] = ((sh[0][lane] + sh[1][lane]) + (sh[2][lane] + sh[3][lane])) + hc;
}

// Source chunks of a launch over nt targets: eight waves per SIMD (two blocks
// of four waves each per CU and SIMD slot) where the targets alone give fewer,
// each chunk at least kMinChunk sources (below that the partials cost more
// than the idle CUs).
constexpr int64_t kMinChunk = 64;
struct Split64 {
  int64_t per;
  int nchunk;
};
Split64 split64(const mf_ctx *ctx, int64_t nt, int64_t ns) {
  const int64_t blocks = (nt + kB - 1) / kB;
  const int64_t want = (static_cast<int64_t>(ctx->num_cu) * 8 + blocks - 1) / blocks;
  const int64_t most = std::max<int64_t>(1, ns / kMinChunk);
  const int64_t nchunk = std::max<int64_t>(1, std::min(want, most));
  Split64 s{};
  s.per = std::max<int64_t>(1, (ns + nchunk - 1) / nchunk);
  s.nchunk = static_cast<int>(std::max<int64_t>(1, (ns + s.per - 1) / s.per));
  return s;
}

// Runs launch(grid, per, out) over the chunks and adds their partials.  These
// entry points need no scratch of their own when the partials cannot be had
// (the workspace would have to grow inside a stream capture, or the allocation
// fails): one chunk then writes the outputs.
template <class Launch>
Status run_chunks(mf_ctx *ctx, int64_t nt, int64_t ns, const double *hconst, double *ox, double *oy,
                  double *oz, const Launch &launch) {
  const double hc[3] = {hconst ? hconst[0] : 0.0, hconst ? hconst[1] : 0.0, hconst ? hconst[2] : 0.0};
  Split64 sp = split64(ctx, nt, ns);
  double *part = nullptr;
  if (sp.nchunk > 1) {
    void *p = nullptr;
    if (workspace_now(ctx, "check64_partial", sizeof(double) * 3 * static_cast<size_t>(nt) * sp.nchunk, &p))
      part = static_cast<double *>(p);
    else
      sp = Split64{std::max<int64_t>(ns, 1), 1};
  }
  const Out64 out = part ? Out64{{part, part + nt, part + 2 * nt}, 3 * nt, {0.0, 0.0, 0.0}}
                         : Out64{{ox, oy, oz}, 0, {hc[0], hc[1], hc[2]}};
  launch(dim3(grid_for(nt, kB), sp.nchunk), sp.per, out);
  MF_LAUNCH_CHECK();
  if (!part) return Status::Ok();
  hipLaunchKernelGGL(reduce64_kernel, dim3(grid_for(nt, 64), 3), dim3(256), 0, ctx->stream, nt,
                     sp.nchunk, part, hc[0], hc[1], hc[2], ox, oy, oz);
  MF_LAUNCH_CHECK();
  return Status::Ok();
}

}  // namespace

Status field_allpairs_f64(mf_ctx *ctx, int64_t nt, const double *tx, const double *ty,
                          const double *tz, int64_t ns, const double *sx, const double *sy,
                          const double *sz, const double *mx, const double *my,
                          const double *mz, double h, const double *hconst, double *ox,
                          double *oy, double *oz) {
  if (nt == 0) return Status::Ok();
  KernelTimer timer(ctx, "field64");
  const FieldConsts64 fc{4.0 * h * h, 1.0 / h, 1.0 / (h * h * h), 1.0 / (h * h * h * h * h)};
  return run_chunks(ctx, nt, ns, hconst, ox, oy, oz, [&](dim3 grid, int64_t per, const Out64 &out) {
    hipLaunchKernelGGL(field64_kernel, grid, dim3(kB), 0, ctx->stream, nt, tx, ty, tz, ns, sx, sy,
                       sz, mx, my, mz, fc, per, out);
  });
}

namespace {
Status force64(mf_ctx *ctx, int64_t n, const double *x, const double *y, const double *z,
               const double *mx, const double *my, const double *mz, double h, int64_t nt,
               const int64_t *idx, double *fx, double *fy, double *fz) {
  if (nt == 0 || n == 0) return Status::Ok();
  KernelTimer timer(ctx, "force64");
  return run_chunks(ctx, nt, n, nullptr, fx, fy, fz, [&](dim3 grid, int64_t per, const Out64 &out) {
    hipLaunchKernelGGL(force64_kernel, grid, dim3(kB), 0, ctx->stream, n, nt, idx, x, y, z, mx, my,
                       mz, h, per, out);
  });
}
}  // namespace

Status force_allpairs_f64(mf_ctx *ctx, int64_t n, const double *x, const double *y,
                          const double *z, const double *mx, const double *my, const double *mz,
                          double h, double *fx, double *fy, double *fz) {
  return force64(ctx, n, x, y, z, mx, my, mz, h, n, nullptr, fx, fy, fz);
}

Status force_subset_f64(mf_ctx *ctx, int64_t n, const double *x, const double *y,
                        const double *z, const double *mx, const double *my, const double *mz,
                        double h, int64_t nt, const int64_t *idx, double *fx, double *fy,
                        double *fz) {
  return force64(ctx, n, x, y, z, mx, my, mz, h, nt, idx, fx, fy, fz);
}

}  // namespace mf
