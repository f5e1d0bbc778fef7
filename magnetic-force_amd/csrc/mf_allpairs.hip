// mf_allpairs.hip -- tiled all-pairs field and force kernels for gfx950.
//
// Replaces the reference's naive kernels (magnetic_solver/magnetic_force.cu):
//   cuda_Apply_G            :8-110    -> field_allpairs_kernel
//   cuda_ext_field_kernel   :120-237  -> field_allpairs_kernel (separate sources),
//                                        field_few_kernel (a few of them)
//   fitted_force_ofM_kernel :516-605  -> force_allpairs_kernel
//   cuda_ext_fitted_force_tensor_kernel :432-512 -> hessian_allpairs_kernel,
//                                        hessian_few_kernel
//
// Design (one wavefront = 16 TPT targets):
//  * Sources live in HBM as 32-byte records {x,y,z,0, mx,my,mz,0}, padded to a
//    whole tile with far-away zero-moment records.
//  * A wave stages 64 records at a time in its own LDS (no barrier: the block
//    is the wave) and reads them back into vector registers: lane l evaluates
//    its TPT targets (l mod 16, + 16, ...) against every fourth record (those
//    of l / 16), so one 24-byte LDS read serves TPT pairs.  A SIMD
//    issues FP32 vector instructions of two waves at once (2.3 cycles each)
//    unless both read a scalar register (4.4), and 9 of a field pair's 20 did
//    while the sources sat in scalar registers.
//  * Sources are cut into tiles of 64 with a precomputed bounding box.  Each
//    wave computes the bounding box of its own targets once; a tile whose
//    box-to-box distance exceeds the smoothing support runs a branch-free
//    far-field loop (pure dipole, one v_rsq_f32 per pair).  Other tiles run
//    the mixed loop, which reads the smoothed coefficients from a table in LDS.
//  * Sums of up to four tiles (64 terms a lane; of one for the force of a set on itself) are
//    FP32; they are accumulated in FP64, so the summation error does not grow with N.
//  * The source range is split into chunks of whole 16-record groups along
//    grid.y to give the 256 CUs enough waves; chunk partials (FP64) are summed
//    in a fixed order by a separate reduction kernel, so results are
//    deterministic.
//  * A record set's field and force on itself (4,096 records or more) evaluate
//    each unordered pair once (field_self_kernel, force_self_kernel below).
//  Measured per launch, at first (scalar sources, closed-form coefficients, chunks
//  of whole tiles), directed kernels now, pairs once: field 22.6 / 8.4 us at 512
//  particles, 65.0 / 52.8 / 41.8 us at 8,192, 33.8 / 28.3 / 22.6 ms at 262,144; force
//  36.9 / 9.8 us, 91.9 / 76.2 / 57.0 us, 49.7 / 40.0 / 29.1 ms.  Field and tensor of
//  4,096 records on 65,520 targets 0.43 / 0.33 ms.  The VALU bounds the large sizes: a
//  directed far field pair is 19 plain instructions at 2.3 cycles and one v_rsq_f32 at 16.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "mf_allpairs.hpp"
#include "mf_pair_once.hpp"
#include "mf_internal.hpp"
#include "mf_pair.hpp"

namespace mf {

namespace {

// ---------------------------------------------------------------------------
// Near-pair coefficient tables (mf_pair.hpp describes their entries).  The
// fits are constexpr: at h = 1 they are the constants of the all-pairs kernels
// (alpha h^5, beta h^3 and the curves times h^4 depend on q alone), which so
// need no table per h; the FMM builds its tables with h included on the host.

// alpha h^5 and beta h^3 of a near pair at q < 2, in FP64 (the forms of the
// mf_pair.hpp header; g unexpanded, which is accurate in FP64).
constexpr void near_coeffs_f64(double q, double &a, double &b) {
  if (q < 1.0) {
    a = 0.8 - 0.5 * q;
    b = -8.0 / 3.0 + q * q * (4.8 - 2.5 * q);
    return;
  }
  const double q3 = q * q * q;
  const double g = -3.0 * (q3 * (((q / 6.0 - 1.2) * q + 3.0) * q - 8.0 / 3.0) + 1.0 / 15.0);
  const double w = (2.0 - q) * (2.0 - q) * (2.0 - q);
  a = (g / q3 - w) / (3.0 * q * q);
  b = g / (3.0 * q3) - w;
}

// cos((2 i + 1) pi / 8): the Chebyshev points of a cubic.
constexpr double kCheb[4] = {0.92387953251128674, 0.38268343236508977, -0.38268343236508977,
                             -0.92387953251128674};

// Power-basis coefficients c[0..3] of the cubic through (t[i], y[i]), i < 4
// (Gaussian elimination with partial pivoting on the Vandermonde system).
constexpr void cubic_through(const double (&t)[4], const double (&y)[4], double (&c)[4]) {
  double m[4][5] = {};
  for (int i = 0; i < 4; ++i) {
    double p = 1.0;
    for (int j = 0; j < 4; ++j, p *= t[i]) m[i][j] = p;
    m[i][4] = y[i];
  }
  auto mag = [](double v) { return v < 0.0 ? -v : v; };
  for (int col = 0; col < 4; ++col) {
    int piv = col;
    for (int i = col + 1; i < 4; ++i)
      if (mag(m[i][col]) > mag(m[piv][col])) piv = i;
    for (int j = 0; j < 5; ++j) {
      const double x = m[col][j];
      m[col][j] = m[piv][j];
      m[piv][j] = x;
    }
    for (int i = col + 1; i < 4; ++i) {
      const double f = m[i][col] / m[col][col];
      for (int j = col; j < 5; ++j) m[i][j] -= f * m[col][j];
    }
  }
  for (int i = 3; i >= 0; --i) {
    double s = m[i][4];
    for (int j = i + 1; j < 4; ++j) s -= m[i][j] * c[j];
    c[i] = s / m[i][i];
  }
}

// Coefficients (ascending powers) of c(t + s) from those of the cubic c(t).
constexpr void shift_cubic(const double *c, double s, double *out) {
  out[0] = ((c[3] * s + c[2]) * s + c[1]) * s + c[0];
  out[1] = (3.0 * c[3] * s + 2.0 * c[2]) * s + c[1];
  out[2] = 3.0 * c[3] * s + c[2];
  out[3] = c[3];
}

// v_rsq_f32 is low by 7.4e-9 in the mean over all significands, and with it the r and the
// q of a table lookup: the tables hold the curves at q (1 + kRsqLow).
constexpr double kRsqLow = 7.4e-9;

// The FP32 coefficients of a cubic over t in [0, 1] (dir = 1) or (-1, 0] (dir = -1).  What
// the rounding of one coefficient takes off is given to the later ones, as their best fit
// to it over the interval: of an error d of the constant term a quarter remains in the
// mean square and a sixteenth in the mean.  Errors of neighbouring pairs, whose distances
// read the same entries, do not average out: with the coefficients simply rounded a field
// of equal moments on a jittered lattice at h = 2 was 3.4e-8 too large.
constexpr void round_cubic(const double *c, int dir, float *out) {
  out[0] = static_cast<float>(c[0]);
  const double e0 = c[0] - static_cast<double>(out[0]);
  const double c1 = c[1] + dir * 7.5 * e0;
  out[1] = static_cast<float>(c1);
  const double e1 = c1 - static_cast<double>(out[1]);
  const double c2 = c[2] - 15.0 * e0 + dir * 3.0 * e1;
  out[2] = static_cast<float>(c2);
  const double e2 = c2 - static_cast<double>(out[2]);
  out[3] = static_cast<float>(c[3] + dir * 8.75 * e0 - 2.1 * e1 + dir * (7.0 / 6.0) * e2);
}

// put(entry, cubic of alpha, cubic of beta) for every entry of the field table,
// alpha times fa and beta times fb.
template <class Put>
constexpr void fill_field_table(double fa, double fb, const Put &put) {
  double t[4] = {};
  for (int i = 0; i < 4; ++i) t[i] = 0.5 + 0.5 * kCheb[i];
  double ca[4] = {}, cb[4] = {};
  for (int k = 0; k < kFieldTabN; ++k) {
    double ya[4] = {}, yb[4] = {};
    for (int i = 0; i < 4; ++i) {
      near_coeffs_f64((k + t[i]) * (2.0 / kFieldTabN) * (1.0 + kRsqLow), ya[i], yb[i]);
      ya[i] *= fa;
      yb[i] *= fb;
    }
    cubic_through(t, ya, ca);
    cubic_through(t, yb, cb);
    put(k, ca, cb);
  }
  double sa[4] = {}, sb[4] = {};  // the last interval's cubics, one interval on
  shift_cubic(ca, 1.0, sa);
  shift_cubic(cb, 1.0, sb);
  put(kFieldTabN, sa, sb);
}

// Fitted curve table of the reference (Dipole_hessian.kern:53-61), highest
// power first.  Kept as data: the force must use exactly these curves.
constexpr double kC1[4][5] = {
    {9.97813616438174e-09, -2.97897856524718e-08, 2.38918644566813e-09, 4.53199938857366e-08,
     2.44617454752747e-11},
    {-2.76473728643294e-09, 2.86975546540539e-08, -9.94582836806651e-08, 1.25129924573675e-07,
     -2.37010166723652e-08},
    {-1.09679990621465e-09, 9.77055663264614e-09, -2.54781238661150e-08, 2.65020634884934e-09,
     5.00787562417835e-08},
    {3.79927162333632e-10, -6.26368404962679e-09, 3.94760528277489e-08, -1.13580541622200e-07,
     1.27491333574323e-07}};
constexpr double kC2[4][5] = {
    {6.69550479838731e-08, -1.61753307173877e-07, 1.68213714992711e-08, 1.34558143036838e-07,
     1.10976027980100e-10},
    {-3.08460139955194e-08, 2.29192245602275e-07, -5.88399621128587e-07, 5.61170054591844e-07,
     -1.14421132829680e-07},
    {3.50477408060213e-09, -5.25956271895141e-08, 2.78876509535747e-07, -6.24199554212217e-07,
     4.91807818904985e-07},
    {7.33485346367840e-10, -9.58855788627803e-09, 4.37085309763591e-08, -7.48004594092261e-08,
     2.34161209605651e-08}};

// put(entry, cubic of C1, cubic of C2 - 3 C1) for every entry of the force table,
// both times scale / (3 mu0 / (4 pi)).
template <class Put>
constexpr void fill_hess_table(double scale, const Put &put) {
  const double f = scale / (3.0 * kMu0 / (4.0 * kPi));
  constexpr int per_unit = kHessTabN / 4;
  double t[4] = {};
  for (int i = 0; i < 4; ++i) t[i] = -0.5 + 0.5 * kCheb[i];
  double cc[4] = {}, cd[4] = {}, first_c[4] = {}, first_d[4] = {};
  for (int e = 1; e <= kHessTabN; ++e) {  // entry e: u in (e - 1, e]
    const int piece = (e - 1) / per_unit;
    double yc[4] = {}, yd[4] = {};
    for (int i = 0; i < 4; ++i) {
      const double q = (e + t[i]) / per_unit * (1.0 + kRsqLow);
      double c1 = 0.0, c2 = 0.0;
      for (int j = 0; j < 5; ++j) {
        c1 = c1 * q + kC1[piece][j];
        c2 = c2 * q + kC2[piece][j];
      }
      yc[i] = f * c1;
      yd[i] = f * (c2 - 3.0 * c1);
    }
    cubic_through(t, yc, cc);
    cubic_through(t, yd, cd);
    put(e, cc, cd);
    if (e == 1)
      for (int j = 0; j < 4; ++j) {
        first_c[j] = cc[j];
        first_d[j] = cd[j];
      }
  }
  double sc[4] = {}, sd[4] = {};
  shift_cubic(cc, 1.0, sc);  // entry kHessTabN + 1 continues the last one
  shift_cubic(cd, 1.0, sd);
  put(kHessTabN + 1, sc, sd);
  shift_cubic(first_c, -1.0, sc);  // entry 0 (u = 0) continues entry 1
  shift_cubic(first_d, -1.0, sd);
  put(0, sc, sd);
}

// The tables at h = 1 in the split layout (split_near_table).
template <int N>
struct UnitTable {
  float v[2][N][4];
};
constexpr UnitTable<kFieldTabEntries> unit_field_table() {
  UnitTable<kFieldTabEntries> t{};
  fill_field_table(1.0, 1.0, [&](int e, const double *a, const double *b) {
    round_cubic(a, 1, t.v[0][e]);
    round_cubic(b, 1, t.v[1][e]);
  });
  return t;
}
constexpr UnitTable<kHessTabEntries> unit_hess_table() {
  UnitTable<kHessTabEntries> t{};
  fill_hess_table(1.0, [&](int e, const double *a, const double *b) {
    round_cubic(a, -1, t.v[0][e]);
    round_cubic(b, -1, t.v[1][e]);
  });
  return t;
}
static __device__ const UnitTable<kFieldTabEntries> d_field_tab __attribute__((aligned(16))) =
    unit_field_table();
static __device__ const UnitTable<kHessTabEntries> d_hess_tab __attribute__((aligned(16))) =
    unit_hess_table();

constexpr float kFieldTabMid = 0.5f, kHessTabMid = -0.5f;  // middle of an entry's t

void store_entry(float *tab, int e, int dir, const double *ca, const double *cb) {
  round_cubic(ca, dir, tab + 8 * e);
  round_cubic(cb, dir, tab + 8 * e + 4);
}

__device__ __forceinline__ float wave_min(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = fminf(v, __shfl_xor(v, off, 64));
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  return v;
}
__device__ __forceinline__ float uniform_f(float v) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

// ---------------------------------------------------------------------------
// Packing and tile boxes.

// One wave per tile of kTile records: the records (padding included) and the
// tile's bounding box (padding excluded) in one pass.
__global__ void pack_tiles_kernel(int64_t n, int64_t ntiles, const float *__restrict__ x,
                                  const float *__restrict__ y, const float *__restrict__ z,
                                  const float *__restrict__ mx, const float *__restrict__ my,
                                  const float *__restrict__ mz, SrcRec *__restrict__ out,
                                  float4 *__restrict__ boxes) {
  const int lane = threadIdx.x & 63;
  const int64_t tile = static_cast<int64_t>(blockIdx.x) * (blockDim.x / 64) + (threadIdx.x >> 6);
  if (tile >= ntiles) return;
  const int64_t i = tile * kTile + lane;
  SrcRec r{kPadCoord, kPadCoord, kPadCoord, 0.f, 0.f, 0.f, 0.f, 0.f};
  float lx = INFINITY, ly = INFINITY, lz = INFINITY;
  float hx = -INFINITY, hy = -INFINITY, hz = -INFINITY;
  if (i < n) {
    lx = hx = r.x = x[i];
    ly = hy = r.y = y[i];
    lz = hz = r.z = z[i];
    r.mx = mx ? mx[i] : 0.f;
    r.my = my ? my[i] : 0.f;
    r.mz = mz ? mz[i] : 0.f;
  }
  out[i] = r;
  lx = wave_min(lx);
  ly = wave_min(ly);
  lz = wave_min(lz);
  hx = wave_max(hx);
  hy = wave_max(hy);
  hz = wave_max(hz);
  if (lane == 0) {
    boxes[2 * tile] = make_float4(lx, ly, lz, 0.f);
    boxes[2 * tile + 1] = make_float4(hx, hy, hz, 0.f);
  }
}

__global__ void pack_moments_kernel(int64_t n, const float *__restrict__ mx,
                                    const float *__restrict__ my, const float *__restrict__ mz,
                                    float scale, SrcRec *__restrict__ out) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float4 m = make_float4(scale * mx[i], scale * my[i], scale * mz[i], 0.f);
  reinterpret_cast<float4 *>(out + i)[1] = m;
}

// Distance^2 between two axis-aligned boxes (0 when they overlap).
__device__ __forceinline__ float box_dist2(float tlx, float tly, float tlz, float thx, float thy,
                                           float thz, float4 slo, float4 shi) {
  const float dx = fmaxf(0.f, fmaxf(tlx - shi.x, slo.x - thx));
  const float dy = fmaxf(0.f, fmaxf(tly - shi.y, slo.y - thy));
  const float dz = fmaxf(0.f, fmaxf(tlz - shi.z, slo.z - thz));
  return dx * dx + dy * dy + dz * dz;
}

// ---------------------------------------------------------------------------
// The wave's share of a launch: targets 16 TPT blockIdx.x + 16 k + (lane mod
// 16), k < TPT; source records [16 sub0, 16 sub1).

constexpr int kSub = 16;    // records per group, the granularity of a chunk
constexpr int kFlush = 4;   // tiles between FP64 accumulations

struct SourceRange {
  int64_t sub0, sub1;
};
__device__ __forceinline__ SourceRange chunk_range(int64_t nsub, int64_t per) {
  const int64_t s0 = static_cast<int64_t>(blockIdx.y) * per;
  return {s0, s0 + per < nsub ? s0 + per : nsub};
}

// Bounding box of the wave's targets (uniform).
struct WaveBox {
  float lx, ly, lz, hx, hy, hz;
};
template <int TPT>
__device__ __forceinline__ WaveBox target_box(const float (&tx)[TPT], const float (&ty)[TPT],
                                              const float (&tz)[TPT]) {
  float v[6] = {tx[0], ty[0], tz[0], tx[0], ty[0], tz[0]};
#pragma unroll
  for (int k = 1; k < TPT; ++k) {
    v[0] = fminf(v[0], tx[k]);
    v[1] = fminf(v[1], ty[k]);
    v[2] = fminf(v[2], tz[k]);
    v[3] = fmaxf(v[3], tx[k]);
    v[4] = fmaxf(v[4], ty[k]);
    v[5] = fmaxf(v[5], tz[k]);
  }
#pragma unroll
  for (int off = 8; off >= 1; off >>= 1)  // the four groups of 16 lanes hold the same targets
#pragma unroll
    for (int a = 0; a < 6; ++a) {
      const float o = __shfl_xor(v[a], off, 64);
      v[a] = a < 3 ? fminf(v[a], o) : fmaxf(v[a], o);
    }
  return {uniform_f(v[0]), uniform_f(v[1]), uniform_f(v[2]),
          uniform_f(v[3]), uniform_f(v[4]), uniform_f(v[5])};
}

// Up to 64 staged records.
struct Staged {
  float4 a[kTile];  // x, y, z, mx
  float2 b[kTile];  // my, mz
};

// Two steps of a tile: the lane's two records, and its TPT targets' distances
// and inverse distances to each (index g TPT + k).  The reciprocal square roots run
// together at raised wave priority: v_rsq_f32 holds its SIMD for about 16 cycles
// where an FMA takes 2.3, and runs that start at once leave the other waves'
// plain VALU work in longer stretches.  262,144 particles with one step and no
// priority / one step / two steps / four: field 29.9 / 28.8 / 28.7 / 29.0 ms, force
// 42.9 / 40.8 / 40.3 / 40.3.
constexpr int kSteps = 2;
template <int TPT>
struct StepPairs {
  float4 u[kSteps];
  float2 v[kSteps];
  float dx[kSteps * TPT], dy[kSteps * TPT], dz[kSteps * TPT], r2[kSteps * TPT], ir[kSteps * TPT];
  __device__ __forceinline__ StepPairs(const Staged &st, int j, int q, const float (&tx)[TPT],
                                       const float (&ty)[TPT], const float (&tz)[TPT]) {
#pragma unroll
    for (int g = 0; g < kSteps; ++g) {
      u[g] = st.a[4 * (j + g) + q];
      v[g] = st.b[4 * (j + g) + q];
#pragma unroll
      for (int k = 0; k < TPT; ++k) {
        const int i = g * TPT + k;
        dx[i] = tx[k] - u[g].x;
        dy[i] = ty[k] - u[g].y;
        dz[i] = tz[k] - u[g].z;
        r2[i] = fmaf(dx[i], dx[i], fmaf(dy[i], dy[i], dz[i] * dz[i]));
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int i = 0; i < kSteps * TPT; ++i) ir[i] = __builtin_amdgcn_rsqf(r2[i]);
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
  }
};

// Walks the wave's sources: stages each tile's part of the range and calls
// body(steps, dist2): `steps` groups of four records are staged (record 4 j + q
// is lane group q's j-th), dist2 is the distance^2 from the wave's targets to
// the tile's box.  flush() runs every kFlush tiles and at the end.  The next
// part's records are loaded before the current one is evaluated.
template <class Body, class Flush>
__device__ __forceinline__ void walk_sources(const SrcRec *__restrict__ src,
                                             const float4 *__restrict__ boxes, SourceRange r,
                                             const WaveBox &t, Staged &st, int lane,
                                             const Body &body, const Flush &flush) {
  const float4 *__restrict__ rec = reinterpret_cast<const float4 *>(src);
  constexpr int kPer = kTile / kSub;  // groups per tile
  auto part = [&](int64_t s) {        // groups of s's tile that belong to the range
    const int64_t e = (s / kPer + 1) * kPer;
    return static_cast<int>((e < r.sub1 ? e : r.sub1) - s);
  };
  // the last record of a short part is read again by the lanes past its end
  auto load = [&](int64_t s, int cnt, float4 &p, float4 &m) {
    const int64_t j = s * kSub + min(lane, cnt * kSub - 1);
    p = rec[2 * j];
    m = rec[2 * j + 1];
  };
  int since = 0;
  int64_t s = r.sub0;
  if (s >= r.sub1) return;
  int cnt = part(s);
  float4 p, m;
  load(s, cnt, p, m);
  while (true) {
    __builtin_amdgcn_wave_barrier();  // the previous part has been read
    st.a[lane] = make_float4(p.x, p.y, p.z, m.x);
    st.b[lane] = make_float2(m.y, m.z);
    __builtin_amdgcn_wave_barrier();
    const int64_t tile = s / kPer;
    const float4 lo = boxes[2 * tile], hi = boxes[2 * tile + 1];
    const int steps = 4 * cnt;
    s += cnt;
    const bool more = s < r.sub1;
    if (more) {
      cnt = part(s);
      load(s, cnt, p, m);
    }
    body(steps, uniform_f(box_dist2(t.lx, t.ly, t.lz, t.hx, t.hy, t.hz, lo, hi)));
    if (++since == kFlush || !more) {
      flush();
      since = 0;
    }
    if (!more) break;
  }
}

// The same over a few sources read from the caller's arrays: each wave stages whole tiles
// and bounds them itself.
template <class Body, class Flush>
__device__ __forceinline__ void walk_arrays(const SourceArrays &src, const WaveBox &t, Staged &st,
                                            int lane, const Body &body, const Flush &flush) {
  for (int s = 0; s < src.n; s += kTile) {
    const int cnt = min(src.n - s, kTile), j = s + lane;
    const bool live = lane < cnt;
    float p[3] = {kPadCoord, kPadCoord, kPadCoord}, m[3] = {0.f, 0.f, 0.f};
    if (live) {
      p[0] = src.x[j];
      p[1] = src.y[j];
      p[2] = src.z[j];
      m[0] = src.mx[j];
      m[1] = src.my[j];
      m[2] = src.mz[j];
    }
    float4 lo, hi;
    lo.x = uniform_f(wave_min(live ? p[0] : INFINITY));
    lo.y = uniform_f(wave_min(live ? p[1] : INFINITY));
    lo.z = uniform_f(wave_min(live ? p[2] : INFINITY));
    hi.x = uniform_f(wave_max(live ? p[0] : -INFINITY));
    hi.y = uniform_f(wave_max(live ? p[1] : -INFINITY));
    hi.z = uniform_f(wave_max(live ? p[2] : -INFINITY));
    __builtin_amdgcn_wave_barrier();  // the previous tile has been read
    st.a[lane] = make_float4(p[0], p[1], p[2], m[0]);
    st.b[lane] = make_float2(m[1], m[2]);
    __builtin_amdgcn_wave_barrier();
    body(4 * ((cnt + kSub - 1) / kSub),
         uniform_f(box_dist2(t.lx, t.ly, t.lz, t.hx, t.hy, t.hz, lo, hi)));
    if ((s / kTile + 1) % kFlush == 0 || s + kTile >= src.n) flush();
  }
}

// A unit table into LDS, its curves times consts.tab_a and tab_b, by `threads`.  Roundings
// of the constants would weigh on all near pairs alike, so the factors are FP32 values and
// what these leave, and the curves are moved by what tab_scale is off: u = (entry + t) is
// high by tab_high of itself, the mean over the entry (at t = `mid`) taken for all of it.
template <int N, class Consts>
__device__ __forceinline__ void load_table(const UnitTable<N> &src, const Consts &consts, float mid,
                                           float4 (&dst)[2 * N], int tid, int threads) {
  const float4 *__restrict__ t = reinterpret_cast<const float4 *>(&src);
  for (int i = tid; i < 2 * N; i += threads) {
    const float4 c = t[i];
    const float2 f = i < N ? consts.tab_a : consts.tab_b;
    const float u = static_cast<float>(i < N ? i : i - N) + mid;
    const float moved = -consts.tab_high * u * c.y * f.x;
    dst[i] = make_float4(fmaf(c.x, f.x, fmaf(c.x, f.y, moved)), fmaf(c.y, f.x, c.y * f.y),
                         fmaf(c.z, f.x, c.z * f.y), fmaf(c.w, f.x, c.w * f.y));
  }
}

// Sum over the four lane groups (the same targets against a quarter of the
// records each).
__device__ __forceinline__ double group_sum(double v) {
  v += __shfl_xor(v, 16, 64);
  v += __shfl_xor(v, 32, 64);
  return v;
}

// ---------------------------------------------------------------------------
// Field: partial[chunk][c][i] = c * sum_{j in chunk} (3 alpha d (d.m) - beta m)_c

// walk(box, staged, body, flush) takes the wave along its sources, put(a, i, v) receives
// target i's sum.
template <int TPT, class Walk, class Put>
__device__ __forceinline__ void field_wave(const Points &tgt, int64_t nt, const FieldConsts &fc,
                                           const Walk &walk, const Put &put) {
  __shared__ Staged st;
  __shared__ float4 s_tab[2 * kFieldTabEntries];
  const int lane = threadIdx.x, c = lane & 15, q = lane >> 4;
  const int64_t tbase = static_cast<int64_t>(blockIdx.x) * (16 * TPT);
  float tx[TPT], ty[TPT], tz[TPT];
#pragma unroll
  for (int k = 0; k < TPT; ++k) {
    const int64_t i = min(tbase + 16 * k + c, nt - 1) * tgt.stride;
    tx[k] = tgt.x[i];
    ty[k] = tgt.y[i];
    tz[k] = tgt.z[i];
  }
  bool have_tab = false;  // read on the first mixed tile
  double acc[TPT][3];
  float a1[TPT][3], a2[TPT][3];
#pragma unroll
  for (int k = 0; k < TPT; ++k)
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      acc[k][a] = 0.0;
      a1[k][a] = a2[k][a] = 0.f;
    }
  auto body = [&](int steps, float dist2) {
    if (dist2 >= fc.near2) {
      // far tile: every pair has q >= 2 (pure dipole)
#pragma unroll 1
      for (int j = 0; j < steps; j += kSteps) {
        const StepPairs<TPT> sp(st, j, q, tx, ty, tz);
#pragma unroll
        for (int i = 0; i < kSteps * TPT; ++i) {
          const int k = i % TPT;
          const float4 u = sp.u[i / TPT];
          const float2 v = sp.v[i / TPT];
          const float dx = sp.dx[i], dy = sp.dy[i], dz = sp.dz[i], ir = sp.ir[i];
          const float ir2 = ir * ir;
          const float ir3 = ir2 * ir;
          const float dm = fmaf(dx, u.w, fmaf(dy, v.x, dz * v.y));
          const float s1 = dm * (ir3 * ir2);
          a1[k][0] = fmaf(dx, s1, a1[k][0]);
          a1[k][1] = fmaf(dy, s1, a1[k][1]);
          a1[k][2] = fmaf(dz, s1, a1[k][2]);
          a2[k][0] = fmaf(u.w, ir3, a2[k][0]);
          a2[k][1] = fmaf(v.x, ir3, a2[k][1]);
          a2[k][2] = fmaf(v.y, ir3, a2[k][2]);
        }
      }
    } else {
      // mixed tile: smoothed near field where q < 2
      if (!have_tab) {
        load_table(d_field_tab, fc, kFieldTabMid, s_tab, lane, 64);
        __builtin_amdgcn_wave_barrier();
        have_tab = true;
      }
#pragma unroll 1
      for (int j = 0; j < steps; j += kSteps) {
        const StepPairs<TPT> sp(st, j, q, tx, ty, tz);
#pragma unroll
        for (int i = 0; i < kSteps * TPT; ++i) {
          const int k = i % TPT;
          const float4 u = sp.u[i / TPT];
          const float2 v = sp.v[i / TPT];
          const float dx = sp.dx[i], dy = sp.dy[i], dz = sp.dz[i], r2 = sp.r2[i], ir = sp.ir[i];
          const float ir2 = ir * ir;
          float beta = ir2 * ir;
          float alpha = beta * ir2;
          if (r2 < fc.near2) field_near_coeffs_tab(s_tab, fc.tab_scale, r2, ir, alpha, beta);
          const float dm = fmaf(dx, u.w, fmaf(dy, v.x, dz * v.y));
          const float s1 = dm * alpha;
          a1[k][0] = fmaf(dx, s1, a1[k][0]);
          a1[k][1] = fmaf(dy, s1, a1[k][1]);
          a1[k][2] = fmaf(dz, s1, a1[k][2]);
          a2[k][0] = fmaf(u.w, beta, a2[k][0]);
          a2[k][1] = fmaf(v.x, beta, a2[k][1]);
          a2[k][2] = fmaf(v.y, beta, a2[k][2]);
        }
      }
    }
  };
  auto flush = [&]() {
#pragma unroll
    for (int k = 0; k < TPT; ++k)
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        acc[k][a] += 3.0 * static_cast<double>(a1[k][a]) - static_cast<double>(a2[k][a]);
        a1[k][a] = a2[k][a] = 0.f;
      }
  };
  walk(target_box<TPT>(tx, ty, tz), st, body, flush);

  const double cfac = 1.0 / (4.0 * kPi);
  const int64_t i = tbase + lane;  // lane group k stores targets 16 k .. 16 k + 15
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    double v = 0.0;
#pragma unroll
    for (int k = 0; k < TPT; ++k) {
      const double sum = group_sum(acc[k][a]);
      v = q == k ? sum : v;
    }
    if (q < TPT && i < nt) put(a, i, v * cfac);
  }
}

template <int TPT>
__global__ __launch_bounds__(64) void field_allpairs_kernel(
    Points tgt, int64_t nt, const SrcRec *__restrict__ src, const float4 *__restrict__ boxes,
    int64_t nsub, int64_t per, FieldConsts fc, int64_t nt_ld, double *__restrict__ partial,
    Skip skip) {
  if (skipped(skip)) return;
  double *out = partial + static_cast<int64_t>(blockIdx.y) * 3 * nt_ld;
  field_wave<TPT>(
      tgt, nt, fc,
      [&](const WaveBox &box, Staged &st, const auto &body, const auto &flush) {
        walk_sources(src, boxes, chunk_range(nsub, per), box, st, threadIdx.x, body, flush);
      },
      [&](int a, int64_t i, double v) { out[a * nt_ld + i] = v; });
}

struct FieldOut {
  float *p[3];
  float hconst[3];
};
template <int TPT>
__global__ __launch_bounds__(64) void field_few_kernel(Points tgt, int64_t nt, SourceArrays src,
                                                       FieldConsts fc, FieldOut out) {
  field_wave<TPT>(
      tgt, nt, fc,
      [&](const WaveBox &box, Staged &st, const auto &body, const auto &flush) {
        walk_arrays(src, box, st, threadIdx.x, body, flush);
      },
      [&](int a, int64_t i, double v) { out.p[a][i] = static_cast<float>(v + out.hconst[a]); });
}

// ---------------------------------------------------------------------------
// Force: targets are the sources themselves (same records), target moment n.
//   F = s sum_j [ d (P (m.n) + R (d.m)(d.n)) + m P (d.n) + n P (d.m) ]
// with s = 3 mu0/(4 pi), accumulated as A_d (3), A_m (3), A_n (1); R = -5 P / r^2
// (far).  -5 goes to the pair, not to n: rounding -5 n once per target would weigh on all of
// its pairs.

template <int TPT>
__global__ __launch_bounds__(64) void force_allpairs_kernel(
    const SrcRec *__restrict__ tgt, int64_t nt, const SrcRec *__restrict__ src,
    const float4 *__restrict__ boxes, int64_t nsub, int64_t per, HessConsts hc, int64_t nt_ld,
    double *__restrict__ partial) {
  __shared__ float4 s_tab[2 * kHessTabEntries];
  __shared__ Staged st;
  const int lane = threadIdx.x, c = lane & 15, q = lane >> 4;
  bool have_tab = false;  // read on the first mixed tile
  const int64_t tbase = static_cast<int64_t>(blockIdx.x) * (16 * TPT);
  float tx[TPT], ty[TPT], tz[TPT], nx[TPT], ny[TPT], nz[TPT];
#pragma unroll
  for (int k = 0; k < TPT; ++k) {
    const SrcRec t = tgt[min(tbase + 16 * k + c, nt - 1)];
    tx[k] = t.x;
    ty[k] = t.y;
    tz[k] = t.z;
    nx[k] = t.mx;
    ny[k] = t.my;
    nz[k] = t.mz;
  }
  double acc[TPT][3];
  float ad[TPT][3], am[TPT][3], an[TPT];
#pragma unroll
  for (int k = 0; k < TPT; ++k) {
    an[k] = 0.f;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      acc[k][a] = 0.0;
      ad[k][a] = am[k][a] = 0.f;
    }
  }
  auto body = [&](int steps, float dist2) {
    if (dist2 > hc.near2) {
#pragma unroll 1
      for (int j = 0; j < steps; j += kSteps) {
        const StepPairs<TPT> sp(st, j, q, tx, ty, tz);
#pragma unroll
        for (int i = 0; i < kSteps * TPT; ++i) {
          const int k = i % TPT;
          const float4 u = sp.u[i / TPT];
          const float2 v = sp.v[i / TPT];
          const float dx = sp.dx[i], dy = sp.dy[i], dz = sp.dz[i], ir = sp.ir[i];
          const float ir2 = ir * ir;
          const float P = ir2 * ir2 * ir;  // r^-5
          const float dm = fmaf(dx, u.w, fmaf(dy, v.x, dz * v.y));
          const float dn = fmaf(dx, nx[k], fmaf(dy, ny[k], dz * nz[k]));
          const float mn = fmaf(u.w, nx[k], fmaf(v.x, ny[k], v.y * nz[k]));
          const float e = P * fmaf(-5.f * ir2 * dm, dn, mn);  // P mn + R dm dn
          const float f1 = P * dn;
          ad[k][0] = fmaf(dx, e, ad[k][0]);
          ad[k][1] = fmaf(dy, e, ad[k][1]);
          ad[k][2] = fmaf(dz, e, ad[k][2]);
          am[k][0] = fmaf(u.w, f1, am[k][0]);
          am[k][1] = fmaf(v.x, f1, am[k][1]);
          am[k][2] = fmaf(v.y, f1, am[k][2]);
          an[k] = fmaf(P, dm, an[k]);
        }
      }
    } else {
      if (!have_tab) {
        load_table(d_hess_tab, hc, kHessTabMid, s_tab, lane, 64);
        __builtin_amdgcn_wave_barrier();
        have_tab = true;
      }
#pragma unroll 1
      for (int j = 0; j < steps; j += kSteps) {
        const StepPairs<TPT> sp(st, j, q, tx, ty, tz);
#pragma unroll
        for (int i = 0; i < kSteps * TPT; ++i) {
          const int k = i % TPT;
          const float4 u = sp.u[i / TPT];
          const float2 v = sp.v[i / TPT];
          const float dx = sp.dx[i], dy = sp.dy[i], dz = sp.dz[i], r2 = sp.r2[i];
          // the clamp keeps a pair at d = 0 finite
          const float ir = __builtin_amdgcn_fmed3f(sp.ir[i], 0.f, 1e12f);
          const float ir2 = ir * ir;
          float c1 = ir2 * ir2, dq = -5.f * c1;  // far curves
          if (!(r2 > hc.near2)) {
            hess_near_curves_tab(s_tab, hc.tab_scale, r2, ir, c1, dq);
            const bool apart = r2 > 0.f;  // nothing at d = 0
            c1 = apart ? c1 : 0.f;
            dq = apart ? dq : 0.f;
          }
          const float P = c1 * ir;
          const float dm = fmaf(dx, u.w, fmaf(dy, v.x, dz * v.y));
          const float dn = fmaf(dx, nx[k], fmaf(dy, ny[k], dz * nz[k]));
          const float mn = fmaf(u.w, nx[k], fmaf(v.x, ny[k], v.y * nz[k]));
          const float e = fmaf(dq * (ir2 * ir), dm * dn, P * mn);
          const float f1 = P * dn;
          ad[k][0] = fmaf(dx, e, ad[k][0]);
          ad[k][1] = fmaf(dy, e, ad[k][1]);
          ad[k][2] = fmaf(dz, e, ad[k][2]);
          am[k][0] = fmaf(u.w, f1, am[k][0]);
          am[k][1] = fmaf(v.x, f1, am[k][1]);
          am[k][2] = fmaf(v.y, f1, am[k][2]);
          an[k] = fmaf(P, dm, an[k]);
        }
      }
    }
  };
  auto flush = [&]() {
#pragma unroll
    for (int k = 0; k < TPT; ++k) {
      const double n3[3] = {nx[k], ny[k], nz[k]};
      const double s = static_cast<double>(an[k]);
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        acc[k][a] += (static_cast<double>(ad[k][a]) + static_cast<double>(am[k][a])) + n3[a] * s;
        ad[k][a] = am[k][a] = 0.f;
      }
      an[k] = 0.f;
    }
  };
  walk_sources(src, boxes, chunk_range(nsub, per), target_box<TPT>(tx, ty, tz), st, lane, body,
               flush);

  const double sfac = 3.0 * kMu0 / (4.0 * kPi);
  double *out = partial + static_cast<int64_t>(blockIdx.y) * 3 * nt_ld;
  const int64_t i = tbase + lane;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    double v = 0.0;
#pragma unroll
    for (int k = 0; k < TPT; ++k) {
      const double sum = group_sum(acc[k][a]);
      v = q == k ? sum : v;
    }
    if (q < TPT && i < nt) out[a * nt_ld + i] = v * sfac;
  }
}

// ---------------------------------------------------------------------------
// One record set against itself, every unordered pair evaluated once.
//
// A unit of work is one wave's 64 records (an i-tile, four targets a lane)
// against one staged j-tile (mf_pair_once.hpp).
//
// A workgroup is W waves with W consecutive i-tiles (a group) walking the same
// j-tiles; the j-sums of its waves meet in LDS and leave in FP64, one slot per
// (group distance d, record): group G takes the j-tiles of groups G, G + 1, ...,
// G + D modulo an odd number of groups 2 D + 1 (the last one may be empty), so every
// group pair is met once and every record gets exactly one sum for each d = 1 .. D.
// The group's own tiles (d = 0) are walked directed, self pairs included.  Chunks of
// the walk along grid.y, each with its i-sums in a slot of its own, give the
// chip enough workgroups; the chunk reduction adds the slots in a fixed order.

constexpr int kSelfTPT = 4;      // 64 targets a wave, 64 = kTile
// Units between FP64 accumulations: the FP32 chains are 16 terms a unit.  The force's terms
// cancel: with four units it was 13 % further from FP64 than the directed kernels' on 12,000
// nearly equal moments, with one it is level (262,144 particles: 29.2 -> 29.8 ms).
constexpr int kFieldSelfFlush = 4, kForceSelfFlush = 1;

struct SelfWalk {
  int ntiles;   // tiles of the record set
  int ngroups;  // odd
  int first, last;  // the launch's units: j-tiles [first, last) of a group's W (D + 1)
  int per;          // units per chunk
  int nchunk;
};

template <class Pairs, class Consts, int W, int NTAB, int FLUSH>
__device__ __forceinline__ void self_walk(const SrcRec *__restrict__ rec,
                                          const float4 *__restrict__ boxes, int64_t n,
                                          const SelfWalk &w, const Consts &consts,
                                          const UnitTable<NTAB> &table, float mid, double fac,
                                          double *__restrict__ partial) {
  __shared__ float4 s_tab[2 * NTAB];
  __shared__ SelfTile st[2];
  __shared__ float jp[2][W][3][kTile];
  __shared__ double s_acc[W][3 * kSelfTPT][64];
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  load_table(table, consts, mid, s_tab, tid, 64 * W);
  const int group = static_cast<int>(blockIdx.x), chunk = static_cast<int>(blockIdx.y);
  const int it = group * W + wave;  // the wave's i-tile
  const bool live = it < w.ntiles;
  Pairs prs(consts, s_tab);
  const int64_t last = static_cast<int64_t>(w.ntiles) * kTile - 1;  // padding included
#pragma unroll
  for (int k = 0; k < kSelfTPT; ++k) {
    const int64_t i = static_cast<int64_t>(it) * kTile + 16 * k + c;
    const SrcRec t = rec[i < last ? i : last];
    prs.tx[k] = t.x;
    prs.ty[k] = t.y;
    prs.tz[k] = t.z;
    prs.nx[k] = t.mx;
    prs.ny[k] = t.my;
    prs.nz[k] = t.mz;
  }
  // the i-tile's box is its targets' (padding excluded)
  const int bt = live ? it : 0;
  const float4 ilo = boxes[2 * bt], ihi = boxes[2 * bt + 1];
  // the lane's FP64 sums live in LDS: 24 registers fewer
  double *acc = &s_acc[wave][0][lane];
#pragma unroll
  for (int k = 0; k < 3 * kSelfTPT; ++k) acc[k * 64] = 0.0;
  prs.clear();
  auto flush = [&]() {
#pragma unroll
    for (int k = 0; k < kSelfTPT; ++k)
#pragma unroll
      for (int a = 0; a < 3; ++a) acc[(3 * k + a) * 64] += prs.sum(k, a);
    prs.clear();
  };

  const int u0 = w.first + chunk * w.per, u1 = min(u0 + w.per, w.last);
  auto tile_of = [&](int u) {
    int g = group + u / W;
    g -= g >= w.ngroups ? w.ngroups : 0;
    return g * W + u % W;
  };
  auto next_unit = [&](int u) {  // the first unit from u on whose j-tile exists
    while (u < u1 && tile_of(u) >= w.ntiles) ++u;
    return u;
  };
  const float4 *__restrict__ rec4 = reinterpret_cast<const float4 *>(rec);
  // wave 0 copies the j-tile
  auto stage = [&](SelfTile &s, int jt) {
    const float4 *g = rec4 + 2 * (static_cast<int64_t>(jt) * kTile + lane);
    copy16_to_lds(g, s.pos);
    copy16_to_lds(g + 1, s.mom);
  };
  int u = next_unit(u0), buf = 0, since = 0;
  if (u < u1 && wave == 0) stage(st[0], tile_of(u));
  wait_vm<0>();  // the copy has landed
  __syncthreads();
  // u, next and buf are uniform over the workgroup: every wave meets every barrier
  while (u < u1) {
    const int next = next_unit(u + 1), jt = tile_of(u);
    const bool both = u >= W;
    // st[buf ^ 1] was last read before the previous barrier
    if (wave == 0 && next < u1) stage(st[buf ^ 1], tile_of(next));
    float jc[3] = {0.f, 0.f, 0.f};
    if (live) {
      const float4 lo = boxes[2 * jt], hi = boxes[2 * jt + 1];
      const bool far = prs.far(uniform_f(box_dist2(ilo.x, ilo.y, ilo.z, ihi.x, ihi.y, ihi.z, lo, hi)));
      if (both) {
        if (far)
          prs.template tile<false, true>(st[buf], c, q, jc);
        else
          prs.template tile<true, true>(st[buf], c, q, jc);
      } else {
        if (far)
          prs.template tile<false, false>(st[buf], c, q, jc);
        else
          prs.template tile<true, false>(st[buf], c, q, jc);
      }
      if (++since == FLUSH) {
        flush();
        since = 0;
      }
    }
    if (both) {
#pragma unroll
      for (int a = 0; a < 3; ++a) jp[buf][wave][a][lane] = jc[a];
    }
    wait_vm<0>();
    __syncthreads();
    if (both && tid < 3 * kTile) {
      // read again only after the next barrier (two buffers)
      const int a = tid / kTile;
      double v = 0.0;
#pragma unroll
      for (int k = 0; k < W; ++k) v += static_cast<double>(jp[buf][k][a][lane]);
      const int64_t j = static_cast<int64_t>(jt) * kTile + lane;
      const int slot = w.nchunk + u / W - max(w.first / W, 1);
      if (j < n) partial[(static_cast<int64_t>(slot) * 3 + a) * n + j] = v * fac;
    }
    u = next;
    buf ^= 1;
  }
  flush();
  double *out = partial + static_cast<int64_t>(chunk) * 3 * n;
  const int64_t i = static_cast<int64_t>(it) * kTile + lane;  // lane group k stores its k-th sixteen
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    double v = 0.0;
#pragma unroll
    for (int k = 0; k < kSelfTPT; ++k) {
      const double sum = group_sum(acc[(3 * k + a) * 64]);
      v = q == k ? sum : v;
    }
    if (i < n) out[a * n + i] = v * fac;
  }
}

template <int W>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(4))) void field_self_kernel(const SrcRec *__restrict__ rec,
                                                            const float4 *__restrict__ boxes,
                                                            int64_t n, SelfWalk w, FieldConsts fc,
                                                            double *__restrict__ partial, Skip skip) {
  if (skipped(skip)) return;
  self_walk<FieldSelf<kSelfTPT>, FieldConsts, W, kFieldTabEntries, kFieldSelfFlush>(
      rec, boxes, n, w, fc, d_field_tab, kFieldTabMid, 1.0 / (4.0 * kPi), partial);
}

template <int W>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(4))) void force_self_kernel(const SrcRec *__restrict__ rec,
                                                            const float4 *__restrict__ boxes,
                                                            int64_t n, SelfWalk w, HessConsts hc,
                                                            double *__restrict__ partial) {
  self_walk<ForceSelf<kSelfTPT>, HessConsts, W, kHessTabEntries, kForceSelfFlush>(
      rec, boxes, n, w, hc, d_hess_tab, kHessTabMid, 3.0 * kMu0 / (4.0 * kPi), partial);
}

// ---------------------------------------------------------------------------
// Force-tensor field at separate targets (the external tensor T_ext of
// eval_hext), walked like the field: partials [chunk][6][nt_ld] (xx yy zz xy
// xz yz).
template <int TPT, class Walk, class Put>
__device__ __forceinline__ void hessian_wave(const Points &tgt, int64_t nt, const HessConsts &hc,
                                             const Walk &walk, const Put &put) {
  __shared__ float4 s_tab[2 * kHessTabEntries];
  __shared__ Staged st;
  const int lane = threadIdx.x, c = lane & 15, q = lane >> 4;
  bool have_tab = false;
  const int64_t tbase = static_cast<int64_t>(blockIdx.x) * (16 * TPT);
  float tx[TPT], ty[TPT], tz[TPT];
#pragma unroll
  for (int k = 0; k < TPT; ++k) {
    const int64_t i = min(tbase + 16 * k + c, nt - 1) * tgt.stride;
    tx[k] = tgt.x[i];
    ty[k] = tgt.y[i];
    tz[k] = tgt.z[i];
  }
  double acc[TPT][6];
  float s[TPT][6];
#pragma unroll
  for (int k = 0; k < TPT; ++k)
#pragma unroll
    for (int a = 0; a < 6; ++a) {
      acc[k][a] = 0.0;
      s[k][a] = 0.f;
    }
  auto pair = [&](const StepPairs<TPT> &sp, int i, bool near) {
    const int k = i % TPT;
    const float dx = sp.dx[i], dy = sp.dy[i], dz = sp.dz[i], r2 = sp.r2[i];
    const float mx = sp.u[i / TPT].w, my = sp.v[i / TPT].x, mz = sp.v[i / TPT].y;
    const float ir = near ? __builtin_amdgcn_fmed3f(sp.ir[i], 0.f, 1e12f) : sp.ir[i];
    const float ir2 = ir * ir;
    float c1 = ir2 * ir2, hq = -2.5f * c1;  // hq: half of R's curve
    if (near && !(r2 > hc.near2)) {
      hess_near_curves_tab(s_tab, hc.tab_scale, r2, ir, c1, hq);
      const bool apart = r2 > 0.f;  // nothing at d = 0
      c1 = apart ? c1 : 0.f;
      hq = apart ? 0.5f * hq : 0.f;
    }
    const float P = c1 * ir;
    const float dm = fmaf(dx, mx, fmaf(dy, my, dz * mz));
    // T_ab = d_a (P m_b + (R/2) dm d_b) + (a <-> b) + delta_ab P dm
    const float h = hq * (ir2 * ir) * dm;
    const float gx = fmaf(P, mx, h * dx), gy = fmaf(P, my, h * dy), gz = fmaf(P, mz, h * dz);
    s[k][0] = fmaf(dx + dx, gx, fmaf(P, dm, s[k][0]));
    s[k][1] = fmaf(dy + dy, gy, fmaf(P, dm, s[k][1]));
    s[k][2] = fmaf(dz + dz, gz, fmaf(P, dm, s[k][2]));
    s[k][3] = fmaf(dx, gy, fmaf(dy, gx, s[k][3]));
    s[k][4] = fmaf(dx, gz, fmaf(dz, gx, s[k][4]));
    s[k][5] = fmaf(dy, gz, fmaf(dz, gy, s[k][5]));
  };
  auto body = [&](int steps, float dist2) {
    if (dist2 > hc.near2) {
#pragma unroll 1
      for (int j = 0; j < steps; j += kSteps) {
        const StepPairs<TPT> sp(st, j, q, tx, ty, tz);
#pragma unroll
        for (int i = 0; i < kSteps * TPT; ++i) pair(sp, i, false);
      }
    } else {
      if (!have_tab) {
        load_table(d_hess_tab, hc, kHessTabMid, s_tab, lane, 64);
        __builtin_amdgcn_wave_barrier();
        have_tab = true;
      }
#pragma unroll 1
      for (int j = 0; j < steps; j += kSteps) {
        const StepPairs<TPT> sp(st, j, q, tx, ty, tz);
#pragma unroll
        for (int i = 0; i < kSteps * TPT; ++i) pair(sp, i, true);
      }
    }
  };
  auto flush = [&]() {
#pragma unroll
    for (int k = 0; k < TPT; ++k)
#pragma unroll
      for (int a = 0; a < 6; ++a) {
        acc[k][a] += static_cast<double>(s[k][a]);
        s[k][a] = 0.f;
      }
  };
  walk(target_box<TPT>(tx, ty, tz), st, body, flush);
  const int64_t i = tbase + lane;
  double v[6];
#pragma unroll
  for (int a = 0; a < 6; ++a) {
    v[a] = 0.0;
#pragma unroll
    for (int k = 0; k < TPT; ++k) {
      const double sum = group_sum(acc[k][a]);
      v[a] = q == k ? sum : v[a];
    }
  }
  if (q < TPT && i < nt) put(i, v);
}

template <int TPT>
__global__ __launch_bounds__(64) void hessian_allpairs_kernel(
    Points tgt, int64_t nt, const SrcRec *__restrict__ src, const float4 *__restrict__ boxes,
    int64_t nsub, int64_t per, HessConsts hc, int64_t nt_ld, double *__restrict__ partial) {
  double *out = partial + static_cast<int64_t>(blockIdx.y) * 6 * nt_ld;
  hessian_wave<TPT>(
      tgt, nt, hc,
      [&](const WaveBox &box, Staged &st, const auto &body, const auto &flush) {
        walk_sources(src, boxes, chunk_range(nsub, per), box, st, threadIdx.x, body, flush);
      },
      [&](int64_t i, const double (&v)[6]) {
#pragma unroll
        for (int a = 0; a < 6; ++a) out[a * nt_ld + i] = v[a];
      });
}

// Destinations of the six tensor components: out[k] (may be null) receives
// component sym[k] (0..5 = xx yy zz xy xz yz) times mu0 3/(4 pi).
struct TensorOut {
  float *p[9];
  int sym[9];
  __device__ __forceinline__ void put(int64_t i, const double (&s)[6]) const {
    const double sfac = 3.0 * kMu0 / (4.0 * kPi);
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      if (!p[k]) continue;
      double v = s[0];
#pragma unroll
      for (int a = 1; a < 6; ++a) v = sym[k] == a ? s[a] : v;  // s stays in registers
      p[k][i] = static_cast<float>(sfac * v);
    }
  }
};

template <int TPT>
__global__ __launch_bounds__(64) void hessian_few_kernel(Points tgt, int64_t nt, SourceArrays src,
                                                         HessConsts hc, TensorOut out) {
  hessian_wave<TPT>(
      tgt, nt, hc,
      [&](const WaveBox &box, Staged &st, const auto &body, const auto &flush) {
        walk_arrays(src, box, st, threadIdx.x, body, flush);
      },
      [&](int64_t i, const double (&v)[6]) { out.put(i, v); });
}

// ---------------------------------------------------------------------------
// Chunk reductions (fixed order => deterministic).  A block takes 256 / W
// targets; its W waves-of-targets add every W-th chunk each, and the sums meet
// in LDS.  With one thread per target (W = 1, the previous form) 8,192 targets
// were 32 blocks walking 64 chunks each: 16.6 us, 5.4 us with W = 4.

template <int W, int NC>
__device__ __forceinline__ bool reduce_chunks(int64_t n, int64_t nt_ld, int nchunk,
                                              const double *__restrict__ partial, int64_t &i,
                                              double (&s)[NC]) {
  constexpr int T = 256 / W;  // targets per block
  const int t = threadIdx.x % T, w = threadIdx.x / T;
  i = static_cast<int64_t>(blockIdx.x) * T + t;
#pragma unroll
  for (int a = 0; a < NC; ++a) s[a] = 0.0;
  if (i < n)
    for (int c = w; c < nchunk; c += W) {
      const double *p = partial + static_cast<int64_t>(c) * NC * nt_ld + i;
#pragma unroll
      for (int a = 0; a < NC; ++a) s[a] += p[a * nt_ld];
    }
  if constexpr (W > 1) {
    __shared__ double sh[W][NC][T];
#pragma unroll
    for (int a = 0; a < NC; ++a) sh[w][a][t] = s[a];
    __syncthreads();
    if (w == 0)
#pragma unroll
      for (int a = 0; a < NC; ++a) {
#pragma unroll
        for (int k = 1; k < W; ++k) s[a] += sh[k][a][t];
      }
  }
  return w == 0 && i < n;
}

template <int W>
__global__ __launch_bounds__(256) void reduce_hessian_kernel(int64_t n, int64_t nt_ld, int nchunk,
                                                             const double *__restrict__ partial,
                                                             TensorOut out) {
  int64_t i;
  double s[6];
  if (!reduce_chunks<W, 6>(n, nt_ld, nchunk, partial, i, s)) return;
  out.put(i, s);
}

template <int W>
__global__ __launch_bounds__(256) void reduce_field_kernel(int64_t n, int64_t nt_ld, int nchunk,
                                                           const double *__restrict__ partial,
                                                           float hc0, float hc1, float hc2,
                                                           float *__restrict__ ox,
                                                           float *__restrict__ oy,
                                                           float *__restrict__ oz) {
  int64_t i;
  double s[3];
  if (!reduce_chunks<W, 3>(n, nt_ld, nchunk, partial, i, s)) return;
  ox[i] = static_cast<float>(s[0] + hc0);
  oy[i] = static_cast<float>(s[1] + hc1);
  oz[i] = static_cast<float>(s[2] + hc2);
}

// The reduction of a conjugate-gradient product: ap = p - g with g the FP32
// rounding of the sum, and the block's part of p . ap.
template <int W>
__global__ __launch_bounds__(256) void reduce_ap_kernel(int64_t n, int64_t nt_ld, int nchunk,
                                                        const double *__restrict__ partial,
                                                        ApOut o) {
  if (skipped(o.skip)) return;
  int64_t i;
  double s[3];
  double dot = 0.0;
  if (reduce_chunks<W, 3>(n, nt_ld, nchunk, partial, i, s)) {
    const float px = o.p[0][i], py = o.p[1][i], pz = o.p[2][i];
    const float ax = px - static_cast<float>(s[0]), ay = py - static_cast<float>(s[1]),
                az = pz - static_cast<float>(s[2]);
    o.ap[0][i] = ax;
    o.ap[1][i] = ay;
    o.ap[2][i] = az;
    dot = static_cast<double>(px) * ax + static_cast<double>(py) * ay + static_cast<double>(pz) * az;
  }
  __shared__ double sh[4];
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) dot += __shfl_xor(dot, off, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = dot;
  __syncthreads();
  if (threadIdx.x == 0) o.dots[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// F_i = sum_chunks partial + Text_i n_i  (Text given as 9 SoA arrays, may be null).
struct Text9 {
  const float *p[9];
};
template <int W>
__global__ __launch_bounds__(256) void reduce_force_kernel(
    int64_t n, int64_t nt_ld, int nchunk, const double *__restrict__ partial,
    const SrcRec *__restrict__ tgt, Text9 text, int has_text, float *__restrict__ fx,
    float *__restrict__ fy, float *__restrict__ fz) {
  int64_t i;
  double s[3];
  if (!reduce_chunks<W, 3>(n, nt_ld, nchunk, partial, i, s)) return;
  if (has_text) {
    // Text rows: dHextdx = (p0,p1,p2), dHextdy = (p3,p4,p5), dHextdz = (p6,p7,p8),
    // glm column a holds (d/dx_a H_x, H_y, H_z); the tensor is symmetric for a
    // curl-free external field, F_r = sum_a T[a][r] n_a (magnetic_force.cu:968-976).
    const double n3[3] = {tgt[i].mx, tgt[i].my, tgt[i].mz};
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      double v = 0.0;
#pragma unroll
      for (int a = 0; a < 3; ++a) v += static_cast<double>(text.p[3 * a + r][i]) * n3[a];
      s[r] += v;
    }
  }
  fx[i] = static_cast<float>(s[0]);
  fy[i] = static_cast<float>(s[1]);
  fz[i] = static_cast<float>(s[2]);
}

}  // namespace

// ---------------------------------------------------------------------------
// Host side.

// v as its FP32 value and what that leaves.
static float2 two_floats(double v) {
  const float hi = static_cast<float>(v);
  return {hi, std::isfinite(hi) ? static_cast<float>(v - static_cast<double>(hi)) : 0.f};
}

FieldConsts make_field_consts(double h) {
  FieldConsts fc{};
  fc.h = static_cast<float>(h);
  fc.near2 = static_cast<float>(4.0 * h * h);
  fc.tab_scale = static_cast<float>(kFieldTabN / (2.0 * h));
  fc.tab_high = static_cast<float>(fc.tab_scale * (2.0 * h) / kFieldTabN - 1.0);
  fc.tab_a = two_floats(1.0 / (h * h * h * h * h));
  fc.tab_b = two_floats(1.0 / (h * h * h));
  return fc;
}

void make_field_table(double h, float *tab) {
  const double ih3 = 1.0 / (h * h * h), ih5 = ih3 / (h * h);
  fill_field_table(ih5, ih3, [&](int e, const double *a, const double *b) { store_entry(tab, e, 1, a, b); });
}

void make_hess_table(double h, float *tab) {
  fill_hess_table(1.0 / (h * h * h * h), [&](int e, const double *a, const double *b) {
    store_entry(tab, e, -1, a, b);
  });
}

void split_near_table(const float *tab, int entries, float *out) {
  for (int e = 0; e < entries; ++e)
    for (int j = 0; j < 4; ++j) {
      out[4 * e + j] = tab[8 * e + j];
      out[4 * (entries + e) + j] = tab[8 * e + 4 + j];
    }
}


HessConsts make_hess_consts(double h) {
  HessConsts hc{};
  hc.h = static_cast<float>(h);
  hc.near2 = static_cast<float>(16.0 * h * h);
  hc.tab_scale = static_cast<float>(kHessTabN / (4.0 * h));
  hc.tab_high = static_cast<float>(hc.tab_scale * (4.0 * h) / kHessTabN - 1.0);
  hc.tab_a = hc.tab_b = two_floats(1.0 / (h * h * h * h));
  return hc;
}

int64_t padded_sources(int64_t n) { return ((n + kTile - 1) / kTile) * kTile; }

Status pack_tiles(mf_ctx *ctx, int64_t n, const float *x, const float *y, const float *z,
                  const float *mx, const float *my, const float *mz, SrcRec *out, float4 *boxes) {
  const int64_t ntiles = padded_sources(n) / kTile;
  if (ntiles == 0) return Status::Ok();
  hipLaunchKernelGGL(pack_tiles_kernel, dim3(grid_for(ntiles, 4)), dim3(256), 0, ctx->stream, n,
                     ntiles, x, y, z, mx, my, mz, out, boxes);
  MF_LAUNCH_CHECK();
  return Status::Ok();
}

Status pack_moments(mf_ctx *ctx, int64_t n, const float *mx, const float *my, const float *mz,
                    float scale, SrcRec *out) {
  if (n == 0) return Status::Ok();
  hipLaunchKernelGGL(pack_moments_kernel, dim3(grid_for(n, 256)), dim3(256), 0, ctx->stream, n,
                     mx, my, mz, scale, out);
  MF_LAUNCH_CHECK();
  return Status::Ok();
}

namespace {
// Targets per lane: 64 targets a wave amortize a staged record over four pairs
// a lane; the tensor's twelve sums a target leave room for two.
constexpr int kFieldTPT = 2;
constexpr int kForceTPT = 2;
constexpr int kHessTPT = 2;

// Launch shape: target waves along grid.x, chunks of whole 16-record groups
// along grid.y.  One fill of the chip (four waves per SIMD) comes first, down
// to two groups a chunk: at 1,859 particles 58 chunks of 32 records take 18.9 us
// a field product, 117 of 16 take 27.3.  Beyond that, equal waves end a launch
// together and the last, partly filled round is lost, so up to 16 fills pay
// (100,000 particles: 5.83 ms with one, 4.87 with four, 4.33 with 16), but each
// chunk costs its partials: not below 32 groups a chunk (8,000 particles: 53 us
// with 17 chunks of 480 records, 64 with 125 of 64).
constexpr int64_t kFillWaves = 16;  // waves per CU of one fill
constexpr int64_t kFills = 16, kGroupsMin = 2, kGroupsFull = 32;
struct Split {
  int64_t nsub, per, nchunk;
  unsigned gx;
};
Split split_sources(const mf_ctx *ctx, int64_t nt, int64_t ns, int tpt, int64_t max_chunks) {
  Split f{};
  f.nsub = (ns + kSub - 1) / kSub;  // a tile's all-padding groups are skipped
  f.gx = static_cast<unsigned>((nt + 16 * tpt - 1) / (16 * tpt));
  const int64_t fill = static_cast<int64_t>(ctx->num_cu) * kFillWaves;
  const int64_t one = std::min((fill + f.gx - 1) / f.gx, f.nsub / kGroupsMin);
  const int64_t many = std::min((fill * kFills + f.gx - 1) / f.gx, f.nsub / kGroupsFull);
  const int64_t nchunk = std::max<int64_t>(std::min(std::max(one, many), max_chunks), 1);
  f.per = std::max<int64_t>((f.nsub + nchunk - 1) / nchunk, 1);
  f.nchunk = std::max<int64_t>((f.nsub + f.per - 1) / f.per, 1);
  return f;
}
constexpr int64_t kMaxChunks = 128;

__global__ void zero_f64_kernel(int64_t n, double *__restrict__ a) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) a[i] = 0.0;
}

// Waves of a reduction block that share a target: four where one thread per
// target would leave CUs without a wave, one beyond.
constexpr int64_t kReduceWide = 65536;
inline bool reduce_wide(int64_t n) { return n < kReduceWide; }
inline dim3 reduce_grid(int64_t n) { return dim3(grid_for(n, reduce_wide(n) ? 64 : 256)); }
}  // namespace

#define MF_REDUCE(kernel, n, ...)                                                               \
  do {                                                                                          \
    if (reduce_wide(n))                                                                         \
      hipLaunchKernelGGL(kernel<4>, reduce_grid(n), dim3(256), 0, ctx->stream, __VA_ARGS__);    \
    else                                                                                        \
      hipLaunchKernelGGL(kernel<1>, reduce_grid(n), dim3(256), 0, ctx->stream, __VA_ARGS__);    \
    MF_LAUNCH_CHECK();                                                                          \
  } while (0)

int64_t field_partial_doubles(int64_t nt, int64_t nchunk) { return 3 * nt * nchunk; }

namespace {
// The chunk sums of the field into `partial`; returns the chunk count.
Status field_chunks(mf_ctx *ctx, const Points &tgt, int64_t nt, const SrcRec *src,
                    const float4 *boxes, const FieldConsts &fc, const Split &f, double *partial,
                    const Skip &skip = {}) {
  if (f.nsub == 0) {
    // a fill kernel, not hipMemsetAsync: callers may capture this in a graph
    hipLaunchKernelGGL(zero_f64_kernel, dim3(grid_for(3 * nt, 256)), dim3(256), 0, ctx->stream,
                       3 * nt, partial);
    MF_LAUNCH_CHECK();
    return Status::Ok();
  }
  KernelTimer timer(ctx, "field");
  hipLaunchKernelGGL(field_allpairs_kernel<kFieldTPT>, dim3(f.gx, static_cast<unsigned>(f.nchunk)),
                     dim3(64), 0, ctx->stream, tgt, nt, src, boxes, f.nsub, f.per, fc, nt, partial,
                     skip);
  MF_LAUNCH_CHECK();
  return Status::Ok();
}
}  // namespace

// Few sources (external magnets): one launch reads the caller's arrays and writes the
// result, where the general path packs records, writes chunk sums and adds them up: field
// and tensor calls of 27 sources, general -> few: 4,096 targets 26.4 -> 19.7 us and 32.4 ->
// 25.7, 1,048,576 42.1 -> 37.8 and 69.4 -> 66.3.  Each wave walks all of the sources, so
// their number is bounded: at 128 the two paths meet (1,048,576 targets: 85.3 -> 84.1 and 148.4 ->
// 149.9), at 512 the few lose (4,096: 26.3 -> 27.2 and 32.2 -> 47.0).  A launch may write
// what another wave has yet to read: outputs that overlap an input take the general path,
// which reads everything first.
constexpr int64_t kFewSources = 128;
bool few_sources(int64_t nt, int64_t ns, const Points &tgt, const SourceArrays &src, float *const *out,
                 int nout) {
  if (ns < 1 || ns > kFewSources) return false;
  auto apart = [](const float *a, int64_t na, const float *b, int64_t nb) {
    const auto pa = reinterpret_cast<uintptr_t>(a), pb = reinterpret_cast<uintptr_t>(b);
    return pa + sizeof(float) * na <= pb || pb + sizeof(float) * nb <= pa;
  };
  for (int k = 0; k < nout; ++k) {
    if (!out[k]) continue;
    for (const float *v : {tgt.x, tgt.y, tgt.z})
      if (!apart(out[k], nt, v, nt)) return false;
    for (const float *v : {src.x, src.y, src.z, src.mx, src.my, src.mz})
      if (!apart(out[k], nt, v, ns)) return false;
  }
  return true;
}

Status field_few_launch(mf_ctx *ctx, const Points &tgt, int64_t nt, const SourceArrays &src,
                        const FieldConsts &fc, const float *hconst, float *ox, float *oy,
                        float *oz) {
  if (nt == 0) return Status::Ok();
  FieldOut out{{ox, oy, oz}, {}};
  for (int a = 0; a < 3; ++a) out.hconst[a] = hconst ? hconst[a] : 0.f;
  KernelTimer timer(ctx, "field");
  hipLaunchKernelGGL(field_few_kernel<kFieldTPT>, dim3(grid_for(nt, 16 * kFieldTPT)), dim3(64), 0,
                     ctx->stream, tgt, nt, src, fc, out);
  MF_LAUNCH_CHECK();
  return Status::Ok();
}

Status hessian_few_launch(mf_ctx *ctx, const Points &tgt, int64_t nt, const SourceArrays &src,
                          const HessConsts &hc, float *const dst[9], const int sym[9]) {
  if (nt == 0) return Status::Ok();
  TensorOut out{};
  for (int k = 0; k < 9; ++k) {
    out.p[k] = dst[k];
    out.sym[k] = sym[k];
  }
  KernelTimer timer(ctx, "hessian");
  hipLaunchKernelGGL(hessian_few_kernel<kHessTPT>, dim3(grid_for(nt, 16 * kHessTPT)), dim3(64), 0,
                     ctx->stream, tgt, nt, src, hc, out);
  MF_LAUNCH_CHECK();
  return Status::Ok();
}

Status field_allpairs_launch_ws(mf_ctx *ctx, const Points &tgt, int64_t nt, const SrcRec *src,
                                const float4 *boxes, int64_t ns, const FieldConsts &fc,
                                const float *hconst, float *ox, float *oy, float *oz,
                                double *partial, int64_t partial_cap) {
  if (nt == 0) return Status::Ok();
  MF_ARG(partial_cap >= field_partial_doubles(nt, 1), "field partial buffer too small");
  const int64_t fit = partial_cap / field_partial_doubles(nt, 1);
  const Split f = split_sources(ctx, nt, ns, kFieldTPT, std::min(fit, kMaxChunks));
  MF_TRY(field_chunks(ctx, tgt, nt, src, boxes, fc, f, partial));
  const float h0 = hconst ? hconst[0] : 0.f, h1 = hconst ? hconst[1] : 0.f,
              h2 = hconst ? hconst[2] : 0.f;
  MF_REDUCE(reduce_field_kernel, nt, nt, nt, static_cast<int>(f.nchunk), partial, h0, h1, h2, ox,
            oy, oz);
  return Status::Ok();
}

namespace {
Status field_workspace(mf_ctx *ctx, int64_t nt, int64_t ns, double **partial, int64_t *cap) {
  const Split f = split_sources(ctx, nt, ns, kFieldTPT, kMaxChunks);
  *cap = field_partial_doubles(nt, f.nchunk);
  void *pw = nullptr;
  MF_TRY(workspace(ctx, "field_partial", sizeof(double) * *cap, &pw));
  *partial = static_cast<double *>(pw);
  return Status::Ok();
}
}  // namespace

Status field_allpairs_launch(mf_ctx *ctx, const Points &tgt, int64_t nt, const SrcRec *src,
                             const float4 *boxes, int64_t ns, const FieldConsts &fc,
                             const float *hconst, float *ox, float *oy, float *oz) {
  if (nt == 0) return Status::Ok();
  double *partial = nullptr;
  int64_t cap = 0;
  MF_TRY(field_workspace(ctx, nt, ns, &partial, &cap));
  return field_allpairs_launch_ws(ctx, tgt, nt, src, boxes, ns, fc, hconst, ox, oy, oz, partial,
                                  cap);
}

namespace {
// Walk of the pair-once kernels.  Four waves a workgroup: two write twice the j-sums
// (262,144 particles: field 24.4 ms, 22.1 with four), eight wait longer for each
// other (22.6).  Up to sixteen fills of the chip (16 waves per CU) with at least four units a
// chunk, but one fill in any case: 15,625 particles take 111 us a field product with
// two to eight units a chunk and 121 with one; 50,000 take 0.88 ms with four fills,
// 0.86 with sixteen.  Below kSelfMin records the directed kernels end first (2,744: field
// 20.0 against 20.5 us, force 21.7 against 23.5; 4,096: 24.2 against 22.2, 28.8 against
// 28.0).
constexpr int kSelfW = 4;
constexpr int64_t kSelfMin = 4096;
constexpr int64_t kSelfUnitsMin = 4;
// The slots grow with the square of n: beyond kSelfBytes the group distances go in
// passes, each folded into one slot before the next.  Where that much cannot be had, half
// as much and so on (self_slots); below kSelfBytesLeast the directed kernels take over.
constexpr int64_t kSelfBytes = int64_t{2} << 30, kSelfBytesLeast = int64_t{128} << 20;
struct SelfSplit {
  SelfWalk w;     // the walk's constants
  int dist;       // group distances 0 .. dist - 1
  int per_pass;   // group distances per pass
  int64_t slots;  // FP64 slots of 3 n: the folded sums if there are several passes, then a pass's
};
int self_chunks(const mf_ctx *ctx, const SelfWalk &w, int units) {
  const int64_t fill = static_cast<int64_t>(ctx->num_cu) * kFillWaves / kSelfW;
  const int64_t one = std::min<int64_t>((fill + w.ngroups - 1) / w.ngroups, units);
  const int64_t many =
      std::min<int64_t>((fill * kFills + w.ngroups - 1) / w.ngroups, units / kSelfUnitsMin);
  return static_cast<int>(std::max<int64_t>(std::max(one, many), 1));
}
SelfSplit self_split(const mf_ctx *ctx, int64_t n, int64_t bytes) {
  SelfSplit f{};
  f.w.ntiles = static_cast<int>((n + kTile - 1) / kTile);
  f.w.ngroups = ((f.w.ntiles + kSelfW - 1) / kSelfW) | 1;
  f.dist = f.w.ngroups / 2 + 1;
  const int64_t fit = std::max<int64_t>(bytes / (24 * n), 2);
  const int chunks = self_chunks(ctx, f.w, kSelfW * f.dist);
  if (chunks + f.dist - 1 <= fit) {
    f.per_pass = f.dist;
    f.slots = chunks + f.dist - 1;
    return f;
  }
  // a pass of d distances takes at most d + self_chunks(d) slots
  f.per_pass = static_cast<int>(std::max<int64_t>(fit - std::min<int64_t>(chunks, fit / 2), 1));
  f.slots = 1 + f.per_pass + self_chunks(ctx, f.w, kSelfW * f.per_pass);
  return f;
}

// Split and slots of a product (kind 0 field, 1 force); false: none can be had now.  What
// was refused is remembered (mf_ctx::self_bytes), so that later products do not ask for it.
bool self_slots(mf_ctx *ctx, int kind, const char *name, int64_t n, SelfSplit *f, double **slots) {
  int64_t &may = ctx->self_bytes[kind];
  while (true) {
    const int64_t bytes = std::min(kSelfBytes, may);
    *f = self_split(ctx, n, bytes);
    const int64_t need = 24 * n * f->slots;
    if (f->per_pass < f->dist && bytes < kSelfBytesLeast) return false;
    void *pw = nullptr;
    if (workspace_now(ctx, name, static_cast<size_t>(need), &pw)) {
      *slots = static_cast<double *>(pw);
      return true;
    }
    if (stream_capturing(ctx)) return false;
    may = std::min(bytes, need) / 2;
  }
}

// sum[i] (+)= the pass's slots.
__global__ void fold_slots_kernel(int64_t n3, int slots, int add, const double *__restrict__ p,
                                  double *__restrict__ sum) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n3) return;
  double s = add ? sum[i] : 0.0;
  for (int k = 0; k < slots; ++k) s += p[k * n3 + i];
  sum[i] = s;
}

// The passes: launch(walk, slots) runs one.  On return the first `nchunk` slots of
// `partial` hold the sums.
template <class Launch>
Status self_passes(mf_ctx *ctx, int64_t n, const SelfSplit &f, double *partial, int *nchunk,
                   const Launch &launch) {
  const bool one = f.per_pass == f.dist;
  double *slots = one ? partial : partial + 3 * n;
  for (int d = 0; d < f.dist; d += f.per_pass) {
    const int d1 = std::min(d + f.per_pass, f.dist);
    SelfWalk w = f.w;
    w.first = kSelfW * d;
    w.last = kSelfW * d1;
    w.nchunk = self_chunks(ctx, w, w.last - w.first);
    w.per = (w.last - w.first + w.nchunk - 1) / w.nchunk;
    w.nchunk = (w.last - w.first + w.per - 1) / w.per;
    launch(w, slots);
    MF_LAUNCH_CHECK();
    *nchunk = w.nchunk + d1 - std::max(d, 1);
    if (!one) {
      hipLaunchKernelGGL(fold_slots_kernel, dim3(grid_for(3 * n, 256)), dim3(256), 0, ctx->stream,
                         3 * n, *nchunk, d > 0 ? 1 : 0, slots, partial);
      MF_LAUNCH_CHECK();
    }
  }
  if (!one) *nchunk = 1;
  return Status::Ok();
}
}  // namespace

namespace {
// The partial sums of the field of a record set on itself.
Status field_self_chunks(mf_ctx *ctx, const SrcRec *rec, const float4 *boxes, int64_t n,
                         const FieldConsts &fc, double **partial, int *nchunk,
                         const Skip &skip = {}) {
  SelfSplit f;
  if (n >= kSelfMin && self_slots(ctx, 0, "field_partial", n, &f, partial)) {
    KernelTimer timer(ctx, "field");
    return self_passes(ctx, n, f, *partial, nchunk, [&](const SelfWalk &w, double *slots) {
      hipLaunchKernelGGL(field_self_kernel<kSelfW>,
                         dim3(static_cast<unsigned>(w.ngroups), static_cast<unsigned>(w.nchunk)),
                         dim3(64 * kSelfW), 0, ctx->stream, rec, boxes, n, w, fc, slots, skip);
    });
  }
  int64_t cap = 0;
  MF_TRY(field_workspace(ctx, n, n, partial, &cap));
  const Split d = split_sources(ctx, n, n, kFieldTPT, kMaxChunks);
  *nchunk = static_cast<int>(d.nchunk);
  return field_chunks(ctx, record_points(rec), n, rec, boxes, fc, d, *partial, skip);
}
}  // namespace

int field_ap_blocks(int64_t n) { return static_cast<int>(reduce_grid(n).x); }

Status field_allpairs_ap(mf_ctx *ctx, const SrcRec *rec, const float4 *boxes, int64_t n,
                         const FieldConsts &fc, const ApOut &out) {
  double *partial = nullptr;
  int nchunk = 0;
  MF_TRY(field_self_chunks(ctx, rec, boxes, n, fc, &partial, &nchunk, out.skip));
  MF_REDUCE(reduce_ap_kernel, n, n, n, nchunk, partial, out);
  return Status::Ok();
}

Status field_self_launch(mf_ctx *ctx, const SrcRec *rec, const float4 *boxes, int64_t n,
                         const FieldConsts &fc, const float *hconst, float *ox, float *oy,
                         float *oz) {
  if (n == 0) return Status::Ok();
  double *partial = nullptr;
  int nchunk = 0;
  MF_TRY(field_self_chunks(ctx, rec, boxes, n, fc, &partial, &nchunk));
  const float h0 = hconst ? hconst[0] : 0.f, h1 = hconst ? hconst[1] : 0.f,
              h2 = hconst ? hconst[2] : 0.f;
  MF_REDUCE(reduce_field_kernel, n, n, n, nchunk, partial, h0, h1, h2, ox, oy, oz);
  return Status::Ok();
}

namespace {
Status force_self_chunks(mf_ctx *ctx, const SrcRec *rec, const float4 *boxes, int64_t n,
                         const HessConsts &hc, double **partial, int *nchunk) {
  SelfSplit f;
  if (n >= kSelfMin && self_slots(ctx, 1, "force_partial", n, &f, partial)) {
    KernelTimer timer(ctx, "force");
    return self_passes(ctx, n, f, *partial, nchunk, [&](const SelfWalk &w, double *slots) {
      hipLaunchKernelGGL(force_self_kernel<kSelfW>,
                         dim3(static_cast<unsigned>(w.ngroups), static_cast<unsigned>(w.nchunk)),
                         dim3(64 * kSelfW), 0, ctx->stream, rec, boxes, n, w, hc, slots);
    });
  }
  const Split d = split_sources(ctx, n, n, kForceTPT, kMaxChunks);
  void *pw = nullptr;
  MF_TRY(workspace(ctx, "force_partial", sizeof(double) * 3 * n * d.nchunk, &pw));
  *partial = static_cast<double *>(pw);
  *nchunk = static_cast<int>(d.nchunk);
  KernelTimer timer(ctx, "force");
  hipLaunchKernelGGL(force_allpairs_kernel<kForceTPT>,
                     dim3(d.gx, static_cast<unsigned>(d.nchunk)), dim3(64), 0, ctx->stream, rec, n,
                     rec, boxes, d.nsub, d.per, hc, n, *partial);
  MF_LAUNCH_CHECK();
  return Status::Ok();
}
}  // namespace

Status force_allpairs_launch(mf_ctx *ctx, const SrcRec *rec, const float4 *boxes, int64_t n,
                             const HessConsts &hc, const float *const *text9, float *fx,
                             float *fy, float *fz) {
  if (n == 0) return Status::Ok();
  double *partial = nullptr;
  int nchunk = 0;
  MF_TRY(force_self_chunks(ctx, rec, boxes, n, hc, &partial, &nchunk));
  Text9 t{};
  int has_text = 0;
  if (text9) {
    has_text = 1;
    for (int k = 0; k < 9; ++k) {
      MF_ARG(text9[k] != nullptr, "text9 entries must be non-null device pointers");
      t.p[k] = text9[k];
    }
  }
  MF_REDUCE(reduce_force_kernel, n, n, n, nchunk, partial, rec, t, has_text, fx,
            fy, fz);
  return Status::Ok();
}

Status hessian_allpairs_launch(mf_ctx *ctx, const Points &tgt, int64_t nt, const SrcRec *src,
                               const float4 *boxes, int64_t ns, const HessConsts &hc,
                               float *const dst[9], const int sym[9]) {
  if (nt == 0) return Status::Ok();
  const Split f = split_sources(ctx, nt, ns, kHessTPT, kMaxChunks);
  void *pw = nullptr;
  MF_TRY(workspace(ctx, "hessian_partial", sizeof(double) * 6 * nt * f.nchunk, &pw));
  double *partial = static_cast<double *>(pw);
  if (f.nsub == 0) {
    hipLaunchKernelGGL(zero_f64_kernel, dim3(grid_for(6 * nt, 256)), dim3(256), 0, ctx->stream,
                       6 * nt, partial);
    MF_LAUNCH_CHECK();
  } else {
    KernelTimer timer(ctx, "hessian");
    hipLaunchKernelGGL(hessian_allpairs_kernel<kHessTPT>,
                       dim3(f.gx, static_cast<unsigned>(f.nchunk)), dim3(64), 0, ctx->stream, tgt,
                       nt, src, boxes, f.nsub, f.per, hc, nt, partial);
    MF_LAUNCH_CHECK();
  }
  TensorOut out{};
  for (int k = 0; k < 9; ++k) {
    out.p[k] = dst[k];
    out.sym[k] = sym[k];
  }
  MF_REDUCE(reduce_hessian_kernel, nt, nt, nt, static_cast<int>(f.nchunk), partial, out);
  return Status::Ok();
}
#undef MF_REDUCE

}  // namespace mf

// Internal: the near-pair coefficient tables, for the CPU tests (not part of
// mf_capi.h).  kind 0 = field (kFieldTabEntries x 8 floats), 1 = force
// (kHessTabEntries x 8), whose second curve is handed out divided by -5: R in units of
// its far form's -5 r^-7.
extern "C" int mf_internal_near_table(int kind, double h, float *out) {
  if (!out || !(h > 0.0)) return 1;
  if (kind == 0) mf::make_field_table(h, out);
  else if (kind == 1) {
    mf::make_hess_table(h, out);
    for (int e = 0; e < mf::kHessTabEntries; ++e)
      for (int j = 4; j < 8; ++j) out[8 * e + j] = static_cast<float>(out[8 * e + j] / -5.0);
  } else return 1;
  return 0;
}
