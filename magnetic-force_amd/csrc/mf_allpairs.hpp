// mf_allpairs.hpp -- host entry points of the all-pairs kernels.
#pragma once

#include <hip/hip_runtime.h>

#include "mf_internal.hpp"
#include "mf_pair.hpp"

namespace mf {

// 32-byte source record: position and moment, both float4-aligned.
struct __attribute__((aligned(32))) SrcRec {
  float x, y, z, w;
  float mx, my, mz, mw;
};

constexpr int kTile = 64;  // sources per tile (bounding-box granularity)

int64_t padded_sources(int64_t n);

// Target positions: element i at x[i * stride], y[i * stride], z[i * stride].
struct Points {
  const float *x, *y, *z;
  int stride;
};
inline Points record_points(const SrcRec *rec) {
  return {&rec->x, &rec->y, &rec->z, static_cast<int>(sizeof(SrcRec) / sizeof(float))};
}

// Packs SoA positions and moments (moments may be null => 0) into
// padded_sources(n) records (padding records are far away, zero moment) and
// writes the bounding box (lo, hi float4 pairs) of every tile of kTile records.
Status pack_tiles(mf_ctx *ctx, int64_t n, const float *x, const float *y, const float *z,
                  const float *mx, const float *my, const float *mz, SrcRec *out, float4 *boxes);
// Rewrites only the moments of the first n records.
Status pack_moments(mf_ctx *ctx, int64_t n, const float *mx, const float *my, const float *mz,
                    float scale, SrcRec *out);

// A few sources, in the caller's arrays.
struct SourceArrays {
  const float *x, *y, *z, *mx, *my, *mz;
  int n;
};
// Whether the launches below take these sources: few of them, and no output (nt
// elements each, null skipped) overlaps an input.
bool few_sources(int64_t nt, int64_t ns, const Points &tgt, const SourceArrays &src, float *const *out,
                 int nout);
Status field_few_launch(mf_ctx *ctx, const Points &tgt, int64_t nt, const SourceArrays &src,
                        const FieldConsts &fc, const float *hconst, float *ox, float *oy, float *oz);
Status hessian_few_launch(mf_ctx *ctx, const Points &tgt, int64_t nt, const SourceArrays &src,
                          const HessConsts &hc, float *const dst[9], const int sym[9]);

// out = hconst + G m over the targets.
Status field_allpairs_launch(mf_ctx *ctx, const Points &tgt, int64_t nt, const SrcRec *src,
                             const float4 *boxes, int64_t ns, const FieldConsts &fc,
                             const float *hconst, float *ox, float *oy, float *oz);
// The same with the chunk partials in caller memory (partial_cap doubles, at
// least field_partial_doubles(nt, 1)); the source chunk count is cut to fit.
// Allocates nothing.
Status field_allpairs_launch_ws(mf_ctx *ctx, const Points &tgt, int64_t nt, const SrcRec *src,
                                const float4 *boxes, int64_t ns, const FieldConsts &fc,
                                const float *hconst, float *ox, float *oy, float *oz,
                                double *partial, int64_t partial_cap);
int64_t field_partial_doubles(int64_t nt, int64_t nchunk);
// A product whose use the host has not decided yet when it is launched: its kernels end at
// once where *rr < below (a solve that has converged).
struct Skip {
  const double *rr = nullptr;  // null: never
  double below = 0.0;
};
#ifdef __HIPCC__
__device__ __forceinline__ bool skipped(const Skip &s) { return s.rr && *s.rr < s.below; }
#endif
// The product of a conjugate-gradient step on one record set (its moments
// packed): ap = p - G m, and dots[b] (b < field_ap_blocks(n)) the parts of
// p . ap.
struct ApOut {
  const float *p[3];
  float *ap[3];
  double *dots;
  Skip skip;
};
// out = hconst + G m of one record set on itself.
Status field_self_launch(mf_ctx *ctx, const SrcRec *rec, const float4 *boxes, int64_t n,
                         const FieldConsts &fc, const float *hconst, float *ox, float *oy,
                         float *oz);
int field_ap_blocks(int64_t n);
Status field_allpairs_ap(mf_ctx *ctx, const SrcRec *rec, const float4 *boxes, int64_t n,
                         const FieldConsts &fc, const ApOut &out);
// F_i = (sum_j B(x_i - x_j)[m_j] + Text_i) m_i over one record set.
Status force_allpairs_launch(mf_ctx *ctx, const SrcRec *rec, const float4 *boxes, int64_t n,
                             const HessConsts &hc, const float *const *text9, float *fx,
                             float *fy, float *fz);
// Force tensor at separate targets: dst[k] (null = skipped) receives the
// symmetric component sym[k] (0..5 = xx yy zz xy xz yz).  boxes: tile boxes
// of the source records.
Status hessian_allpairs_launch(mf_ctx *ctx, const Points &tgt, int64_t nt, const SrcRec *src,
                               const float4 *boxes, int64_t ns, const HessConsts &hc,
                               float *const dst[9], const int sym[9]);

// FP64 check path (mf_check64.hip).
Status field_allpairs_f64(mf_ctx *ctx, int64_t nt, const double *tx, const double *ty,
                          const double *tz, int64_t ns, const double *sx, const double *sy,
                          const double *sz, const double *mx, const double *my,
                          const double *mz, double h, const double *hconst, double *ox,
                          double *oy, double *oz);
Status force_allpairs_f64(mf_ctx *ctx, int64_t n, const double *x, const double *y,
                          const double *z, const double *mx, const double *my, const double *mz,
                          double h, double *fx, double *fy, double *fz);

Status force_subset_f64(mf_ctx *ctx, int64_t n, const double *x, const double *y,
                        const double *z, const double *mx, const double *my, const double *mz,
                        double h, int64_t nt, const int64_t *idx, double *fx, double *fy,
                        double *fz);

}  // namespace mf
