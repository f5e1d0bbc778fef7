// mf_pair_once.hpp -- a block of targets in registers against a staged tile of
// records, each unordered pair evaluated once for both of its particles.
//
// The distance, its inverse root and the radial coefficients of a pair serve
// both particles, and the force on one is minus the force on the other.  A wave
// holds 16 TPT targets (lane c of each 16-lane row: targets c, c + 16, ...) and a
// tile of 64 records in LDS, 16 for each row: at step s lane c takes record
// (s + c) mod 16 of its row's sixteen, and the sums for that record move one lane
// down the row with it, so after 16 steps lane l holds the sums of record l over
// the wave's targets.  Sums of either side that are combined in the end (the field's two,
// the force's term along the particle's own moment) are kept apart until then.  64 evaluated far pairs cost 96 (field) and 121 (force) cycles
// at TPT = 4, where two directed ones cost 130 and 182.
#pragma once

#include <hip/hip_runtime.h>

#include "mf_allpairs.hpp"
#include "mf_pair.hpp"

namespace mf {

constexpr float kPadCoord = 1.0e18f;  // far-away position of padding records

struct SelfTile {  // 64 records
  float4 pos[kTile], mom[kTile];
};

// Copies 16 bytes a lane from global memory into LDS (lane l's at lds + 16 l), with no
// register held; the copy has landed once vmcnt says so.
__device__ __forceinline__ void copy16_to_lds(const float4 *g, float4 *lds) {
  __builtin_amdgcn_global_load_lds(
      reinterpret_cast<const __attribute__((address_space(1))) void *>(
          reinterpret_cast<uintptr_t>(g)),
      reinterpret_cast<__attribute__((address_space(3))) void *>(reinterpret_cast<uintptr_t>(lds)),
      16, 0, 0);
}

// Waits until at most N of the wave's memory operations are outstanding (copies
// into LDS and stores retire in order); no access moves across it.
template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// The value of the next lane up in the 16-lane row (cyclic).
__device__ __forceinline__ float row_next(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x12F, 0xf, 0xf, false));
}

// Distances and inverse distances of the lane's record (u.xyz) to its targets
// k0 .. k0 + K - 1; one run of roots at raised priority, as in StepPairs.
template <int K>
struct SelfPairs {
  float dx[K], dy[K], dz[K], r2[K], ir[K];
  template <int TPT>
  __device__ __forceinline__ SelfPairs(const float4 &u, int k0, const float (&tx)[TPT],
                                       const float (&ty)[TPT], const float (&tz)[TPT]) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      dx[k] = tx[k0 + k] - u.x;
      dy[k] = ty[k0 + k] - u.y;
      dz[k] = tz[k0 + k] - u.z;
      r2[k] = fmaf(dx[k], dx[k], fmaf(dy[k], dy[k], dz[k] * dz[k]));
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int k = 0; k < K; ++k) ir[k] = __builtin_amdgcn_rsqf(r2[k]);
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
  }
};

template <int TPT>
struct FieldSelf {
  const FieldConsts &fc;
  const float4 *tab;
  float tx[TPT], ty[TPT], tz[TPT], nx[TPT], ny[TPT], nz[TPT];
  float a1[TPT][3], a2[TPT][3];
  __device__ __forceinline__ FieldSelf(const FieldConsts &consts, const float4 *t)
      : fc(consts), tab(t) {}
  __device__ __forceinline__ bool far(float dist2) const { return dist2 >= fc.near2; }
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int k = 0; k < TPT; ++k)
#pragma unroll
      for (int a = 0; a < 3; ++a) a1[k][a] = a2[k][a] = 0.f;
  }
  // target k's sum since the last clear, component a
  __device__ __forceinline__ double sum(int k, int a) const {
    return 3.0 * static_cast<double>(a1[k][a]) - static_cast<double>(a2[k][a]);
  }
  // jc (BOTH): the sums of the lane's record
  template <bool MIXED, bool BOTH>
  __device__ __forceinline__ void tile(const SelfTile &st, int c, int q, float (&jc)[3]) {
    float j1[3] = {0.f, 0.f, 0.f}, j2[3] = {0.f, 0.f, 0.f};
#pragma unroll 1
    for (int s = 0; s < 16; ++s) {
      const int r = 16 * q + ((s + c) & 15);
      const float4 u = st.pos[r], v = st.mom[r];
      float b1[3] = {0.f, 0.f, 0.f}, b2[3] = {0.f, 0.f, 0.f};
      constexpr int K = MIXED ? 1 : TPT;  // with the table, fewer pairs' registers
#pragma unroll
      for (int k0 = 0; k0 < TPT; k0 += K) {
        const SelfPairs<K> p(u, k0, tx, ty, tz);
#pragma unroll
        for (int i = 0; i < K; ++i) {
          const int k = k0 + i;
          const float ir2 = p.ir[i] * p.ir[i];
          float beta = ir2 * p.ir[i];
          float alpha = beta * ir2;
          if constexpr (MIXED) {
            if (p.r2[i] < fc.near2) {
              field_near_coeffs_tab(tab, fc.tab_scale, p.r2[i], p.ir[i], alpha, beta);
            }
          }
          const float dm = fmaf(p.dx[i], v.x, fmaf(p.dy[i], v.y, p.dz[i] * v.z));
          const float s1 = dm * alpha;
          a1[k][0] = fmaf(p.dx[i], s1, a1[k][0]);
          a1[k][1] = fmaf(p.dy[i], s1, a1[k][1]);
          a1[k][2] = fmaf(p.dz[i], s1, a1[k][2]);
          a2[k][0] = fmaf(v.x, beta, a2[k][0]);
          a2[k][1] = fmaf(v.y, beta, a2[k][1]);
          a2[k][2] = fmaf(v.z, beta, a2[k][2]);
          if constexpr (BOTH) {
            const float dn = fmaf(p.dx[i], nx[k], fmaf(p.dy[i], ny[k], p.dz[i] * nz[k]));
            const float s2 = dn * alpha;
            b1[0] = fmaf(p.dx[i], s2, b1[0]);
            b1[1] = fmaf(p.dy[i], s2, b1[1]);
            b1[2] = fmaf(p.dz[i], s2, b1[2]);
            b2[0] = fmaf(nx[k], beta, b2[0]);
            b2[1] = fmaf(ny[k], beta, b2[1]);
            b2[2] = fmaf(nz[k], beta, b2[2]);
          }
        }
      }
      if constexpr (BOTH) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          j1[a] = row_next(j1[a]) + b1[a];
          j2[a] = row_next(j2[a]) + b2[a];
        }
      }
    }
    if constexpr (BOTH) {
#pragma unroll
      for (int a = 0; a < 3; ++a)
        jc[a] = static_cast<float>(3.0 * static_cast<double>(row_next(j1[a])) -
                                   static_cast<double>(row_next(j2[a])));
    }
  }
};

// The pair force f = d e + m f1 + n g1 on the target is -f on the record:
// f1 = P (d.n), g1 = P (d.m), e = P (m.n) + R (d.m)(d.n), R = -5 P / r^2 (far).
template <int TPT>
struct ForceSelf {
  const HessConsts &hc;
  const float4 *tab;
  float tx[TPT], ty[TPT], tz[TPT], nx[TPT], ny[TPT], nz[TPT];
  float ad[TPT][3], am[TPT][3], an[TPT];
  __device__ __forceinline__ ForceSelf(const HessConsts &consts, const float4 *t)
      : hc(consts), tab(t) {}
  __device__ __forceinline__ bool far(float dist2) const { return dist2 > hc.near2; }
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int k = 0; k < TPT; ++k) {
#pragma unroll
      for (int a = 0; a < 3; ++a) ad[k][a] = am[k][a] = 0.f;
      an[k] = 0.f;
    }
  }
  __device__ __forceinline__ double sum(int k, int a) const {
    float n = a == 0 ? nx[k] : a == 1 ? ny[k] : nz[k];
    // not converted ahead of the caller's walk: 24 registers held through every tile
    asm volatile("" : "+v"(n));
    return (static_cast<double>(ad[k][a]) + static_cast<double>(am[k][a])) +
           static_cast<double>(n) * static_cast<double>(an[k]);
  }
  // jc (BOTH): the sums of the lane's record
  template <bool MIXED, bool BOTH>
  __device__ __forceinline__ void tile(const SelfTile &st, int c, int q, float (&jc)[3]) {
    float j[3] = {0.f, 0.f, 0.f}, jf = 0.f;
#pragma unroll 1
    for (int s = 0; s < 16; ++s) {
      const int r = 16 * q + ((s + c) & 15);
      const float4 u = st.pos[r], v = st.mom[r];
      float b[3] = {0.f, 0.f, 0.f}, bf = 0.f;
      constexpr int K = MIXED ? 1 : TPT;  // with the table, fewer pairs' registers
#pragma unroll
      for (int k0 = 0; k0 < TPT; k0 += K) {
        const SelfPairs<K> p(u, k0, tx, ty, tz);
#pragma unroll
        for (int i = 0; i < K; ++i) {
          const int k = k0 + i;
          const float dm = fmaf(p.dx[i], v.x, fmaf(p.dy[i], v.y, p.dz[i] * v.z));
          const float dn = fmaf(p.dx[i], nx[k], fmaf(p.dy[i], ny[k], p.dz[i] * nz[k]));
          const float mn = fmaf(v.x, nx[k], fmaf(v.y, ny[k], v.z * nz[k]));
          float P, e;
          if constexpr (MIXED) {
            // the clamp keeps a pair at d = 0 finite
            const float ir = __builtin_amdgcn_fmed3f(p.ir[i], 0.f, 1e12f);
            const float ir2 = ir * ir;
            float c1 = ir2 * ir2, dq = -5.f * c1;  // far curves
            if (!(p.r2[i] > hc.near2)) {
              hess_near_curves_tab(tab, hc.tab_scale, p.r2[i], ir, c1, dq);
              const bool apart = p.r2[i] > 0.f;  // nothing at d = 0
              c1 = apart ? c1 : 0.f;
              dq = apart ? dq : 0.f;
            }
            P = c1 * ir;
            e = fmaf(dq * (ir2 * ir), dm * dn, P * mn);
          } else {
            const float ir2 = p.ir[i] * p.ir[i];
            P = ir2 * ir2 * p.ir[i];
            e = P * fmaf(-5.f * ir2 * dm, dn, mn);
          }
          const float f1 = P * dn, g1 = P * dm;
          ad[k][0] = fmaf(p.dx[i], e, ad[k][0]);
          ad[k][1] = fmaf(p.dy[i], e, ad[k][1]);
          ad[k][2] = fmaf(p.dz[i], e, ad[k][2]);
          am[k][0] = fmaf(v.x, f1, am[k][0]);
          am[k][1] = fmaf(v.y, f1, am[k][1]);
          am[k][2] = fmaf(v.z, f1, am[k][2]);
          an[k] += g1;
          if constexpr (BOTH) {
            b[0] = fmaf(nx[k], g1, fmaf(p.dx[i], e, b[0]));
            b[1] = fmaf(ny[k], g1, fmaf(p.dy[i], e, b[1]));
            b[2] = fmaf(nz[k], g1, fmaf(p.dz[i], e, b[2]));
            bf += f1;
          }
        }
      }
      if constexpr (BOTH) {
#pragma unroll
        for (int a = 0; a < 3; ++a) j[a] = row_next(j[a]) + b[a];
        jf = row_next(jf) + bf;
      }
    }
    if constexpr (BOTH) {
      const float4 v = st.mom[16 * q + c];
      const double f = static_cast<double>(row_next(jf));
      jc[0] = static_cast<float>(-(static_cast<double>(v.x) * f + static_cast<double>(row_next(j[0]))));
      jc[1] = static_cast<float>(-(static_cast<double>(v.y) * f + static_cast<double>(row_next(j[1]))));
      jc[2] = static_cast<float>(-(static_cast<double>(v.z) * f + static_cast<double>(row_next(j[2]))));
    }
  }
};

}  // namespace mf
