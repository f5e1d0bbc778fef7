// mf_sort.hip -- device radix sort and scans for the octree build (rocPRIM).
// Kept in its own translation unit: the rocPRIM templates are slow to compile.
#include <cstring>

#include <hip/hip_runtime.h>
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include "mf_sort.hpp"

namespace mf {

Status sort_pairs_u64_i32(mf_ctx *ctx, const uint64_t *keys_in, uint64_t *keys_out,
                          const int32_t *vals_in, int32_t *vals_out, int64_t n, int begin_bit,
                          int end_bit) {
  if (n == 0) return Status::Ok();
  size_t bytes = 0;
  MF_HIP(rocprim::radix_sort_pairs(nullptr, bytes, keys_in, keys_out, vals_in, vals_out,
                                   static_cast<size_t>(n), begin_bit, end_bit, ctx->stream));
  void *tmp = nullptr;
  MF_TRY(workspace(ctx, "sort_tmp", bytes + 16, &tmp));
  MF_HIP(rocprim::radix_sort_pairs(tmp, bytes, keys_in, keys_out, vals_in, vals_out,
                                   static_cast<size_t>(n), begin_bit, end_bit, ctx->stream));
  return Status::Ok();
}

namespace {
// One workgroup, each thread a run of up to 16: two launches and the host side of rocPRIM's
// device scan take longer than the scan of a small tree (a plan build has four: 4,000
// particles 390 -> 326 to 375 us in all).
constexpr int kScanThreads = 1024;
constexpr int64_t kScanSmall = 16 * kScanThreads;
__global__ __launch_bounds__(kScanThreads) void scan_small_kernel(int n, const int32_t *in, int32_t *out) {
  __shared__ int32_t s_wave[kScanThreads / 64];
  const int per = (n + kScanThreads - 1) / kScanThreads, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int i0 = min(static_cast<int>(threadIdx.x) * per, n), i1 = min(i0 + per, n);
  int32_t sum = 0;
  for (int i = i0; i < i1; ++i) sum += in[i];
  int32_t incl = sum;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int32_t v = __shfl_up(incl, o, 64);
    if (lane >= o) incl += v;
  }
  if (lane == 63) s_wave[w] = incl;
  __syncthreads();
  int32_t run = incl - sum;
  for (int k = 0; k < w; ++k) run += s_wave[k];
  for (int i = i0; i < i1; ++i) {
    const int32_t v = in[i];
    out[i] = run;
    run += v;
  }
}
}  // namespace

Status exclusive_scan_i32(mf_ctx *ctx, const int32_t *in, int32_t *out, int64_t n) {
  if (n == 0) return Status::Ok();
  if (n <= kScanSmall) {
    hipLaunchKernelGGL(scan_small_kernel, dim3(1), dim3(kScanThreads), 0, ctx->stream,
                       static_cast<int>(n), in, out);
    MF_LAUNCH_CHECK();
    return Status::Ok();
  }
  size_t bytes = 0;
  MF_HIP(rocprim::exclusive_scan(nullptr, bytes, in, out, 0, static_cast<size_t>(n),
                                 rocprim::plus<int32_t>(), ctx->stream));
  void *tmp = nullptr;
  MF_TRY(workspace(ctx, "scan_tmp", bytes + 16, &tmp));
  MF_HIP(rocprim::exclusive_scan(tmp, bytes, in, out, 0, static_cast<size_t>(n),
                                 rocprim::plus<int32_t>(), ctx->stream));
  return Status::Ok();
}

}  // namespace mf
