// Row copies by an index map: dst row r = src row map[r], zeros where map[r] is outside
// [0, n_src) (NaN where it is kRowNan).  The fused head forms dl and runs the dh GEMM on the rows
// whose outputs are not all zero (head.lm_head_ce_kl_loss(skip_masked_rows=True)): the compact dh
// (and, on request, dl) is scattered back with zero rows between.  HBM-bound: each byte is read
// and written once, with non-temporal 16-byte accesses (the rows are not read again soon).
#include "ns_internal.h"
#include "ns_profile.h"

namespace ns {
namespace {

typedef uint32_t u32x4r_t __attribute__((ext_vector_type(4)));

// One thread per 16-byte chunk (W = 16) or 4-byte word (W = 4) of a destination row.
template <int W>
__global__ __launch_bounds__(256) void copy_rows_kernel(const char* __restrict__ src, int64_t ld_src, int64_t n_src,
                                                        const int64_t* __restrict__ map, int64_t n_dst,
                                                        int64_t row_bytes, char* __restrict__ dst, int64_t ld_dst) {
  const int64_t per_row = row_bytes / W;
  const int64_t total = n_dst * per_row;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int64_t r = i / per_row, c = i - r * per_row;
    const int64_t s = map[r];
    char* to = dst + r * ld_dst + c * W;
    if constexpr (W == 16) {
      const uint32_t none = s == kRowNan ? 0xffffffffu : 0u;
      u32x4r_t x = {none, none, none, none};
      if (s >= 0 && s < n_src) x = __builtin_nontemporal_load(reinterpret_cast<const u32x4r_t*>(src + s * ld_src + c * W));
      __builtin_nontemporal_store(x, reinterpret_cast<u32x4r_t*>(to));
    } else {
      uint32_t x = s == kRowNan ? 0xffffffffu : 0u;
      if (s >= 0 && s < n_src) x = *reinterpret_cast<const uint32_t*>(src + s * ld_src + c * W);
      *reinterpret_cast<uint32_t*>(to) = x;
    }
  }
}

// The kept rows' places: 1024 threads walk the rows, each wave's kept lanes counted by ballot, the
// waves' counts summed through LDS.  One workgroup: 32 steps at N = 32,768, and the host waits for
// the count.
constexpr int kKeptThreads = 1024;
__global__ __launch_bounds__(kKeptThreads) void kept_rows_kernel(const float* __restrict__ weights,
                                                                 const uint8_t* __restrict__ valid, int64_t n,
                                                                 int64_t* __restrict__ index,
                                                                 int64_t* __restrict__ count) {
  __shared__ int part[kKeptThreads / 64];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  int64_t base = 0;
  for (int64_t r0 = 0; r0 < n; r0 += kKeptThreads) {
    const int64_t r = r0 + threadIdx.x;
    const bool keep = r < n && (valid[r] != 0 || weights[r] != 0.f);
    const uint64_t m = __ballot(keep);
    if (lane == 0) part[wave] = __popcll(m);
    __syncthreads();
    int before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < kKeptThreads / 64; ++w) {
      before += w < wave ? part[w] : 0;
      all += part[w];
    }
    if (r < n) index[r] = keep ? base + before + __popcll(m & ((uint64_t(1) << lane) - 1)) : -1;
    base += all;
    __syncthreads();
  }
  if (threadIdx.x == 0) count[0] = base;
}

}  // namespace

hipError_t kept_rows(const float* weights, const uint8_t* valid, int64_t n, int64_t* index, int64_t* count,
                     hipStream_t st) {
  NS_TIMED("kept_rows", st);
  hipLaunchKernelGGL(kept_rows_kernel, dim3(1), dim3(kKeptThreads), 0, st, weights, valid, n, index, count);
  return hipGetLastError();
}

hipError_t copy_rows(const void* src, int64_t ld_src, int64_t n_src, const int64_t* map, int64_t n_dst,
                     int64_t row_bytes, void* dst, int64_t ld_dst, hipStream_t st) {
  if (n_dst == 0 || row_bytes == 0) return hipSuccess;
  const bool vec = row_bytes % 16 == 0 && ld_src % 16 == 0 && ld_dst % 16 == 0 &&
                   (reinterpret_cast<uintptr_t>(src) & 15u) == 0 && (reinterpret_cast<uintptr_t>(dst) & 15u) == 0;
  const int64_t items = n_dst * (row_bytes / (vec ? 16 : 4));
  const int64_t blocks = (items + 255) / 256 < 8192 ? (items + 255) / 256 : 8192;
  NS_TIMED("copy_rows", st);
  if (vec)
    hipLaunchKernelGGL(copy_rows_kernel<16>, dim3((unsigned)blocks), dim3(256), 0, st, static_cast<const char*>(src),
                       ld_src, n_src, map, n_dst, row_bytes, static_cast<char*>(dst), ld_dst);
  else
    hipLaunchKernelGGL(copy_rows_kernel<4>, dim3((unsigned)blocks), dim3(256), 0, st, static_cast<const char*>(src),
                       ld_src, n_src, map, n_dst, row_bytes, static_cast<char*>(dst), ld_dst);
  return hipGetLastError();
}

}  // namespace ns
