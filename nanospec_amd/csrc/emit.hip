// Second pass of the fused head over kept tile values: accept rate and dl (objective.py:39-46,
// 70-80) from the draft logits that pass 1's epilogue left in the workspace, the teacher rows
// and the row log-normalisers.  It replaces a second run of the whole head GEMM
// (head_kernel<EMIT> in lmhead.hip, still used where no workspace for the values is given): at
// N = 4096, d = 5120, V = 248,320 that run took 8.4 ms, most of it MFMA work done before.
//
// The values come as the accumulators held them (kZTile in ns_internal.h): 32 tokens x 128
// vocab entries of one wave as 16 KB, lane after lane.  A wave here takes one such block, so
// each of its lanes holds the entries head_kernel<EMIT>'s lane holds and adds them in the same
// order: dl and the accept sums are the same bits on either path.
#include "ns_profile.h"
#include "ns_tiles.h"

namespace ns {
namespace {

constexpr int kThreads = 256;   // 4 waves as 2 (vocab halves) x 2 (token halves), independent

struct EmitParams {
  const float* z;           // [tt][vt] tiles of kZTile
  const void* teacher;      // [n or nt, V]
  int64_t ldt;
  const int64_t* trows;     // teacher row of each token (null: its own)
  int64_t nt;
  const int64_t* labels;
  const float* weights;
  const float* row_stats;
  float c_ce, c_kl, inv_acc;
  uint16_t* dl;             // or null
  int64_t ldd;
  // with drows, token t's dl goes to row drows[t] of ndl; a token whose drows is outside [0, ndl)
  // has none, and its teacher row is not read
  const int64_t* drows;
  int64_t ndl;
  int64_t n, v;
  int vt;
  float* asum;              // [vt][2][rows]: each 128-entry half tile's sum min(p, t)
  float* ksum;              // likewise sum t (u - z) (LSE), or null
  int64_t rows;
};

// Workgroup: step s (tokens 32 s .. + 31 of both 128-token halves) of one 256 x 256 tile.
// Memory-bound: 4 + 2 bytes read and 2 written per entry (bf16 teacher), every load of a wave
// issued before its first use (24 KB a wave, 12 waves a CU).
template <typename TT, bool LSE, bool MAP>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(sizeof(TT) == 2 ? 3 : 2)))
void emit_tiles_kernel(EmitParams p) {
  using R = Rows<TT>;
  __shared__ __attribute__((aligned(16))) char lds_raw[4][R::kBytes];
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int wm = wv >> 1, wn = wv & 1;
  // vocab tiles fastest: workgroups that run together read and write neighbouring columns of the
  // same 64 rows (at N = 4096, V = 248,320: 1.38 ms, against 1.50 ms with the steps fastest)
  const int vt = blockIdx.x % p.vt, s = blockIdx.x / p.vt;
  const int64_t tb = (int64_t)blockIdx.y * 256 + wn * 128 + 32 * s;
  if (tb >= p.n) return;   // the whole wave; no workgroup barrier follows
  const int64_t vb = (int64_t)vt * 256 + wm * 128;
  const int64_t t = tb + r, tc = t < p.n ? t : p.n - 1;
  float* const asum = p.asum + ((int64_t)vt * 2 + wm) * p.rows;
  float* const ksum = LSE ? p.ksum + ((int64_t)vt * 2 + wm) * p.rows : nullptr;
  if (vb >= p.v) {
    if (h == 0 && t < p.n) {
      asum[t] = 0.f;
      if (LSE) ksum[t] = 0.f;
    }
    return;
  }
  // this lane's token's row of dl, -1: none (n and ndl are below 2^31); a wave without any leaves,
  // its tokens' sums are not read
  int dmine = (int)t;
  if (MAP) {
    const int64_t m = t < p.n ? p.drows[t] : -1;
    dmine = m >= 0 && m < p.ndl ? (int)m : -1;
    if (!__any(dmine >= 0)) return;
  }
  lds_t* const lds = (lds_t*)lds_raw[wv];
  const bool full = vb + 128 <= p.v;

  // the kept values
  const f32x4_t* zp = reinterpret_cast<const f32x4_t*>(p.z + ((int64_t)blockIdx.y * p.vt + vt) * kZTile) +
                      (s * 4 + wv) * 16 * 64 + lane;
  f32x4_t zv[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) zv[k] = __builtin_nontemporal_load(zp + k * 64);
  // the teacher rows (rows past N re-read the last one, pieces past V the first; neither is used)
  const TT* const teacher = static_cast<const TT*>(p.teacher);
  const int64_t col = vb + R::kPer * R::piece(lane);
  const int64_t colc = col < p.v ? col : vb;
  u32x4_t uv[R::kLoads];
#pragma unroll
  for (int i = 0; i < R::kLoads; ++i) {
    int64_t tr = tb + R::row(i, lane);
    tr = tr < p.n ? tr : p.n - 1;
    // a row without dl reads the step's first (a branch here made every load wait: 8.5 ms at
    // N = 2048 for 0.5)
    if (MAP) tr = __shfl(dmine, R::row(i, lane)) >= 0 ? tr : tb;
    if (p.trows) {
      tr = p.trows[tr];
      tr = tr >= 0 && tr < p.nt ? tr : 0;   // its log-normaliser is NaN
    }
    uv[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(teacher + tr * p.ldt + colc));
  }
  const float* rs = p.row_stats + tc * kRowStatWidth;
  const float lzl = rs[kLseZ] * kLog2e, lul = rs[kLseU] * kLog2e;
  const int64_t y = p.labels[tc];
  const float w = p.weights[tc] * p.inv_acc;
  // an ignored row has no CE term: dl = w c_kl (p - t) (its label matches no entry)
  const float cp = y == kIgnoreIndex ? w * p.c_kl : w * (p.c_ce + p.c_kl), ct = w * p.c_kl;
  const int64_t yr = y - vb;
  // this lane holds entry y
  const bool mine = t < p.n && yr >= 0 && yr < 128 && y < p.v && (int)((yr >> 2) & 1) == h;
  float uy = 0.f;
  if (p.dl && mine) {
    int64_t tr = tc;
    if (p.trows) {
      tr = p.trows[tc];
      tr = tr >= 0 && tr < p.nt ? tr : 0;
    }
    uy = load1(teacher + tr * p.ldt + y);
  }
#pragma unroll
  for (int i = 0; i < R::kLoads; ++i) R::put(lds, i, lane, uv[i]);
  wave_lds_sync();

  float aloc = 0.f, kloc = 0.f;
  auto chunk = [&](int k) {
    float u[4], d[4];
    R::get(lds, k, r, h, u);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float pp = fast_exp2(__builtin_fmaf(zv[k][q], kLog2e, -lzl));
      const float tt = fast_exp2(__builtin_fmaf(u[q], kLog2e, -lul));
      aloc += min_nonneg(pp, tt);
      // KL's sum t (u - z)
      if (LSE) kloc = __builtin_fmaf(tt, u[q] - zv[k][q], kloc);
      d[q] = __builtin_fmaf(cp, pp, -ct * tt);
    }
    const u32x2_t o = {pack_bf16x2(d[0], d[1]), pack_bf16x2(d[2], d[3])};
    *reinterpret_cast<__attribute__((address_space(3))) u32x2_t*>(lds + R::off(k, r, h)) = o;
  };
  if (full) {
#pragma unroll
    for (int k = 0; k < 16; ++k) chunk(k);
  } else {   // V % 8 == 0: each chunk is wholly inside or outside
#pragma unroll
    for (int k = 0; k < 16; ++k)
      if (vb + 8 * k < p.v) chunk(k);
  }
  aloc = half_sum(aloc);
  if (LSE) kloc = half_sum(kloc);
  if (h == 0 && t < p.n) {
    asum[t] = aloc;
    if (LSE) ksum[t] = kloc;
  }
  if (!p.dl) return;
  if (mine) {
    // the label entry with its -c_ce term, over this lane's own store; z_y is pass 1's value
    const float pp = fast_exp2(__builtin_fmaf(rs[kZy], kLog2e, -lzl));
    const float tt = fast_exp2(__builtin_fmaf(uy, kLog2e, -lul));
    *reinterpret_cast<__attribute__((address_space(3))) uint16_t*>(lds + R::off((int)(yr >> 3), r, h) +
                                                                   2 * (int)(yr & 3)) =
        f32_to_bf16(__builtin_fmaf(cp, pp, -ct * tt) - w * p.c_ce);
  }
  wave_lds_sync();
  // out as rows: 16 lanes per token, 256 bytes
  const int c = lane & 15;
  const int64_t ocol = vb + 8 * c;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int row = 4 * i + (lane >> 4);
    const u32x4_t x = R::out(lds, row, c);
    const int64_t dr = MAP ? (int64_t)__shfl(dmine, row) : tb + row;
    if ((MAP ? dr >= 0 : dr < p.n) && ocol < p.v)
      __builtin_nontemporal_store(x, reinterpret_cast<u32x4_t*>(p.dl + dr * p.ldd + ocol));
  }
}

// Row sums of the half tiles' partials in the order head_kernel<EMIT> and row_parts_kernel add
// them: each vocab half's tiles of a split in tile order, the halves, then the splits in order.
// kSumRows rows x 256 / kSumRows split lanes per workgroup: 16 rows, or 4 past 48 splits (few
// rows: with 16, N = 224, 256 splits took 30 us for 15, N = 1001, 64 splits 23 for 15; N = 2048,
// 32 splits 15 us for 24 the other way round).
template <bool LSE, int kSumRows>
__global__ __launch_bounds__(256) void emit_rows_kernel(const float* __restrict__ asum, const float* __restrict__ ksum,
                                                        int64_t rows, int vt, int splits, int64_t n,
                                                        float* __restrict__ row_stats, int64_t* __restrict__ drows,
                                                        int64_t ndl) {
  extern __shared__ float sh[];   // [LSE ? 2 : 1][splits][kSumRows]
  const int rl = threadIdx.x % kSumRows, l = threadIdx.x / kSumRows;
  const int64_t r = (int64_t)blockIdx.x * kSumRows + rl;
  const int64_t rc = r < n ? r : n - 1;
  for (int sp = l; sp < splits; sp += 256 / kSumRows) {
    const int v0 = (int)((int64_t)sp * vt / splits), v1 = (int)((int64_t)(sp + 1) * vt / splits);
    float a0 = 0.f, a1 = 0.f, k0 = 0.f, k1 = 0.f;
#pragma unroll 4
    for (int j = v0; j < v1; ++j) {
      a0 += asum[(int64_t)(2 * j) * rows + rc];
      a1 += asum[(int64_t)(2 * j + 1) * rows + rc];
      if (LSE) {
        k0 += ksum[(int64_t)(2 * j) * rows + rc];
        k1 += ksum[(int64_t)(2 * j + 1) * rows + rc];
      }
    }
    sh[sp * kSumRows + rl] = a0 + a1;
    if (LSE) sh[(splits + sp) * kSumRows + rl] = k0 + k1;
  }
  __syncthreads();
  if (l > 0 || r >= n) return;
  float* rs = row_stats + r * kRowStatWidth;
  if (drows && (drows[r] < 0 || drows[r] >= ndl)) {
    // a row without dl: accept 0, or NaN (and marked) where its dl is 0 * NaN
    const float none = accept_rate_of(0.f, rs[kLseZ], rs[kLseU]);
    rs[kAccept] = none;
    drows[r] = none == 0.f ? -1 : kRowNan;
    return;
  }
  float a = sh[rl];
  for (int sp = 1; sp < splits; ++sp) a += sh[sp * kSumRows + rl];
  rs[kAccept] = accept_rate_of(a, rs[kLseZ], rs[kLseU]);
  if (LSE) {
    float k = sh[splits * kSumRows + rl];
    for (int sp = 1; sp < splits; ++sp) k += sh[(splits + sp) * kSumRows + rl];
    rs[kKL] = k - rs[kLseU] + rs[kLseZ];
  }
}

template <typename TT, bool LSE, bool MAP>
hipError_t launch(const EmitParams& p, int splits, float* row_stats, hipStream_t st) {
  const int tt = (int)((p.n + 255) / 256);
  {
    NS_TIMED("head_emit", st);
    hipLaunchKernelGGL((emit_tiles_kernel<TT, LSE, MAP>), dim3((unsigned)p.vt * 4, (unsigned)tt), dim3(kThreads), 0, st, p);
    if (const hipError_t e = hipGetLastError(); e != hipSuccess) return e;
  }
  NS_TIMED("row_parts", st);
  const int rows = splits > 48 ? 4 : 16;
  const dim3 grid((unsigned)((p.n + rows - 1) / rows));
  const size_t lds = (size_t)splits * rows * sizeof(float) * (LSE ? 2 : 1);
  if (rows == 4)
    hipLaunchKernelGGL((emit_rows_kernel<LSE, 4>), grid, dim3(256), lds, st, p.asum, p.ksum, p.rows, p.vt, splits, p.n,
                       row_stats, const_cast<int64_t*>(p.drows), p.ndl);
  else
    hipLaunchKernelGGL((emit_rows_kernel<LSE, 16>), grid, dim3(256), lds, st, p.asum, p.ksum, p.rows, p.vt, splits,
                       p.n, row_stats, const_cast<int64_t*>(p.drows), p.ndl);
  return hipGetLastError();
}

}  // namespace

size_t emit_workspace_bytes(int64_t n, int64_t v) {
  const int64_t tt = (n + 255) / 256, vt = (v + 255) / 256;
  return align_up((size_t)(tt * vt * kZTile) * sizeof(float), 256) +
         2 * align_up((size_t)(vt * 2 * tt * 256) * sizeof(float), 256);
}

hipError_t emit_from_tiles(void* ws, const void* teacher, int tdt, int64_t ldt, const TeacherSpec& ts, int64_t v,
                           const SlotArgs& a, int splits, void* dl, int64_t ldd, int64_t* drows, int64_t ndl,
                           float* row_stats, hipStream_t st) {
  EmitParams p = {};
  const int64_t tt = (a.n + 255) / 256;
  p.vt = (int)((v + 255) / 256);
  p.rows = tt * 256;
  const size_t bz = align_up((size_t)(tt * p.vt * kZTile) * sizeof(float), 256);
  const size_t bs = align_up((size_t)(p.vt * 2 * p.rows) * sizeof(float), 256);
  char* c = static_cast<char*>(ws);
  p.z = reinterpret_cast<const float*>(c);
  p.asum = reinterpret_cast<float*>(c + bz);
  p.ksum = reinterpret_cast<float*>(c + bz + bs);
  p.teacher = teacher; p.ldt = ldt;
  p.trows = ts.rows; p.nt = ts.nt;
  p.labels = a.labels; p.weights = a.weights; p.row_stats = row_stats;
  p.c_ce = a.c_ce; p.c_kl = a.c_kl; p.inv_acc = a.inv_acc;
  p.dl = static_cast<uint16_t*>(dl); p.ldd = ldd;
  p.drows = drows; p.ndl = ndl;
  p.n = a.n; p.v = v;
  if (drows)
    return tdt == kBF16 ? launch<uint16_t, false, true>(p, splits, row_stats, st)
                        : launch<float, false, true>(p, splits, row_stats, st);
  if (tdt == kBF16)
    return ts.lse ? launch<uint16_t, true, false>(p, splits, row_stats, st)
                  : launch<uint16_t, false, false>(p, splits, row_stats, st);
  return ts.lse ? launch<float, true, false>(p, splits, row_stats, st)
                : launch<float, false, false>(p, splits, row_stats, st);
}

}  // namespace ns
