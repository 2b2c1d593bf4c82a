// The head GEMM for few rows (at most kThinRows): a narrow tile that is bound by reading W once.
//
// The 256 x 256 tiles of lmhead.hip spend a whole token tile of matrix-core and LDS work however
// few tokens there are, which kept such a pass at 4.2 TB/s of W (N = 7, d = 5120, V = 248,320:
// 0.60 ms).  Here a wave takes 128 vocab rows and all tokens (NB blocks of 32).  Its weight rows come
// straight into LDS, 128 bytes of a row at a time as coalesced pieces, in two stages that no other
// wave reads; the hidden rows are shared by the workgroup.  With one stage multiplied in a quarter
// of the time the next takes to arrive, memory sets the pace: 0.43 ms, 5.9 TB/s.  (Loading the
// fragments from memory by the lanes that use them, 32 bytes of 32 rows an instruction and no
// LDS, ran no faster than the wide tile.)
//
// Every accumulator entry runs the MFMA instruction of lmhead.hip over K in the same order, and
// the epilogue folds a wave's 128 entries per token as that kernel does, so logits, statistics and
// partial sums are the same bits.
#include "ns_profile.h"
#include "ns_tiles.h"

namespace ns {
namespace {

enum { THIN_STATS = 0, THIN_STORE = 1 };

struct ThinParams {
  const uint16_t* hidden;   // [n or nh, d]
  const uint16_t* weight;   // [V, d]
  int64_t ldh, ldw, n, d, v;
  const int64_t* hrows;     // hidden row of each token (STORE; null: its own) of nh
  int64_t nh;
  const int64_t* prev;      // Markov head as a second K segment (r > 0)
  const uint16_t *w1, *w2;
  int64_t ldw1, ldw2, r;
  const uint16_t* markov;   // dense addend [n, V] or null
  int64_t ldm;
  const void* teacher;      // STATS
  int64_t ldt;
  const int64_t* trows;
  int64_t nt;
  const int64_t* labels;
  float* z;                 // STATS: tiles of kZTile (one token tile)
  float* zy;
  uint16_t* out;            // STORE: [n, V]
  int64_t ldo;
  RowPart* tpart;           // [vt][2][n] partials of each half tile (STORE: or null)
  int vt;
  bool stagger;
};

// Weight rows whose pitch is a multiple of 4 KB meet the same memory channels while all workgroups walk
// K in step.  Where W comes from memory the workgroups of an XCD then start apart: projections in us
// together / apart, n = 8 and 56: V = 248,320, d = 2048 255 / 231, 268 / 246; V = 65,536, d = 4096 127 /
// 116, 131 / 122; V = 98,304, d = 2048 (384 MB) 83 / 81, 110 / 108; V = 40,960, d = 4096 (320 MB) 71 / 67,
// 74 / 74.  A smaller W is held by the Infinity Cache (256 MB) and the delay is a tail: V = 65,536, d =
// 2048 41 / 42, 43 / 47; V = 32,768 22 / 27, 33 / 38; V = 8192 20 / 23, 32 / 35.  (n = 120: unchanged
// below 700 MB, 288 / 268 at V = 248,320.)
constexpr int64_t kStaggerBytes = int64_t(5) << 26;

// LDS of a workgroup of W waves: each wave's own two stages of its 128 weight rows (64 K entries,
// 128 bytes a row, lds_off's swizzle), then the stages of the NB x 32 hidden rows they share: three,
// or two with a second barrier a stage where three do not fit (128 rows, four waves).
constexpr int kAStage = 128 * 128;
constexpr int b_stage(int nb) { return nb * 32 * 128; }
constexpr int b_stages(int w, int nb) { return w * 2 * kAStage + 3 * b_stage(nb) <= 160 * 1024 ? 3 : 2; }
constexpr int thin_lds(int w, int nb) { return w * 2 * kAStage + b_stages(w, nb) * b_stage(nb); }

// One K segment of KT 64-entry stages: acc += weight rows . hidden rows.  Stage t + 1 is in flight
// while stage t is multiplied (a short while of a stage's time: the pass waits for memory), its
// hidden rows go out after a barrier that finds their buffer read by every wave, its weight rows
// once the wave has read stage t - 1 (no other wave reads them).
template <int W, int NB>
__device__ __forceinline__ void thin_segment(f32x16_t (&acc)[4][NB], const char* wbase, const DmaTile<128, 1>& ta,
                                             const char* hbase, const DmaTile<32 * NB, W>& tb, int KT, lds_t* lds,
                                             int wv, int lane) {
  constexpr int NIB = DmaTile<32 * NB, W>::NI, BS = b_stages(W, NB);
  lds_t* const la = lds + wv * 2 * kAStage;
  lds_t* const lb = lds + W * 2 * kAStage;
  const int r = lane & 31, h = lane >> 5;
  auto k_of = [&](int t) -> int64_t { return (int64_t)(t < KT - 1 ? t : KT - 1) * 128; };   // past the end: unused
  auto fill_a = [&](int t) {
#pragma unroll
    for (int i = 0; i < 16; ++i) ta.issue_asm(wbase + k_of(t), la + (t & 1) * kAStage, 0, i);
  };
  auto fill_b = [&](int t) {
#pragma unroll
    for (int i = 0; i < NIB; ++i) tb.issue_asm(hbase + k_of(t), lb + (t % BS) * b_stage(NB), wv, i);
  };
  fill_b(0);
  fill_a(0);
  fill_b(1);
  fill_a(1);
  for (int t = 0; t < KT; ++t) {
    vm_barrier<16 + NIB>();   // stage t landed in every wave; every wave is past stage t - 1
    if (BS == 3) fill_b(t + 2);
    const lds_t* a = la + (t & 1) * kAStage;
    const lds_t* b = lb + (t % BS) * b_stage(NB);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      bf16x8_t fa[4], fb[NB];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        fa[i] = *reinterpret_cast<const __attribute__((address_space(3))) bf16x8_t*>(a + lds_off(32 * i + r, kk * 2 + h));
#pragma unroll
      for (int j = 0; j < NB; ++j)
        fb[j] = *reinterpret_cast<const __attribute__((address_space(3))) bf16x8_t*>(b + lds_off(32 * j + r, kk * 2 + h));
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
    }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): this wave has read its stage
    if (BS == 2) __builtin_amdgcn_s_barrier();   // every wave has read the shared rows
    asm volatile("" ::: "memory");
    if (BS == 2) fill_b(t + 2);
    fill_a(t + 2);
  }
  fill_barrier();   // nothing in flight, every wave done with the shared stages
}

template <int MODE, typename TT, bool LSE, int NB, int W>
__global__ __launch_bounds__(64 * W) void thin_kernel(ThinParams p) {
  // STATS: LSE = the teacher's log-normaliser is given (no teacher read); STORE: LSE = the stored
  // values' log-sum-exp partials are formed
  constexpr bool kReadU = MODE == THIN_STATS && !LSE;
  static_assert(Rows<uint16_t>::kBytes + Rows<float>::kBytes <= 2 * kAStage, "the epilogue's rows");
  __shared__ __attribute__((aligned(16))) char lds_raw[thin_lds(W, NB)];
  lds_t* const lds = (lds_t*)lds_raw;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int vt = (int)blockIdx.x * (W / 2) + (wv >> 1), wm = wv & 1;
  // a wave past the last entry runs along on the last row (the waves share barriers)
  const int64_t vb = (int64_t)vt * 256 + wm * 128;
  const bool none = vb >= p.v;
  const bool full = vb + 128 <= p.v;

  // an XCD's workgroups start up to 7 us apart (kStaggerBytes)
  if (p.stagger)
    for (int q = (int)(blockIdx.x / kNumXcd) % 8; q > 0; --q) __builtin_amdgcn_s_sleep(32);

  f32x16_t acc[4][NB];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  {
    const int64_t w0 = none ? p.v - 1 : vb;
    DmaTile<128, 1> ta;
    DmaTile<32 * NB, W> tb;
    // the hidden rows' fill offsets: row(token) of a [.., ld] matrix
    auto hidden_rows = [&](int64_t ld, auto&& row) {
#pragma unroll
      for (int i = 0; i < DmaTile<32 * NB, W>::NI; ++i) {
        const int q = (wv * DmaTile<32 * NB, W>::NI + i) * 8 + (lane >> 3);
        tb.off[i] = (uint32_t)(row(q < p.n ? q : p.n - 1) * ld * 2 + ((lane & 7) ^ swz(q)) * 16);
      }
    };
    ta.init(p.ldw * 2, w0, p.v, 0);
    hidden_rows(p.ldh, [&](int64_t t) -> int64_t {
      if (MODE != THIN_STORE || !p.hrows) return t;
      const int64_t x = p.hrows[t];
      return x >= 0 && x < p.nh ? x : 0;
    });
    thin_segment<W, NB>(acc, reinterpret_cast<const char*>(p.weight + w0 * p.ldw), ta,
                        reinterpret_cast<const char*>(p.hidden), tb, (int)(p.d / 64), lds, wv, lane);
    if (MODE == THIN_STATS && p.r > 0) {
      ta.init(p.ldw2 * 2, w0, p.v, 0);
      hidden_rows(p.ldw1, [&](int64_t t) -> int64_t {
        const int64_t x = p.prev[t];
        return x >= 0 && x < p.v ? x : 0;
      });
      thin_segment<W, NB>(acc, reinterpret_cast<const char*>(p.w2 + w0 * p.ldw2), ta,
                          reinterpret_cast<const char*>(p.w1), tb, (int)(p.r / 64), lds, wv, lane);
    }
  }
  if (vt >= p.vt) return;
  RowPart* const tp = p.tpart ? p.tpart + ((int64_t)vt * 2 + wm) * p.n : nullptr;
  if (none) {   // no entry in this half tile: its partials are still merged
    RowPart rp;
    rp.mz = rp.mu = kNegBig;
    rp.sz = rp.su = rp.A = rp.pad0 = rp.pad1 = rp.pad2 = 0.f;
    if (tp)
      for (int64_t t = lane; t < p.n; t += 64) tp[t] = rp;
    return;
  }
  // opaque from here: the epilogue's addresses are formed after the K loop, not held across it
  asm volatile("" : "+v"(lane));
  r = lane & 31;
  h = lane >> 5;
  // (the wave's own stages are free: the K loop ended with a barrier)
  lds_t* const lm = lds + wv * 2 * kAStage;
  lds_t* const lu = lm + Rows<uint16_t>::kBytes;
  const float nan = __builtin_nanf("");
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int64_t tb = 32 * j, t = tb + r, tc = t < p.n ? t : p.n - 1;
    if (tb >= p.n) break;   // the whole wave
    PairState ploc = pair_init();
    LseState lloc = {kNegBig, 0.f};
    bool ubad = false, bad = false;   // teacher row; Markov id or gathered hidden row out of range
    if (MODE == THIN_STATS && p.r > 0) {
      const int64_t id = p.prev[tc];
      bad = id < 0 || id >= p.v;
    }
    if (MODE == THIN_STORE && p.hrows) {
      const int64_t hr = p.hrows[tc];
      bad = hr < 0 || hr >= p.nh;
    }
    {
      wave_lds_sync();   // the previous block's rows are read
      // the dense addend's and the teacher's rows, whole pieces into LDS (rows past N re-read the
      // last, pieces past V the first; neither is used)
      if (p.markov) {
        using R = Rows<uint16_t>;
        const int64_t col = vb + 8 * R::piece(lane), colc = col < p.v ? col : vb;
        u32x4_t x[R::kLoads];
#pragma unroll
        for (int i = 0; i < R::kLoads; ++i) {
          int64_t row = tb + R::row(i, lane);
          row = row < p.n ? row : p.n - 1;
          x[i] = *reinterpret_cast<const u32x4_t*>(p.markov + row * p.ldm + colc);
        }
#pragma unroll
        for (int i = 0; i < R::kLoads; ++i) R::put(lm, i, lane, x[i]);
      }
      if constexpr (kReadU) {
        using R = Rows<TT>;
        const int64_t col = vb + R::kPer * R::piece(lane), colc = col < p.v ? col : vb;
        const TT* const u = static_cast<const TT*>(p.teacher);
        u32x4_t x[R::kLoads];
#pragma unroll
        for (int i = 0; i < R::kLoads; ++i) {
          int64_t row = tb + R::row(i, lane);
          row = row < p.n ? row : p.n - 1;
          if (p.trows) {
            row = p.trows[row];
            row = row >= 0 && row < p.nt ? row : 0;
          }
          x[i] = *reinterpret_cast<const u32x4_t*>(u + row * p.ldt + colc);
        }
#pragma unroll
        for (int i = 0; i < R::kLoads; ++i) R::put(lu, i, lane, x[i]);
        if (p.trows) {
          const int64_t tr = p.trows[tc];
          ubad = tr < 0 || tr >= p.nt;
        }
      }
      wave_lds_sync();
      const int64_t y = MODE == THIN_STATS ? p.labels[tc] : -1;
      const int64_t yr = y - vb;
      const bool mine = MODE == THIN_STATS && t < p.n && yr >= 0 && yr < 128 && y < p.v && (int)((yr >> 2) & 1) == h;
      float zy = 0.f;
#pragma unroll
      for (int hs = 0; hs < 2; ++hs) {
        float z[32], u[32];
#pragma unroll
        for (int c = 0; c < 8; ++c) {
          const int k = 8 * hs + c;   // chunk: rows 32 (k / 4) + 8 (k % 4) + 4 h .. of the half tile
          const bool ok = full || vb + 8 * k < p.v;
          float mk[4] = {0.f, 0.f, 0.f, 0.f};
          if (p.markov) Rows<uint16_t>::get(lm, k, r, h, mk);
          if constexpr (kReadU) Rows<TT>::get(lu, k, r, h, u + 4 * c);
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            float& zq = z[4 * c + q];
            zq = acc[k >> 2][j][4 * (k & 3) + q] + mk[q];
            if (MODE == THIN_STORE && bad) zq = nan;
            zq = ok ? zq : kNegBig;
            if (kReadU) u[4 * c + q] = ok ? u[4 * c + q] : kNegBig;
            if (MODE == THIN_STATS) zy = 8 * k + 4 * h + q == (int)yr ? zq : zy;
          }
          if (MODE == THIN_STATS) {
            const f32x4_t zc = {z[4 * c], z[4 * c + 1], z[4 * c + 2], z[4 * c + 3]};
            // step j % 4 of token half j / 4 (here 0): emit.hip reads it back with the same lanes
            reinterpret_cast<f32x4_t*>(p.z + (int64_t)vt * kZTile)[((j * 4 + wm * 2) * 16 + k) * 64 + lane] = zc;
          } else {
            const u32x2_t o = {pack_bf16x2(z[4 * c], z[4 * c + 1]), pack_bf16x2(z[4 * c + 2], z[4 * c + 3])};
            *reinterpret_cast<__attribute__((address_space(3))) u32x2_t*>(lm + Rows<uint16_t>::off(k, r, h)) = o;
          }
        }
        const bool any = full || vb + 64 * hs < p.v;
        if (any) {
          if constexpr (kReadU) {
            pair_update<32>(ploc, z, u);
          } else if constexpr (MODE == THIN_STATS) {
            lse_update<32>(lloc, z);
          } else if (LSE) {   // of the values as stored
#pragma unroll
            for (int i = 0; i < 32; ++i) z[i] = bf16_to_f32(f32_to_bf16(z[i]));
            lse_update<32>(lloc, z);
          }
        }
      }
      if (mine) p.zy[t] = bad ? nan : zy;
      if (MODE == THIN_STORE) {
        wave_lds_sync();
        const int c = lane & 15;
        const int64_t col = vb + 8 * c;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int row = 4 * i + (lane >> 4);
          const u32x4_t x = Rows<uint16_t>::out(lm, row, c);
          if (tb + row < p.n && col < p.v) *reinterpret_cast<u32x4_t*>(p.out + (tb + row) * p.ldo + col) = x;
        }
      }
    }
    if (!tp) continue;
    RowPart rp;
    rp.pad0 = rp.pad1 = rp.pad2 = 0.f;
    if constexpr (kReadU) {
      PairState loc = half_merge(ploc);
      if (bad) { loc.mz = nan; loc.sz = nan; }
      if (ubad) { loc.mu = nan; loc.su = nan; loc.A = nan; }
      rp.mz = loc.mz; rp.sz = loc.sz; rp.mu = loc.mu; rp.su = loc.su; rp.A = loc.A;
    } else {
      LseState loc = half_merge(lloc);
      if (MODE == THIN_STATS && bad) loc = {nan, nan};
      rp.mz = loc.m; rp.sz = loc.s; rp.mu = kNegBig; rp.su = 0.f; rp.A = 0.f;
    }
    if (h == 0 && t < p.n) tp[t] = rp;
  }
}

template <int MODE, typename TT, bool LSE>
hipError_t launch_thin(const ThinParams& args, const char* name, hipStream_t st) {
  NS_TIMED(name, st);
  ThinParams p = args;
  p.stagger = p.ldw % 2048 == 0 && p.v * p.d * 2 >= kStaggerBytes;
  // 512 vocab rows a workgroup, or 256 where those would leave CUs without one
  const bool wide = p.vt > kThinWide;
  const dim3 grid((unsigned)(wide ? (p.vt + 1) / 2 : p.vt));
  if (p.n <= 32 && wide)
    hipLaunchKernelGGL((thin_kernel<MODE, TT, LSE, 1, 4>), grid, dim3(256), 0, st, p);
  else if (p.n <= 32)
    hipLaunchKernelGGL((thin_kernel<MODE, TT, LSE, 1, 2>), grid, dim3(128), 0, st, p);
  else if (p.n <= 64 && wide)
    hipLaunchKernelGGL((thin_kernel<MODE, TT, LSE, 2, 4>), grid, dim3(256), 0, st, p);
  else if (p.n <= 64)
    hipLaunchKernelGGL((thin_kernel<MODE, TT, LSE, 2, 2>), grid, dim3(128), 0, st, p);
  else   // more than 64 rows come only with kThinWide
    hipLaunchKernelGGL((thin_kernel<MODE, TT, LSE, 4, 4>), grid, dim3(256), 0, st, p);
  return hipGetLastError();
}

}  // namespace

size_t thin_workspace_bytes(int64_t n, int64_t v) {
  return align_up((size_t)((v + 255) / 256 * 2 * n) * sizeof(RowPart), 256);
}

hipError_t thin_stats(const ThinHead& x, const SlotArgs& a, const TeacherSpec& ts, const void* teacher, int tdt,
                      int64_t ldt, float* z, float* zy, RowPart* tpart, hipStream_t st) {
  ThinParams p = {};
  p.hidden = x.hidden; p.weight = x.weight; p.ldh = x.ldh; p.ldw = x.ldw;
  p.n = a.n; p.d = x.d; p.v = x.v;
  p.markov = x.markov; p.ldm = x.ldm;
  if (x.factors) {
    p.prev = x.factors->prev;
    p.w1 = static_cast<const uint16_t*>(x.factors->w1);
    p.w2 = static_cast<const uint16_t*>(x.factors->w2);
    p.ldw1 = x.factors->ldw1; p.ldw2 = x.factors->ldw2; p.r = x.factors->r;
  }
  p.teacher = teacher; p.ldt = ldt;
  p.trows = ts.rows; p.nt = ts.nt;
  p.labels = a.labels;
  p.z = z; p.zy = zy; p.tpart = tpart;
  p.vt = (int)((x.v + 255) / 256);
  if (ts.lse) return launch_thin<THIN_STATS, uint16_t, true>(p, "head_stats", st);
  if (tdt == kBF16) return launch_thin<THIN_STATS, uint16_t, false>(p, "head_stats", st);
  return launch_thin<THIN_STATS, float, false>(p, "head_stats", st);
}

hipError_t thin_store(const ThinHead& x, const int64_t* rows, int64_t nrows, int64_t n, void* out, int64_t ldo,
                      RowPart* tpart, hipStream_t st) {
  ThinParams p = {};
  p.hidden = x.hidden; p.weight = x.weight; p.ldh = x.ldh; p.ldw = x.ldw;
  p.n = n; p.d = x.d; p.v = x.v;
  p.hrows = rows; p.nh = nrows;
  p.markov = x.markov; p.ldm = x.ldm;
  p.out = static_cast<uint16_t*>(out); p.ldo = ldo;
  p.tpart = tpart;
  p.vt = (int)((x.v + 255) / 256);
  if (!tpart) return launch_thin<THIN_STORE, uint16_t, false>(p, "head_linear", st);
  return launch_thin<THIN_STORE, uint16_t, true>(p, "head_linear_lse", st);
}

}  // namespace ns
