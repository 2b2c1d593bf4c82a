// Internal launch interface shared by the kernel sources and the C ABI layer.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <atomic>

#include "ns_common.h"

namespace ns {

// Inputs shared by every objective entry point (all device pointers).
struct SlotArgs {
  const int64_t* labels;   // [N] target token ids (prepared.target_ids)
  const float* weights;    // [N] w = valid * exp(-slot/gamma) (prepared.weights)
  const uint8_t* valid;    // [N] supervision validity (prepared.valid, torch.bool)
  int64_t n;               // rows (draft slots)
  int64_t k;               // slots per block (accept_len prefix axis)
  float c_ce, c_kl;        // objective.ce, objective.kl
  float inv_acc;           // 1 / accumulation_steps
};

// ---- logits-level streaming path (stream.hip) -----------------------------
int stream_splits(int64_t n, int64_t v);
size_t stream_workspace_bytes(int64_t n, int64_t v);
hipError_t stream_forward(const void* z, int zdt, int64_t ldz, const void* u, int udt, int64_t ldu,
                          int64_t v, const SlotArgs& a, void* dl, int64_t ldd, float* row_stats,
                          float* metrics, void* ws, hipStream_t st);
hipError_t stream_backward(const void* z, int zdt, int64_t ldz, const void* u, int udt, int64_t ldu,
                           int64_t v, const SlotArgs& a, const float* row_stats, void* dl, int64_t ldd,
                           hipStream_t st);

// ---- shared tails (stream.hip) ---------------------------------------------
// Teacher logits as the producer left them: objective row t reads teacher row rows[t]
// (rows null: row t) of nt rows; lse (null: formed in pass 1) holds one log-normaliser per
// teacher row.
struct TeacherSpec {
  const int64_t* rows;
  int64_t nt;
  const float* lse;
};
// Vocab splits of a head plan at most (one a CU): a row merge over half tiles forms each split's state
// in a thread of its own.
constexpr int kMaxHeadSplits = 256;
// Merge first-pass partials part1[N][S] (+ z_y[N]) into row_stats (lse_z, lse_u, ce, kl, z_y).
// With ts (its lse given) lse_u comes from ts and KL is left to the finalize.  tiles > 0: part1
// holds the partials of half vocab tiles instead, [tiles][2][N], of which each of S splits takes a
// contiguous range (S <= kMaxHeadSplits).
hipError_t launch_merge(const RowPart* part1, const float* zy, int64_t v, int splits, const SlotArgs& a,
                        float* row_stats, hipStream_t st, const TeacherSpec* ts = nullptr, int tiles = 0);
// Sum accept partials parta[N][S], form block lengths and the six metrics; with partk
// (pass-2 sums of t (u - z)), KL = sum partk - lse_u + lse_z first.  parta NULL: the metrics
// alone, from complete row_stats; metrics NULL: the row sums alone.
hipError_t launch_finalize(const float* parta, int splits, const SlotArgs& a, float* row_stats,
                           float* metrics, hipStream_t st, const float* partk = nullptr);
// lse[t] = log-sum-exp from (max, sum-exp) partials part1[N][S] (mz, sz), fixed order.
hipError_t launch_lse_merge(const RowPart* part1, int splits, int64_t n, float* lse, hipStream_t st, int tiles = 0);

// ---- final_norm around the head (norm.hip) ------------------------------------
constexpr int64_t kMaxNormD = 16384;   // hidden sizes the rms-norm kernels hold in registers
// rms_norm backward operands (ops.py:55-66): x the forward's input, inv its [N] inverse
// RMS, w the norm weight [d]; outputs dx [N, d] and wgrad [d] (overwritten), all bf16
struct NormBwd {
  const uint16_t* x;
  int64_t ldx;
  const float* inv;
  const uint16_t* w;
  uint16_t* dx;
  int64_t lddx;
  uint16_t* wgrad;
};
int norm_rows_per_block(int64_t n);
size_t norm_bwd_workspace_bytes(int64_t n, int64_t d);
hipError_t rms_norm_forward(const void* x, int64_t ldx, const void* weight, int64_t n, int64_t d, float eps,
                            void* out, int64_t ldo, void* normalized, int64_t ldn, float* inv, hipStream_t st);
// dy from split-K partials part[ksplit][N][d] (dh_out, if not NULL, receives bf16 dh) or,
// with part == NULL, from the bf16 tensor dy
hipError_t rms_norm_backward_rows(const float* part, int ksplit, const void* dy, int64_t lddy, const NormBwd& nb,
                                  void* dh_out, int64_t lddh, int64_t n, int64_t d, void* ws, hipStream_t st);

// ---- fused LM-head path (lmhead.hip) ---------------------------------------
// Markov head in factored form: logits += W1[prev] . W2^T (rank r, r % 64 == 0).
struct MarkovFactors {
  const int64_t* prev;   // [N] previous-token ids
  const void* w1;        // [V, r] bf16, row stride ldw1
  const void* w2;        // [V, r] bf16, row stride ldw2
  int64_t ldw1, ldw2, r;
};
// Workspace of the fused forward: required (partials of all rows in one plan), min (partials by
// windows of rows, as the full one: the same bits), and the full one, which also holds one
// window's tile values (kZTile): pass 2 then forms dl from pass 1's values instead of running
// the GEMM again.
size_t lmhead_required_bytes(int64_t n, int64_t v);
size_t lmhead_min_workspace_bytes(int64_t n, int64_t v);
size_t lmhead_workspace_bytes(int64_t n, int64_t v, int64_t d);
size_t lmhead_rows_workspace_bytes(int64_t n, int64_t v);   // with drows: always with the tile values
// Raises the dynamic-LDS limit of every head instantiation lmhead_forward can launch, on the
// current device (done lazily at launch otherwise; this lets a caller do it before capture).
hipError_t lmhead_forward_prepare();
// lmhead_forward's parts: pass 1 and the merge (row_stats' log-normalisers, CE, KL, z_label),
// then pass 2 with the per-row accept (and teacher-once KL) sums and, when metrics is not
// NULL, the metrics
constexpr int kHeadStats = 1, kHeadEmit = 2, kHeadParts = kHeadStats | kHeadEmit;
hipError_t lmhead_forward(const void* hidden, int64_t ldh, const void* weight, int64_t ldw,
                          const void* markov, int64_t ldm, const MarkovFactors* factors, const void* teacher,
                          int tdt, int64_t ldt, int64_t d, int64_t v, const SlotArgs& a, const TeacherSpec* ts,
                          void* dl, int64_t ldd, float* row_stats, float* metrics, void* ws, size_t ws_bytes,
                          hipStream_t st, int parts = kHeadParts, int64_t* drows = nullptr, int64_t ndl = 0);
// dl row index of every row that is supervised (valid or a non-zero weight), in order, -1 for
// the others; count[0] = how many
hipError_t kept_rows(const float* weights, const uint8_t* valid, int64_t n, int64_t* index, int64_t* count,
                     hipStream_t st);

// ---- second pass over kept tile values (emit.hip) ------------------------------
// One 256 x 256 tile of draft logits (fp32, Markov addend included) as pass 1's accumulators hold
// it: block (s, wave) = 32 tokens x 128 vocab entries, 16 KB at ((s * 4 + wave) * 16 + k) * 256
// floats for chunk k = 0..15, 4 floats per lane: token 128 (wave & 1) + 32 s + lane % 32, entries
// 128 (wave >> 1) + 8 k + 4 (lane / 32) + 0..3.
constexpr int64_t kZTile = 256 * 256;
// A window's values (at the workspace's start, [token tiles][vocab tiles] of kZTile) and the
// partial sums after them.
size_t emit_workspace_bytes(int64_t n, int64_t v);
// accept rates (with ts.lse also KL) into row_stats and dl (if not NULL) of a window of a.n rows;
// `splits`: the vocab splits whose order the row sums follow.  With drows (ts.lse null) row t's dl
// goes to row drows[t] of ndl; rows mapped outside [0, ndl) have none, their accept rate is 0 (NaN
// when a log-normaliser is not finite) and their drows becomes -1 (kRowNan).
constexpr int64_t kRowNan = INT64_MIN;
hipError_t emit_from_tiles(void* ws, const void* teacher, int tdt, int64_t ldt, const TeacherSpec& ts, int64_t v,
                           const SlotArgs& a, int splits, void* dl, int64_t ldd, int64_t* drows, int64_t ndl,
                           float* row_stats, hipStream_t st);
// dst row r = src row map[r] (row_bytes bytes), or zeros where map[r] is outside [0, n_src), or
// bytes of 0xFF (NaN in bf16 and fp32) where map[r] is kRowNan
hipError_t copy_rows(const void* src, int64_t ld_src, int64_t n_src, const int64_t* map, int64_t n_dst,
                     int64_t row_bytes, void* dst, int64_t ld_dst, hipStream_t st);
// Pass 2 of lmhead_forward alone: dl for a.inv_acc from the row_stats a forward over the
// same inputs wrote (same kernel, so the same bits a forward with that inv_acc emits).
// Workspace: lmhead_workspace_bytes.
hipError_t lmhead_emit_dlogits(const void* hidden, int64_t ldh, const void* weight, int64_t ldw,
                               const void* markov, int64_t ldm, const MarkovFactors* factors, const void* teacher,
                               int tdt, int64_t ldt, int64_t d, int64_t v, const SlotArgs& a,
                               const TeacherSpec* ts, const float* row_stats, void* dl, int64_t ldd, void* ws,
                               hipStream_t st);
// dh workspace; r > 0 adds the Markov column tiles' partials, norm the rms-norm
// backward's column partials
size_t lmhead_bwd_workspace_bytes(int64_t n, int64_t v, int64_t d, int64_t r = 0, bool norm = false);
// what a call needs at least: with less than the above it takes as many K splits as fit
size_t lmhead_bwd_required_bytes(int64_t n, int64_t v, int64_t d, int64_t r = 0, bool norm = false);
hipError_t lmhead_backward(const void* dl, int64_t ldd, const void* weight, int64_t ldw, void* dh,
                           int64_t lddh, int64_t n, int64_t v, int64_t d, void* ws, size_t ws_bytes,
                           hipStream_t st);
// dh = dl . weight and, when r > 0, dprev = dl . w2 (fp32 [N, r], row stride r) in the same
// GEMM.  With norm, the split-K reduction is the rms-norm backward: dx and the norm weight's
// gradient are written, and dh only if dh is not NULL.
hipError_t lmhead_backward_ext(const void* dl, int64_t ldd, const void* weight, int64_t ldw, const void* w2,
                               int64_t ldw2, int64_t r, void* dh, int64_t lddh, float* dprev, const NormBwd* norm,
                               int64_t n, int64_t v, int64_t d, void* ws, size_t ws_bytes, hipStream_t st);
// Markov-head backward (markov.hip): dh (or, with norm, dx and the norm weight's gradient),
// w2_grad = dl^T . w1[prev] (overwritten) and w1_grad.index_add_(prev, dl . w2)
// (accumulated, deterministic order)
size_t markov_bwd_workspace_bytes(int64_t n, int64_t v, int64_t d, int64_t r);
size_t markov_bwd_required_bytes(int64_t n, int64_t v, int64_t d, int64_t r);
hipError_t markov_backward(const void* dl, int64_t ldd, const void* weight, int64_t ldw, const MarkovFactors& f,
                           void* dh, int64_t lddh, const NormBwd* norm, void* w1_grad, int64_t ldg1, void* w2_grad,
                           int64_t ldg2, int64_t n, int64_t v, int64_t d, void* ws, size_t ws_bytes, hipStream_t st);
hipError_t lmhead_linear(const void* x, int64_t ldx, const void* weight, int64_t ldw, const void* addend,
                         int64_t lda, void* out, int64_t ldo, int64_t n, int64_t v, int64_t d,
                         hipStream_t st);
// The projection as a teacher-logit producer: out = x[rows] . weight^T (+ addend) with,
// when lse is not NULL, lse[t] = log-sum-exp of out's bf16 row t; rows (null: row t)
// index nrows rows of x.  Workspace with lse: at least linear_lse_required_bytes; with
// lmhead_linear_lse_workspace_bytes few rows take thin.hip's kernel too.
size_t linear_lse_required_bytes(int64_t n, int64_t v);
size_t lmhead_linear_lse_workspace_bytes(int64_t n, int64_t v);
hipError_t lmhead_linear_lse(const void* x, int64_t ldx, const int64_t* rows, int64_t nrows, const void* weight,
                             int64_t ldw, const void* addend, int64_t lda, void* out, int64_t ldo, float* lse,
                             int64_t n, int64_t v, int64_t d, void* ws, size_t ws_bytes, hipStream_t st);

// ---- the head GEMM for few rows (thin.hip) ----------------------------------------
constexpr int64_t kThinRows = 128;   // up to 64 rows of any vocabulary, above with vocab tiles > kThinWide
constexpr int64_t kThinWide = 512;
struct ThinHead {
  const uint16_t *hidden, *weight, *markov;
  int64_t ldh, ldw, ldm, d, v;
  const MarkovFactors* factors;
};
// partials of each 128-entry half tile
size_t thin_workspace_bytes(int64_t n, int64_t v);
// Pass 1 of a.n <= kThinRows rows: z (one token tile of kZTile per vocab tile), z_label and the half
// tiles' partials tpart[vocab tiles][2][n], which launch_merge turns into the bits that
// head_kernel<STATS> and it form.
hipError_t thin_stats(const ThinHead& x, const SlotArgs& a, const TeacherSpec& ts, const void* teacher, int tdt,
                      int64_t ldt, float* z, float* zy, RowPart* tpart, hipStream_t st);
// The projection of n <= kThinRows rows, and with tpart its log-sum-exp partials.
hipError_t thin_store(const ThinHead& x, const int64_t* rows, int64_t nrows, int64_t n, void* out, int64_t ldo,
                      RowPart* tpart, hipStream_t st);

// ---- FP8 teacher head (fp8.hip) ---------------------------------------------
size_t fp8_workspace_bytes(int64_t n, int64_t v, int64_t d);
hipError_t fp8_quantize_rows(const void* x, int64_t ldx, int64_t n, int64_t d, uint8_t* q, float* xs,
                             hipStream_t st);
// lse (null: not formed): log-sum-exp of each stored bf16 output row, from the epilogue
hipError_t fp8_teacher_logits(const void* x, int64_t ldx, const uint8_t* wq, int64_t ldw,
                              const float* scale, void* out, int64_t ldo, float* lse, int64_t n, int64_t v,
                              int64_t d, void* ws, hipStream_t st);

// ---- slot preparation (prepare.hip) -----------------------------------------
hipError_t prepare_slots(const int64_t* ids, const float* loss_mask, const int64_t* anchors,
                         const uint8_t* keep, int64_t b, int64_t s, int64_t nb, int64_t k,
                         float gamma, int64_t* target_ids, int64_t* previous, float* weights,
                         uint8_t* valid, int64_t* teacher_indices, hipStream_t st);

// ---- pooled-normalisation tail (pooled.hip) ------------------------------------
// out[4] = (loss, accept_len, gradient factor, pooled denominator) from [count][6] metrics
hipError_t pooled_tail(const float* metrics, int64_t count, int64_t world_size, int64_t accumulation_steps,
                       float* out, hipStream_t st);
// grad[0..n) *= *factor in place (bf16 or fp32)
hipError_t scale_gradient(void* grad, int dtype, int64_t n, const float* factor, hipStream_t st);

// Groups of splits that the sums of split-K partials are formed in: each group's contiguous share
// (group g: splits [g * ksplit / G, (g + 1) * ksplit / G)) in order, then the groups in order.
__host__ __device__ inline int split_groups(int ksplit) { return ksplit <= 8 ? 1 : ksplit <= 24 ? 4 : 16; }

inline size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

// Raises a kernel's dynamic-LDS limit to `bytes` on the current device.  The attribute
// belongs to each device's copy of the kernel, so `done` keeps one bit per device id (ids
// of 64 and up set it on every call); concurrent first calls may both set it, harmlessly.
inline hipError_t ensure_dynamic_lds(const void* fn, int bytes, std::atomic<uint64_t>& done) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  const uint64_t bit = dev >= 0 && dev < 64 ? (uint64_t(1) << dev) : 0;
  if (bit && (done.load(std::memory_order_relaxed) & bit)) return hipSuccess;
  e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (e == hipSuccess && bit) done.fetch_or(bit, std::memory_order_relaxed);
  return e;
}

}  // namespace ns
