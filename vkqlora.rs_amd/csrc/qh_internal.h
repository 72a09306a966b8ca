// qh_internal.h -- declarations shared by the runtime (runtime.cpp) and the
// gfx950 kernels (k_*.hip).  Not part of the public ABI.
#pragma once
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <utility>

namespace qh {

// Kernel timing: when the runtime arms `g_launch_timing` around a call, the
// next kernel launched through qh_launch gets the two events stamped by the
// GPU at that kernel's own start and end (hipExtLaunchKernelGGL), so host
// launch gaps never enter the measurement.
struct LaunchTiming {
  hipEvent_t start = nullptr, stop = nullptr;
};
extern thread_local LaunchTiming g_launch_timing;

template <typename... KArgs, typename... Args>
hipError_t qh_launch(void (*k)(KArgs...), dim3 grid, dim3 block, uint32_t shmem,
                     hipStream_t s, Args &&...args) {
  static_assert(sizeof...(KArgs) == sizeof...(Args), "kernel argument count");
  if (g_launch_timing.start) {
    const LaunchTiming t = g_launch_timing;
    g_launch_timing = LaunchTiming();
    hipExtLaunchKernelGGL(k, grid, block, shmem, s, t.start, t.stop, 0,
                          static_cast<KArgs>(std::forward<Args>(args))...);
  } else {
    k<<<grid, block, shmem, s>>>(static_cast<KArgs>(std::forward<Args>(args))...);
  }
  return hipGetLastError();
}

// Device view of a quantized weight (rows x cols, flat row-major index).
struct DevQW {
  int64_t rows, cols, n, bs, nb;
  const uint8_t *codes;
  int kind;  // 0 = fp32 scales, 1 = int8 codes + fp32 absmax per 256 blocks
  const float *scales;
  const uint8_t *scale_codes;
  const float *absmax;
};

// Operand storage forms of the GEMM tile engine.  The engine computes
// C[m][n] = sum_k A[m][k] * B[k][n]; an operand with "rows" r (m for A, n
// for B) and reduction index k is stored either
//   ROWK: element (r, k) at p[r * ld + k]   (k contiguous), or
//   KROW: element (r, k) at p[k * ld + r]   (r contiguous).
enum Form { ROWK = 0, KROW = 1 };
enum Elem { E_F32 = 0, E_BF16 = 1, E_NF4 = 2 };

struct Operand {
  const void *p;
  int64_t ld;
  int form;  // Form
  int elem;  // Elem
  float scale;  // multiplies the operand when staged (1.0f = none)
};

struct GemmArgs {
  int64_t M, N;
  // segment 1: reduction over K with operands A, B (B may be NF4)
  Operand A, B;
  int64_t K;
  DevQW qw;  // valid when B.elem == E_NF4
  // segment 2 (optional, K2 == 0 = none): extra reduction with fp32 operands
  Operand A2, B2;
  int64_t K2;
  // output C[m * ldc + n] = alpha * acc; with split-K, split z writes to
  // C + z * split_stride and only covers its K range of segment 1.
  float *C;
  int64_t ldc;
  float alpha;
  int splits;
  int64_t split_stride;
};

// ---- k_gemm_bf16.hip: the NF4 GEMMs on bf16 MFMA ----
// Up to kMaxBf16Segs weights, each with its LoRA term, in one launch.
//  w_form ROWK (forward): every segment s reads the shared activations A
//   (M x K, row stride lda) and writes its own output
//   C_s (M x len_s) = alpha * (A . W_s^T + A2_s . B2_s),  W_s: len_s x K.
//  w_form KROW (input gradient): one output C (M x N) sums all segments,
//   C = alpha * sum_s (A_s . W_s + A2_s . B2_s),  A_s: M x len_s (row stride
//   lda_s), W_s: len_s x N; K = sum of len_s.
// A / A_s are bf16 or (a_f32) fp32 split into bf16 hi and lo parts.  The
// LoRA term: fp32 A2_s (M x K2_s, row-major, lda2) times B2_s scaled by
// b2scale, B2_s[k][n] = p[n * ldb2 + k] (ROWK) or p[k * ldb2 + n] (KROW).
constexpr int kMaxBf16Segs = 4;
struct Bf16Seg {
  DevQW w;
  const void *A;  // KROW: this segment's activations
  int64_t lda;
  const float *A2, *B2;
  int64_t lda2, ldb2, K2;
  float b2scale;
  float *C;  // ROWK: this segment's output
  int64_t ldc;
  int64_t len;    // ROWK: output columns; KROW: reduction length
  int64_t tile0;  // ROWK: first output tile (set by the launcher)
};
struct Bf16GemmArgs {
  int64_t M, N, K;  // N: all output columns, K: the whole reduction
  const void *A;    // ROWK: the shared activations
  int64_t lda;
  float *C;  // KROW: the output
  int64_t ldc;
  float alpha;
  int beta;  // 1: C += alpha (sum) (a residual already in C)
  int64_t split_stride;  // set by the launcher when the reduction is split
  int nseg;
  Bf16Seg seg[kMaxBf16Segs];
};
// True when the bf16-MFMA kernels take this weight (64-element blocks that
// never straddle a row) with activations `a` (row stride lda, K columns read).
bool bf16_gemm_ok(const DevQW &w, const void *a, int64_t lda, int64_t K);
// Reduction splits the bf16 kernels use for (M x N) outputs over K: > 1
// needs splits * M * N floats of partial sums.
int bf16_gemm_splits(int64_t M, int64_t N, int64_t K);
// About what they take for it (us), with fp32 or bf16 activations; `split`: in
// those splits (grouped forwards run in one).
double bf16_gemm_us(int64_t M, int64_t N, int64_t K, bool f32, bool split);
hipError_t launch_gemm_bf16(const Bf16GemmArgs &g, int w_form, int a_f32, int splits,
                            float *partial, hipStream_t s);
// Dense C = alpha sum_k A(m, k) B(n, k) on bf16 MFMA (fp32 operands as hi +
// lo parts), one output side at most 64 (the LoRA-rank products T1, Ds,
// grad_A, grad_B); A(m, k) at a[m lda + k] (ROWK) or a[k lda + m] (KROW), B
// the same with n.  Splits > 1 need dense_bf16_splits(M, N, K) * M * N floats
// of partial sums.
bool dense_bf16_ok(int64_t M, int64_t N, int64_t K, int a_form, const void *a, int64_t lda,
                   int b_form, const void *b, int64_t ldb);
int dense_bf16_splits(int64_t M, int64_t N, int64_t K);
hipError_t launch_dense_bf16(const void *a, int a_form, int a_f32, int64_t lda, const void *b,
                             int b_form, int b_f32, int64_t ldb, float *c, int64_t ldc,
                             int64_t M, int64_t N, int64_t K, float alpha, float *partial,
                             hipStream_t s);

// ---- k_quant.hip ----
hipError_t launch_quantize(const float *w, int64_t n, int64_t bs, int dq,
                           uint8_t *codes, float *scales, uint8_t *scale_codes,
                           float *absmax, float *scratch, hipStream_t s);
hipError_t launch_block_scales(const DevQW &w, float *out, hipStream_t s);
hipError_t launch_dequantize(const DevQW &w, float *out, hipStream_t s);

// ---- k_gemm.hip ----
// Runs the tile engine; splits > 1 needs `partial` (splits * M * N floats)
// and reduces into args.C deterministically.
// True when the tile engine runs (M x N) on 128x128 tiles (else 64x64).
bool gemm_uses_t128(int64_t M, int64_t N);
hipError_t launch_gemm(const GemmArgs &args, float *partial, hipStream_t s);
// C (M x N, row stride ldc) = the sum of `splits` partial (M x N) matrices
// stored back to back in `part`, added in split order (beta 1: C += that sum).
hipError_t launch_reduce_splits(const float *part, int splits, int64_t M, int64_t N, float *C,
                                int64_t ldc, hipStream_t s, int beta = 0);
// Tile-engine eligibility of a quantized B operand: block_size 64 and
// whole blocks per row of the reduction form.
bool nf4_fast_ok(const DevQW &w);

// ---- k_gemv.hip ----
// y[m][n] = sum_k x[m][k] W[n][k] + s * sum_j t1[m][j] * lb[n][j]  (M <= 4)
hipError_t launch_gemv(const DevQW &w, const void *x, int x_bf16, int64_t M,
                       const float *t1, const float *lb, int64_t r, float s,
                       float *y, hipStream_t st);
bool gemv_ok(const DevQW &w, int64_t M);
// T1 = X A^T for the GEMV path (K % 4 == 0, 16-byte aligned rows).
hipError_t launch_lora_t1(const void *x, int x_bf16, int64_t M, int64_t K, const float *a,
                          int64_t r, float *t1, hipStream_t st);
// The T1 of several layers with the same batch in one launch (per layer
// x: M x K, a: r x K, t1: M x r; the bits of launch_lora_t1).
constexpr int kMaxT1Jobs = 8;
struct T1Job {
  const void *x;
  const float *a;
  float *t1;
  int64_t K;
  int r;
};
struct T1Jobs {
  T1Job j[kMaxT1Jobs];
  int count;
};
hipError_t launch_lora_t1_jobs(const T1Jobs &jobs, int x_bf16, int64_t M, hipStream_t st);

// ---- decode (k_dstream.hip, k_dsplit.hip) ----
// `tickets` is the context's zero-initialised counter array of
// kTicketWords words (plus the one-launch kernel's words after it); every
// kernel leaves its counters at zero, and calls sharing it must be
// stream-ordered.  decode_ok: the shapes the MFMA decode kernels take
// (batch <= 16, r <= 64, block 64, in_dim % 256 == 0, aligned parts).
constexpr int kTicketWords = 16384;
constexpr int kDecodeTileCounterBase = 64;
constexpr int64_t kDecodeMaxTiles = kTicketWords - kDecodeTileCounterBase;
bool decode_ok(const DevQW &w, int64_t M, int64_t r);
// ---- k_dstream.hip ----
// Decode GEMV in one launch per layer (at most one workgroup per CU, one
// round) for batches of 1 and 2 rows, T1 = X A^T included.  It keeps 16
// launch counters (uint64) at tickets[kStreamEpochWord..] and tagged T1
// partials in the kStreamT1Words words after the kTicketWords counter
// words (both zero before the first launch); calls sharing them must be
// stream-ordered.
constexpr int kStreamEpochWord = 32;
constexpr int kStreamT1Words = 128 * 64 * 2;
// The second layer of a two-layer launch keeps its own 16 launch counters
// (32 words) and tagged T1 partials (kStreamT1Words words) from this word on.
constexpr int kStreamSlot2Word = kTicketWords + kStreamT1Words;
constexpr int kTicketsTotalWords = kStreamSlot2Word + 32 + kStreamT1Words;
// Two independent batch-1 layers in one launch (k_dstream2): each layer as
// launch_decode_stream would compute it, bit for bit.
bool decode_stream2_ok(const DevQW &w1, int64_t r1, const DevQW &w2, int64_t r2);
hipError_t launch_decode_stream2(const DevQW &w1, const void *x1, const float *a1, int64_t r1,
                                 const float *lb1, float s1, float *y1, float *t1_out1,
                                 const DevQW &w2, const void *x2, const float *a2, int64_t r2,
                                 const float *lb2, float s2, float *y2, float *t1_out2,
                                 int x_bf16, unsigned *tickets, bool force_t1_recompute,
                                 hipStream_t st);
// True when one launch serves the layer (batch 1-2, one round, T1 slices
// that fit a producer lane).
bool decode_stream_ok(const DevQW &w, int64_t M, int64_t r);
hipError_t launch_decode_stream(const DevQW &w, const void *x, int x_bf16, int64_t M,
                                const float *a, int64_t r, const float *lb, float s, float *y,
                                float *t1_out, unsigned *tickets, bool force_t1_recompute,
                                hipStream_t st);

// ---- k_dsplit.hip ----
// Decode GEMV for batches of 1-16 rows whose T1 = X A^T was computed by an
// earlier launch: one pass over the packed weight for the whole batch, K
// split into S slices across workgroups, the slices summed in order by the
// last workgroup of each group of R tiles (tickets from
// kDecodeTileCounterBase; calls sharing them must be stream-ordered).  A
// plan covers 1 / share of the CUs (share 2: one layer of a two-layer
// launch); the bits depend on the plan's S alone.
struct SplitPlan {
  int R = 0, S = 0, RW = 0, groups = 0, G = 0, Mt = 0;
  size_t part_floats = 0;  // scratch for the slices' partial sums (S > 1)
  uint32_t lds = 0;
  bool ok = false;
};
SplitPlan split_plan(const DevQW &w, int64_t M, int64_t r, int share = 1);
// True when two layers' plans (share 2) can run in one launch.
bool split_pair(SplitPlan &a, SplitPlan &b);
struct SplitLayerIn {
  DevQW w;
  const void *x;    // M x K
  const float *t1;  // M x r (r > 0)
  const float *lb;  // N x r (nullptr: no adapter)
  int64_t r;
  float s;
  float *y;         // M x N
  float *part;      // plan.part_floats floats (S > 1)
};
hipError_t launch_decode_split(int count, const SplitLayerIn *in, const SplitPlan *plans,
                               int64_t M, int x_bf16, unsigned *tickets, hipStream_t st);

// ---- k_plane.hip: large GEMMs through bf16 operand planes ----
// An operand (rows x K) as planes: fp32 p[r * ld + k] (PLANE_ROWK) or
// p[k * ld + r] (PLANE_KROW), times scale, as hi and lo parts; bf16
// p[r * ld + k] as one part; NF4 weight rows (r = W row) or columns (r = W
// column, K = W rows; rows % 64 == 0) as hi and lo parts.
enum PlaneForm { PLANE_ROWK, PLANE_KROW, PLANE_NF4_ROW, PLANE_NF4_COL };
struct PlaneSrc {
  int form, bf16;
  const void *p;
  int64_t ld, rows, K;
  float scale;
  DevQW w;
  void *dst;
};
// Whether an M x N output over K with an adapter of rank r (0: none) and fp32 or
// bf16 activations goes through planes (PLANE_NF4_ROW: where plane_codes_ok too).
bool plane_ok(int64_t M, int64_t N, int64_t K, int64_t r, bool f32);
// Whether the codes can be read as weight rows: 16 bytes at a time.
inline bool plane_codes_ok(const DevQW &w) { return ((uintptr_t)w.codes & 15) == 0; }
// About what they then take (us).
double plane_us(int64_t M, int64_t N, int64_t K, bool f32);
// Bytes of an A operand's (M rows) and a B operand's (N rows) planes.
size_t plane_a_bytes(int64_t M, int64_t K, int parts);
size_t plane_b_bytes(int64_t N, int64_t K);
hipError_t launch_planes(const PlaneSrc *src, int count, hipStream_t st);  // count <= 4
// C (M x N) = A . B^T + A2 . B2^T (+ C with beta), the sums of k_gemm_bf16.hip's
// unsplit kernels in their order.
struct PlaneGemm {
  const void *a, *b, *a2, *b2;
  int a_parts;
  int64_t M, N, K, K2;
  float *c;
  int64_t ldc;
  int beta;
};
hipError_t launch_plane_gemm(const PlaneGemm &p, hipStream_t st);

// ---- k_slim.hip ----
// The forward for few tokens: up to kMaxSlimSegs layers with the same batch
// in one pair of launches (launch_slim_prep, then launch_slim).  Layers with
// the same xp share their X.  The plan's tickets start at
// kDecodeTileCounterBase; calls sharing them must be stream-ordered.
constexpr int kMaxSlimSegs = 4;
struct SlimPlan {
  bool ok = false;
  int G = 0, P = 0, R = 0, chunks = 0;
  uint32_t lds = 0;
  double us = 0;  // about what the two launches take
  int S[kMaxSlimSegs] = {}, groups[kMaxSlimSegs] = {}, nz[kMaxSlimSegs] = {};
  size_t part_floats[kMaxSlimSegs] = {};  // scratch of the K slices' sums
  size_t xp_bytes[kMaxSlimSegs] = {};     // scratch of the X planes
};
struct SlimIn {
  DevQW w;
  const void *x;   // M x K
  const float *a;  // r x K
  int64_t r;       // 0: no adapter
  const float *lb; // N x r
  float s;
  float *t1p;      // nz x M x r partial T1s, written by the preparation (r > 0)
  float *t1;       // M x r, their sum (or nullptr)
  float *y;        // M x N
  int beta;        // 1: y += the result
  void *xp;        // plan.xp_bytes (16-byte aligned)
  float *part;     // plan.part_floats
};
bool slim_ok(const DevQW &w, const void *x, int x_bf16, const float *a, int64_t M, int64_t r);
SlimPlan slim_plan(int count, const DevQW *w, const int64_t *r, int64_t M, int x_bf16);
hipError_t launch_slim_prep(int count, const SlimIn *in, const SlimPlan &p, int64_t M,
                            int x_bf16, hipStream_t st);
hipError_t launch_slim(int count, const SlimIn *in, const SlimPlan &p, int64_t M,
                       unsigned *tickets, hipStream_t st);

// ---- k_elem.hip ----
hipError_t launch_axpy_inplace(float *y, const float *x, int64_t n,
                               hipStream_t s);  // y += x
hipError_t launch_zero(float *y, int64_t n, hipStream_t s);
hipError_t launch_bf16_to_f32(const uint16_t *x, float *y, int64_t n,
                              hipStream_t s);

// ---- k_adam.hip ----
struct AdamTensor {
  float *p;
  const float *g;
  uint8_t *m_codes, *v_codes;
  float *m_scales, *v_scales;
  int64_t numel, nblocks, block_offset;  // block_offset: prefix over tensors
  float b1t, b2t;
  double inv_b1t, inv_b2t;  // 1 / (double)b1t and 1 / (double)b2t
};
hipError_t launch_adam(const AdamTensor *d_tensors, int ntensors,
                       int64_t total_blocks, int64_t block_size, float lr,
                       float beta1, float beta2, float eps, hipStream_t s);

// Block glue around the projections (k_block.hip).
// x_copy (optional, not aliasing x or y): x is also copied there as read.
hipError_t launch_rmsnorm(const float *x, const float *w, float *y, int64_t rows, int h,
                          float eps, hipStream_t s, float *x_copy = nullptr);
int rmsnorm_dw_slices(int64_t rows);
// scratch of launch_rmsnorm_bwd when dw is wanted (floats)
size_t rmsnorm_dw_scratch_floats(int64_t rows, int h);
// add (optional, not aliasing dx): dx = rmsnorm_backward's dx + add.
hipError_t launch_rmsnorm_bwd(const float *x, const float *w, const float *dy, float *dx,
                              float *dw, float *scratch, int64_t rows, int h, float eps,
                              hipStream_t s, const float *add = nullptr);
hipError_t launch_swiglu(const float *gate, const float *up, float *act, int64_t n,
                         hipStream_t s);
hipError_t launch_swiglu_bwd(const float *gate, const float *up, const float *d_act, float *dg,
                             float *du, int64_t n, hipStream_t s);
// terms: seq floats of scratch
hipError_t launch_softmax_ce(const float *logits, const uint32_t *targets, int64_t seq,
                             int64_t vocab, float *loss, float *dlogits, float *terms,
                             hipStream_t s);

// LoRA-rank GEMMs with an (M x r) output, r <= 64, K <= 2048 (k_rank.hip):
// out[m][j] = alpha * sum_k P[m][k] Q(j, k); P row-major (ldp) in fp32 or
// bf16; Q(j, k) = q[j * ldq + k] (q_kmajor = 0) or q[k * ldq + j] (1).
// A list of independent rank GEMMs for one launch (blockIdx.y = job).
// k_rank_gemm job: out (M x r, row stride ldo) = alpha * P (M x k, stride
// ldp) . Q(j, k) with Q = A (r x k, stride ldq) or, q_kmajor, B (k x r).
// k_rank_tgemm job: out(c, j) = alpha * sum_m P[m][c] * Q[m][j] for c < k
// (the job's column count), P (M x k) and Q (M x r, stride ldq), stored at
// out[c * ldo + j] or, out_t, out[j * ldo + c].
struct RankJob {
  const void *p;
  int64_t ldp;
  const float *q;
  int64_t ldq;
  float *out;
  int64_t ldo;
  int64_t k;
  int r;
  int out_t;
  float alpha;
};
constexpr int kMaxRankJobs = 6;
struct RankJobs {
  RankJob j[kMaxRankJobs];
  int count;
};
hipError_t launch_rank_gemms(const RankJobs &jobs, int p_bf16, int q_kmajor, int64_t M,
                             hipStream_t s);
hipError_t launch_rank_tgemms(const RankJobs &jobs, int big_bf16, int64_t M, hipStream_t s);
bool rank_gemm_ok(int64_t K, int64_t r);
hipError_t launch_rank_gemm(const void *P, int p_bf16, int64_t ldp, const float *Q, int q_kmajor,
                            int64_t ldq, float *out, int64_t ldo, int64_t M, int64_t K, int64_t r,
                            float alpha, hipStream_t s);

// The LoRA-rank GEMMs reducing over M <= 2048 tokens (k_rank.hip):
// out(c, j) = alpha * sum_m Big[m][c] Small[m][j], Big (M x C, ldb) fp32 or
// bf16, Small (M x r, lds) fp32; out[c * ldo + j] (out_t = 0) or
// out[j * ldo + c] (out_t = 1).
bool rank_tgemm_ok(int64_t M, int64_t r);
hipError_t launch_rank_tgemm(const void *Big, int big_bf16, int64_t ldb, const float *Small,
                             int64_t lds, float *out, int64_t ldo, int out_t, int64_t M,
                             int64_t C, int64_t r, float alpha, hipStream_t s);

}  // namespace qh
