// runtime.cpp -- host side of the C ABI declared in include/qlora_hip.h.
//
// Context and stream management, argument validation with the reference's
// accept/reject rules and messages, staging of host slices, choice of
// kernel per shape, and the 8-bit Adam state that lives in HBM.
#include "qlora_hip.h"
#include "qh_host.h"

#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>
#include <vector>

#include "dev_buf.h"
#include "qh_internal.h"

using qh::Carve;
using qh::check;
using qh::DevBuf;
using qh::DevQW;
using qh::GemmArgs;
using qh::GpuError;
using qh::Operand;

namespace {

thread_local std::string g_err;

qh_status fail(qh_status st, const std::string &msg) {
  // Display formats of QloraError (qlora-core/src/error.rs:16-24).
  switch (st) {
    case QH_ERR_SHAPE_MISMATCH: g_err = "shape mismatch: " + msg; break;
    case QH_ERR_INVALID_CONFIG: g_err = "invalid config: " + msg; break;
    case QH_ERR_GPU: g_err = "gpu error: " + msg; break;
    // IoError's Display formats (qlora-io/src/error.rs:15-20)
    case QH_ERR_MALFORMED: g_err = "malformed input: " + msg; break;
    case QH_ERR_UNSUPPORTED: g_err = "unsupported: " + msg; break;
    default: g_err = msg; break;
  }
  return st;
}

std::string fmt(const char *f, ...) __attribute__((format(printf, 1, 2)));
std::string fmt(const char *f, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, f);
  vsnprintf(buf, sizeof buf, f, ap);
  va_end(ap);
  return buf;
}

// Where a call's device scratch comes from: the context's growable buffer,
// or a fixed region of known capacity (the allocation-free entry point,
// whose callers have checked the size before any launch).
struct ScratchSrc {
  DevBuf *grow = nullptr;
  char *fixed = nullptr;
  size_t cap = 0;
  std::vector<char *> bind(Carve &c, hipStream_t s) {
    if (grow) return c.bind(*grow, s);
    if (c.total() > cap) throw GpuError{"scratch larger than the fixed region"};
    return c.bind_at(fixed);
  }
};

inline size_t div_ceil(size_t a, size_t b) { return (a + b - 1) / b; }

bool mul_overflows(size_t a, size_t b, size_t *out) {
  return __builtin_mul_overflow(a, b, out);
}

}  // namespace

struct TimedLaunch {
  std::string name;
  hipEvent_t start, stop;
};

struct qh_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  std::mutex mu;
  DevBuf stage[10];  // host-API staging
  DevBuf scratch;    // internal scratch of the fused paths
  // Operand planes of the large GEMMs, two orders of magnitude above the rest:
  // a buffer of their own, so that the scratch does not move when they grow.
  DevBuf planes;
  DevBuf block_tmp[2];  // intermediate activations of the MLP block calls
  // Zero-initialised counters of kernels whose last workgroup finishes a
  // reduction; each such kernel leaves its counter at zero again.
  unsigned *tickets = nullptr;
  char name[256] = {0};
  bool timing = false;
  uint32_t test_flags = 0;  // QH_TEST_* hooks
  // This device's copy of the allocation-free backward's scratch region
  // (from hipGetSymbolAddress), or null with the error that prevented it.
  void *noalloc = nullptr;
  hipError_t noalloc_err = hipSuccess;
  std::vector<TimedLaunch> pending;
  std::vector<hipEvent_t> event_pool;
  std::map<std::string, std::pair<uint64_t, double>> totals;
};

namespace {

hipEvent_t take_event(qh_ctx *c) {
  if (!c->event_pool.empty()) {
    hipEvent_t e = c->event_pool.back();
    c->event_pool.pop_back();
    return e;
  }
  hipEvent_t e;
  check(hipEventCreate(&e), "hipEventCreate");
  return e;
}

// Arms the GPU-stamped start/stop events of the next qh_launch while timing
// is on (never during stream capture).
struct Timed {
  qh_ctx *c;
  const char *name;
  hipEvent_t a = nullptr, b = nullptr;
  Timed(qh_ctx *ctx, const char *n, hipStream_t st) : c(ctx), name(n) {
    if (!c->timing) return;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone)
      return;
    a = take_event(c);
    b = take_event(c);
    qh::g_launch_timing.start = a;
    qh::g_launch_timing.stop = b;
  }
  ~Timed() {
    if (!a) return;
    if (qh::g_launch_timing.start == nullptr) {
      c->pending.push_back({name, a, b});  // consumed by a launch
    } else {
      qh::g_launch_timing = qh::LaunchTiming();
      c->event_pool.push_back(a);
      c->event_pool.push_back(b);
    }
  }
};

template <class F>
void timed(qh_ctx *c, const char *name, hipStream_t s, F &&f) {
  Timed t(c, name, s);
  check(f(), name);
}

void drain_timing(qh_ctx *c) {
  for (auto &t : c->pending) {
    check(hipEventSynchronize(t.stop), "hipEventSynchronize");
    float ms = 0.0f;
    check(hipEventElapsedTime(&ms, t.start, t.stop), "hipEventElapsedTime");
    auto &slot = c->totals[t.name];
    slot.first += 1;
    slot.second += ms;
    c->event_pool.push_back(t.start);
    c->event_pool.push_back(t.stop);
  }
  c->pending.clear();
}

}  // namespace

struct qh_dweight {
  qh_ctx *ctx;
  qh_qweight view;  // device pointers
  void *codes = nullptr, *scales = nullptr, *absmax = nullptr;
};

struct ParamStateDev {
  size_t numel = 0, nb = 0;
  uint8_t *m_codes = nullptr, *v_codes = nullptr;
  float *m_scales = nullptr, *v_scales = nullptr;
  uint64_t step = 0;
};

struct qh_adam8bit {
  qh_ctx *ctx;
  qh_adam_config cfg;
  std::vector<ParamStateDev> states;
  DevBuf stage_p, stage_g;
};

namespace {

// Device-pointer entry points run on the caller's stream; NULL is the HIP
// null stream (ordered with the caller's other default-stream work).  The
// context's own stream serves only the blocking host-slice entry points.
hipStream_t pick_stream(qh_ctx *ctx, void *stream) {
  (void)ctx;
  return (hipStream_t)stream;
}

DevQW make_devqw(const qh_qweight &w) {
  DevQW d;
  d.rows = (int64_t)w.rows;
  d.cols = (int64_t)w.cols;
  d.n = (int64_t)(w.rows * w.cols);
  d.bs = (int64_t)w.block_size;
  d.nb = w.block_size ? (d.n + d.bs - 1) / d.bs : 0;
  d.codes = w.codes;
  d.kind = w.scale_kind;
  d.scales = w.scales;
  d.scale_codes = w.scale_codes;
  d.absmax = w.absmax;
  return d;
}

// QuantizedTensor invariants (quant.rs:171-207): block_size > 0 and no
// rows*cols overflow; the scale kind must be one of the two stores.
qh_status validate_weight(const qh_qweight *w) {
  if (!w) return fail(QH_ERR_SHAPE_MISMATCH, "weight descriptor is NULL");
  if (w->block_size == 0)
    return fail(QH_ERR_INVALID_CONFIG, "block_size must be > 0");
  size_t n;
  if (mul_overflows(w->rows, w->cols, &n))
    return fail(QH_ERR_INVALID_CONFIG, "rows*cols overflow");
  if (w->scale_kind != QH_SCALES_F32 && w->scale_kind != QH_SCALES_DQ_INT8)
    return fail(QH_ERR_INVALID_CONFIG, "unknown scale kind");
  return QH_OK;
}

// LoraAdapter::new (lora.rs:28-61) against the layer's dims.
qh_status validate_lora(const qh_lora *l, size_t in_dim, size_t out_dim) {
  if (!l) return QH_OK;
  if (l->r == 0) return fail(QH_ERR_INVALID_CONFIG, "rank r must be > 0");
  if ((l->a_len && !l->a) || (l->b_len && !l->b))
    return fail(QH_ERR_SHAPE_MISMATCH, "the adapter's A or B is NULL");
  if (l->a_len != l->r * in_dim)
    return fail(QH_ERR_SHAPE_MISMATCH,
                fmt("a.len() = %zu but r*in_dim = %zu", l->a_len, l->r * in_dim));
  if (l->b_len != out_dim * l->r)
    return fail(QH_ERR_SHAPE_MISMATCH,
                fmt("b.len() = %zu but out_dim*r = %zu", l->b_len, out_dim * l->r));
  return QH_OK;
}

// Scale kind and pointer for one weight: upload to staging for host calls.
size_t scale_bytes(const qh_qweight &w, size_t *am_bytes) {
  size_t n = w.rows * w.cols;
  size_t nb = div_ceil(n, w.block_size);
  if (w.scale_kind == QH_SCALES_F32) {
    *am_bytes = 0;
    return nb * 4;
  }
  *am_bytes = div_ceil(nb, 256) * 4;
  return nb;
}

// Copies a host weight into device staging buffers and returns a device
// view of it.
DevQW upload_weight(qh_ctx *ctx, const qh_qweight &w, int slot, hipStream_t s) {
  size_t n = w.rows * w.cols;
  size_t cb = div_ceil(n, 2), amb = 0;
  size_t sb = scale_bytes(w, &amb);
  Carve c;
  size_t ic = c.add(cb + 16), is = c.add(sb + 16), ia = c.add(amb + 16);
  auto p = c.bind(ctx->stage[slot]);
  if (cb) check(hipMemcpyAsync(p[ic], w.codes, cb, hipMemcpyHostToDevice, s), "upload codes");
  qh_qweight d = w;
  d.codes = (const uint8_t *)p[ic];
  if (w.scale_kind == QH_SCALES_F32) {
    if (sb) check(hipMemcpyAsync(p[is], w.scales, sb, hipMemcpyHostToDevice, s), "upload scales");
    d.scales = (const float *)p[is];
  } else {
    if (sb) check(hipMemcpyAsync(p[is], w.scale_codes, sb, hipMemcpyHostToDevice, s), "upload scale codes");
    if (amb) check(hipMemcpyAsync(p[ia], w.absmax, amb, hipMemcpyHostToDevice, s), "upload absmax");
    d.scale_codes = (const uint8_t *)p[is];
    d.absmax = (const float *)p[ia];
  }
  return make_devqw(d);
}

float *upload_f32(qh_ctx *ctx, int slot, const float *h, size_t n, hipStream_t s) {
  float *d = (float *)ctx->stage[slot].ensure(n * 4 + 16);
  if (n) check(hipMemcpyAsync(d, h, n * 4, hipMemcpyHostToDevice, s), "upload");
  return d;
}

float *alloc_f32(qh_ctx *ctx, int slot, size_t n) {
  return (float *)ctx->stage[slot].ensure(n * 4 + 16);
}

void download_f32(float *h, const float *d, size_t n, hipStream_t s) {
  if (n) check(hipMemcpyAsync(h, d, n * 4, hipMemcpyDeviceToHost, s), "download");
}

Operand op(const void *p, int64_t ld, int form, int elem, float scale = 1.0f) {
  Operand o;
  o.p = p;
  o.ld = ld;
  o.form = form;
  o.elem = elem;
  o.scale = scale;
  return o;
}

GemmArgs gemm_args(int64_t M, int64_t N, int64_t K, Operand A, Operand B,
                   float *C, int64_t ldc, float alpha) {
  GemmArgs g;
  std::memset(&g, 0, sizeof g);
  g.M = M;
  g.N = N;
  g.K = K;
  g.A = A;
  g.B = B;
  g.C = C;
  g.ldc = ldc;
  g.alpha = alpha;
  g.splits = 1;
  g.K2 = 0;
  g.A2 = op(nullptr, 0, qh::ROWK, qh::E_F32);
  g.B2 = op(nullptr, 0, qh::ROWK, qh::E_F32);
  return g;
}

// Split-K factor for outputs that cover too few tiles to fill 256 CUs.
// Split-K of the LoRA-rank GEMMs (one side r <= 64): each workgroup's K loop
// is a chain of dependent 32-wide steps whose loads the tile engine hides
// only one step ahead, so a skinny GEMM is paced by load latency.  Split K
// until about 4 workgroups per CU (1024) run, each keeping >= 4 steps.
int choose_splits(int64_t M, int64_t N, int64_t K) {
  int64_t tiles = div_ceil(M, 64) * div_ceil(N, 64);
  if (M >= 128 && N >= 128 && (M / 128) * (N / 128) >= 64) return 1;
  if (tiles >= 256) return 1;
  int64_t sp = 1024 / (tiles ? tiles : 1);
  if (sp > 32) sp = 32;
  int64_t kmax = K / 128;
  if (sp > kmax) sp = kmax;
  return sp < 1 ? 1 : (int)sp;
}

// Split-K of the base NF4 GEMMs (forward, grad_x) on 64x64 tiles: at C4's
// shapes (2048 tokens, 576-1536 features) 96-768 tiles leave most CUs with
// one workgroup that walks 18-48 dependent K steps.  Same target as above,
// at most 8 splits and 64 MB of partial sums.
int base_splits(int64_t M, int64_t N, int64_t K) {
  if (qh::gemm_uses_t128(M, N)) return 1;
  const int64_t tiles = div_ceil(M, 64) * div_ceil(N, 64);
  if (tiles >= 1024) return 1;
  int64_t sp = div_ceil(1024, tiles ? tiles : 1);
  if (sp > 8) sp = 8;
  if (sp > K / 128) sp = K / 128;
  while (sp > 1 && (size_t)(sp * M * N * 4) > ((size_t)64 << 20)) --sp;
  return sp < 1 ? 1 : (int)sp;
}

size_t partial_floats(const GemmArgs &g) {
  return g.splits > 1 ? (size_t)g.splits * g.M * g.N : 0;
}

// A LoRA-rank product (T1, Ds, grad_A, grad_B) on the dense bf16-MFMA
// kernel: C = alpha sum_k A(m, k) B(n, k), taken where the rank kernels'
// reduction limit (2048) is passed and the operands allow it.
struct DenseOp {
  const void *a;
  int af, a32;
  int64_t lda;
  const void *b;
  int bf, b32;
  int64_t ldb;
  float *c;
  int64_t ldc, M, N, K;
  float alpha;
  bool ok() const { return qh::dense_bf16_ok(M, N, K, af, a, lda, bf, b, ldb); }
  size_t partial_bytes() const {
    const int sp = qh::dense_bf16_splits(M, N, K);
    return sp > 1 ? (size_t)sp * M * N * 4 : 0;
  }
  hipError_t run(float *partial, hipStream_t s) const {
    return qh::launch_dense_bf16(a, af, a32, lda, b, bf, b32, ldb, c, ldc, M, N, K, alpha,
                                 partial, s);
  }
};

// T1 = X . A^T (M x r): X(m, k) along k, A(j, k) along k.
DenseOp dense_t1(const void *x, int xe, int64_t M, int64_t K, const qh_lora *l, float *t1) {
  return DenseOp{x, qh::ROWK, xe == qh::E_F32, K, l->a, qh::ROWK, 1, K, t1, (int64_t)l->r,
                 M, (int64_t)l->r, K, 1.0f};
}

// T1 = X . A^T (M x r) on its own (lora.rs:94-97), for the shapes where no
// GEMM follows it.
void t1_dev(qh_ctx *ctx, const void *x, int xe, int64_t M, int64_t K, const qh_lora *l,
            float *t1, hipStream_t s) {
  const int64_t r = (int64_t)l->r;
  if (qh::rank_gemm_ok(K, r)) {
    timed(ctx, "t1_gemm", s, [&] {
      return qh::launch_rank_gemm(x, xe == qh::E_BF16, K, l->a, 0, K, t1, r, M, K, r, 1.0f, s);
    });
    return;
  }
  const DenseOp dt = dense_t1(x, xe, M, K, l, t1);
  if (dt.ok()) {
    Carve c;
    size_t ip = c.add(dt.partial_bytes());
    auto p = c.bind(ctx->scratch, s);
    timed(ctx, "t1_gemm", s, [&] { return dt.run((float *)p[ip], s); });
    return;
  }
  GemmArgs g = gemm_args(M, r, K, op(x, K, qh::ROWK, xe), op(l->a, K, qh::ROWK, qh::E_F32),
                         t1, r, 1.0f);
  g.splits = choose_splits(M, r, K);
  Carve c;
  size_t ip = c.add(partial_floats(g) * 4);
  auto p = c.bind(ctx->scratch, s);
  timed(ctx, "t1_gemm", s, [&] { return qh::launch_gemm(g, (float *)p[ip], s); });
}

void zero_dev(float *p, size_t n, hipStream_t s) {
  if (n) check(qh::launch_zero(p, (int64_t)n, s), "zero fill");
}

// True when forward_dev serves this layer with one k_dstream launch (batch
// 1-2, T1 in the launch): the layers a two-layer launch may pair.
bool takes_stream(const DevQW &W, const qh_lora *l, const void *x, int64_t M) {
  const int64_t K = W.cols, r = l ? (int64_t)l->r : 0;
  if (M == 0 || K == 0 || W.rows == 0) return false;
  const bool aligned = (((uintptr_t)x) & 15) == 0 && (K % 8) == 0 &&
                       (!l || (((uintptr_t)l->a) & 15) == 0);
  return aligned && qh::decode_ok(W, M, r) && qh::decode_stream_ok(W, M, r);
}

// True when forward_dev serves this layer with the split decode kernel after
// a T1 launch (the layers a group computes T1 for in one launch).
bool takes_split(const DevQW &W, const qh_lora *l, const void *x, int64_t M) {
  const int64_t K = W.cols, r = l ? (int64_t)l->r : 0;
  if (M == 0 || K == 0 || W.rows == 0) return false;
  const bool aligned = (((uintptr_t)x) & 15) == 0 && (K % 8) == 0 &&
                       (!l || (((uintptr_t)l->a) & 15) == 0);
  // the LoRA B rows are copied to LDS in 16-byte units
  const bool b_aligned = !l || (((uintptr_t)l->b) & 15) == 0;
  return aligned && b_aligned && qh::decode_ok(W, M, r) && !qh::decode_stream_ok(W, M, r) &&
         qh::split_plan(W, M, r).ok;
}

// True when forward_dev with `accumulate` can add its result to y in the
// GEMM (the few-token kernel, operand planes and k_nf4_bf16, by their epilogue or
// the reduction of their split sums: what is true here may take any of the
// three); otherwise a caller that wants y += forward(x) computes into a buffer and
// adds.
static bool forward_accumulates(const DevQW &W, const qh_lora *l, const void *x, size_t batch) {
  const int64_t M = (int64_t)batch, N = W.rows, K = W.cols;
  if (M == 0 || K == 0 || N == 0) return false;
  const int64_t r = l ? (int64_t)l->r : 0;
  const bool aligned = (((uintptr_t)x) & 15) == 0 && (K % 8) == 0 &&
                       (!l || (((uintptr_t)l->a) & 15) == 0);
  if (aligned && (qh::decode_ok(W, M, r) || (r <= 64 && qh::gemv_ok(W, M)))) return false;
  return qh::nf4_fast_ok(W) && qh::bf16_gemm_ok(W, x, K, K);
}

// ---- the forward for few tokens (k_slim.hip) ------------------------------
bool takes_slim(const DevQW &W, const qh_lora *l, const void *x, int xdt, int64_t M) {
  return qh::slim_ok(W, x, xdt == QH_BF16, l ? l->a : nullptr, M, l ? (int64_t)l->r : 0);
}

// About what the tile kernels take for T1 (us), fitted with bf16_gemm_us: a rank
// launch up to K = 2048, else the dense kernel and its reduction.
double t1_us(int64_t M, int64_t K, int64_t r, bool f32) {
  if (r == 0) return 0.0;
  const double k = (double)K * 1e-3, mk = (double)M * (double)K * 1e-6;
  if (!qh::rank_gemm_ok(K, r)) return (f32 ? 11.3 : 10.6) + k + 1.6 * mk;
  return (f32 ? 2.9 : 3.2) + k * ((f32 ? 3.55 : 8.5) + 3.6 * (double)((r + 15) / 16 - 1)) + 1.6 * mk;
}
double tile_forward_us(const DevQW &W, const qh_lora *l, int xdt, int64_t M) {
  const bool f32 = xdt != QH_BF16;
  return qh::bf16_gemm_us(M, W.rows, W.cols, f32, true) + t1_us(M, W.cols, l ? (int64_t)l->r : 0, f32);
}

// `count` layers, each on its own x (layers with the same x share its
// preparation); with `beta` y += the result.  False, with nothing launched,
// where its scratch cannot be had (see Carve::try_bind), no plan covers the
// group, or the tile kernels' `tile_us` is clearly below the plan's (see
// slim_plan): the caller runs the layers on the tile kernels.  Their scratch for
// these layers is `tile_bytes`, and the buffer grows to that as well: what
// this kernel needs does not rise with the token count, so a capture of fewer
// tokens than the calls before it may find too little for it, but not for
// the tiles, which then need no more than those calls would have.
bool slim_dev(qh_ctx *ctx, size_t count, const DevQW *W, const qh_lora *const *l,
              const void *const *x, int xdt, int64_t M, float *const *y, float *const *t1_out,
              int beta, size_t tile_bytes, double tile_us, hipStream_t s) {
  if (count > (size_t)qh::kMaxSlimSegs) return false;
  const int xb = xdt == QH_BF16, n = (int)count;
  int64_t rs[qh::kMaxSlimSegs] = {};
  for (int i = 0; i < n; ++i) rs[i] = l[i] ? (int64_t)l[i]->r : 0;
  const qh::SlimPlan pl = qh::slim_plan(n, W, rs, M, xb);
  bool lora = false;
  for (int i = 0; i < n; ++i) lora = lora || rs[i] > 0;
  if (!pl.ok || pl.us > tile_us + (lora ? 1.0 : 0.2)) return false;
  Carve c;
  size_t it[qh::kMaxSlimSegs], ix[qh::kMaxSlimSegs], ip[qh::kMaxSlimSegs];
  int own[qh::kMaxSlimSegs];
  for (int i = 0; i < n; ++i) {
    own[i] = i;
    for (int j = 0; j < i && own[i] == i; ++j)
      if (x[j] == x[i] && W[j].cols == W[i].cols) own[i] = own[j];
    it[i] = c.add((size_t)pl.nz[i] * M * rs[i] * 4);
    ix[i] = c.add(own[i] == i ? pl.xp_bytes[i] : 0);
    ip[i] = c.add(pl.part_floats[i] * 4);
  }
  Carve both = c;
  if (tile_bytes > c.total()) both.add(tile_bytes - c.total());
  std::vector<char *> p;
  if (!both.try_bind(ctx->scratch, s, &p) && !c.try_bind(ctx->scratch, s, &p)) return false;
  qh::SlimIn in[qh::kMaxSlimSegs] = {};
  for (int i = 0; i < n; ++i) {
    in[i].w = W[i], in[i].x = x[i], in[i].y = y[i], in[i].beta = beta;
    in[i].xp = p[ix[own[i]]], in[i].part = (float *)p[ip[i]];
    if (l[i]) {
      in[i].a = l[i]->a, in[i].lb = l[i]->b, in[i].r = rs[i];
      in[i].s = l[i]->alpha / (float)l[i]->r;  // lora.rs:64-66
      in[i].t1p = (float *)p[it[i]];
      in[i].t1 = t1_out ? t1_out[i] : nullptr;
    }
  }
  timed(ctx, "slim_prep", s, [&] { return qh::launch_slim_prep(n, in, pl, M, xb, s); });
  timed(ctx, "forward_slim", s, [&] { return qh::launch_slim(n, in, pl, M, ctx->tickets, s); });
  return true;
}

// ---- large GEMMs through operand planes (k_plane.hip) ---------------------
// Slots of one GEMM's planes (A, the weight, the LoRA term's two).
struct PlaneSlots {
  size_t a, b, a2, b2;
  PlaneSlots(Carve &c, bool on, int64_t M, int64_t N, int64_t K, int64_t r, int parts)
      : a(c.add(on ? qh::plane_a_bytes(M, K, parts) : 0)),
        b(c.add(on ? qh::plane_b_bytes(N, K) : 0)),
        a2(c.add(on && r ? qh::plane_a_bytes(M, r, 2) : 0)),
        b2(c.add(on && r ? qh::plane_b_bytes(N, r) : 0)) {}
};

// C (M x N) = X . op(W)^T + P2 . (scale Q2)^T (+ C with beta): the forward
// (w_form PLANE_NF4_ROW: X M x K, P2 = T1, Q2 = B, N x r) or the input gradient
// (PLANE_NF4_COL: X = dY, P2 = Ds, Q2 = A^T, A r x N).
void plane_gemm_dev(qh_ctx *ctx, const std::vector<char *> &p, const PlaneSlots &ps, const char *name,
                    const DevQW &W, int w_form, const void *x, int a32, int64_t M, int64_t N,
                    int64_t K, const float *p2, const float *q2, int64_t r, float scale, float *c,
                    int beta, hipStream_t s) {
  qh::PlaneSrc src[4] = {};
  src[0].form = qh::PLANE_ROWK, src[0].bf16 = !a32, src[0].p = x, src[0].ld = K, src[0].rows = M;
  src[0].K = K, src[0].scale = 1.0f, src[0].dst = p[ps.a];
  src[1].form = w_form, src[1].w = W, src[1].rows = N, src[1].K = K, src[1].dst = p[ps.b];
  if (r) {
    src[2].form = qh::PLANE_ROWK, src[2].p = p2, src[2].ld = r, src[2].rows = M, src[2].K = r;
    src[2].scale = 1.0f, src[2].dst = p[ps.a2];
    src[3].form = w_form == qh::PLANE_NF4_ROW ? qh::PLANE_ROWK : qh::PLANE_KROW;
    src[3].p = q2, src[3].ld = w_form == qh::PLANE_NF4_ROW ? r : N, src[3].rows = N, src[3].K = r;
    src[3].scale = scale, src[3].dst = p[ps.b2];
  }
  timed(ctx, "planes", s, [&] { return qh::launch_planes(src, r ? 4 : 2, s); });
  const qh::PlaneGemm g{p[ps.a], p[ps.b], p[ps.a2], p[ps.b2], a32 ? 2 : 1, M, N, K, r, c, N, beta};
  timed(ctx, name, s, [&] { return qh::launch_plane_gemm(g, s); });
}

// What the forward of one layer (M, K, N > 0) runs on the tile kernels, and its
// scratch.
struct TileForward {
  bool fast, bf16;                         // whole 64-element row blocks; on bf16 MFMA
  bool t1_rank = false, t1_dense = false;  // T1's kernel (else the tile engine)
  GemmArgs gt1{};
  DenseOp dt1{};
  int y_splits;
  Carve c;
  size_t i_t1, i_w32, i_p1, i_p2;
  TileForward(const DevQW &W, const qh_lora *l, const void *x, int xe, int64_t M,
              const float *t1_out) {
    const int64_t N = W.rows, K = W.cols, r = l ? (int64_t)l->r : 0;
    fast = qh::nf4_fast_ok(W);
    bf16 = fast && qh::bf16_gemm_ok(W, x, K, K);
    if (l) {
      t1_rank = qh::rank_gemm_ok(K, r);
      gt1 = gemm_args(M, r, K, op(x, K, qh::ROWK, xe), op(l->a, K, qh::ROWK, qh::E_F32),
                      nullptr, r, 1.0f);
      dt1 = dense_t1(x, xe, M, K, l, nullptr);
      t1_dense = !t1_rank && dt1.ok();
      gt1.splits = t1_rank || t1_dense ? 1 : choose_splits(M, r, K);
    }
    y_splits = bf16 ? qh::bf16_gemm_splits(M, N, K) : base_splits(M, N, K);
    i_t1 = c.add(l && !t1_out ? (size_t)M * r * 4 : 0);
    i_w32 = c.add(fast ? 0 : (size_t)W.n * 4);
    i_p1 = c.add(!l ? 0 : t1_dense ? dt1.partial_bytes() : partial_floats(gt1) * 4);
    i_p2 = c.add(y_splits > 1 ? (size_t)y_splits * M * N * 4 : 0);
  }
};

// ---- fused forward on device pointers -----------------------------------
// With `accumulate` y += the result; only the paths that forward_accumulates names
// do that, every other path refuses it before launching anything
// (forward_add_dev picks).
void forward_dev(qh_ctx *ctx, const DevQW &W, const qh_lora *l, const void *x,
                 int xdt, size_t batch, float *y, float *t1_out, hipStream_t s,
                 bool accumulate = false) {
  const int64_t M = (int64_t)batch, N = W.rows, K = W.cols;
  const bool lora = l != nullptr;
  const int64_t r = lora ? (int64_t)l->r : 0;
  const float sc = lora ? l->alpha / (float)l->r : 0.0f;  // lora.rs:64-66
  const int xe = xdt == QH_BF16 ? qh::E_BF16 : qh::E_F32;
  auto writes_y = [&](const char *path) {
    if (accumulate) check(hipErrorInvalidValue, path);  // y would be overwritten
  };
  if (M == 0) return;
  if (K == 0) {  // empty reductions: Y = 0 and T1 = 0 (qlora.rs:86-107)
    writes_y("forward_dev: y += on the empty-reduction path");
    zero_dev(y, (size_t)M * N, s);
    if (lora && t1_out) zero_dev(t1_out, (size_t)M * r, s);
    return;
  }
  if (N == 0) {  // no outputs, but the caller may still want T1
    if (lora && t1_out) t1_dev(ctx, x, xe, M, K, l, t1_out, s);
    return;
  }
  if (takes_slim(W, l, x, xdt, M) &&
      slim_dev(ctx, 1, &W, &l, &x, xdt, M, &y, &t1_out, accumulate ? 1 : 0,
               TileForward(W, l, x, xe, M, t1_out).c.total(), tile_forward_us(W, l, xdt, M), s))
    return;
  // Small batches: the MFMA decode kernels (batch <= 16, K % 256 == 0), else
  // the VALU GEMV (batch <= 4, K % 64 == 0); both need 16-byte aligned rows
  // of X and A.
  const bool aligned = (((uintptr_t)x) & 15) == 0 && (K % 8) == 0 &&
                       (!lora || (((uintptr_t)l->a) & 15) == 0);
  const bool decode = aligned && qh::decode_ok(W, M, r);
  const bool gemv = aligned && !decode && r <= 64 && qh::gemv_ok(W, M);

  if (gemv) {
    writes_y("forward_dev: y += on the GEMV path");
    Carve cg;
    size_t i_t1 = cg.add(lora && !t1_out ? (size_t)M * r * 4 : 0);
    auto pg = cg.bind(ctx->scratch, s);
    float *t1 = lora ? (t1_out ? t1_out : (float *)pg[i_t1]) : nullptr;
    const int xb = xe == qh::E_BF16;
    if (lora)
      timed(ctx, "lora_t1", s, [&] { return qh::launch_lora_t1(x, xb, M, K, l->a, r, t1, s); });
    timed(ctx, "gemv", s, [&] {
      return qh::launch_gemv(W, x, xb, M, t1, lora ? l->b : nullptr, r, sc, y, s);
    });
    return;
  }

  // Batch 1-2 in one launch with T1 inside it where the layer fits one
  // round; other decode batches (3-16, and 1-2 past that) stream the weight
  // once for the whole batch on the split kernel after a T1 launch.
  if (decode && qh::decode_stream_ok(W, M, r)) {
    writes_y("forward_dev: y += on the decode path");
    const int xb = xe == qh::E_BF16;
    timed(ctx, "decode_stream", s, [&] {
      return qh::launch_decode_stream(W, x, xb, M, lora ? l->a : nullptr, r,
                                      lora ? l->b : nullptr, sc, y, t1_out, ctx->tickets,
                                      (ctx->test_flags & QH_TEST_FORCE_T1_RECOMPUTE) != 0, s);
    });
    return;
  }
  if (decode && (!lora || (((uintptr_t)l->b) & 15) == 0)) {
    const qh::SplitPlan sp = qh::split_plan(W, M, r);
    if (sp.ok) {
      writes_y("forward_dev: y += on the split decode path");
      Carve cs;
      size_t i_t1 = cs.add(lora && !t1_out ? (size_t)M * r * 4 : 0);
      size_t i_pt = cs.add(sp.part_floats * 4);
      auto ps = cs.bind(ctx->scratch, s);
      float *t1 = lora ? (t1_out ? t1_out : (float *)ps[i_t1]) : nullptr;
      const int xb = xe == qh::E_BF16;
      if (lora)
        timed(ctx, "decode_t1", s,
              [&] { return qh::launch_lora_t1(x, xb, M, K, l->a, r, t1, s); });
      const qh::SplitLayerIn in{W, x, t1, lora ? l->b : nullptr, r, sc, y, (float *)ps[i_pt]};
      timed(ctx, "decode_split", s,
            [&] { return qh::launch_decode_split(1, &in, &sp, M, xb, ctx->tickets, s); });
      return;
    }
  }

  // NF4 weights in whole 64-element row blocks run on bf16 MFMA (the weight
  // as hi / lo bf16 parts); others on the fp32 tile engine
  TileForward f(W, l, x, xe, M, t1_out);
  const bool fast = f.fast, bf16 = f.bf16;
  if (!bf16) writes_y("forward_dev: y += on the fp32 tile engine");
  // large GEMMs through operand planes where their memory can be had
  bool plane = bf16 && qh::plane_codes_ok(W) && qh::plane_ok(M, N, K, r, xe == qh::E_F32);
  Carve cp;
  const PlaneSlots slots(cp, plane, M, N, K, r, xe == qh::E_F32 ? 2 : 1);
  std::vector<char *> pp;
  plane = plane && cp.try_bind(ctx->planes, s, &pp);
  auto p = f.c.bind(ctx->scratch, s);
  float *t1 = lora ? (t1_out ? t1_out : (float *)p[f.i_t1]) : nullptr;

  if (lora && f.t1_rank) {
    timed(ctx, "t1_gemm", s, [&] {
      return qh::launch_rank_gemm(x, xe == qh::E_BF16, K, l->a, 0, K, t1, r, M, K, r, 1.0f, s);
    });
  } else if (lora && f.t1_dense) {
    f.dt1.c = t1;
    timed(ctx, "t1_gemm", s, [&] { return f.dt1.run((float *)p[f.i_p1], s); });
  } else if (lora) {
    f.gt1.C = t1;
    timed(ctx, "t1_gemm", s, [&] { return qh::launch_gemm(f.gt1, (float *)p[f.i_p1], s); });
  }
  Operand B;
  if (fast) {
    B = op(W.codes, K, qh::ROWK, qh::E_NF4);
  } else {
    float *w32 = (float *)p[f.i_w32];
    timed(ctx, "dequantize", s, [&] { return qh::launch_dequantize(W, w32, s); });
    B = op(w32, K, qh::ROWK, qh::E_F32);
  }
  if (plane) {
    plane_gemm_dev(ctx, pp, slots, "forward_gemm_bf16", W, qh::PLANE_NF4_ROW, x, xe == qh::E_F32, M,
                   N, K, t1, lora ? l->b : nullptr, r, sc, y, accumulate ? 1 : 0, s);
    return;
  }
  if (bf16) {
    // bf16 MFMA against the weight's hi / lo bf16 parts (X exact when bf16,
    // split into hi / lo when fp32), the LoRA term T1 . (s B)^T in the same
    // kernel
    qh::Bf16GemmArgs b{};
    b.M = M, b.N = N, b.K = K, b.A = x, b.lda = K, b.alpha = 1.0f, b.nseg = 1;
    b.beta = accumulate ? 1 : 0;
    qh::Bf16Seg &q = b.seg[0];
    q.w = W, q.len = N, q.C = y, q.ldc = N;
    if (lora) q.A2 = t1, q.lda2 = r, q.B2 = l->b, q.ldb2 = r, q.b2scale = sc, q.K2 = r;
    timed(ctx, "forward_gemm_bf16", s,
          [&] {
            return qh::launch_gemm_bf16(b, qh::ROWK, xe == qh::E_F32, f.y_splits,
                                        (float *)p[f.i_p2], s);
          });
    return;
  }
  GemmArgs gm = gemm_args(M, N, K, op(x, K, qh::ROWK, xe), B, y, N, 1.0f);
  gm.qw = W;
  if (lora) {
    gm.K2 = r;
    gm.A2 = op(t1, r, qh::ROWK, qh::E_F32);
    gm.B2 = op(l->b, r, qh::ROWK, qh::E_F32, sc);
  }
  gm.splits = f.y_splits;
  timed(ctx, "forward_gemm", s, [&] { return qh::launch_gemm(gm, (float *)p[f.i_p2], s); });
}

// y += forward(x): in the bf16 GEMM's epilogue (or its split-K reduction)
// where that path serves the shape (x + v rounds as v + x: the same bits
// as the add), else into `tmp` and one add.
void forward_add_dev(qh_ctx *ctx, const DevQW &W, const qh_lora *l, const void *x, int xdt,
                     size_t batch, float *y, float *t1_out, DevBuf &tmp, hipStream_t s) {
  if (forward_accumulates(W, l, x, batch)) {
    forward_dev(ctx, W, l, x, xdt, batch, y, t1_out, s, true);
    return;
  }
  float *t = (float *)tmp.ensure(batch * (size_t)W.rows * 4, s);
  forward_dev(ctx, W, l, x, xdt, batch, t, t1_out, s);
  timed(ctx, "residual_add", s, [&] {
    return qh::launch_axpy_inplace(y, t, (int64_t)(batch * (size_t)W.rows), s);
  });
}

// ---- fused backward on device pointers ----------------------------------
// With `plan_bytes` set, nothing is launched: the scratch bytes the call
// would need are stored there.  `src` (default: the context's growable
// buffer) provides the scratch.
// Whether backward_dev can add its input gradient into gx (the bf16-MFMA
// path's epilogue or split-K reduction does gx + result, the bits of a
// separate add); the other paths write gx.
bool backward_accumulates(const DevQW &W, const void *dy, size_t batch) {
  return batch > 0 && W.rows > 0 && W.cols > 0 && qh::nf4_fast_ok(W) &&
         qh::bf16_gemm_ok(W, dy, W.rows, W.rows);
}

void backward_dev(qh_ctx *ctx, const DevQW &W, const qh_lora *l, const void *x,
                  const void *dy, int adt, size_t batch, const float *t1_in,
                  float *gx, float *ga, float *gb, hipStream_t s,
                  ScratchSrc *src = nullptr, size_t *plan_bytes = nullptr,
                  bool accumulate = false) {
  if (accumulate && !backward_accumulates(W, dy, batch))
    check(hipErrorInvalidValue, "backward_dev: accumulate on a path that writes grad_x");
  const int64_t M = (int64_t)batch, N = W.rows, K = W.cols;
  const bool lora = l != nullptr;
  const int64_t r = lora ? (int64_t)l->r : 0;
  const float sc = lora ? l->alpha / (float)l->r : 0.0f;
  const int ae = adt == QH_BF16 ? qh::E_BF16 : qh::E_F32;
  const bool fast = qh::nf4_fast_ok(W);
  // Empty reductions (qlora.rs:116-165): with in_dim = 0, T1 = 0, so
  // grad_B = 0 and grad_x, grad_A are empty; with out_dim = 0, Ds = 0, so
  // grad_x = 0 and grad_A = 0; with no tokens, grad_A = grad_B = 0.
  if (K == 0 || N == 0 || M == 0) {
    if (plan_bytes) {
      *plan_bytes = 0;
      return;
    }
    if (lora) {
      zero_dev(gb, (size_t)N * r, s);
      zero_dev(ga, (size_t)r * K, s);
    }
    zero_dev(gx, (size_t)M * K, s);
    return;
  }

  GemmArgs gt1{}, gds{}, ggb{}, gga{};
  const bool t1_rank = lora && qh::rank_gemm_ok(K, r);
  const bool ds_rank = lora && qh::rank_gemm_ok(N, r);
  // (grad_A / grad_B of wide layers go to the dense kernel even within the
  // rank kernel's token limit: measured faster from 8192 features up)
  const bool g_rank = lora && qh::rank_tgemm_ok(M, r) && std::max(N, K) < 8192;
  // the dense bf16 kernel where the rank kernels do not reach
  const int a32 = ae == qh::E_F32;
  DenseOp dt1{}, dds{}, dgb{}, dga{};
  bool t1_dense = false, ds_dense = false, gb_dense = false, ga_dense = false;
  if (lora) {
    dt1 = dense_t1(x, ae, M, K, l, nullptr);
    // Ds = s dY . B: dY(m, n) along n, B(j, n) = B[n][j] across n
    dds = DenseOp{dy, qh::ROWK, a32, N, l->b, qh::KROW, 1, r, nullptr, r, M, r, N, sc};
    // grad_B = s dY^T . T1: dY(n, m) = dY[m][n] and T1(j, m) = T1[m][j], across m
    // (T1 is the caller's t1_in or aligned scratch: the check sees which)
    dgb = DenseOp{dy, qh::KROW, a32, N, t1_in, qh::KROW, 1, r, gb, r, N, r, M, sc};
    // grad_A = Ds^T . X: Ds(j, m) = Ds[m][j] and X(k, m) = X[m][k], across m
    dga = DenseOp{nullptr, qh::KROW, 1, r, x, qh::KROW, a32, K, ga, K, r, K, M, 1.0f};
    t1_dense = !t1_in && !t1_rank && dt1.ok();
    ds_dense = !ds_rank && dds.ok();
    gb_dense = !g_rank && dgb.ok();
    ga_dense = !g_rank && dga.ok();
  }
  if (lora) {
    gt1 = gemm_args(M, r, K, op(x, K, qh::ROWK, ae), op(l->a, K, qh::ROWK, qh::E_F32),
                    nullptr, r, 1.0f);
    gt1.splits = t1_rank || t1_dense ? 1 : choose_splits(M, r, K);
    // Ds = s * dY . B   (qlora.rs:143,149)
    gds = gemm_args(M, r, N, op(dy, N, qh::ROWK, ae), op(l->b, r, qh::KROW, qh::E_F32),
                    nullptr, r, sc);
    gds.splits = ds_rank || ds_dense ? 1 : choose_splits(M, r, N);
    // grad_B = (s * dY)^T . T1  (qlora.rs:147)
    ggb = gemm_args(N, r, M, op(dy, N, qh::KROW, ae), op(nullptr, r, qh::KROW, qh::E_F32),
                    gb, r, sc);
    ggb.splits = g_rank || gb_dense ? 1 : choose_splits(N, r, M);
    // grad_A = Ds^T . X  (qlora.rs:151)
    gga = gemm_args(r, K, M, op(nullptr, r, qh::KROW, qh::E_F32), op(x, K, qh::KROW, ae),
                    ga, K, 1.0f);
    gga.splits = g_rank || ga_dense ? 1 : choose_splits(r, K, M);
  }
  Carve c;
  size_t i_t1 = c.add(lora && !t1_in ? (size_t)M * r * 4 : 0);
  size_t i_ds = c.add(lora ? (size_t)M * r * 4 : 0);
  size_t i_w32 = c.add(fast ? 0 : (size_t)W.n * 4);
  size_t i_p1 = c.add(!lora ? 0 : t1_dense ? dt1.partial_bytes() : partial_floats(gt1) * 4);
  size_t i_p2 = c.add(!lora ? 0 : ds_dense ? dds.partial_bytes() : partial_floats(gds) * 4);
  size_t i_p3 = c.add(!lora ? 0 : gb_dense ? dgb.partial_bytes() : partial_floats(ggb) * 4);
  size_t i_p4 = c.add(!lora ? 0 : ga_dense ? dga.partial_bytes() : partial_floats(gga) * 4);
  const bool bf16 = fast && qh::bf16_gemm_ok(W, dy, N, N);
  const int gx_splits = bf16 ? qh::bf16_gemm_splits(M, K, N) : base_splits(M, K, N);
  const size_t i_p5 = c.add(gx_splits > 1 ? (size_t)gx_splits * M * K * 4 : 0);
  if (plan_bytes) {
    *plan_bytes = c.total();
    return;
  }
  // the input gradient through operand planes where their memory can be had
  // (never in the fixed region, whose bound is part of the interface)
  bool plane = bf16 && !src && qh::plane_ok(M, K, N, r, a32);
  Carve cp;
  const PlaneSlots slots(cp, plane, M, K, N, r, a32 ? 2 : 1);
  std::vector<char *> pp;
  plane = plane && cp.try_bind(ctx->planes, s, &pp);
  ScratchSrc grow{&ctx->scratch, nullptr, 0};
  auto p = (src ? *src : grow).bind(c, s);

  const float *t1 = nullptr;
  float *ds = nullptr;
  if (lora) {
    if (t1_in) {
      t1 = t1_in;
    } else if (t1_rank) {
      float *t1w = (float *)p[i_t1];
      timed(ctx, "t1_gemm", s, [&] {
        return qh::launch_rank_gemm(x, ae == qh::E_BF16, K, l->a, 0, K, t1w, r, M, K, r, 1.0f,
                                    s);
      });
      t1 = t1w;
    } else if (t1_dense) {
      dt1.c = (float *)p[i_t1];
      timed(ctx, "t1_gemm", s, [&] { return dt1.run((float *)p[i_p1], s); });
      t1 = dt1.c;
    } else {
      gt1.C = (float *)p[i_t1];
      timed(ctx, "t1_gemm", s, [&] { return qh::launch_gemm(gt1, (float *)p[i_p1], s); });
      t1 = gt1.C;
    }
    ds = (float *)p[i_ds];
    if (ds_rank) {
      timed(ctx, "ds_gemm", s, [&] {
        return qh::launch_rank_gemm(dy, ae == qh::E_BF16, N, l->b, 1, r, ds, r, M, N, r, sc, s);
      });
    } else if (ds_dense) {
      dds.c = ds;
      timed(ctx, "ds_gemm", s, [&] { return dds.run((float *)p[i_p2], s); });
    } else {
      gds.C = ds;
      timed(ctx, "ds_gemm", s, [&] { return qh::launch_gemm(gds, (float *)p[i_p2], s); });
    }
    if (g_rank) {
      // grad_B (N x r) = s dY^T T1 and grad_A (r x K) = Ds^T X as two jobs
      // of one launch (each job's sums are those of its own launch)
      qh::RankJobs jg{};
      jg.count = 2;
      jg.j[0] = qh::RankJob{dy, N, t1, r, gb, r, N, (int)r, 0, sc};
      jg.j[1] = qh::RankJob{x, K, ds, r, ga, K, K, (int)r, 1, 1.0f};
      timed(ctx, "grad_ab_gemm", s,
            [&] { return qh::launch_rank_tgemms(jg, ae == qh::E_BF16, M, s); });
    } else {
      if (gb_dense) {
        dgb.b = t1;
        timed(ctx, "grad_b_gemm", s, [&] { return dgb.run((float *)p[i_p3], s); });
      } else {
        ggb.B.p = t1;
        timed(ctx, "grad_b_gemm", s, [&] { return qh::launch_gemm(ggb, (float *)p[i_p3], s); });
      }
      if (ga_dense) {
        dga.a = ds;
        timed(ctx, "grad_a_gemm", s, [&] { return dga.run((float *)p[i_p4], s); });
      } else {
        gga.A.p = ds;
        timed(ctx, "grad_a_gemm", s, [&] { return qh::launch_gemm(gga, (float *)p[i_p4], s); });
      }
    }
  }
  if (plane) {
    plane_gemm_dev(ctx, pp, slots, "grad_x_gemm_bf16", W, qh::PLANE_NF4_COL, dy, a32, M, K, N, ds,
                   lora ? l->a : nullptr, r, 1.0f, gx, accumulate ? 1 : 0, s);
    return;
  }
  if (bf16) {
    // grad_x = dY . W + Ds . A on bf16 MFMA (dY exact when bf16, split when fp32)
    qh::Bf16GemmArgs b{};
    b.M = M, b.N = K, b.K = N, b.C = gx, b.ldc = K, b.alpha = 1.0f, b.nseg = 1;
    b.beta = accumulate ? 1 : 0;
    qh::Bf16Seg &q = b.seg[0];
    q.w = W, q.A = dy, q.lda = N, q.len = N;
    if (lora) q.A2 = ds, q.lda2 = r, q.B2 = l->a, q.ldb2 = K, q.b2scale = 1.0f, q.K2 = r;
    timed(ctx, "grad_x_gemm_bf16", s,
          [&] {
            return qh::launch_gemm_bf16(b, qh::KROW, ae == qh::E_F32, gx_splits,
                                        (float *)p[i_p5], s);
          });
    return;
  }
  Operand B;
  if (fast) {
    B = op(W.codes, K, qh::KROW, qh::E_NF4);
  } else {
    float *w32 = (float *)p[i_w32];
    timed(ctx, "dequantize", s, [&] { return qh::launch_dequantize(W, w32, s); });
    B = op(w32, K, qh::KROW, qh::E_F32);
  }
  GemmArgs gm = gemm_args(M, K, N, op(dy, N, qh::ROWK, ae), B, gx, K, 1.0f);
  gm.qw = W;
  if (lora) {
    gm.K2 = r;
    gm.A2 = op(ds, r, qh::ROWK, qh::E_F32);
    gm.B2 = op(l->a, K, qh::KROW, qh::E_F32);
  }
  gm.splits = gx_splits;
  timed(ctx, "grad_x_gemm", s, [&] { return qh::launch_gemm(gm, (float *)p[i_p5], s); });
}

// ---- projections that read the same activations -------------------------
// q / k / v of one normed input, or gate / up: their T1s in one rank
// launch and their base GEMMs in one segmented bf16-MFMA launch (forward);
// Ds, then grad_A and grad_B, in one rank launch each and the input gradient
// summed over the group in one segmented launch (backward).  Taken when
// every member fits those kernels; otherwise the members run one by one.
constexpr size_t kMaxShared = 3;  // members: 2 rank jobs each in one launch

bool shared_ok(size_t count, const DevQW *W, const qh_lora *const *l, const void *x,
               const void *const *dy, int64_t M, bool f32) {
  if (count < 2 || count > kMaxShared || count > (size_t)qh::kMaxBf16Segs) return false;
  const int64_t K = W[0].cols;
  // Members that are all large GEMMs run through operand planes one by one where
  // that is faster than one launch of the group (by both estimates, see plane_ok):
  // three forwards of 1024 x 4352 over 640 in fp32 take 120 us through planes and 78
  // in one launch, of 2048 x 4096 over 4096 545 and 609, their input gradients 589
  // and 745.
  bool planes = true;
  double us = 0;
  int64_t sum = 0;
  for (size_t i = 0; i < count && planes; ++i) {
    const int64_t N = W[i].rows, r = l[i] ? (int64_t)l[i]->r : 0;
    planes = dy ? qh::plane_ok(M, K, N, r, f32)
                : qh::plane_codes_ok(W[i]) && qh::plane_ok(M, N, K, r, f32);
    us += dy ? qh::plane_us(M, K, N, f32) : qh::plane_us(M, N, K, f32);
    sum += N;
  }
  if (planes && us < 0.98 * (dy ? qh::bf16_gemm_us(M, K, sum, f32, true)
                                : qh::bf16_gemm_us(M, sum, K, f32, false)))
    return false;
  for (size_t i = 0; i < count; ++i) {
    if (W[i].cols != K || W[i].rows == 0 || W[i].kind != W[0].kind) return false;
    if (!qh::nf4_fast_ok(W[i]) || !qh::bf16_gemm_ok(W[i], x, K, K)) return false;
    if (dy && !qh::bf16_gemm_ok(W[i], dy[i], W[i].rows, W[i].rows)) return false;
    const qh_lora *li = l[i];
    if (li) {
      const int64_t r = (int64_t)li->r;
      if (!qh::rank_gemm_ok(K, r) || !qh::rank_gemm_ok(W[i].rows, r) ||
          !qh::rank_tgemm_ok(M, r))
        return false;
    }
  }
  return M > 16 && K > 0;  // decode-sized batches take the GEMV kernels
}

void forward_shared_dev(qh_ctx *ctx, size_t count, const DevQW *W, const qh_lora *const *l,
                        const void *x, int xdt, size_t batch, float *const *y,
                        float *const *t1_out, hipStream_t s) {
  const int64_t M = (int64_t)batch, K = W[0].cols;
  const int xe = xdt == QH_BF16 ? qh::E_BF16 : qh::E_F32;
  bool slim = count <= (size_t)qh::kMaxSlimSegs;
  for (size_t i = 0; i < count && slim; ++i) slim = takes_slim(W[i], l[i], x, xdt, M);
  const bool shared = shared_ok(count, W, l, x, nullptr, M, xe == qh::E_F32);
  if (slim) {
    const void *const xs[qh::kMaxSlimSegs] = {x, x, x, x};
    size_t tile_bytes = 0;
    double tile_us = 0;
    int64_t rows = 0, r = 0;
    for (size_t i = 0; i < count; ++i) {
      const float *t1i = t1_out ? t1_out[i] : nullptr;
      rows += W[i].rows, r = std::max(r, l[i] ? (int64_t)l[i]->r : 0);
      if (shared)
        tile_bytes += l[i] && !t1i ? (size_t)M * l[i]->r * 4 + 256 : 0;
      else
        tile_bytes = std::max(tile_bytes, TileForward(W[i], l[i], x, xe, M, t1i).c.total()),
        tile_us += tile_forward_us(W[i], l[i], xdt, M);
    }
    if (shared)
      tile_us = qh::bf16_gemm_us(M, rows, K, xdt != QH_BF16, false) + t1_us(M, K, r, xdt != QH_BF16);
    if (slim_dev(ctx, count, W, l, xs, xdt, M, y, t1_out, 0, tile_bytes, tile_us, s)) return;
  }
  if (!shared) {
    for (size_t i = 0; i < count; ++i)
      forward_dev(ctx, W[i], l[i], x, xdt, batch, y[i], t1_out ? t1_out[i] : nullptr, s);
    return;
  }
  Carve c;
  size_t it[kMaxShared];
  for (size_t i = 0; i < count; ++i)
    it[i] = c.add(l[i] && !(t1_out && t1_out[i]) ? (size_t)M * l[i]->r * 4 : 0);
  auto p = c.bind(ctx->scratch, s);
  float *t1[kMaxShared];
  qh::RankJobs jt{};
  for (size_t i = 0; i < count; ++i) {
    t1[i] = nullptr;
    if (!l[i]) continue;
    t1[i] = t1_out && t1_out[i] ? t1_out[i] : (float *)p[it[i]];
    jt.j[jt.count++] = qh::RankJob{x, K, l[i]->a, K, t1[i], (int64_t)l[i]->r, K,
                                   (int)l[i]->r, 0, 1.0f};
  }
  if (jt.count)
    timed(ctx, "t1_gemm", s,
          [&] { return qh::launch_rank_gemms(jt, xe == qh::E_BF16, 0, M, s); });
  qh::Bf16GemmArgs b{};
  b.M = M, b.K = K, b.A = x, b.lda = K, b.alpha = 1.0f, b.nseg = (int)count;
  for (size_t i = 0; i < count; ++i) {
    qh::Bf16Seg &q = b.seg[i];
    const int64_t N = W[i].rows;
    q.w = W[i], q.len = N, q.C = y[i], q.ldc = N;
    if (l[i]) {
      const int64_t r = (int64_t)l[i]->r;
      q.A2 = t1[i], q.lda2 = r, q.B2 = l[i]->b, q.ldb2 = r, q.K2 = r;
      q.b2scale = l[i]->alpha / (float)l[i]->r;  // lora.rs:64-66
    }
    b.N += N;
  }
  timed(ctx, "forward_gemm_bf16", s,
        [&] { return qh::launch_gemm_bf16(b, qh::ROWK, xe == qh::E_F32, 1, nullptr, s); });
}

// gx = sum over the members of their input gradients (summed in the GEMM's
// accumulators: the same value as adding the members' gradients, rounded
// differently).
void backward_shared_dev(qh_ctx *ctx, size_t count, const DevQW *W, const qh_lora *const *l,
                         const void *x, const void *const *dy, int adt, size_t batch,
                         const float *const *t1_in, float *gx, float *const *ga,
                         float *const *gb, hipStream_t s) {
  const int64_t M = (int64_t)batch, K = W[0].cols;
  if (!shared_ok(count, W, l, x, dy, M, adt != QH_BF16)) {
    // members after the first add their input gradient into gx: in the
    // GEMM's epilogue where the path allows it, else through a separate add
    for (size_t i = 0; i < count; ++i) {
      const float *t1i = t1_in ? t1_in[i] : nullptr;
      if (i == 0 || backward_accumulates(W[i], dy[i], batch)) {
        backward_dev(ctx, W[i], l[i], x, dy[i], adt, batch, t1i, gx, ga[i], gb[i], s, nullptr,
                     nullptr, i > 0);
        continue;
      }
      float *tmp = (float *)ctx->block_tmp[1].ensure((size_t)M * K * 4, s);
      backward_dev(ctx, W[i], l[i], x, dy[i], adt, batch, t1i, tmp, ga[i], gb[i], s);
      timed(ctx, "residual_add", s,
            [&] { return qh::launch_axpy_inplace(gx, tmp, (int64_t)(M * K), s); });
    }
    return;
  }
  const int ae = adt == QH_BF16 ? qh::E_BF16 : qh::E_F32;
  const int ab = ae == qh::E_BF16;
  int64_t nsum = 0;
  for (size_t i = 0; i < count; ++i) nsum += W[i].rows;
  const int splits = qh::bf16_gemm_splits(M, K, nsum);
  Carve c;
  size_t it[kMaxShared], id[kMaxShared];
  for (size_t i = 0; i < count; ++i) {
    const size_t mr = l[i] ? (size_t)M * l[i]->r * 4 : 0;
    it[i] = c.add(l[i] && !(t1_in && t1_in[i]) ? mr : 0);
    id[i] = c.add(mr);
  }
  const size_t ip = c.add(splits > 1 ? (size_t)splits * M * K * 4 : 0);
  auto p = c.bind(ctx->scratch, s);
  const float *t1[kMaxShared];
  float *ds[kMaxShared];
  qh::RankJobs jt{}, jd{}, jg{};
  for (size_t i = 0; i < count; ++i) {
    t1[i] = nullptr, ds[i] = nullptr;
    if (!l[i]) continue;
    const int64_t N = W[i].rows, r = (int64_t)l[i]->r;
    const float sc = l[i]->alpha / (float)l[i]->r;
    if (t1_in && t1_in[i]) {
      t1[i] = t1_in[i];
    } else {
      t1[i] = (float *)p[it[i]];
      jt.j[jt.count++] = qh::RankJob{x, K, l[i]->a, K, (float *)p[it[i]], r, K, (int)r, 0, 1.0f};
    }
    ds[i] = (float *)p[id[i]];
    // Ds = s dY . B (qlora.rs:143, 149)
    jd.j[jd.count++] = qh::RankJob{dy[i], N, l[i]->b, r, ds[i], r, N, (int)r, 0, sc};
    // grad_B = s dY^T . T1 (N x r), grad_A = Ds^T . X (r x K) (qlora.rs:147, 151)
    jg.j[jg.count++] = qh::RankJob{dy[i], N, t1[i], r, gb[i], r, N, (int)r, 0, sc};
    jg.j[jg.count++] = qh::RankJob{x, K, ds[i], r, ga[i], K, K, (int)r, 1, 1.0f};
  }
  if (jt.count)
    timed(ctx, "t1_gemm", s, [&] { return qh::launch_rank_gemms(jt, ab, 0, M, s); });
  if (jd.count) {
    timed(ctx, "ds_gemm", s, [&] { return qh::launch_rank_gemms(jd, ab, 1, M, s); });
    timed(ctx, "grad_ab_gemm", s, [&] { return qh::launch_rank_tgemms(jg, ab, M, s); });
  }
  qh::Bf16GemmArgs b{};
  b.M = M, b.N = K, b.K = nsum, b.C = gx, b.ldc = K, b.alpha = 1.0f, b.nseg = (int)count;
  for (size_t i = 0; i < count; ++i) {
    qh::Bf16Seg &q = b.seg[i];
    const int64_t N = W[i].rows;
    q.w = W[i], q.A = dy[i], q.lda = N, q.len = N;
    if (l[i]) {
      const int64_t r = (int64_t)l[i]->r;
      q.A2 = ds[i], q.lda2 = r, q.B2 = l[i]->a, q.ldb2 = K, q.b2scale = 1.0f, q.K2 = r;
    }
  }
  timed(ctx, "grad_x_gemm_bf16", s, [&] {
    return qh::launch_gemm_bf16(b, qh::KROW, ae == qh::E_F32, splits, (float *)p[ip], s);
  });
}

// Plain GEMMs (gpu_matmul*): C = A.B, A^T.B, A.B^T.
void matmul_dev(qh_ctx *ctx, int opk, const float *a, const float *b, size_t m,
                size_t k, size_t n, float *c, hipStream_t s) {
  GemmArgs g;
  if (opk == QH_MM_NN) {
    g = gemm_args(m, n, k, op(a, k, qh::ROWK, qh::E_F32), op(b, n, qh::KROW, qh::E_F32), c, n, 1.0f);
  } else if (opk == QH_MM_NT) {
    g = gemm_args(m, n, k, op(a, k, qh::ROWK, qh::E_F32), op(b, k, qh::ROWK, qh::E_F32), c, n, 1.0f);
  } else {
    // C(k x n) = A(m x k)^T B(m x n): rows of C index A's columns.
    g = gemm_args(k, n, m, op(a, k, qh::KROW, qh::E_F32), op(b, n, qh::KROW, qh::E_F32), c, n, 1.0f);
  }
  g.splits = choose_splits(g.M, g.N, g.K);
  Carve cv;
  size_t ip = cv.add(partial_floats(g) * 4);
  auto p = cv.bind(ctx->scratch, s);
  timed(ctx, "matmul", s, [&] { return qh::launch_gemm(g, (float *)p[ip], s); });
}

template <class F>
qh_status guarded(qh_ctx *ctx, F &&f) {
  if (!ctx) return fail(QH_ERR_GPU, "context is NULL");
  std::lock_guard<std::mutex> lk(ctx->mu);
  try {
    check(hipSetDevice(ctx->device), "hipSetDevice");
    return f();
  } catch (const GpuError &e) {
    (void)hipGetLastError();  // do not leave the failure for the caller's next HIP call
    qh::g_launch_timing = qh::LaunchTiming();
    return fail(QH_ERR_GPU, e.msg);
  } catch (const std::bad_alloc &) {
    return fail(QH_ERR_GPU, "host allocation failed");
  } catch (...) {
    return fail(QH_ERR_GPU, "unexpected failure");
  }
}

}  // namespace

// ---- the allocation-free backward's scratch region --------------------------
// One region per GPU, in the library's code object: every device the library
// runs on holds its own copy until the process ends.  In host code the
// array's name is only a handle for hipGetSymbolAddress, never an address:
// kernels get the per-device address that call returns.
static __device__ __align__(256) unsigned char scratch[QH_NOALLOC_SCRATCH_BYTES];

namespace {

// The region's address on `dev`, looked up once per device (with `dev`
// current, as the lookup requires) and kept for every later context.
hipError_t noalloc_region(int dev, void **out) {
  static std::mutex mu;
  static std::map<int, void *> addr;
  std::lock_guard<std::mutex> lk(mu);
  auto it = addr.find(dev);
  if (it != addr.end()) {
    *out = it->second;
    return hipSuccess;
  }
  void *p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess) return e;
  addr[dev] = p;
  *out = p;
  return hipSuccess;
}

// Timing off for the duration of a call (it would create events).
struct NoTiming {
  qh_ctx *c;
  bool was;
  explicit NoTiming(qh_ctx *ctx) : c(ctx), was(ctx->timing) { c->timing = false; }
  ~NoTiming() { c->timing = was; }
};

}  // namespace

// ===========================================================================
extern "C" {

uint32_t qh_abi_version(void) { return QH_ABI_VERSION; }

const char *qh_last_error(void) { return g_err.c_str(); }

qh_status qh_ctx_create(qh_ctx **out) {
  if (!out) return fail(QH_ERR_GPU, "out is NULL");
  *out = nullptr;
  int n = 0;
  hipError_t e = hipGetDeviceCount(&n);
  if (e == hipErrorNoDevice || (e == hipSuccess && n == 0) ||
      e == hipErrorInsufficientDriver) {
    (void)hipGetLastError();
    return fail(QH_NO_DEVICE, "no GPU device is visible");
  }
  if (e != hipSuccess) return fail(QH_ERR_GPU, hipGetErrorString(e));
  qh_ctx *c = new (std::nothrow) qh_ctx();
  if (!c) return fail(QH_ERR_GPU, "host allocation failed");
  if (hipGetDevice(&c->device) != hipSuccess) c->device = 0;
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, c->device) == hipSuccess)
    snprintf(c->name, sizeof c->name, "%s (%s)", prop.name, prop.gcnArchName);
  if ((e = hipSetDevice(c->device)) != hipSuccess ||
      (e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking)) != hipSuccess ||
      (e = hipMalloc((void **)&c->tickets, (size_t)qh::kTicketsTotalWords * 4)) != hipSuccess ||
      (e = hipMemset(c->tickets, 0, (size_t)qh::kTicketsTotalWords * 4)) != hipSuccess ||
      (e = hipDeviceSynchronize()) != hipSuccess) {
    if (c->tickets) (void)hipFree(c->tickets);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
    return fail(QH_ERR_GPU, hipGetErrorString(e));
  }
  // The allocation-free backward's region on this device (the device is
  // current here); a failure is kept and reported by that entry point only.
  c->noalloc_err = noalloc_region(c->device, &c->noalloc);
  if (c->noalloc_err != hipSuccess) (void)hipGetLastError();
  *out = c;
  return QH_OK;
}

void qh_ctx_destroy(qh_ctx *ctx) {
  if (!ctx) return;
  (void)hipSetDevice(ctx->device);
  if (ctx->stream) {
    (void)hipStreamSynchronize(ctx->stream);
    (void)hipStreamDestroy(ctx->stream);
  }
  for (auto &b : ctx->stage) b.release();
  ctx->scratch.release();
  ctx->planes.release();
  for (auto &b : ctx->block_tmp) b.release();
  if (ctx->tickets) (void)hipFree(ctx->tickets);
  delete ctx;
}

qh_status qh_ctx_device_name(qh_ctx *ctx, char *buf, size_t len) {
  if (!ctx || !buf || !len) return fail(QH_ERR_GPU, "bad arguments");
  snprintf(buf, len, "%s", ctx->name);
  return QH_OK;
}

qh_status qh_ctx_synchronize(qh_ctx *ctx) {
  return guarded(ctx, [&] {
    check(hipStreamSynchronize(ctx->stream), "hipStreamSynchronize");
    return QH_OK;
  });
}

qh_status qh_ctx_set_timing(qh_ctx *ctx, int enable) {
  return guarded(ctx, [&] {
    ctx->timing = enable != 0;
    return QH_OK;
  });
}

qh_status qh_ctx_set_test_flags(qh_ctx *ctx, uint32_t flags) {
  if (!ctx) return fail(QH_ERR_GPU, "context is NULL");
  std::lock_guard<std::mutex> lk(ctx->mu);
  ctx->test_flags = flags;
  return QH_OK;
}

qh_status qh_ctx_timing_report(qh_ctx *ctx, char *buf, size_t len, int reset) {
  return guarded(ctx, [&] {
    drain_timing(ctx);
    std::string out;
    for (const auto &kv : ctx->totals)
      out += fmt("%s %llu %.6f\n", kv.first.c_str(), (unsigned long long)kv.second.first,
                 kv.second.second);
    if (buf && len) snprintf(buf, len, "%s", out.c_str());
    if (reset) ctx->totals.clear();
    return QH_OK;
  });
}

size_t qh_codes_len(size_t rows, size_t cols) { return div_ceil(rows * cols, 2); }
size_t qh_num_blocks(size_t rows, size_t cols, size_t bs) {
  return bs ? div_ceil(rows * cols, bs) : 0;
}
size_t qh_num_absmax(size_t rows, size_t cols, size_t bs) {
  return div_ceil(qh_num_blocks(rows, cols, bs), 256);
}
size_t qh_storage_bytes(const qh_qweight *w) {
  if (!w || !w->block_size) return 0;
  size_t nb = qh_num_blocks(w->rows, w->cols, w->block_size);
  size_t sb = w->scale_kind == QH_SCALES_F32 ? nb * 4 : nb + div_ceil(nb, 256) * 4;
  return qh_codes_len(w->rows, w->cols) + sb;
}

// ---- quantization ---------------------------------------------------------
qh_status qh_quantize_nf4(qh_ctx *ctx, const float *w, size_t w_len,
                          size_t rows, size_t cols, size_t block_size,
                          int double_quant, uint8_t *codes, float *scales,
                          uint8_t *scale_codes, float *absmax) {
  // quant.rs:110-119: validate, overflow, then length.
  if (block_size == 0) return fail(QH_ERR_INVALID_CONFIG, "block_size must be > 0");
  size_t n;
  if (mul_overflows(rows, cols, &n)) return fail(QH_ERR_INVALID_CONFIG, "rows*cols overflow");
  if (w_len != n)
    return fail(QH_ERR_SHAPE_MISMATCH, fmt("weights.len() = %zu but rows*cols = %zu", w_len, n));
  return guarded(ctx, [&] {
    hipStream_t s = ctx->stream;
    const size_t nb = div_ceil(n, block_size), nsb = div_ceil(nb, 256);
    const size_t cb = div_ceil(n, 2);
    Carve c;
    size_t iw = c.add(n * 4), ic = c.add(cb + 16), is = c.add(nb * 4 + 16),
           isc = c.add(nb + 16), ia = c.add(nsb * 4 + 16), it = c.add(nb * 4 + 16);
    auto p = c.bind(ctx->stage[0]);
    if (n) check(hipMemcpyAsync(p[iw], w, n * 4, hipMemcpyHostToDevice, s), "upload");
    timed(ctx, "quantize", s, [&] { return qh::launch_quantize((float *)p[iw], (int64_t)n, (int64_t)block_size,
                              double_quant ? 1 : 0, (uint8_t *)p[ic], (float *)p[is],
                              (uint8_t *)p[isc], (float *)p[ia], (float *)p[it], s); });
    if (cb) check(hipMemcpyAsync(codes, p[ic], cb, hipMemcpyDeviceToHost, s), "download");
    if (double_quant) {
      if (nb) check(hipMemcpyAsync(scale_codes, p[isc], nb, hipMemcpyDeviceToHost, s), "download");
      if (nsb) check(hipMemcpyAsync(absmax, p[ia], nsb * 4, hipMemcpyDeviceToHost, s), "download");
    } else if (nb) {
      check(hipMemcpyAsync(scales, p[is], nb * 4, hipMemcpyDeviceToHost, s), "download");
    }
    check(hipStreamSynchronize(s), "sync");
    return QH_OK;
  });
}

qh_status qh_quantize_nf4_dev(qh_ctx *ctx, const float *d_w, size_t rows,
                              size_t cols, size_t block_size, int double_quant,
                              uint8_t *d_codes, float *d_scales,
                              uint8_t *d_scale_codes, float *d_absmax,
                              void *stream) {
  if (block_size == 0) return fail(QH_ERR_INVALID_CONFIG, "block_size must be > 0");
  size_t n;
  if (mul_overflows(rows, cols, &n)) return fail(QH_ERR_INVALID_CONFIG, "rows*cols overflow");
  return guarded(ctx, [&] {
    hipStream_t s = pick_stream(ctx, stream);
    float *tmp = nullptr;
    if (double_quant && block_size != 64)
      tmp = (float *)ctx->scratch.ensure(div_ceil(n, block_size) * 4 + 16, s);
    timed(ctx, "quantize", s, [&] { return qh::launch_quantize(d_w, (int64_t)n, (int64_t)block_size, double_quant ? 1 : 0,
                              d_codes, d_scales, d_scale_codes, d_absmax, tmp, s); });
    return QH_OK;
  });
}

qh_status qh_block_scales(qh_ctx *ctx, const qh_qweight *w, float *out) {
  qh_status st = validate_weight(w);
  if (st != QH_OK) return st;
  return guarded(ctx, [&] {
    hipStream_t s = ctx->stream;
    DevQW d = upload_weight(ctx, *w, 0, s);
    float *o = alloc_f32(ctx, 1, (size_t)d.nb);
    timed(ctx, "block_scales", s, [&] { return qh::launch_block_scales(d, o, s); });
    download_f32(out, o, (size_t)d.nb, s);
    check(hipStreamSynchronize(s), "sync");
    return QH_OK;
  });
}

qh_status qh_dequantize(qh_ctx *ctx, const qh_qweight *w, float *out) {
  qh_status st = validate_weight(w);
  if (st != QH_OK) return st;
  return guarded(ctx, [&] {
    hipStream_t s = ctx->stream;
    DevQW d = upload_weight(ctx, *w, 0, s);
    float *o = alloc_f32(ctx, 1, (size_t)d.n);
    timed(ctx, "dequantize", s, [&] { return qh::launch_dequantize(d, o, s); });
    download_f32(out, o, (size_t)d.n, s);
    check(hipStreamSynchronize(s), "sync");
    return QH_OK;
  });
}

qh_status qh_dequantize_dev(qh_ctx *ctx, const qh_qweight *w, float *d_out,
                            void *stream) {
  qh_status st = validate_weight(w);
  if (st != QH_OK) return st;
  return guarded(ctx, [&] {
    hipStream_t s = pick_stream(ctx, stream);
    timed(ctx, "dequantize", s, [&] { return qh::launch_dequantize(make_devqw(*w), d_out, s); });
    return QH_OK;
  });
}

// ---- GEMMs ------------------------------------------------------------------
static qh_status matmul_host(qh_ctx *ctx, int opk, const char *name,
                             const float *a, size_t a_len, const float *b,
                             size_t b_len, size_t m, size_t k, size_t n,
                             float *c) {
  // kernels.rs:151-160 (NN, NT) and :231-240 (TN): empty output first,
  // then the length check.
  size_t out_len;
  if (opk == QH_MM_TN) {
    if (k == 0 || n == 0) return QH_OK;
    if (a_len != m * k || b_len != m * n)
      return fail(QH_ERR_SHAPE_MISMATCH,
                  fmt("%s: a.len() = %zu, b.len() = %zu, expected %zu*%zu and %zu*%zu",
                      name, a_len, b_len, m, k, m, n));
    out_len = k * n;
  } else {
    if (m == 0 || n == 0) return QH_OK;
    size_t bl = opk == QH_MM_NN ? k * n : n * k;
    if (a_len != m * k || b_len != bl)
      return fail(QH_ERR_SHAPE_MISMATCH,
                  opk == QH_MM_NN
                      ? fmt("%s: a.len() = %zu, b.len() = %zu, expected %zu*%zu and %zu*%zu",
                            name, a_len, b_len, m, k, k, n)
                      : fmt("%s: a.len() = %zu, b.len() = %zu, expected %zu*%zu and %zu*%zu",
                            name, a_len, b_len, m, k, n, k));
    out_len = m * n;
  }
  return guarded(ctx, [&] {
    hipStream_t s = ctx->stream;
    float *da = upload_f32(ctx, 0, a, a_len, s);
    float *db = upload_f32(ctx, 1, b, b_len, s);
    float *dc = alloc_f32(ctx, 2, out_len);
    matmul_dev(ctx, opk, da, db, m, k, n, dc, s);
    download_f32(c, dc, out_len, s);
    check(hipStreamSynchronize(s), "sync");
    return QH_OK;
  });
}

qh_status qh_matmul(qh_ctx *ctx, const float *a, size_t a_len, const float *b,
                    size_t b_len, size_t m, size_t k, size_t n, float *c) {
  return matmul_host(ctx, QH_MM_NN, "gpu_matmul", a, a_len, b, b_len, m, k, n, c);
}
qh_status qh_matmul_trans_a(qh_ctx *ctx, const float *a, size_t a_len,
                            const float *b, size_t b_len, size_t m, size_t k,
                            size_t n, float *c) {
  return matmul_host(ctx, QH_MM_TN, "gpu_matmul_trans_a", a, a_len, b, b_len, m, k, n, c);
}
qh_status qh_matmul_trans_b(qh_ctx *ctx, const float *a, size_t a_len,
                            const float *b, size_t b_len, size_t m, size_t k,
                            size_t n, float *c) {
  return matmul_host(ctx, QH_MM_NT, "gpu_matmul_trans_b", a, a_len, b, b_len, m, k, n, c);
}

qh_status qh_matmul_dev(qh_ctx *ctx, int opk, const float *d_a, const float *d_b,
                        size_t m, size_t k, size_t n, float *d_c, void *stream) {
  if (opk != QH_MM_NN && opk != QH_MM_NT && opk != QH_MM_TN)
    return fail(QH_ERR_INVALID_CONFIG, "unknown matmul op");
  return guarded(ctx, [&] {
    matmul_dev(ctx, opk, d_a, d_b, m, k, n, d_c, pick_stream(ctx, stream));
    return QH_OK;
  });
}

// ---- the layer ------------------------------------------------------------------
qh_status qh_qlora_forward(qh_ctx *ctx, const qh_qweight *w, const qh_lora *lora,
                           const float *x, size_t x_len, size_t batch, float *y) {
  qh_status st = validate_weight(w);
  if (st != QH_OK) return st;
  const size_t in_dim = w->cols, out_dim = w->rows;
  if ((st = validate_lora(lora, in_dim, out_dim)) != QH_OK) return st;
  if (x_len != batch * in_dim)
    return fail(QH_ERR_SHAPE_MISMATCH,
                fmt("x.len() = %zu but batch*in_dim = %zu", x_len, batch * in_dim));
  return guarded(ctx, [&] {
    hipStream_t s = ctx->stream;
    DevQW d = upload_weight(ctx, *w, 0, s);
    float *dx = upload_f32(ctx, 1, x, x_len, s);
    float *dy = alloc_f32(ctx, 2, batch * out_dim);
    qh_lora dl{};
    if (lora) {
      dl = *lora;
      dl.a = upload_f32(ctx, 3, lora->a, lora->a_len, s);
      dl.b = upload_f32(ctx, 4, lora->b, lora->b_len, s);
    }
    forward_dev(ctx, d, lora ? &dl : nullptr, dx, QH_F32, batch, dy, nullptr, s);
    download_f32(y, dy, batch * out_dim, s);
    check(hipStreamSynchronize(s), "sync");
    return QH_OK;
  });
}

qh_status qh_qlora_backward(qh_ctx *ctx, const qh_qweight *w, const qh_lora *lora,
                            const float *x, size_t x_len, const float *dy,
                            size_t dy_len, size_t batch, float *grad_x,
                            float *grad_a, float *grad_b) {
  qh_status st = validate_weight(w);
  if (st != QH_OK) return st;
  const size_t in_dim = w->cols, out_dim = w->rows;
  if ((st = validate_lora(lora, in_dim, out_dim)) != QH_OK) return st;
  // qlora.rs:119-132
  if (x_len != batch * in_dim)
    return fail(QH_ERR_SHAPE_MISMATCH,
                fmt("x.len() = %zu but batch*in_dim = %zu", x_len, batch * in_dim));
  if (dy_len != batch * out_dim)
    return fail(QH_ERR_SHAPE_MISMATCH,
                fmt("dy.len() = %zu but batch*out_dim = %zu", dy_len, batch * out_dim));
  return guarded(ctx, [&] {
    hipStream_t s = ctx->stream;
    DevQW d = upload_weight(ctx, *w, 0, s);
    float *dx = upload_f32(ctx, 1, x, x_len, s);
    float *ddy = upload_f32(ctx, 2, dy, dy_len, s);
    float *dgx = alloc_f32(ctx, 5, batch * in_dim);
    qh_lora dl{};
    float *dga = nullptr, *dgb = nullptr;
    if (lora) {
      dl = *lora;
      dl.a = upload_f32(ctx, 3, lora->a, lora->a_len, s);
      dl.b = upload_f32(ctx, 4, lora->b, lora->b_len, s);
      dga = alloc_f32(ctx, 6, lora->r * in_dim);
      dgb = alloc_f32(ctx, 7, out_dim * lora->r);
    }
    backward_dev(ctx, d, lora ? &dl : nullptr, dx, ddy, QH_F32, batch, nullptr, dgx, dga,
                 dgb, s);
    download_f32(grad_x, dgx, batch * in_dim, s);
    if (lora) {
      download_f32(grad_a, dga, lora->r * in_dim, s);
      download_f32(grad_b, dgb, out_dim * lora->r, s);
    }
    check(hipStreamSynchronize(s), "sync");
    return QH_OK;
  });
}

// A device buffer that a call reads or writes must not be NULL: the kernels
// would dereference it.  `elems` is the buffer's element count for the call.
static qh_status need_buf(const void *p, size_t elems, const char *what) {
  if (p == nullptr && elems != 0)
    return fail(QH_ERR_SHAPE_MISMATCH, fmt("%s is NULL but holds %zu elements", what, elems));
  return QH_OK;
}

qh_status qh_qlora_forward_dev(qh_ctx *ctx, const qh_qweight *w, const qh_lora *lora,
                               const void *d_x, int x_dtype, size_t batch, float *d_y,
                               float *d_t1, void *stream) {
  qh_status st = validate_weight(w);
  if (st != QH_OK) return st;
  if ((st = validate_lora(lora, w->cols, w->rows)) != QH_OK) return st;
  if (x_dtype != QH_F32 && x_dtype != QH_BF16)
    return fail(QH_ERR_INVALID_CONFIG, "x_dtype must be QH_F32 or QH_BF16");
  if ((st = need_buf(d_x, batch * w->cols, "x")) != QH_OK ||
      (st = need_buf(d_y, batch * w->rows, "y")) != QH_OK ||
      (st = need_buf(w->codes, w->rows * w->cols, "the weight's codes")) != QH_OK)
    return st;
  return guarded(ctx, [&] {
    forward_dev(ctx, make_devqw(*w), lora, d_x, x_dtype, batch, d_y, d_t1,
                pick_stream(ctx, stream));
    return QH_OK;
  });
}

// Layer-indexed errors: "<kind>: layer i: <text>".
static qh_status layer_error(qh_status st, size_t i) {
  const size_t pos = g_err.find(": ");
  if (pos != std::string::npos) g_err.insert(pos + 2, fmt("layer %zu: ", i));
  return st;
}

qh_status qh_qlora_forward_group_dev(qh_ctx *ctx, size_t count, const qh_qweight *ws,
                                     const qh_lora *const *loras, const void *const *d_xs,
                                     int x_dtype, size_t batch, float *const *d_ys,
                                     float *const *d_t1s, void *stream) {
  if (count == 0) return QH_OK;
  if (!ws || !d_xs || !d_ys)
    return fail(QH_ERR_SHAPE_MISMATCH, "ws, d_xs and d_ys must be given for count > 0");
  if (x_dtype != QH_F32 && x_dtype != QH_BF16)
    return fail(QH_ERR_INVALID_CONFIG, "x_dtype must be QH_F32 or QH_BF16");
  for (size_t i = 0; i < count; ++i) {
    const qh_qweight *w = &ws[i];
    const qh_lora *l = loras ? loras[i] : nullptr;
    qh_status st = validate_weight(w);
    if (st == QH_OK) st = validate_lora(l, w->cols, w->rows);
    if (st == QH_OK) st = need_buf(d_xs[i], batch * w->cols, "x");
    if (st == QH_OK) st = need_buf(d_ys[i], batch * w->rows, "y");
    if (st == QH_OK) st = need_buf(w->codes, w->rows * w->cols, "the weight's codes");
    if (st != QH_OK) return layer_error(st, i);
  }
  return guarded(ctx, [&] {
    hipStream_t s = pick_stream(ctx, stream);
    const int xb = x_dtype == QH_BF16;
    const bool force = (ctx->test_flags & QH_TEST_FORCE_T1_RECOMPUTE) != 0;
    std::vector<char> done(count, 0);
    if (batch >= 2 && batch <= 16) {
      // Layers on the split kernel (3-16 rows, and 2 rows past the one-launch
      // kernel): the adapters' T1 of all of them in one launch (the caller's
      // T1 buffer where given, else scratch), then the weight streams, two
      // layers per split launch where their plans pair (the same bits in
      // every such call; within rounding of per-layer calls).
      const int64_t M = (int64_t)batch;
      std::vector<size_t> idx;
      for (size_t i = 0; i < count; ++i) {
        const qh_lora *l = loras ? loras[i] : nullptr;
        const DevQW W = make_devqw(ws[i]);
        if (l && takes_split(W, l, d_xs[i], M)) idx.push_back(i);
      }
      if (idx.size() >= 2) {
        // split layers in order, two per launch (each planned for half of
        // the CUs) where both plan that way, else one per launch
        std::vector<qh::SplitPlan> plan(idx.size());
        std::vector<char> paired(idx.size(), 0);  // first of a pair
        for (size_t q = 0; q < idx.size(); ++q) {
          const size_t i = idx[q];
          const DevQW W = make_devqw(ws[i]);
          plan[q] = qh::split_plan(W, M, loras[i]->r);
        }
        for (size_t q = 0; q + 1 < idx.size(); ++q) {
          if (!plan[q].ok || !plan[q + 1].ok) continue;
          qh::SplitPlan a = qh::split_plan(make_devqw(ws[idx[q]]), M, loras[idx[q]]->r, 2);
          qh::SplitPlan b =
              qh::split_plan(make_devqw(ws[idx[q + 1]]), M, loras[idx[q + 1]]->r, 2);
          if (qh::split_pair(a, b)) {
            plan[q] = a;
            plan[q + 1] = b;
            paired[q] = 1;
            ++q;
          }
        }
        Carve c;
        std::vector<size_t> slot(idx.size()), pslot(idx.size());
        for (size_t q = 0; q < idx.size(); ++q) {
          const size_t i = idx[q];
          slot[q] = c.add(d_t1s && d_t1s[i] ? 0 : (size_t)M * loras[i]->r * 4);
          pslot[q] = c.add(plan[q].ok ? plan[q].part_floats * 4 : 0);
        }
        auto p = c.bind(ctx->scratch, s);
        std::vector<float *> t1(idx.size());
        for (size_t q = 0; q < idx.size(); ++q)
          t1[q] = d_t1s && d_t1s[idx[q]] ? d_t1s[idx[q]] : (float *)p[slot[q]];
        for (size_t q0 = 0; q0 < idx.size(); q0 += qh::kMaxT1Jobs) {
          qh::T1Jobs jobs{};
          jobs.count = (int)std::min<size_t>(qh::kMaxT1Jobs, idx.size() - q0);
          for (int q = 0; q < jobs.count; ++q) {
            const size_t i = idx[q0 + q];
            jobs.j[q] = qh::T1Job{d_xs[i], loras[i]->a, t1[q0 + q], (int64_t)ws[i].cols,
                                  (int)loras[i]->r};
          }
          timed(ctx, "decode_t1", s,
                [&] { return qh::launch_lora_t1_jobs(jobs, xb, M, s); });
        }
        auto split_in = [&](size_t q) {
          const size_t i = idx[q];
          const qh_lora *l = loras[i];
          return qh::SplitLayerIn{make_devqw(ws[i]), d_xs[i], t1[q], l->b, (int64_t)l->r,
                                  l->alpha / (float)l->r, d_ys[i], (float *)p[pslot[q]]};
        };
        for (size_t q = 0; q < idx.size(); ++q) {
          const size_t i = idx[q];
          if (plan[q].ok) {
            if (paired[q]) {
              const qh::SplitPlan pp[2] = {plan[q], plan[q + 1]};
              const qh::SplitLayerIn in[2] = {split_in(q), split_in(q + 1)};
              timed(ctx, "decode_split", s, [&] {
                return qh::launch_decode_split(2, in, pp, M, xb, ctx->tickets, s);
              });
              done[i] = done[idx[q + 1]] = 1;
              ++q;
              continue;
            }
            const qh::SplitLayerIn in = split_in(q);
            timed(ctx, "decode_split", s, [&] {
              return qh::launch_decode_split(1, &in, &plan[q], M, xb, ctx->tickets, s);
            });
            done[i] = 1;
          }
        }
      }
    }
    for (size_t i = 0; i < count; ++i) {
      if (done[i]) continue;
      const qh_lora *l1 = loras ? loras[i] : nullptr;
      float *t1o1 = d_t1s ? d_t1s[i] : nullptr;
      const DevQW W1 = make_devqw(ws[i]);
      if (batch == 1 && i + 1 < count && takes_stream(W1, l1, d_xs[i], 1)) {
        const qh_lora *l2 = loras ? loras[i + 1] : nullptr;
        const DevQW W2 = make_devqw(ws[i + 1]);
        const int64_t r1 = l1 ? (int64_t)l1->r : 0, r2 = l2 ? (int64_t)l2->r : 0;
        if (takes_stream(W2, l2, d_xs[i + 1], 1) && qh::decode_stream2_ok(W1, r1, W2, r2)) {
          float *t1o2 = d_t1s ? d_t1s[i + 1] : nullptr;
          timed(ctx, "decode_stream2", s, [&] {
            return qh::launch_decode_stream2(
                W1, d_xs[i], l1 ? l1->a : nullptr, r1, l1 ? l1->b : nullptr,
                l1 ? l1->alpha / (float)l1->r : 0.0f, d_ys[i], t1o1, W2, d_xs[i + 1],
                l2 ? l2->a : nullptr, r2, l2 ? l2->b : nullptr,
                l2 ? l2->alpha / (float)l2->r : 0.0f, d_ys[i + 1], t1o2, xb, ctx->tickets,
                force, s);
          });
          ++i;
          continue;
        }
      }
      forward_dev(ctx, W1, l1, d_xs[i], x_dtype, batch, d_ys[i], t1o1, s);
    }
    return QH_OK;
  });
}

constexpr size_t kMaxSharedApi = 8;

qh_status qh_qlora_forward_shared_dev(qh_ctx *ctx, size_t count, const qh_qweight *ws,
                                      const qh_lora *const *loras, const void *d_x,
                                      int x_dtype, size_t batch, float *const *d_ys,
                                      float *const *d_t1s, void *stream) {
  if (count == 0) return QH_OK;
  if (count > kMaxSharedApi) return fail(QH_ERR_INVALID_CONFIG, "more than 8 layers");
  if (!ws || !d_ys) return fail(QH_ERR_SHAPE_MISMATCH, "ws and d_ys must be given");
  if (x_dtype != QH_F32 && x_dtype != QH_BF16)
    return fail(QH_ERR_INVALID_CONFIG, "x_dtype must be QH_F32 or QH_BF16");
  for (size_t i = 0; i < count; ++i) {
    const qh_qweight *w = &ws[i];
    qh_status st = validate_weight(w);
    if (st == QH_OK && w->cols != ws[0].cols)
      st = fail(QH_ERR_SHAPE_MISMATCH, fmt("in_dim %zu differs from layer 0's %zu", w->cols,
                                           ws[0].cols));
    if (st == QH_OK) st = validate_lora(loras ? loras[i] : nullptr, w->cols, w->rows);
    if (st == QH_OK) st = need_buf(d_x, batch * w->cols, "x");
    if (st == QH_OK) st = need_buf(d_ys[i], batch * w->rows, "y");
    if (st == QH_OK) st = need_buf(w->codes, w->rows * w->cols, "the weight's codes");
    if (st != QH_OK) return layer_error(st, i);
  }
  return guarded(ctx, [&] {
    DevQW W[kMaxSharedApi];
    const qh_lora *L[kMaxSharedApi];
    for (size_t i = 0; i < count; ++i) {
      W[i] = make_devqw(ws[i]);
      L[i] = loras ? loras[i] : nullptr;
    }
    forward_shared_dev(ctx, count, W, L, d_x, x_dtype, batch, d_ys, d_t1s,
                       pick_stream(ctx, stream));
    return QH_OK;
  });
}

static qh_status validate_backward_dev(const qh_qweight *w, const qh_lora *lora,
                                       const void *d_x, const void *d_dy, int act_dtype,
                                       size_t batch, float *d_grad_x, float *d_grad_a,
                                       float *d_grad_b);

qh_status qh_qlora_backward_shared_dev(qh_ctx *ctx, size_t count, const qh_qweight *ws,
                                       const qh_lora *const *loras, const void *d_x,
                                       const void *const *d_dys, int act_dtype, size_t batch,
                                       const float *const *d_t1s, float *d_grad_x,
                                       float *const *d_grad_as, float *const *d_grad_bs,
                                       void *stream) {
  if (count == 0) return QH_OK;
  if (count > kMaxSharedApi) return fail(QH_ERR_INVALID_CONFIG, "more than 8 layers");
  if (!ws || !d_dys) return fail(QH_ERR_SHAPE_MISMATCH, "ws and d_dys must be given");
  for (size_t i = 0; i < count; ++i) {
    const qh_lora *l = loras ? loras[i] : nullptr;
    qh_status st = QH_OK;
    if (ws[i].cols != ws[0].cols)
      st = fail(QH_ERR_SHAPE_MISMATCH, fmt("in_dim %zu differs from layer 0's %zu", ws[i].cols,
                                           ws[0].cols));
    if (st == QH_OK && l && (!d_grad_as || !d_grad_bs))
      st = fail(QH_ERR_SHAPE_MISMATCH, "an adapter's gradient buffer is NULL");
    if (st == QH_OK)
      st = validate_backward_dev(&ws[i], l, d_x, d_dys[i], act_dtype, batch, d_grad_x,
                                 l ? d_grad_as[i] : nullptr, l ? d_grad_bs[i] : nullptr);
    if (st != QH_OK) return layer_error(st, i);
  }
  return guarded(ctx, [&] {
    DevQW W[kMaxSharedApi];
    const qh_lora *L[kMaxSharedApi];
    float *GA[kMaxSharedApi], *GB[kMaxSharedApi];
    for (size_t i = 0; i < count; ++i) {
      W[i] = make_devqw(ws[i]);
      L[i] = loras ? loras[i] : nullptr;
      GA[i] = L[i] ? d_grad_as[i] : nullptr;
      GB[i] = L[i] ? d_grad_bs[i] : nullptr;
    }
    backward_shared_dev(ctx, count, W, L, d_x, d_dys, act_dtype, batch, d_t1s, d_grad_x, GA,
                        GB, pick_stream(ctx, stream));
    return QH_OK;
  });
}

static qh_status validate_backward_dev(const qh_qweight *w, const qh_lora *lora,
                                       const void *d_x, const void *d_dy, int act_dtype,
                                       size_t batch, float *d_grad_x, float *d_grad_a,
                                       float *d_grad_b) {
  qh_status st = validate_weight(w);
  if (st != QH_OK) return st;
  if ((st = validate_lora(lora, w->cols, w->rows)) != QH_OK) return st;
  if (act_dtype != QH_F32 && act_dtype != QH_BF16)
    return fail(QH_ERR_INVALID_CONFIG, "act_dtype must be QH_F32 or QH_BF16");
  const size_t in_dim = w->cols, out_dim = w->rows, r = lora ? lora->r : 0;
  // grad_A and grad_B are written whenever an adapter is given, even when
  // they come out zero
  if ((st = need_buf(d_grad_a, r * in_dim, "grad_a")) != QH_OK ||
      (st = need_buf(d_grad_b, out_dim * r, "grad_b")) != QH_OK ||
      (st = need_buf(d_dy, batch * out_dim, "dy")) != QH_OK ||
      (st = need_buf(d_grad_x, batch * in_dim, "grad_x")) != QH_OK ||
      (st = need_buf(d_x, lora ? batch * in_dim : 0, "x")) != QH_OK ||
      (st = need_buf(w->codes, w->rows * w->cols, "the weight's codes")) != QH_OK)
    return st;
  return QH_OK;
}

qh_status qh_qlora_backward_dev(qh_ctx *ctx, const qh_qweight *w, const qh_lora *lora,
                                const void *d_x, const void *d_dy, int act_dtype,
                                size_t batch, const float *d_t1, float *d_grad_x,
                                float *d_grad_a, float *d_grad_b, void *stream) {
  qh_status st = validate_backward_dev(w, lora, d_x, d_dy, act_dtype, batch, d_grad_x,
                                       d_grad_a, d_grad_b);
  if (st != QH_OK) return st;
  return guarded(ctx, [&] {
    backward_dev(ctx, make_devqw(*w), lora, d_x, d_dy, act_dtype, batch, d_t1, d_grad_x,
                 d_grad_a, d_grad_b, pick_stream(ctx, stream));
    return QH_OK;
  });
}

qh_status qh_qlora_backward_dev_noalloc(qh_ctx *ctx, const qh_qweight *w, const qh_lora *lora,
                                        const void *d_x, const void *d_dy, int act_dtype,
                                        size_t batch, const float *d_t1, float *d_grad_x,
                                        float *d_grad_a, float *d_grad_b, void *stream) {
  qh_status st = validate_backward_dev(w, lora, d_x, d_dy, act_dtype, batch, d_grad_x,
                                       d_grad_a, d_grad_b);
  if (st != QH_OK) return st;
  // The plan of qh_qlora_backward_dev without operand planes (the same bits);
  // its scratch must fit the region.
  size_t need = 0;
  backward_dev(ctx, make_devqw(*w), lora, d_x, d_dy, act_dtype, batch, d_t1, d_grad_x,
               d_grad_a, d_grad_b, nullptr, nullptr, &need);
  if (need > QH_NOALLOC_SCRATCH_BYTES)
    return fail(QH_ERR_INVALID_CONFIG,
                fmt("the call needs %zu bytes of scratch but the allocation-free backward has "
                    "%zu",
                    need, (size_t)QH_NOALLOC_SCRATCH_BYTES));
  return guarded(ctx, [&] {
    if (!ctx->noalloc)
      throw GpuError{std::string("no scratch region on this device: ") +
                     hipGetErrorString(ctx->noalloc_err)};
    NoTiming nt(ctx);
    ScratchSrc src{nullptr, (char *)ctx->noalloc, (size_t)QH_NOALLOC_SCRATCH_BYTES};
    backward_dev(ctx, make_devqw(*w), lora, d_x, d_dy, act_dtype, batch, d_t1, d_grad_x,
                 d_grad_a, d_grad_b, pick_stream(ctx, stream), &src);
    return QH_OK;
  });
}

// ---- Adam -------------------------------------------------------------------
void qh_adam_config_default(qh_adam_config *cfg) {
  if (!cfg) return;
  cfg->lr = 1e-3f;
  cfg->beta1 = 0.9f;
  cfg->beta2 = 0.999f;
  cfg->eps = 1e-8f;
  cfg->block_size = 256;
  cfg->max_resident_pages = SIZE_MAX;
}

qh_status qh_adam8bit_create(qh_ctx *ctx, const qh_adam_config *cfg,
                             qh_adam8bit **out) {
  if (!out || !cfg) return fail(QH_ERR_INVALID_CONFIG, "NULL argument");
  *out = nullptr;
  // optim.rs:63-80
  if (cfg->lr <= 0.0f || !std::isfinite(cfg->lr))
    return fail(QH_ERR_INVALID_CONFIG, "lr must be positive and finite");
  if (!(cfg->beta1 >= 0.0f && cfg->beta1 < 1.0f) || !(cfg->beta2 >= 0.0f && cfg->beta2 < 1.0f))
    return fail(QH_ERR_INVALID_CONFIG, "betas must be in (0, 1)");
  if (cfg->block_size == 0 || cfg->max_resident_pages == 0)
    return fail(QH_ERR_INVALID_CONFIG, "block_size and max_resident_pages must be > 0");
  if (cfg->block_size > 4096)
    return fail(QH_ERR_INVALID_CONFIG,
                "block_size > 4096 exceeds the GPU kernel's LDS staging");
  if (!ctx) return fail(QH_ERR_GPU, "context is NULL");
  qh_adam8bit *o = new (std::nothrow) qh_adam8bit();
  if (!o) return fail(QH_ERR_GPU, "host allocation failed");
  o->ctx = ctx;
  o->cfg = *cfg;
  *out = o;
  return QH_OK;
}

static void free_state(ParamStateDev &st) {
  if (st.m_codes) (void)hipFree(st.m_codes);
  if (st.v_codes) (void)hipFree(st.v_codes);
  if (st.m_scales) (void)hipFree(st.m_scales);
  if (st.v_scales) (void)hipFree(st.v_scales);
  st = ParamStateDev();
}

void qh_adam8bit_destroy(qh_adam8bit *o) {
  if (!o) return;
  (void)hipSetDevice(o->ctx->device);
  (void)hipStreamSynchronize(o->ctx->stream);
  for (auto &st : o->states) free_state(st);
  o->stage_p.release();
  o->stage_g.release();
  delete o;
}

static void init_state(ParamStateDev &st, size_t numel, size_t bs, hipStream_t s) {
  free_state(st);
  st.numel = numel;
  st.nb = div_ceil(numel, bs);
  check(hipMalloc(&st.m_codes, numel + 16), "hipMalloc");
  check(hipMalloc(&st.v_codes, numel + 16), "hipMalloc");
  check(hipMalloc(&st.m_scales, st.nb * 4 + 16), "hipMalloc");
  check(hipMalloc(&st.v_scales, st.nb * 4 + 16), "hipMalloc");
  check(hipMemsetAsync(st.m_codes, 0, numel + 16, s), "memset");
  check(hipMemsetAsync(st.v_codes, 0, numel + 16, s), "memset");
  check(hipMemsetAsync(st.m_scales, 0, st.nb * 4 + 16, s), "memset");
  check(hipMemsetAsync(st.v_scales, 0, st.nb * 4 + 16, s), "memset");
  st.step = 0;
}

// Adam8bit::step (optim.rs:164-199): tensors before the first length
// mismatch are stepped, then the mismatch is reported.
static qh_status adam_step_core(qh_adam8bit *o, float *const *d_params,
                                const float *const *d_grads, const size_t *lens,
                                size_t count, size_t mismatch_at,
                                qh_adam_stats *stats, hipStream_t s) {
  const qh_adam_config &c = o->cfg;
  std::vector<qh::AdamTensor> ts;
  size_t pages = 0;
  int64_t blocks = 0;
  for (size_t i = 0; i < count && i < mismatch_at; ++i) {
    if (o->states.size() <= i) o->states.emplace_back();
    ParamStateDev &st = o->states[i];
    if (st.m_codes == nullptr || st.numel != lens[i]) init_state(st, lens[i], c.block_size, s);
    st.step += 1;
    const float t = (float)st.step;
    qh::AdamTensor at;
    at.p = d_params[i];
    at.g = d_grads[i];
    at.m_codes = st.m_codes;
    at.v_codes = st.v_codes;
    at.m_scales = st.m_scales;
    at.v_scales = st.v_scales;
    at.numel = (int64_t)st.numel;
    at.nblocks = (int64_t)st.nb;
    at.block_offset = blocks;
    at.b1t = 1.0f - powf(c.beta1, t);  // optim.rs:209-210
    at.b2t = 1.0f - powf(c.beta2, t);
    at.inv_b1t = 1.0 / (double)at.b1t;
    at.inv_b2t = 1.0 / (double)at.b2t;
    blocks += at.nblocks;
    pages += st.nb;
    ts.push_back(at);
  }
  if (!ts.empty())
    timed(o->ctx, "adam", s, [&] {
      return qh::launch_adam(ts.data(), (int)ts.size(), blocks, (int64_t)c.block_size,
                             c.lr, c.beta1, c.beta2, c.eps, s);
    });
  if (stats) {
    stats->pages_streamed = pages;
    stats->state_bytes = qh_adam8bit_state_bytes(o);
  }
  return QH_OK;
}

qh_status qh_adam8bit_step(qh_adam8bit *o, float *const *params,
                           const size_t *param_lens, const float *const *grads,
                           const size_t *grad_lens, size_t count,
                           qh_adam_stats *stats) {
  if (!o) return fail(QH_ERR_INVALID_CONFIG, "optimizer is NULL");
  size_t mismatch = count;
  for (size_t i = 0; i < count; ++i)
    if (param_lens[i] != grad_lens[i]) {
      mismatch = i;
      break;
    }
  qh_ctx *ctx = o->ctx;
  qh_status st = guarded(ctx, [&] {
    hipStream_t s = ctx->stream;
    size_t tot = 0;
    for (size_t i = 0; i < mismatch; ++i) tot += param_lens[i];
    float *dp = (float *)o->stage_p.ensure(tot * 4 + 16);
    float *dg = (float *)o->stage_g.ensure(tot * 4 + 16);
    std::vector<float *> pp(mismatch);
    std::vector<const float *> gp(mismatch);
    size_t off = 0;
    for (size_t i = 0; i < mismatch; ++i) {
      pp[i] = dp + off;
      gp[i] = dg + off;
      if (param_lens[i]) {
        check(hipMemcpyAsync(pp[i], params[i], param_lens[i] * 4, hipMemcpyHostToDevice, s), "upload");
        check(hipMemcpyAsync((void *)gp[i], grads[i], param_lens[i] * 4, hipMemcpyHostToDevice, s), "upload");
      }
      off += (param_lens[i] + 3) / 4 * 4;
    }
    adam_step_core(o, pp.data(), gp.data(), param_lens, mismatch, mismatch, stats, s);
    for (size_t i = 0; i < mismatch; ++i)
      if (param_lens[i])
        check(hipMemcpyAsync(params[i], pp[i], param_lens[i] * 4, hipMemcpyDeviceToHost, s), "download");
    check(hipStreamSynchronize(s), "sync");
    return QH_OK;
  });
  if (st != QH_OK) return st;
  if (mismatch < count)
    return fail(QH_ERR_SHAPE_MISMATCH, fmt("param %zu: len = %zu but grad len = %zu", mismatch,
                                           param_lens[mismatch], grad_lens[mismatch]));
  return QH_OK;
}

qh_status qh_adam8bit_step_dev(qh_adam8bit *o, float *const *d_params,
                               const float *const *d_grads, const size_t *lens,
                               size_t count, qh_adam_stats *stats, void *stream) {
  if (!o) return fail(QH_ERR_INVALID_CONFIG, "optimizer is NULL");
  qh_ctx *ctx = o->ctx;
  return guarded(ctx, [&] {
    return adam_step_core(o, d_params, d_grads, lens, count, count, stats,
                          pick_stream(ctx, stream));
  });
}

size_t qh_adam8bit_state_bytes(const qh_adam8bit *o) {
  // optim.rs:128-131: m and v codes plus 4-byte scales for both.
  if (!o) return 0;
  size_t t = 0;
  for (const auto &st : o->states) t += 2 * st.numel + 2 * st.nb * 4;
  return t;
}

qh_status qh_adam8bit_get_state(qh_adam8bit *o, size_t idx, uint8_t *m_codes,
                                float *m_scales, uint8_t *v_codes, float *v_scales,
                                uint64_t *step) {
  if (!o) return fail(QH_ERR_INVALID_CONFIG, "optimizer is NULL");
  if (idx >= o->states.size()) return fail(QH_ERR_SHAPE_MISMATCH, "no state at this index");
  qh_ctx *ctx = o->ctx;
  return guarded(ctx, [&] {
    hipStream_t s = ctx->stream;
    const ParamStateDev &st = o->states[idx];
    check(hipStreamSynchronize(s), "sync");
    if (st.numel) {
      check(hipMemcpy(m_codes, st.m_codes, st.numel, hipMemcpyDeviceToHost), "download");
      check(hipMemcpy(v_codes, st.v_codes, st.numel, hipMemcpyDeviceToHost), "download");
      check(hipMemcpy(m_scales, st.m_scales, st.nb * 4, hipMemcpyDeviceToHost), "download");
      check(hipMemcpy(v_scales, st.v_scales, st.nb * 4, hipMemcpyDeviceToHost), "download");
    }
    if (step) *step = st.step;
    return QH_OK;
  });
}

// ---- the glue of a decoder block (qlora-model/src/llama.rs) -------------------
static qh_status check_rows(size_t len, size_t h, const char *what, size_t *rows) {
  if (h == 0) return fail(QH_ERR_SHAPE_MISMATCH, "hidden size (w.len()) is 0");
  if (h > (size_t)INT32_MAX) return fail(QH_ERR_INVALID_CONFIG, "hidden size above 2^31-1");
  if (len % h != 0)
    return fail(QH_ERR_SHAPE_MISMATCH,
                fmt("%s.len() = %zu is not a multiple of the hidden size %zu", what, len, h));
  *rows = len / h;
  return QH_OK;
}

static qh_status check_dev_rows(size_t rows, size_t h) {
  size_t n;
  if (h > (size_t)INT32_MAX) return fail(QH_ERR_INVALID_CONFIG, "hidden size above 2^31-1");
  if (mul_overflows(rows, h, &n)) return fail(QH_ERR_SHAPE_MISMATCH, "rows*h overflows");
  if (rows > 0 && h == 0) return fail(QH_ERR_SHAPE_MISMATCH, "hidden size is 0");
  return QH_OK;
}

static float *dw_scratch(qh_ctx *ctx, size_t rows, size_t h, hipStream_t s) {
  return (float *)ctx->scratch.ensure(qh::rmsnorm_dw_scratch_floats((int64_t)rows, (int)h) * 4,
                                      s);
}

qh_status qh_rmsnorm(qh_ctx *ctx, const float *x, size_t x_len, const float *w, size_t h,
                     float eps, float *y) {
  size_t rows;
  qh_status st = check_rows(x_len, h, "x", &rows);
  if (st != QH_OK) return st;
  return guarded(ctx, [&] {
    hipStream_t s = ctx->stream;
    float *dx = upload_f32(ctx, 0, x, x_len, s);
    float *dw = upload_f32(ctx, 1, w, h, s);
    timed(ctx, "rmsnorm", s, [&] {
      return qh::launch_rmsnorm(dx, dw, dx, (int64_t)rows, (int)h, eps, s);
    });
    download_f32(y, dx, x_len, s);
    check(hipStreamSynchronize(s), "sync");
    return QH_OK;
  });
}

qh_status qh_rmsnorm_dev(qh_ctx *ctx, const float *d_x, const float *d_w, size_t rows,
                         size_t h, float eps, float *d_y, void *stream) {
  qh_status st = check_dev_rows(rows, h);
  if (st != QH_OK) return st;
  return guarded(ctx, [&] {
    hipStream_t s = pick_stream(ctx, stream);
    timed(ctx, "rmsnorm", s, [&] {
      return qh::launch_rmsnorm(d_x, d_w, d_y, (int64_t)rows, (int)h, eps, s);
    });
    return QH_OK;
  });
}

qh_status qh_rmsnorm_backward(qh_ctx *ctx, const float *x, size_t x_len, const float *w,
                              size_t h, const float *dy, size_t dy_len, float eps, float *dx,
                              float *dw) {
  size_t rows;
  qh_status st = check_rows(x_len, h, "x", &rows);
  if (st != QH_OK) return st;
  if (dy_len != x_len)
    return fail(QH_ERR_SHAPE_MISMATCH, fmt("dy.len() = %zu but x.len() = %zu", dy_len, x_len));
  return guarded(ctx, [&] {
    hipStream_t s = ctx->stream;
    float *d_x = upload_f32(ctx, 0, x, x_len, s);
    float *d_w = upload_f32(ctx, 1, w, h, s);
    float *d_dy = upload_f32(ctx, 2, dy, dy_len, s);
    float *d_dw = dw ? alloc_f32(ctx, 3, h) : nullptr;
    // dx over dy only without dw: the dw stage reads dy after dx is written
    float *d_dx = dw ? alloc_f32(ctx, 4, x_len) : d_dy;
    float *scr = dw ? dw_scratch(ctx, rows, h, s) : nullptr;
    timed(ctx, "rmsnorm_backward", s, [&] {
      return qh::launch_rmsnorm_bwd(d_x, d_w, d_dy, d_dx, d_dw, scr, (int64_t)rows, (int)h,
                                    eps, s);
    });
    download_f32(dx, d_dx, x_len, s);
    if (dw) download_f32(dw, d_dw, h, s);
    check(hipStreamSynchronize(s), "sync");
    return QH_OK;
  });
}

qh_status qh_rmsnorm_backward_dev(qh_ctx *ctx, const float *d_x, const float *d_w,
                                  const float *d_dy, size_t rows, size_t h, float eps,
                                  float *d_dx, float *d_dw, void *stream) {
  qh_status st = check_dev_rows(rows, h);
  if (st != QH_OK) return st;
  if (d_dw && rows > 0 && d_dx == d_dy)
    return fail(QH_ERR_INVALID_CONFIG, "dx may alias dy only when dw is not requested");
  return guarded(ctx, [&] {
    hipStream_t s = pick_stream(ctx, stream);
    float *scr = d_dw ? dw_scratch(ctx, rows, h, s) : nullptr;
    timed(ctx, "rmsnorm_backward", s, [&] {
      return qh::launch_rmsnorm_bwd(d_x, d_w, d_dy, d_dx, d_dw, scr, (int64_t)rows, (int)h,
                                    eps, s);
    });
    return QH_OK;
  });
}

qh_status qh_swiglu(qh_ctx *ctx, const float *gate, size_t gate_len, const float *up,
                    size_t up_len, float *act) {
  if (gate_len != up_len)
    return fail(QH_ERR_SHAPE_MISMATCH,
                fmt("gate.len() = %zu but up.len() = %zu", gate_len, up_len));
  return guarded(ctx, [&] {
    hipStream_t s = ctx->stream;
    float *d_g = upload_f32(ctx, 0, gate, gate_len, s);
    float *d_u = upload_f32(ctx, 1, up, up_len, s);
    timed(ctx, "swiglu", s, [&] { return qh::launch_swiglu(d_g, d_u, d_g, (int64_t)gate_len, s); });
    download_f32(act, d_g, gate_len, s);
    check(hipStreamSynchronize(s), "sync");
    return QH_OK;
  });
}

qh_status qh_swiglu_dev(qh_ctx *ctx, const float *d_gate, const float *d_up, size_t n,
                        float *d_act, void *stream) {
  return guarded(ctx, [&] {
    hipStream_t s = pick_stream(ctx, stream);
    timed(ctx, "swiglu", s, [&] { return qh::launch_swiglu(d_gate, d_up, d_act, (int64_t)n, s); });
    return QH_OK;
  });
}

qh_status qh_swiglu_backward(qh_ctx *ctx, const float *gate, const float *up,
                             const float *d_act, size_t n, float *dg, float *du) {
  return guarded(ctx, [&] {
    hipStream_t s = ctx->stream;
    float *d_g = upload_f32(ctx, 0, gate, n, s);
    float *d_u = upload_f32(ctx, 1, up, n, s);
    float *d_a = upload_f32(ctx, 2, d_act, n, s);
    timed(ctx, "swiglu_backward", s, [&] {
      return qh::launch_swiglu_bwd(d_g, d_u, d_a, d_g, d_u, (int64_t)n, s);
    });
    download_f32(dg, d_g, n, s);
    download_f32(du, d_u, n, s);
    check(hipStreamSynchronize(s), "sync");
    return QH_OK;
  });
}

qh_status qh_swiglu_backward_dev(qh_ctx *ctx, const float *d_gate, const float *d_up,
                                 const float *d_act, size_t n, float *d_dg, float *d_du,
                                 void *stream) {
  return guarded(ctx, [&] {
    hipStream_t s = pick_stream(ctx, stream);
    timed(ctx, "swiglu_backward", s, [&] {
      return qh::launch_swiglu_bwd(d_gate, d_up, d_act, d_dg, d_du, (int64_t)n, s);
    });
    return QH_OK;
  });
}

static qh_status check_ce(size_t seq, size_t vocab) {
  size_t n;
  if (mul_overflows(seq, vocab, &n)) return fail(QH_ERR_SHAPE_MISMATCH, "seq*vocab overflows");
  if (seq > 0 && vocab == 0) return fail(QH_ERR_SHAPE_MISMATCH, "vocab is 0");
  if (seq > (size_t)INT32_MAX) return fail(QH_ERR_INVALID_CONFIG, "seq above 2^31-1");
  return QH_OK;
}

qh_status qh_softmax_cross_entropy(qh_ctx *ctx, const float *logits, size_t logits_len,
                                   const uint32_t *targets, size_t seq, size_t vocab,
                                   float *loss, float *dlogits) {
  qh_status st = check_ce(seq, vocab);
  if (st != QH_OK) return st;
  if (logits_len != seq * vocab)
    return fail(QH_ERR_SHAPE_MISMATCH,
                fmt("logits.len() = %zu but seq*vocab = %zu", logits_len, seq * vocab));
  for (size_t t = 0; t < seq; t++)
    if ((size_t)targets[t] >= vocab)
      return fail(QH_ERR_SHAPE_MISMATCH,
                  fmt("target %u at position %zu is out of range for vocab %zu", targets[t], t,
                      vocab));
  return guarded(ctx, [&] {
    hipStream_t s = ctx->stream;
    float *d_l = upload_f32(ctx, 0, logits, logits_len, s);
    uint32_t *d_t = (uint32_t *)ctx->stage[1].ensure(seq * 4 + 16);
    if (seq) check(hipMemcpyAsync(d_t, targets, seq * 4, hipMemcpyHostToDevice, s), "upload");
    float *d_loss = alloc_f32(ctx, 2, 1);
    float *terms = (float *)ctx->scratch.ensure(seq * 4 + 16, s);
    timed(ctx, "softmax_cross_entropy", s, [&] {
      return qh::launch_softmax_ce(d_l, d_t, (int64_t)seq, (int64_t)vocab, d_loss, d_l, terms, s);
    });
    download_f32(dlogits, d_l, logits_len, s);
    download_f32(loss, d_loss, 1, s);
    check(hipStreamSynchronize(s), "sync");
    return QH_OK;
  });
}

qh_status qh_softmax_cross_entropy_dev(qh_ctx *ctx, const float *d_logits,
                                       const uint32_t *d_targets, size_t seq, size_t vocab,
                                       float *d_loss, float *d_dlogits, void *stream) {
  qh_status st = check_ce(seq, vocab);
  if (st != QH_OK) return st;
  return guarded(ctx, [&] {
    hipStream_t s = pick_stream(ctx, stream);
    float *terms = (float *)ctx->scratch.ensure(seq * 4 + 16, s);
    timed(ctx, "softmax_cross_entropy", s, [&] {
      return qh::launch_softmax_ce(d_logits, d_targets, (int64_t)seq, (int64_t)vocab, d_loss,
                                   d_dlogits, terms, s);
    });
    return QH_OK;
  });
}

// ---- packed NF4 files: host views into HBM ------------------------------------
qh_status qh_weight_upload_dev(qh_ctx *ctx, const qh_qweight *w, uint8_t *d_codes,
                               float *d_scales, uint8_t *d_scale_codes, float *d_absmax,
                               void *stream) {
  qh_status st = validate_weight(w);
  if (st != QH_OK) return st;
  const bool dq = w->scale_kind == QH_SCALES_DQ_INT8;
  if (!d_codes || (dq ? (!d_scale_codes || !d_absmax) : !d_scales))
    return fail(QH_ERR_SHAPE_MISMATCH, "a device buffer for the weight's parts is NULL");
  return guarded(ctx, [&] {
    hipStream_t s = pick_stream(ctx, stream);
    const size_t n = w->rows * w->cols, nb = div_ceil(n, w->block_size);
    if (n) check(hipMemcpyAsync(d_codes, w->codes, div_ceil(n, 2), hipMemcpyHostToDevice, s),
                 "upload codes");
    if (dq) {
      if (nb) check(hipMemcpyAsync(d_scale_codes, w->scale_codes, nb, hipMemcpyHostToDevice, s),
                    "upload scale codes");
      if (nb) check(hipMemcpyAsync(d_absmax, w->absmax, div_ceil(nb, 256) * 4,
                                   hipMemcpyHostToDevice, s), "upload absmax");
    } else if (nb) {
      check(hipMemcpyAsync(d_scales, w->scales, nb * 4, hipMemcpyHostToDevice, s),
            "upload scales");
    }
    return QH_OK;
  });
}

// ---- a decoder block's MLP on device (qlora-model llama.rs) --------------------
static qh_status validate_mlp(const qh_mlp_block *b) {
  if (!b) return fail(QH_ERR_SHAPE_MISMATCH, "block descriptor is NULL");
  const size_t h = b->hidden, f = b->inter;
  if (h == 0 || f == 0) return fail(QH_ERR_SHAPE_MISMATCH, "hidden and inter must be > 0");
  if (h > (size_t)INT32_MAX) return fail(QH_ERR_INVALID_CONFIG, "hidden size above 2^31-1");
  if (!b->norm_w) return fail(QH_ERR_SHAPE_MISMATCH, "norm weight is NULL");
  qh_status st;
  const qh_qweight *ws[3] = {&b->gate, &b->up, &b->down};
  const qh_lora *ls[3] = {b->gate_lora, b->up_lora, b->down_lora};
  const size_t rows[3] = {f, f, h}, cols[3] = {h, h, f};
  const char *nm[3] = {"gate", "up", "down"};
  for (int i = 0; i < 3; ++i) {
    if ((st = validate_weight(ws[i])) != QH_OK) return st;
    if (ws[i]->rows != rows[i] || ws[i]->cols != cols[i])
      return fail(QH_ERR_SHAPE_MISMATCH,
                  fmt("%s weight is %zu x %zu but the block needs %zu x %zu", nm[i], ws[i]->rows,
                      ws[i]->cols, rows[i], cols[i]));
    if ((st = validate_lora(ls[i], cols[i], rows[i])) != QH_OK) return st;
  }
  return QH_OK;
}

static qh_status validate_cache(const qh_mlp_block *b, const qh_mlp_cache *c) {
  if (!c || !c->x_mid || !c->xn || !c->gate || !c->up || !c->act)
    return fail(QH_ERR_SHAPE_MISMATCH, "cache buffers must not be NULL");
  return QH_OK;
}

qh_status qh_mlp_forward_dev(qh_ctx *ctx, const qh_mlp_block *b, float *d_x, size_t seq,
                             const qh_mlp_cache *c, void *stream) {
  qh_status st = validate_mlp(b);
  if (st != QH_OK) return st;
  if ((st = validate_cache(b, c)) != QH_OK) return st;
  return guarded(ctx, [&] {
    if (seq == 0) return QH_OK;
    hipStream_t s = pick_stream(ctx, stream);
    const size_t h = b->hidden, f = b->inter;
    // llama.rs:449-463: xn = rmsnorm(x); gate, up; act = silu(gate) * up;
    // x += down(act).  The block input is kept for the backward's norm (the
    // norm kernel writes the copy as it reads x).
    timed(ctx, "rmsnorm", s, [&] {
      return qh::launch_rmsnorm(d_x, b->norm_w, c->xn, (int64_t)seq, (int)h, b->eps, s,
                                c->x_mid);
    });
    {
      const DevQW W[2] = {make_devqw(b->gate), make_devqw(b->up)};
      const qh_lora *L[2] = {b->gate_lora, b->up_lora};
      float *Y[2] = {c->gate, c->up};
      float *T[2] = {b->gate_lora ? c->t1_gate : nullptr, b->up_lora ? c->t1_up : nullptr};
      forward_shared_dev(ctx, 2, W, L, c->xn, QH_F32, seq, Y, T, s);
    }
    timed(ctx, "swiglu", s, [&] {
      return qh::launch_swiglu(c->gate, c->up, c->act, (int64_t)(seq * f), s);
    });
    forward_add_dev(ctx, make_devqw(b->down), b->down_lora, c->act, QH_F32, seq, d_x,
                    b->down_lora ? c->t1_down : nullptr, ctx->block_tmp[0], s);
    return QH_OK;
  });
}

qh_status qh_mlp_backward_dev(qh_ctx *ctx, const qh_mlp_block *b, const qh_mlp_cache *c,
                              const float *d_dx_out, size_t seq, float *d_dx_in,
                              float *const *d_grad_a, float *const *d_grad_b, void *stream) {
  qh_status st = validate_mlp(b);
  if (st != QH_OK) return st;
  if ((st = validate_cache(b, c)) != QH_OK) return st;
  if (d_dx_in == d_dx_out && seq > 0)
    return fail(QH_ERR_INVALID_CONFIG, "dx_in must not alias dx_out (read at the end)");
  const qh_lora *ls[3] = {b->gate_lora, b->up_lora, b->down_lora};
  for (int i = 0; i < 3; ++i)
    if (ls[i] && (!d_grad_a || !d_grad_b || !d_grad_a[i] || !d_grad_b[i]))
      return fail(QH_ERR_SHAPE_MISMATCH, "an adapter's gradient buffer is NULL");
  return guarded(ctx, [&] {
    if (seq == 0) return QH_OK;
    hipStream_t s = pick_stream(ctx, stream);
    const size_t h = b->hidden, f = b->inter;
    // llama.rs:554-574 (MLP branch of block_backward)
    float *d_act = (float *)ctx->block_tmp[0].ensure(seq * f * 4, s);
    backward_dev(ctx, make_devqw(b->down), b->down_lora, c->act, d_dx_out, QH_F32, seq,
                 b->down_lora ? c->t1_down : nullptr, d_act,
                 b->down_lora ? d_grad_a[2] : nullptr, b->down_lora ? d_grad_b[2] : nullptr, s);
    // dg over the cached gate, du over the cached up (the cache is consumed)
    timed(ctx, "swiglu_backward", s, [&] {
      return qh::launch_swiglu_bwd(c->gate, c->up, d_act, c->gate, c->up, (int64_t)(seq * f), s);
    });
    {
      // dxn = dxn_gate + dxn_up (llama.rs:563-567)
      const DevQW W[2] = {make_devqw(b->gate), make_devqw(b->up)};
      const qh_lora *L[2] = {b->gate_lora, b->up_lora};
      const void *DY[2] = {c->gate, c->up};
      const float *T[2] = {b->gate_lora ? c->t1_gate : nullptr, b->up_lora ? c->t1_up : nullptr};
      float *GA[2] = {b->gate_lora ? d_grad_a[0] : nullptr, b->up_lora ? d_grad_a[1] : nullptr};
      float *GB[2] = {b->gate_lora ? d_grad_b[0] : nullptr, b->up_lora ? d_grad_b[1] : nullptr};
      backward_shared_dev(ctx, 2, W, L, c->xn, DY, QH_F32, seq, T, d_dx_in, GA, GB, s);
    }
    // dx_mid = rmsnorm_backward(x_mid, w, dxn).dx + dx_out (dw is discarded,
    // llama.rs:568): the residual added by the norm kernel as it writes dx
    timed(ctx, "rmsnorm_backward", s, [&] {
      return qh::launch_rmsnorm_bwd(c->x_mid, b->norm_w, d_dx_in, d_dx_in, nullptr, nullptr,
                                    (int64_t)seq, (int)h, b->eps, s, d_dx_out);
    });
    return QH_OK;
  });
}

// ---- a decoder block's attention projections on device (llama.rs) -------------
static qh_status validate_attn(const qh_attn_block *b) {
  if (!b) return fail(QH_ERR_SHAPE_MISMATCH, "block descriptor is NULL");
  const size_t h = b->hidden, kv = b->kv_dim;
  if (h == 0 || kv == 0) return fail(QH_ERR_SHAPE_MISMATCH, "hidden and kv_dim must be > 0");
  if (h > (size_t)INT32_MAX) return fail(QH_ERR_INVALID_CONFIG, "hidden size above 2^31-1");
  if (!b->norm_w) return fail(QH_ERR_SHAPE_MISMATCH, "norm weight is NULL");
  qh_status st;
  const qh_qweight *ws[4] = {&b->q, &b->k, &b->v, &b->o};
  const qh_lora *ls[4] = {b->q_lora, b->k_lora, b->v_lora, b->o_lora};
  const size_t rows[4] = {h, kv, kv, h};
  const char *nm[4] = {"q", "k", "v", "o"};
  for (int i = 0; i < 4; ++i) {
    if ((st = validate_weight(ws[i])) != QH_OK) return st;
    if (ws[i]->rows != rows[i] || ws[i]->cols != h)
      return fail(QH_ERR_SHAPE_MISMATCH,
                  fmt("%s weight is %zu x %zu but the block needs %zu x %zu", nm[i], ws[i]->rows,
                      ws[i]->cols, rows[i], h));
    if ((st = validate_lora(ls[i], h, rows[i])) != QH_OK) return st;
  }
  return QH_OK;
}

static qh_status validate_attn_cache(const qh_attn_cache *c) {
  if (!c || !c->x_in || !c->xn || !c->attn)
    return fail(QH_ERR_SHAPE_MISMATCH, "cache buffers must not be NULL");
  return QH_OK;
}

qh_status qh_attn_qkv_forward_dev(qh_ctx *ctx, const qh_attn_block *b, const float *d_x,
                                  size_t seq, const qh_attn_cache *c, float *d_q, float *d_k,
                                  float *d_v, void *stream) {
  qh_status st = validate_attn(b);
  if (st != QH_OK) return st;
  if ((st = validate_attn_cache(c)) != QH_OK) return st;
  if (seq > 0 && (!d_x || !d_q || !d_k || !d_v))
    return fail(QH_ERR_SHAPE_MISMATCH, "x, q, k and v must not be NULL");
  return guarded(ctx, [&] {
    if (seq == 0) return QH_OK;
    hipStream_t s = pick_stream(ctx, stream);
    const size_t h = b->hidden;
    // llama.rs:426-434: the block input kept (written by the norm kernel as
    // it reads x), xn = rmsnorm(x), q, k, v of xn
    timed(ctx, "rmsnorm", s, [&] {
      return qh::launch_rmsnorm(d_x, b->norm_w, c->xn, (int64_t)seq, (int)h, b->eps, s,
                                c->x_in);
    });
    const DevQW W[3] = {make_devqw(b->q), make_devqw(b->k), make_devqw(b->v)};
    const qh_lora *L[3] = {b->q_lora, b->k_lora, b->v_lora};
    float *Y[3] = {d_q, d_k, d_v};
    float *T[3] = {b->q_lora ? c->t1_q : nullptr, b->k_lora ? c->t1_k : nullptr,
                   b->v_lora ? c->t1_v : nullptr};
    forward_shared_dev(ctx, 3, W, L, c->xn, QH_F32, seq, Y, T, s);
    return QH_OK;
  });
}

qh_status qh_attn_o_forward_dev(qh_ctx *ctx, const qh_attn_block *b, float *d_x, size_t seq,
                                const qh_attn_cache *c, void *stream) {
  qh_status st = validate_attn(b);
  if (st != QH_OK) return st;
  if ((st = validate_attn_cache(c)) != QH_OK) return st;
  if (seq > 0 && !d_x) return fail(QH_ERR_SHAPE_MISMATCH, "x must not be NULL");
  return guarded(ctx, [&] {
    if (seq == 0) return QH_OK;
    hipStream_t s = pick_stream(ctx, stream);
    // llama.rs:436-439: x += o(attn)
    forward_add_dev(ctx, make_devqw(b->o), b->o_lora, c->attn, QH_F32, seq, d_x,
                    b->o_lora ? c->t1_o : nullptr, ctx->block_tmp[0], s);
    return QH_OK;
  });
}

qh_status qh_attn_o_backward_dev(qh_ctx *ctx, const qh_attn_block *b, const qh_attn_cache *c,
                                 const float *d_dx_mid, size_t seq, float *d_dattn,
                                 float *d_grad_a_o, float *d_grad_b_o, void *stream) {
  qh_status st = validate_attn(b);
  if (st != QH_OK) return st;
  if ((st = validate_attn_cache(c)) != QH_OK) return st;
  if (seq > 0 && (!d_dx_mid || !d_dattn))
    return fail(QH_ERR_SHAPE_MISMATCH, "dx_mid and dattn must not be NULL");
  if (b->o_lora && (!d_grad_a_o || !d_grad_b_o))
    return fail(QH_ERR_SHAPE_MISMATCH, "an adapter's gradient buffer is NULL");
  return guarded(ctx, [&] {
    if (seq == 0) return QH_OK;
    hipStream_t s = pick_stream(ctx, stream);
    // llama.rs:577: (o_ab, d_attn) = proj_backward(o, attn_out, dx_mid)
    backward_dev(ctx, make_devqw(b->o), b->o_lora, c->attn, d_dx_mid, QH_F32, seq,
                 b->o_lora ? c->t1_o : nullptr, d_dattn, b->o_lora ? d_grad_a_o : nullptr,
                 b->o_lora ? d_grad_b_o : nullptr, s);
    return QH_OK;
  });
}

qh_status qh_attn_qkv_backward_dev(qh_ctx *ctx, const qh_attn_block *b, const qh_attn_cache *c,
                                   const float *d_dq, const float *d_dk, const float *d_dv,
                                   const float *d_dx_mid, size_t seq, float *d_dx_in,
                                   float *const *d_grad_a, float *const *d_grad_b,
                                   void *stream) {
  qh_status st = validate_attn(b);
  if (st != QH_OK) return st;
  if ((st = validate_attn_cache(c)) != QH_OK) return st;
  if (seq > 0 && (!d_dq || !d_dk || !d_dv || !d_dx_mid || !d_dx_in))
    return fail(QH_ERR_SHAPE_MISMATCH, "dq, dk, dv, dx_mid and dx_in must not be NULL");
  if (d_dx_in == d_dx_mid && seq > 0)
    return fail(QH_ERR_INVALID_CONFIG, "dx_in must not alias dx_mid (read at the end)");
  const qh_lora *ls[3] = {b->q_lora, b->k_lora, b->v_lora};
  for (int i = 0; i < 3; ++i)
    if (ls[i] && (!d_grad_a || !d_grad_b || !d_grad_a[i] || !d_grad_b[i]))
      return fail(QH_ERR_SHAPE_MISMATCH, "an adapter's gradient buffer is NULL");
  return guarded(ctx, [&] {
    if (seq == 0) return QH_OK;
    hipStream_t s = pick_stream(ctx, stream);
    const size_t h = b->hidden;
    // llama.rs:580-601: dxn = (dxn_q + dxn_k) + dxn_v, then the norm's dx and
    // the residual's straight path
    const DevQW W[3] = {make_devqw(b->q), make_devqw(b->k), make_devqw(b->v)};
    const qh_lora *L[3] = {b->q_lora, b->k_lora, b->v_lora};
    const void *DY[3] = {d_dq, d_dk, d_dv};
    const float *T[3] = {b->q_lora ? c->t1_q : nullptr, b->k_lora ? c->t1_k : nullptr,
                         b->v_lora ? c->t1_v : nullptr};
    float *GA[3], *GB[3];
    for (int i = 0; i < 3; ++i) {
      GA[i] = L[i] ? d_grad_a[i] : nullptr;
      GB[i] = L[i] ? d_grad_b[i] : nullptr;
    }
    backward_shared_dev(ctx, 3, W, L, c->xn, DY, QH_F32, seq, T, d_dx_in, GA, GB, s);
    // dx_in = dx_norm + dx_mid (llama.rs:596-601; a + b rounds as b + a),
    // the residual added by the norm kernel as it writes dx
    timed(ctx, "rmsnorm_backward", s, [&] {
      return qh::launch_rmsnorm_bwd(c->x_in, b->norm_w, d_dx_in, d_dx_in, nullptr, nullptr,
                                    (int64_t)seq, (int)h, b->eps, s, d_dx_mid);
    });
    return QH_OK;
  });
}

// ---- library-owned device weights ---------------------------------------------
qh_status qh_weight_upload(qh_ctx *ctx, const qh_qweight *host, qh_dweight **out) {
  if (!out) return fail(QH_ERR_SHAPE_MISMATCH, "out is NULL");
  *out = nullptr;
  qh_status st = validate_weight(host);
  if (st != QH_OK) return st;
  const bool dq = host->scale_kind == QH_SCALES_DQ_INT8;
  const size_t n = host->rows * host->cols, nb = div_ceil(n, host->block_size);
  if (n && (!host->codes || (dq ? (!host->scale_codes || !host->absmax) : !host->scales)))
    return fail(QH_ERR_SHAPE_MISMATCH, "a part of the host weight is NULL");
  qh_dweight *d = new (std::nothrow) qh_dweight();
  if (!d) return fail(QH_ERR_GPU, "host allocation failed");
  d->ctx = ctx;
  st = guarded(ctx, [&] {
    const size_t cb = div_ceil(n, 2), sb = dq ? nb : nb * 4, ab = dq ? div_ceil(nb, 256) * 4 : 0;
    check(hipMalloc(&d->codes, cb ? cb : 1), "hipMalloc codes");
    check(hipMalloc(&d->scales, sb ? sb : 1), "hipMalloc scales");
    if (dq) check(hipMalloc(&d->absmax, ab ? ab : 4), "hipMalloc absmax");
    hipStream_t s = ctx->stream;
    if (cb) check(hipMemcpyAsync(d->codes, host->codes, cb, hipMemcpyHostToDevice, s), "upload");
    if (sb)
      check(hipMemcpyAsync(d->scales, dq ? (const void *)host->scale_codes : host->scales, sb,
                           hipMemcpyHostToDevice, s), "upload");
    if (ab) check(hipMemcpyAsync(d->absmax, host->absmax, ab, hipMemcpyHostToDevice, s), "upload");
    check(hipStreamSynchronize(s), "sync");
    return QH_OK;
  });
  if (st != QH_OK) {
    qh_dweight_destroy(d);
    return st;
  }
  d->view = *host;
  d->view.codes = (const uint8_t *)d->codes;
  d->view.scales = dq ? nullptr : (const float *)d->scales;
  d->view.scale_codes = dq ? (const uint8_t *)d->scales : nullptr;
  d->view.absmax = dq ? (const float *)d->absmax : nullptr;
  *out = d;
  return QH_OK;
}

qh_status qh_dweight_view(const qh_dweight *w, qh_qweight *view) {
  if (!w || !view) return fail(QH_ERR_SHAPE_MISMATCH, "weight handle or view is NULL");
  *view = w->view;
  return QH_OK;
}

void qh_dweight_destroy(qh_dweight *w) {
  if (!w) return;
  if (w->ctx) {
    std::lock_guard<std::mutex> lk(w->ctx->mu);
    (void)hipSetDevice(w->ctx->device);
    if (w->codes) (void)hipFree(w->codes);
    if (w->scales) (void)hipFree(w->scales);
    if (w->absmax) (void)hipFree(w->absmax);
  }
  delete w;
}

}  // extern "C"

namespace qh {
qh_status host_fail(qh_status st, const std::string &msg) { return fail(st, msg); }
}  // namespace qh
