/*
 * qlora_hip.h -- C ABI of the MI355X (gfx950) QloraLinear hot path.
 *
 * Drop-in boundary for stuarch/VkQLoRA.rs `qlora-wgpu` (the GPU backend of
 * the QLoRA linear layer) plus GPU versions of the two CPU-only pieces of
 * `qlora-core` it is used with: `QuantizedTensor::quantize` and
 * `Adam8bit::step`.  Every entry point names the reference interface it
 * replaces (paths relative to the reference tree).
 *
 * Conventions
 *  - Plain pointers and sizes only.  Host-memory entry points take
 *    borrowed host slices plus their lengths, validate them with the
 *    reference's rules and messages, run on the GPU and return only when
 *    the result is in the caller's buffers (the reference blocks in
 *    `pollster::block_on` / `device.poll(Wait)`: qlora-wgpu/src/context.rs:34,
 *    kernels.rs:413).
 *  - `*_dev` entry points take device pointers that are already resident in
 *    HBM, enqueue on `stream` (a hipStream_t; NULL = the HIP null stream)
 *    and return without synchronising.  Sizes are trusted.
 *  - The caller allocates every output at its exact size.  Opaque handles
 *    (qh_ctx, qh_adam8bit) are the only library-owned memory.
 *  - Errors never cross the ABI as exceptions: every call returns a
 *    qh_status whose values map 1:1 onto `QloraError`
 *    (qlora-core/src/error.rs:6-14), and qh_last_error() returns the
 *    message in the reference's Display format ("shape mismatch: ...",
 *    "invalid config: ...", "gpu error: ...", error.rs:16-24).
 *  - A qh_ctx may be shared between threads; calls on one context are
 *    serialised by a mutex inside it.
 */
#ifndef QLORA_HIP_H
#define QLORA_HIP_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define QH_API __attribute__((visibility("default")))
#define QH_ABI_VERSION 1u

typedef enum qh_status {
  QH_OK = 0,
  QH_ERR_SHAPE_MISMATCH = 1, /* QloraError::ShapeMismatch (error.rs:8) */
  QH_ERR_INVALID_CONFIG = 2, /* QloraError::InvalidConfig (error.rs:10) */
  QH_ERR_GPU = 3,            /* QloraError::Gpu (error.rs:12) */
  QH_NO_DEVICE = 4, /* try_new_blocking() -> Ok(None) (context.rs:50-53) */
  QH_ERR_MALFORMED = 5,  /* qlora-io IoError::Malformed (qlora-io/src/error.rs:8) */
  QH_ERR_UNSUPPORTED = 6 /* qlora-io IoError::Unsupported (error.rs:10) */
} qh_status;

/* Scale storage of a quantized weight: `ScaleStore` (quant.rs:84-89). */
typedef enum qh_scale_kind {
  QH_SCALES_F32 = 0,     /* ScaleStore::F32: one fp32 absmax per block */
  QH_SCALES_DQ_INT8 = 1  /* ScaleStore::Int8: i8 code per block, fp32
                            absmax per 256 blocks (double quantization) */
} qh_scale_kind;

typedef enum qh_dtype { QH_F32 = 0, QH_BF16 = 1 } qh_dtype;

typedef enum qh_matmul_op {
  QH_MM_NN = 0, /* C(m,n) = A(m,k) B(k,n)        lora.rs:129-142 */
  QH_MM_TN = 1, /* C(k,n) = A(m,k)^T B(m,n)      lora.rs:148-162 */
  QH_MM_NT = 2  /* C(m,n) = A(m,k) B(n,k)^T      lora.rs:169-183 */
} qh_matmul_op;

/* A row-major (rows x cols) NF4 weight: `QuantizedTensor` (quant.rs:93-100).
 * codes: ceil(n/2) bytes, element 2i in the low nibble of byte i.
 * F32 scales: `scales`, ceil(n/block_size) floats.
 * DQ scales:  `scale_codes` (i8 bit-cast to u8), ceil(n/block_size) bytes,
 *             and `absmax`, ceil(num_blocks/256) floats. */
typedef struct qh_qweight {
  size_t rows, cols, block_size;
  const uint8_t *codes;
  int32_t scale_kind; /* qh_scale_kind */
  const float *scales;
  const uint8_t *scale_codes;
  const float *absmax;
} qh_qweight;

/* `LoraAdapter` (lora.rs:16-24): A (r x in_dim), B (out_dim x r), row-major,
 * scale alpha / r (lora.rs:64-66).  Pass NULL for "no adapter". */
typedef struct qh_lora {
  const float *a;
  size_t a_len;
  const float *b;
  size_t b_len;
  size_t r;
  float alpha;
} qh_lora;

typedef struct qh_ctx qh_ctx;

/* ---- context: GpuContext (qlora-wgpu/src/context.rs:18-115) ------------ */
QH_API uint32_t qh_abi_version(void);
/* GpuContext::try_new_blocking (context.rs:33).  QH_NO_DEVICE when no
 * MI355X is visible (*out stays NULL), QH_ERR_GPU on runtime failure. */
QH_API qh_status qh_ctx_create(qh_ctx **out);
/* Gives back the device memory that the context's calls grew it to: scratch of
 * the largest call, and from the first call with large GEMMs on their operand
 * planes, up to 2 GiB.  Destroy HIP graphs captured on the context first: they
 * hold addresses in that memory. */
QH_API void qh_ctx_destroy(qh_ctx *ctx);
/* Message of the last failing call on this thread ("" if none). */
QH_API const char *qh_last_error(void);
/* Device name / gfx arch of the context's GPU. */
QH_API qh_status qh_ctx_device_name(qh_ctx *ctx, char *buf, size_t len);
/* Wait for all work on the context's stream. */
QH_API qh_status qh_ctx_synchronize(qh_ctx *ctx);
/* Kernel timing (no counterpart in the reference, whose dispatches carry
 * no timestamps: kernels.rs:383).  While enabled, every hot-path kernel
 * launch is bracketed by HIP events recorded on its own stream.  The report
 * waits for those events and writes one line per kernel name:
 * "<name> <launches> <total_ms>\n"; `reset` clears the totals. */
QH_API qh_status qh_ctx_set_timing(qh_ctx *ctx, int enable);
QH_API qh_status qh_ctx_timing_report(qh_ctx *ctx, char *buf, size_t len,
                                      int reset);
/* Test hooks (no counterpart in the reference): flags that force the rare
 * paths of the kernels from the host so that tests can check them.
 * QH_TEST_FORCE_T1_RECOMPUTE: the one-launch decode GEMV takes the path of a
 * workgroup whose awaited T1 slices never arrive (it computes them itself),
 * which must give the same bits as the normal path.  Products leave the
 * flags at 0 (their value after qh_ctx_create). */
#define QH_TEST_FORCE_T1_RECOMPUTE 1u
QH_API qh_status qh_ctx_set_test_flags(qh_ctx *ctx, uint32_t flags);

/* ---- layout helpers (quant.rs:93-100, 223-257) ------------------------- */
QH_API size_t qh_codes_len(size_t rows, size_t cols);
QH_API size_t qh_num_blocks(size_t rows, size_t cols, size_t block_size);
QH_API size_t qh_num_absmax(size_t rows, size_t cols, size_t block_size);
/* QuantizedTensor::storage_bytes (quant.rs:229-235). */
QH_API size_t qh_storage_bytes(const qh_qweight *w);

/* ---- quantization ------------------------------------------------------ */
/* QuantizedTensor::quantize (quant.rs:104-154) with nearest_nf4_code
 * (:263-278) and double_quantize_scales (:283-299).  Bit-exact.
 * double_quant == 0 fills `scales`; otherwise `scale_codes` and `absmax`. */
QH_API qh_status qh_quantize_nf4(qh_ctx *ctx, const float *w, size_t w_len,
                                 size_t rows, size_t cols, size_t block_size,
                                 int double_quant, uint8_t *codes,
                                 float *scales, uint8_t *scale_codes,
                                 float *absmax);
/* QuantizedTensor::block_scales (quant.rs:212-221): decoded fp32 scales. */
QH_API qh_status qh_block_scales(qh_ctx *ctx, const qh_qweight *w,
                                 float *out);
/* gpu_dequantize (qlora-wgpu/src/kernels.rs:44-103) ==
 * QuantizedTensor::dequantize (quant.rs:157-167).  Bit-exact fp32. */
QH_API qh_status qh_dequantize(qh_ctx *ctx, const qh_qweight *w, float *out);

/* ---- GEMMs: gpu_matmul{,_trans_a,_trans_b} (kernels.rs:140-257) -------- */
QH_API qh_status qh_matmul(qh_ctx *ctx, const float *a, size_t a_len,
                           const float *b, size_t b_len, size_t m, size_t k,
                           size_t n, float *c);
QH_API qh_status qh_matmul_trans_a(qh_ctx *ctx, const float *a, size_t a_len,
                                   const float *b, size_t b_len, size_t m,
                                   size_t k, size_t n, float *c);
QH_API qh_status qh_matmul_trans_b(qh_ctx *ctx, const float *a, size_t a_len,
                                   const float *b, size_t b_len, size_t m,
                                   size_t k, size_t n, float *c);

/* ---- the layer ---------------------------------------------------------- */
/* gpu_qlora_forward (kernels.rs:262-296) == QloraLinear::forward
 * (qlora.rs:86-107).  y: batch x out_dim. */
QH_API qh_status qh_qlora_forward(qh_ctx *ctx, const qh_qweight *w,
                                  const qh_lora *lora, const float *x,
                                  size_t x_len, size_t batch, float *y);
/* gpu_qlora_backward (kernels.rs:301-353) == QloraLinear::backward
 * (qlora.rs:116-165).  grad_x: batch x in_dim; grad_a (r x in_dim) and
 * grad_b (out_dim x r) are written only when lora != NULL. */
QH_API qh_status qh_qlora_backward(qh_ctx *ctx, const qh_qweight *w,
                                   const qh_lora *lora, const float *x,
                                   size_t x_len, const float *dy,
                                   size_t dy_len, size_t batch, float *grad_x,
                                   float *grad_a, float *grad_b);

/* ---- paged 8-bit Adam: Adam8bit (qlora-core/src/optim.rs:32-249) ------- */
typedef struct qh_adam_config { /* AdamConfig (optim.rs:32-60) */
  float lr, beta1, beta2, eps;
  size_t block_size;
  size_t max_resident_pages; /* SIZE_MAX = everything resident */
} qh_adam_config;

typedef struct qh_adam_stats { /* AdamStats (optim.rs:135-141) */
  size_t pages_streamed;
  size_t state_bytes;
} qh_adam_stats;

typedef struct qh_adam8bit qh_adam8bit;

/* AdamConfig::default (optim.rs:49-60). */
QH_API void qh_adam_config_default(qh_adam_config *cfg);
/* Adam8bit::new (optim.rs:155-161): validates the config. */
QH_API qh_status qh_adam8bit_create(qh_ctx *ctx, const qh_adam_config *cfg,
                                    qh_adam8bit **out);
QH_API void qh_adam8bit_destroy(qh_adam8bit *opt);
/* Adam8bit::step (optim.rs:164-199) on host slices: params updated in
 * place.  Bit-exact with the reference's f32 arithmetic. */
QH_API qh_status qh_adam8bit_step(qh_adam8bit *opt, float *const *params,
                                  const size_t *param_lens,
                                  const float *const *grads,
                                  const size_t *grad_lens, size_t count,
                                  qh_adam_stats *stats);
/* Same step on device-resident params/grads, enqueued on `stream`. */
QH_API qh_status qh_adam8bit_step_dev(qh_adam8bit *opt,
                                      float *const *d_params,
                                      const float *const *d_grads,
                                      const size_t *lens, size_t count,
                                      qh_adam_stats *stats, void *stream);
/* Adam8bit::state_bytes (optim.rs:201-204). */
QH_API size_t qh_adam8bit_state_bytes(const qh_adam8bit *opt);
/* Copy the int8 state of parameter `idx` to host memory (m/v codes: numel
 * bytes, m/v scales: ceil(numel/block_size) floats). */
QH_API qh_status qh_adam8bit_get_state(qh_adam8bit *opt, size_t idx,
                                       uint8_t *m_codes, float *m_scales,
                                       uint8_t *v_codes, float *v_scales,
                                       uint64_t *step);

/* ---- device-resident hot path (async on `stream`) ----------------------- */
/* All pointers are device pointers; `w` describes device buffers.  Calls on
 * one context share its scratch, launch counters and T1 exchange words: keep
 * them ordered on one stream (or use one context per stream). */
QH_API qh_status qh_quantize_nf4_dev(qh_ctx *ctx, const float *d_w,
                                     size_t rows, size_t cols,
                                     size_t block_size, int double_quant,
                                     uint8_t *d_codes, float *d_scales,
                                     uint8_t *d_scale_codes, float *d_absmax,
                                     void *stream);
QH_API qh_status qh_dequantize_dev(qh_ctx *ctx, const qh_qweight *w,
                                   float *d_out, void *stream);
QH_API qh_status qh_matmul_dev(qh_ctx *ctx, int op, const float *d_a,
                               const float *d_b, size_t m, size_t k, size_t n,
                               float *d_c, void *stream);
/* Fused forward.  x: batch x in_dim in `x_dtype` (QH_BF16 = bf16
 * activations, upcast exactly).  d_t1 (optional, batch x r fp32) receives
 * X.A^T for reuse by the backward. */
QH_API qh_status qh_qlora_forward_dev(qh_ctx *ctx, const qh_qweight *w,
                                      const qh_lora *lora, const void *d_x,
                                      int x_dtype, size_t batch, float *d_y,
                                      float *d_t1, void *stream);
/* Forward of `count` independent layers on one stream: layer i gets what
 * qh_qlora_forward_dev(ctx, &ws[i], loras[i], d_xs[i], x_dtype, batch,
 * d_ys[i], d_t1s ? d_t1s[i] : NULL, stream) gives (loras[i] NULL = no
 * adapter).  No counterpart in the reference, whose forward takes one layer
 * per call (qlora-wgpu/src/kernels.rs:262-296): at batch 1, consecutive
 * layers that the one-launch decode kernel serves run in pairs, one launch
 * per pair (the two layers' workgroups side by side on every CU), bit for
 * bit as in their own launches; at batches of 2-16 the layers whose T1
 * comes from a launch before their weight stream get that T1 from one
 * launch for all of them, and consecutive ones share a split-K launch, each
 * planned for half of the CUs -- its K slices then meet in another order
 * than in the layer's own launch (within the fp32 tolerance; the same bits
 * from call to call).  As in a decoder block's independent projections
 * (q / k / v, gate / up) or two layers of a decode step.  Arguments are
 * validated for every layer before any launch. */
QH_API qh_status qh_qlora_forward_group_dev(qh_ctx *ctx, size_t count,
                                            const qh_qweight *ws,
                                            const qh_lora *const *loras,
                                            const void *const *d_xs, int x_dtype,
                                            size_t batch, float *const *d_ys,
                                            float *const *d_t1s, void *stream);
/* Fused backward.  x and dy in `act_dtype`.  d_t1: X.A^T from the forward
 * (NULL = recompute). */
QH_API qh_status qh_qlora_backward_dev(qh_ctx *ctx, const qh_qweight *w,
                                       const qh_lora *lora, const void *d_x,
                                       const void *d_dy, int act_dtype,
                                       size_t batch, const float *d_t1,
                                       float *d_grad_x, float *d_grad_a,
                                       float *d_grad_b, void *stream);
/* Allocation-free fused backward: no counterpart in the reference.  For
 * callers that cannot allocate device memory (code under HIP graph capture,
 * tight serving loops, harnesses that forbid hipMalloc).  Arguments and
 * results, bit for bit, are those of qh_qlora_backward_dev, but its scratch
 * (T1 when d_t1 is NULL, Ds = s.dY.B, split-K partial sums) lives in a fixed
 * region of QH_NOALLOC_SCRATCH_BYTES that each GPU holds from the first context
 * created on it until the process ends; the call allocates nothing.  So it
 * has no room for the operand planes of large input gradients, and computes
 * those at the speed of the kernel without them.  A call that
 * would need more scratch fails with QH_ERR_INVALID_CONFIG before any
 * launch.  Every call on one GPU shares that GPU's region: calls that
 * overlap on one GPU (other streams, other contexts, other threads) race,
 * and the caller must order them.  Kernel timing (qh_ctx_set_timing) does
 * not apply to it. */
#define QH_NOALLOC_SCRATCH_BYTES ((size_t)64 << 20)
QH_API qh_status qh_qlora_backward_dev_noalloc(qh_ctx *ctx, const qh_qweight *w,
                                               const qh_lora *lora, const void *d_x,
                                               const void *d_dy, int act_dtype,
                                               size_t batch, const float *d_t1,
                                               float *d_grad_x, float *d_grad_a,
                                               float *d_grad_b, void *stream);

/* ---- the glue of a decoder block around its projections ----------------
 * qlora-model/src/llama.rs calls these between the QLoRA projections of
 * `block_forward` / `block_backward` (llama.rs:417-602).  All fp32,
 * row-major.  The host-slice forms validate lengths (QH_ERR_SHAPE_MISMATCH)
 * and block; the `_dev` forms enqueue on `stream` and trust their sizes. */

/* rmsnorm_in_place (llama.rs:730-739): y = x / sqrt(mean(x^2) + eps) * w for
 * each of `rows` rows of h; y may alias x. */
QH_API qh_status qh_rmsnorm(qh_ctx *ctx, const float *x, size_t x_len,
                            const float *w, size_t h, float eps, float *y);
QH_API qh_status qh_rmsnorm_dev(qh_ctx *ctx, const float *d_x, const float *d_w,
                                size_t rows, size_t h, float eps, float *d_y,
                                void *stream);
/* rmsnorm_backward (llama.rs:605-628): dx (rows x h) and, unless dw is NULL,
 * dw (h).  block_backward discards dw (llama.rs:568, 594); pass NULL to skip
 * it.  dx may alias dy only when dw is NULL (the dw pass reads dy after dx
 * is written; the device form rejects that aliasing). */
QH_API qh_status qh_rmsnorm_backward(qh_ctx *ctx, const float *x, size_t x_len,
                                     const float *w, size_t h, const float *dy,
                                     size_t dy_len, float eps, float *dx,
                                     float *dw);
QH_API qh_status qh_rmsnorm_backward_dev(qh_ctx *ctx, const float *d_x,
                                         const float *d_w, const float *d_dy,
                                         size_t rows, size_t h, float eps,
                                         float *d_dx, float *d_dw,
                                         void *stream);
/* MLP activation (llama.rs:452-456, 516-518): act = silu(gate) * up over n
 * elements; act may alias gate or up. */
QH_API qh_status qh_swiglu(qh_ctx *ctx, const float *gate, size_t gate_len,
                           const float *up, size_t up_len, float *act);
QH_API qh_status qh_swiglu_dev(qh_ctx *ctx, const float *d_gate,
                               const float *d_up, size_t n, float *d_act,
                               void *stream);
/* Its backward (llama.rs:559-562, 520-527): dg = d_act * up * silu'(gate),
 * du = d_act * silu(gate); dg may alias gate, du may alias up. */
QH_API qh_status qh_swiglu_backward(qh_ctx *ctx, const float *gate,
                                    const float *up, const float *d_act,
                                    size_t n, float *dg, float *du);
QH_API qh_status qh_swiglu_backward_dev(qh_ctx *ctx, const float *d_gate,
                                        const float *d_up, const float *d_act,
                                        size_t n, float *d_dg, float *d_du,
                                        void *stream);
/* softmax_cross_entropy (llama.rs:487-514): *loss = mean over seq rows of
 * -log softmax(logits)[target]; dlogits = (softmax - onehot) / seq, row-major
 * (seq x vocab), may alias logits.  The host form rejects a target >= vocab
 * (the reference panics on it); the device form gives a NaN loss for one and
 * leaves out its one-hot term. */
QH_API qh_status qh_softmax_cross_entropy(qh_ctx *ctx, const float *logits,
                                          size_t logits_len,
                                          const uint32_t *targets, size_t seq,
                                          size_t vocab, float *loss,
                                          float *dlogits);
QH_API qh_status qh_softmax_cross_entropy_dev(qh_ctx *ctx,
                                              const float *d_logits,
                                              const uint32_t *d_targets,
                                              size_t seq, size_t vocab,
                                              float *d_loss, float *d_dlogits,
                                              void *stream);

/* ---- library-owned device weights ----------------------------------------
 * A packed weight uploaded once and kept in HBM (the device-resident form a
 * model stack holds; the reference re-uploads W on every call,
 * qlora-wgpu/src/kernels.rs:60-75, 268-276).  The view is a qh_qweight of
 * device pointers for the *_dev entry points; it stays valid until
 * qh_dweight_destroy, which must come before the context's destroy. */
typedef struct qh_dweight qh_dweight;
/* Allocates HBM, copies the host weight (validated like qh_qweight
 * everywhere else) and waits for the copy. */
QH_API qh_status qh_weight_upload(qh_ctx *ctx, const qh_qweight *host,
                                  qh_dweight **out);
QH_API qh_status qh_dweight_view(const qh_dweight *w, qh_qweight *view);
QH_API void qh_dweight_destroy(qh_dweight *w);

/* Projections that read the same activations: the q / k / v projections of
 * one normed input, or gate / up (no counterpart in the reference, whose
 * layers run one call each: qlora-wgpu/src/kernels.rs:262-353).  All layers
 * share in_dim; count <= 8.  The forward gives each layer i what
 * qh_qlora_forward_dev(ctx, &ws[i], loras[i], d_x, x_dtype, batch, d_ys[i],
 * d_t1s ? d_t1s[i] : NULL, stream) gives, within the GEMM tolerance; the
 * backward writes each layer's grad_A / grad_B as qh_qlora_backward_dev does
 * and d_grad_x = the sum of the layers' input gradients (qlora-model's
 * block_backward sums them: llama.rs:563-567, 580-593).  Groups of 2-3
 * layers that fit the grouped kernels run as one launch per stage (T1, the
 * base GEMMs; Ds, grad_A with grad_B, the input gradient); others run layer
 * by layer.  loras[i] NULL = no adapter (its gradient entries are ignored). */
QH_API qh_status qh_qlora_forward_shared_dev(qh_ctx *ctx, size_t count,
                                             const qh_qweight *ws,
                                             const qh_lora *const *loras,
                                             const void *d_x, int x_dtype,
                                             size_t batch, float *const *d_ys,
                                             float *const *d_t1s, void *stream);
QH_API qh_status qh_qlora_backward_shared_dev(
    qh_ctx *ctx, size_t count, const qh_qweight *ws, const qh_lora *const *loras,
    const void *d_x, const void *const *d_dys, int act_dtype, size_t batch,
    const float *const *d_t1s, float *d_grad_x, float *const *d_grad_as,
    float *const *d_grad_bs, void *stream);

/* ---- a decoder block's MLP on device ----------------------------------------
 * The MLP half of `block_forward` / `block_backward` (qlora-model/src/
 * llama.rs:449-463, 554-574) with its three projections as QLoRA layers
 * (`Proj::Qlora`, llama.rs:106-140): activations stay in HBM from the norm
 * to the residual add, all on `stream`.  Device pointers throughout. */
typedef struct qh_mlp_block {
  size_t hidden, inter;
  float eps;                /* LlamaConfig::rms_eps */
  const float *norm_w;      /* mlp_norm, hidden floats */
  qh_qweight gate, up;      /* inter x hidden */
  qh_qweight down;          /* hidden x inter */
  const qh_lora *gate_lora, *up_lora, *down_lora; /* NULL = no adapter */
} qh_mlp_block;

/* Activations the forward keeps for the backward (caller-owned device
 * buffers; the backward consumes gate and up). */
typedef struct qh_mlp_cache {
  float *x_mid;             /* seq x hidden: the block's input */
  float *xn;                /* seq x hidden: rmsnorm(x_mid) */
  float *gate, *up, *act;   /* seq x inter */
  float *t1_gate, *t1_up, *t1_down; /* seq x r of each adapter (or NULL) */
} qh_mlp_cache;

/* x (seq x hidden) <- x + down(silu(gate(xn)) * up(xn)), xn = rmsnorm(x). */
QH_API qh_status qh_mlp_forward_dev(qh_ctx *ctx, const qh_mlp_block *blk,
                                    float *d_x, size_t seq,
                                    const qh_mlp_cache *cache, void *stream);
/* dx_in = dL/d(block input) from dx_out = dL/d(block output) (separate
 * buffers: dx_out is read after dx_in is first written); adapter
 * gradients in gate, up, down order (d_grad_a[i]: r x in, d_grad_b[i]:
 * out x r), entries of projections without an adapter are ignored. */
QH_API qh_status qh_mlp_backward_dev(qh_ctx *ctx, const qh_mlp_block *blk,
                                     const qh_mlp_cache *cache,
                                     const float *d_dx_out, size_t seq,
                                     float *d_dx_in, float *const *d_grad_a,
                                     float *const *d_grad_b, void *stream);

/* ---- a decoder block's attention projections on device ----------------------
 * The attention half of `block_forward` / `block_backward` (qlora-model/src/
 * llama.rs:426-439, 577-601) around the attention itself, which stays with
 * the caller: RMSNorm and the q/k/v QLoRA projections before it, the o
 * projection and the residual add after it, and their backward.  Device
 * pointers throughout, all work on `stream`. */
typedef struct qh_attn_block {
  size_t hidden, kv_dim;    /* kv_dim = kv_heads * head_dim */
  float eps;                /* LlamaConfig::rms_eps */
  const float *norm_w;      /* attn_norm, hidden floats */
  qh_qweight q;             /* hidden x hidden */
  qh_qweight k, v;          /* kv_dim x hidden */
  qh_qweight o;             /* hidden x hidden */
  const qh_lora *q_lora, *k_lora, *v_lora, *o_lora; /* NULL = no adapter */
} qh_attn_block;

/* Activations kept for the backward (caller-owned device buffers). */
typedef struct qh_attn_cache {
  float *x_in;              /* seq x hidden: the block's input */
  float *xn;                /* seq x hidden: rmsnorm(x_in) */
  float *attn;              /* seq x hidden: the attention output (the
                               caller writes it; the o projection reads it) */
  float *t1_q, *t1_k, *t1_v, *t1_o; /* seq x r of each adapter (or NULL) */
} qh_attn_cache;

/* llama.rs:426-434: xn = rmsnorm(x); q = q(xn) (seq x hidden), k = k(xn),
 * v = v(xn) (seq x kv_dim).  x is not changed (a copy goes to the cache). */
QH_API qh_status qh_attn_qkv_forward_dev(qh_ctx *ctx, const qh_attn_block *blk,
                                         const float *d_x, size_t seq,
                                         const qh_attn_cache *cache, float *d_q,
                                         float *d_k, float *d_v, void *stream);
/* llama.rs:436-439: x (seq x hidden) <- x + o(cache->attn). */
QH_API qh_status qh_attn_o_forward_dev(qh_ctx *ctx, const qh_attn_block *blk,
                                       float *d_x, size_t seq,
                                       const qh_attn_cache *cache, void *stream);
/* llama.rs:577: the o projection's backward from dx_mid = dL/d(x after
 * the attention residual): d_attn (seq x hidden) and o's adapter gradients
 * (ignored without an adapter). */
QH_API qh_status qh_attn_o_backward_dev(qh_ctx *ctx, const qh_attn_block *blk,
                                        const qh_attn_cache *cache,
                                        const float *d_dx_mid, size_t seq,
                                        float *d_dattn, float *d_grad_a_o,
                                        float *d_grad_b_o, void *stream);
/* llama.rs:580-601: q/k/v backward from the attention's dq, dk, dv, the sum
 * (dxn_q + dxn_k) + dxn_v, RMSNorm's dx (its dw discarded, llama.rs:594)
 * and the residual: dx_in = dx_mid + dx_norm (dx_in must not alias dx_mid).
 * Adapter gradients in q, k, v order; entries of projections without an
 * adapter are ignored. */
QH_API qh_status qh_attn_qkv_backward_dev(qh_ctx *ctx, const qh_attn_block *blk,
                                          const qh_attn_cache *cache,
                                          const float *d_dq, const float *d_dk,
                                          const float *d_dv, const float *d_dx_mid,
                                          size_t seq, float *d_dx_in,
                                          float *const *d_grad_a,
                                          float *const *d_grad_b, void *stream);

/* ---- packed NF4 files -----------------------------------------------------
 * No counterpart in the reference: its quantized weights leave `quantize`
 * only as fp32 (QuantizedWeight.scales, qlora-python/src/lib.rs:101) and
 * qlora-io writes and reads fp32 tensors (npz.rs:46, safetensors.rs:25).  A
 * safetensors file holding, per weight <name>, "<name>.nf4_codes" (U8),
 * then "<name>.nf4_scale_codes" (U8, the int8 codes bit-cast) and
 * "<name>.nf4_absmax" (F32), or "<name>.nf4_scales" (F32), plus
 * "__metadata__" {"format": "qlora-hip-nf4/1", "<name>": "rows,cols,bs"}.
 * Readers that convert every tensor to fp32 (qlora-io's read_safetensors)
 * still parse it.  The writer puts every F32 part first, so with buf
 * 4-byte aligned each F32 view is aligned; files with U8 parts first (an
 * earlier writer of this format, other safetensors writers) are read too,
 * and their F32 views may then be unaligned: copy them byte-wise (memcpy,
 * qh_weight_upload_dev) rather than reading them as floats.  Malformed files
 * return QH_ERR_MALFORMED, other dtypes QH_ERR_UNSUPPORTED, part lengths
 * that disagree with the shape QH_ERR_SHAPE_MISMATCH (the from_raw_parts
 * rule, quant.rs:170-197). */
/* File size for `count` host-resident weights named names[i]. */
QH_API qh_status qh_nf4_file_size(const qh_qweight *ws, const char *const *names,
                                  size_t count, size_t *bytes);
/* Write the file into buf (buf_len must equal qh_nf4_file_size's bytes). */
QH_API qh_status qh_nf4_file_write(const qh_qweight *ws, const char *const *names,
                                   size_t count, uint8_t *buf, size_t buf_len);
/* Number of weights in a file image. */
QH_API qh_status qh_nf4_file_count(const uint8_t *buf, size_t len,
                                   size_t *count);
/* Weight `index` (file order): its name and a view whose pointers point
 * into buf (no copy). */
QH_API qh_status qh_nf4_file_entry(const uint8_t *buf, size_t len,
                                   size_t index, char *name, size_t name_len,
                                   qh_qweight *view);
QH_API qh_status qh_nf4_file_find(const uint8_t *buf, size_t len,
                                  const char *name, qh_qweight *view);
/* Copy a host-resident weight (e.g. a view into a file image) into device
 * buffers of its part sizes, on `stream` (asynchronous for pinned host
 * memory): the packed form loads straight into HBM, no fp32 and no
 * quantize on the way. */
QH_API qh_status qh_weight_upload_dev(qh_ctx *ctx, const qh_qweight *w,
                                      uint8_t *d_codes, float *d_scales,
                                      uint8_t *d_scale_codes, float *d_absmax,
                                      void *stream);

#ifdef __cplusplus
}
#endif
#endif /* QLORA_HIP_H */
