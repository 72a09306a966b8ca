// k_gemm_bf16.hip -- the large NF4 GEMMs of a QLoRA layer on bf16 MFMA (gfx950).
//
// The forward and the input gradient (qlora-core/src/qlora.rs:86-165, the
// reference's mm_nt / mm_nn WGSL kernels qlora-wgpu/shaders/gemm.wgsl:34-98):
//
//   forward  C = X . W^T + T1 . (s B)^T    (W: N x K, C: M x N)
//   grad_x   C = dY . W + Ds . A           (W: K x N as stored, C: M x N)
//
// on v_mfma_f32_32x32x16_bf16 with fp32 accumulation.  The dequantized
// weight w = L[code] * block_scale (fp32, bit-exact with quant.rs:157-167)
// is split into two bf16 parts, w = wh + wl + d with |d| <= 2^-16 |w|.
//  * bf16 activations (XF = 0) are exact in bf16: a product runs as two
//    MFMAs, x.wh + x.wl.
//  * fp32 activations (XF = 1) are split the same way: xh.wh + xh.wl +
//    xl.wh, three MFMAs, leaving out xl.wl (~2^-16 of the product); the
//    bf16 MFMA rate is 16 times the fp32 one, so three of them still beat
//    one fp32 MFMA five-fold.
//  * The LoRA segment (fp32 operands) always runs as three MFMAs.
//
// Tiles: large problems use 512 threads = 8 waves (two per SIMD, so that one
// wave's dequant work and waits overlap the other's MFMAs) in a 2 x 4 grid;
// a block computes 256 x BN outputs (BN = 256 or 128), a wave 128 x BN/4 of
// 32 x 32 MFMA tiles whose accumulators stay in registers for the whole
// reduction.  Small problems (a few hundred 256-row tiles or fewer: a decoder
// block's projections at a few thousand tokens) use 256 threads = 4 waves in
// a 2 x 2 grid on 64 x 64 tiles, several blocks per CU, loads two steps
// ahead, and split the reduction across blocks when the tiles alone cannot
// fill the GPU (partial sums reduced in a fixed order by a second kernel).
// The reduction runs in steps of 32 through two LDS stages: while the MFMAs
// read one stage, the next step's activations and codes are already in
// registers (loaded at the top of the step) and are dequantized, split and
// written to the other stage after the MFMAs; one barrier per step.
// LDS rows hold 32 bf16 (64 bytes) as four 16-byte granules; granule g of
// row r sits at position g ^ ((r >> 2) & 3), so that the fragment reads of
// 16 consecutive rows that one LDS cycle serves (16 lanes x 16 bytes over
// the 64 four-byte banks) fall in 16 distinct bank groups without padding.
#include <type_traits>

#include "qh_internal.h"
#include "qh_nf4.h"

namespace qh {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

constexpr int kBK = 32;          // reduction per step = one LDS row

// Block shape: T threads (T / 64 waves in a 2 x T/128 grid), BM x BN outputs;
// a step reduces KS x 32 (KS LDS sub-tiles between two barriers) and its
// global loads are issued PF steps before its MFMAs.
template <int T_, int BM_, int BN_, int PF_ = 1, int KS_ = 1, int PP_ = 0>
struct Cfg {
  static constexpr int T = T_, BM = BM_, BN = BN_, PF = PF_, KS = KS_, PP = PP_;
  static_assert(PF == 1 || PF == 2, "prefetch depth");
  static_assert(KS == 1 || KS == 2, "sub-tiles per step");
  static_assert(!PP || (PF == 1 && KS == 1 && T == 512), "ping-pong blocks");
  static constexpr int WGN = T / 128;              // wave grid: 2 x WGN
  static constexpr int WTM = BM / 2, WTN = BN / WGN;  // one wave's outputs
  static constexpr int TM = WTM / 32, TN = WTN / 32;  // 32 x 32 MFMA tiles per wave
  static_assert(TM >= 1 && TN >= 1 && WTM % 32 == 0 && WTN % 32 == 0, "wave tile");
  static_assert(BN <= T && BM % (T / 4) == 0, "staging maps");
};
using CfgL256 = Cfg<512, 256, 256, 1, 1, 1>;
using CfgL128 = Cfg<512, 256, 128, 1, 1, 1>;
using CfgM = Cfg<512, 128, 128, 2, 2>;
using CfgM1 = Cfg<512, 128, 128, 2, 1>;  // half the LDS: two blocks per CU
using CfgS = Cfg<256, 64, 64, 2, 2>;

__constant__ float c_lut_bf[17] = QH_NF4_LUT17_INIT;  // the codebook (quant.rs:27-44)

// Element offset of granule g (8 elements) of LDS row `row`.
__device__ __forceinline__ int sw(int row, int g) { return row * kBK + 8 * (g ^ ((row >> 2) & 3)); }

// Two floats as a bf16 pair (round to nearest even).
__device__ __forceinline__ uint32_t pk_bf16(float a, float b) {
  const bf16x2_t h = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(uint32_t, h);
}
__device__ __forceinline__ float bf16_lo_f(uint32_t p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float bf16_hi_f(uint32_t p) { return __uint_as_float(p & 0xffff0000u); }

// hi and lo bf16 parts of two floats: hi = bf16(v), lo = bf16(v - hi).
__device__ __forceinline__ void split2(float a, float b, uint32_t &hi, uint32_t &lo) {
  hi = pk_bf16(a, b);
  // opaque to the compiler, which otherwise converts a again to rebuild
  // bf16(a) as a float instead of shifting the word it has
  asm("" : "+v"(hi));
  lo = pk_bf16(a - bf16_lo_f(hi), b - bf16_hi_f(hi));
}

// Block scale (quant.rs:212-221): fp32, or fl(fl(c / 127) * absmax).  c / 127
// is the double product with the double reciprocal of 127 rounded once to
// float, which is the IEEE float quotient bit for bit (an exact quotient of
// two floats lies at least 2^-49 relatively from every float midpoint; the
// product is within 2^-52), without a float division.
struct ScaleRef {
  float a;    // the fp32 scale, or the super-block absmax
  int32_t c;  // the int8 scale code
};
// KIND is the weight's scale store (0: fp32 scales, 1: int8 codes + absmax);
// a template parameter so that the step loop's loads are the same on every
// path and the compiler can wait for exactly the ones a step needs.
template <int KIND>
__device__ __forceinline__ ScaleRef load_scale(const DevQW &w, int64_t blk) {
  if constexpr (KIND == 0) return ScaleRef{w.scales[blk], 127};
  else return ScaleRef{w.absmax[blk >> 8], (int32_t)(int8_t)w.scale_codes[blk]};
}
template <int KIND>
__device__ __forceinline__ float decode_scale(ScaleRef r) {
  if constexpr (KIND == 0) return r.a;
  else return (float)((double)(float)r.c * (1.0 / 127.0)) * r.a;
}

// ---- activation tile: BM rows x 32 of a row-major (rows x K) matrix ----------
// Thread t owns rows t / 4 + (T / 4) v and granule t % 4 (elements 8 (t % 4)
// ... + 8).  bf16 (XF = 0) is copied; fp32 (XF = 1) is split into hi and lo.
// The tiles take thread t = threadIdx.x % C::T, so that a half-size C lets
// each half of a block stage its own half of a tile.  Rows and elements past
// the matrix are loaded from a valid address and zeroed when written to LDS,
// not when loaded: nothing touches loaded data before its LDS write, so the
// MFMAs issued in between never wait for those loads.
template <int XF, class C>
struct ActTile;

template <class C>
struct ActTile<0, C> {
  static constexpr int P = C::BM / (C::T / 4);  // passes
  uint4 v[P];
  uint32_t okm;  // bit i: pass i in range
  __device__ __forceinline__ void load(const void *pv, int64_t ld, int64_t m0, int64_t M,
                                       int64_t k0, int64_t K) {
    const uint16_t *p = (const uint16_t *)pv;
    const int c = (threadIdx.x % C::T) & 3;
    okm = 0;
#pragma unroll
    for (int i = 0; i < P; ++i) {
      const int64_t row = m0 + ((threadIdx.x % C::T) >> 2) + (C::T / 4) * i, k = k0 + 8 * c;
      const bool ok = row < M && k < K;
      v[i] = *(const uint4 *)(p + (ok ? row * ld + k : 0));
      okm |= (uint32_t)ok << i;
    }
  }
  __device__ __forceinline__ void store(uint16_t *Sh, uint16_t *) const {
    const int c = (threadIdx.x % C::T) & 3;
#pragma unroll
    for (int i = 0; i < P; ++i) {
      // out-of-range rows and elements become zeros: one AND per word with
      // an all-ones or all-zeros mask, no branch
      const uint32_t mk = 0u - ((okm >> i) & 1u);
      const uint4 t = make_uint4(v[i].x & mk, v[i].y & mk, v[i].z & mk, v[i].w & mk);
      *(uint4 *)(Sh + sw(((threadIdx.x % C::T) >> 2) + (C::T / 4) * i, c)) = t;
    }
  }
};

template <class C>
struct ActTile<1, C> {
  static constexpr int P = C::BM / (C::T / 4);  // passes
  float4 v[P][2];
  uint32_t okm;  // bit i: pass i in range
  __device__ __forceinline__ void load(const void *pv, int64_t ld, int64_t m0, int64_t M,
                                       int64_t k0, int64_t K) {
    const float *p = (const float *)pv;
    const int c = (threadIdx.x % C::T) & 3;
    okm = 0;
#pragma unroll
    for (int i = 0; i < P; ++i) {
      const int64_t row = m0 + ((threadIdx.x % C::T) >> 2) + (C::T / 4) * i, k = k0 + 8 * c;
      const bool ok = row < M && k < K;
      const float *q = p + (ok ? row * ld + k : 0);
      v[i][0] = *(const float4 *)q;
      v[i][1] = *(const float4 *)(q + 4);
      okm |= (uint32_t)ok << i;
    }
  }
  __device__ __forceinline__ void store(uint16_t *Sh, uint16_t *Sl) const {
    const int c = (threadIdx.x % C::T) & 3;
#pragma unroll
    for (int i = 0; i < P; ++i) {
      const float4 t0 = v[i][0], t1 = v[i][1];
      uint32_t h[4], l[4];
      split2(t0.x, t0.y, h[0], l[0]);
      split2(t0.z, t0.w, h[1], l[1]);
      split2(t1.x, t1.y, h[2], l[2]);
      split2(t1.z, t1.w, h[3], l[3]);
      // out-of-range rows and elements become zeros (whatever their loaded
      // bits split to): one AND per word, no branch
      const uint32_t mk = 0u - ((okm >> i) & 1u);
      const int o = sw(((threadIdx.x % C::T) >> 2) + (C::T / 4) * i, c);
      *(uint4 *)(Sh + o) = make_uint4(h[0] & mk, h[1] & mk, h[2] & mk, h[3] & mk);
      *(uint4 *)(Sl + o) = make_uint4(l[0] & mk, l[1] & mk, l[2] & mk, l[3] & mk);
    }
  }
};

// ---- NF4 tile, forward orientation: BN W rows (output columns) x 32 ----------
// W row n = n0 + t / TPR, elements (t % TPR) * EPT ... + EPT of the step
// (within one 64-element block, so one scale).
template <class C, int KIND>
struct WTileRow {
  static constexpr int TPR = C::T / C::BN;      // threads per W row: 2 or 4
  static constexpr int EPT = kBK / TPR;         // elements per thread: 16 or 8
  static_assert(TPR == 2 || TPR == 4, "threads per W row");
  uint2 c;        // EPT / 2 code bytes
  ScaleRef sr;
  bool in;        // in range (else the elements are written as zeros)
  __device__ __forceinline__ void load(const DevQW &w, int64_t n0, int64_t k0) {
    const int64_t n = n0 + (threadIdx.x % C::T) / TPR;
    const int64_t k = k0 + ((threadIdx.x % C::T) % TPR) * EPT;
    const bool ok = n < w.rows && k < w.cols;
    const int64_t e = ok ? n * w.cols + k : 0;
    if (EPT == 16) c = *(const uint2 *)(w.codes + (e >> 1));
    else c = make_uint2(*(const uint32_t *)(w.codes + (e >> 1)), 0u);
    sr = load_scale<KIND>(w, e >> 6);
    in = ok;
  }
  __device__ __forceinline__ void store(uint16_t *Sh, uint16_t *Sl, const float *lut) const {
    const int row = (threadIdx.x % C::T) / TPR, g0 = ((threadIdx.x % C::T) % TPR) * (EPT / 8);
    const float s = in ? decode_scale<KIND>(sr) : 0.0f;
    const uint32_t cw[2] = {c.x, c.y};
#pragma unroll
    for (int q = 0; q < EPT / 8; ++q) {  // 8 elements = one code word = one granule
      float f[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = lut[(cw[q] >> (4 * e)) & 15u] * s;
      uint32_t h[4], l[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) split2(f[2 * e], f[2 * e + 1], h[e], l[e]);
      const int o = sw(row, g0 + q);
      *(uint4 *)(Sh + o) = make_uint4(h[0], h[1], h[2], h[3]);
      *(uint4 *)(Sl + o) = make_uint4(l[0], l[1], l[2], l[3]);
    }
  }
};

// ---- NF4 tile, input-gradient orientation: 32 W rows (the reduction) x BN
// W columns (the outputs), row-major in LDS (row stride ldb_t(BN)), read
// column-wise by the LDS transpose loads (mma below).  Thread t holds EPT
// consecutive columns (t % TPR) * EPT of W row k0 + t / TPR: one code load
// and one block scale, as in the forward.
__host__ __device__ constexpr int ldb_t(int bn) { return bn + 32; }  // 64 bytes of padding

template <class C, int KIND, int LDB = ldb_t(C::BN)>
struct WTileKRow {
  static constexpr int EPT = C::BN * kBK / C::T;  // columns per thread: 16 or 8
  static constexpr int TPR = C::BN / EPT;          // threads per W row
  static_assert(EPT == 16 || EPT == 8, "columns per thread");
  static_assert(TPR * kBK == C::T, "one W row per TPR threads");
  uint2 c;        // EPT / 2 code bytes
  ScaleRef sr;
  bool in;        // in range (else the elements are written as zeros)
  __device__ __forceinline__ void load(const DevQW &w, int64_t n0, int64_t k0) {
    const int64_t n = k0 + (threadIdx.x % C::T) / TPR;                 // W row (reduction)
    const int64_t col = n0 + ((threadIdx.x % C::T) % TPR) * EPT;       // W column (output)
    const bool ok = n < w.rows && col < w.cols;               // cols % 64 == 0
    const int64_t e = ok ? n * w.cols + col : 0;
    if (EPT == 16) c = *(const uint2 *)(w.codes + (e >> 1));
    else c = make_uint2(*(const uint32_t *)(w.codes + (e >> 1)), 0u);
    sr = load_scale<KIND>(w, e >> 6);
    in = ok;
  }
  __device__ __forceinline__ void store(uint16_t *Sh, uint16_t *Sl, const float *lut) const {
    const int row = (threadIdx.x % C::T) / TPR, c0 = ((threadIdx.x % C::T) % TPR) * EPT;
    const float s = in ? decode_scale<KIND>(sr) : 0.0f;
    const uint32_t cw[2] = {c.x, c.y};
#pragma unroll
    for (int q = 0; q < EPT / 8; ++q) {  // 8 columns = one code word
      float f[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = lut[(cw[q] >> (4 * e)) & 15u] * s;
      uint32_t h[4], l[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) split2(f[2 * e], f[2 * e + 1], h[e], l[e]);
      const int o = row * LDB + c0 + 8 * q;
      *(uint4 *)(Sh + o) = make_uint4(h[0], h[1], h[2], h[3]);
      *(uint4 *)(Sl + o) = make_uint4(l[0], l[1], l[2], l[3]);
    }
  }
};

// ---- LoRA segment tiles (fp32 operands, split into hi / lo) -----------------
// R rows x 32 of a row-major fp32 matrix (element (row, k) at p[row * ld + k]),
// scaled by `scale`: thread t of T owns rows t / 8 + (T / 8) v, elements
// 4 (t % 8) ... + 4.
template <int R, int T>
__device__ __forceinline__ void stage_f32_rowk(const float *p, int64_t ld, int64_t r0, int64_t rlim,
                                               int64_t k0, int64_t klim, float scale,
                                               uint16_t *Sh, uint16_t *Sl) {
  static_assert(R % (T / 8) == 0, "rows per pass");
  const int c = threadIdx.x & 7;
#pragma unroll
  for (int i = 0; i < R / (T / 8); ++i) {
    const int rl = (threadIdx.x >> 3) + (T / 8) * i;
    const int64_t row = r0 + rl, k = k0 + 4 * c;
    float f[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) f[j] = (row < rlim && k + j < klim) ? p[row * ld + k + j] * scale : 0.0f;
    uint32_t h0, h1, l0, l1;
    split2(f[0], f[1], h0, l0);
    split2(f[2], f[3], h1, l1);
    const int o = sw(rl, c >> 1) + 4 * (c & 1);
    *(uint2 *)(Sh + o) = make_uint2(h0, h1);
    *(uint2 *)(Sl + o) = make_uint2(l0, l1);
  }
}

// 32 x R of a row-major fp32 matrix (element (col, k) at p[k * ld + col]),
// scaled, into the input gradient's row-major B layout (row k, column col,
// row stride ldb_t(R)): thread t owns reduction rows t / (R / 4) + KS v and
// columns 4 (t % (R / 4)) ... + 4.
template <int R, int T>
__device__ __forceinline__ void stage_f32_krow(const float *p, int64_t ld, int64_t c0, int64_t clim,
                                               int64_t k0, int64_t klim, float scale,
                                               uint16_t *Sh, uint16_t *Sl) {
  constexpr int CG = R / 4, KS = T / CG;
  static_assert(KS <= kBK && kBK % KS == 0, "reduction rows per pass");
  const int cl = 4 * (threadIdx.x % CG);
#pragma unroll
  for (int i = 0; i < kBK / KS; ++i) {
    const int kl = threadIdx.x / CG + KS * i;
    const int64_t k = k0 + kl;
    float f[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t col = c0 + cl + j;
      f[j] = (k < klim && col < clim) ? p[k * ld + col] * scale : 0.0f;
    }
    uint32_t h0, h1, l0, l1;
    split2(f[0], f[1], h0, l0);
    split2(f[2], f[3], h1, l1);
    const int o = kl * ldb_t(R) + cl;
    *(uint2 *)(Sh + o) = make_uint2(h0, h1);
    *(uint2 *)(Sl + o) = make_uint2(l0, l1);
  }
}

// ---- the kernel --------------------------------------------------------------
// WF = ROWK: forward (W rows are the output columns); WF = KROW: grad_x (W
// rows are the reduction).  XF: activations bf16 (0) or fp32 (1).  Waves in
// a 2 x WGN grid, each WTM x WTN of the block's BM x BN outputs.  LDS per
// stage: Ah[BM][32], Al[BM][32], Bh[BN][32], Bl[BN][32]; two stages, then the
// 16-entry codebook.  gridDim.y > 1 splits the reduction: block (x, z)
// covers steps [z S / Z, (z + 1) S / Z) of the S 32-wide steps and writes its
// partial sums to C + z * split_stride; the LoRA segment goes to split 0.
template <class C, int WF, int XF, int KIND>
__global__ __launch_bounds__(C::T, 2) void k_nf4_bf16(Bf16GemmArgs g, int tiles_n) {
  constexpr int TM = C::TM, TN = C::TN, BM = C::BM, BN = C::BN, KS = C::KS;
  // B: the forward's W rows as 32-element LDS rows; the input gradient's
  // 32 W rows row-major (ldb_t(BN) per row)
  constexpr int A_ELEMS = BM * kBK, B_ELEMS = WF == ROWK ? BN * kBK : kBK * ldb_t(BN);
  constexpr int SUB = 2 * A_ELEMS + 2 * B_ELEMS;  // one 32-wide sub-tile
  constexpr int STAGE = KS * SUB;
  extern __shared__ __align__(16) uint16_t smem[];
  float *lut = (float *)(smem + 2 * STAGE);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, h = lane >> 5;
  const int wm0 = (wave / C::WGN) * C::WTM, wn0 = (wave % C::WGN) * C::WTN;
  // Blocks go to the 8 XCDs round robin (block b to XCD b % 8): give each
  // XCD a contiguous run of tiles (whole rows of them), so that the blocks
  // sharing an activation panel share an L2.
  const int nb = (int)gridDim.x;
  int tb = (int)blockIdx.x;
  if (nb % 8 == 0) tb = (tb % 8) * (nb / 8) + tb / 8;
  const int64_t m0 = (int64_t)(tb / tiles_n) * BM, nt = tb % tiles_n;
  // forward: the output tile's segment (the tiles of segment s start at
  // seg[s].tile0); input gradient: one output, all segments reduced
  int sg = 0;
  if (WF == ROWK)
    while (sg + 1 < g.nseg && nt >= g.seg[sg + 1].tile0) ++sg;
  const int64_t n0 = (nt - (WF == ROWK ? g.seg[sg].tile0 : 0)) * BN;
  const int64_t n_end = WF == ROWK ? g.seg[sg].len : g.N;  // output columns
  const int z = (int)blockIdx.y, nz = (int)gridDim.y;
  if (tid < 16) lut[tid] = c_lut_bf[tid];

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

  // Input gradient: the B operand of lane l (column l % 32 of the MFMA's
  // 32, reduction rows 8 (l / 32) ... + 8) from the row-major W tile by two
  // LDS transpose loads.  Within each 16 lanes, ds_read_b64_tr_b16 gives
  // lane i element i % 4 of the 8-byte pieces read by lanes i / 4 + 4 q,
  // q = 0..3: lane i reads columns c0 + 4 (i % 4) ... + 4 of row r0 + i / 4
  // (+ 4 for the second load), and receives rows r0 ... r0 + 3 (+ 4) of
  // column c0 + i.
  typedef short v4s __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) v4s lds_v4s;
  auto tr_operand = [&](const uint16_t *B, int r0, int c0, int ln) {
    const int i = ln & 15;
    const uint16_t *p = B + (r0 + (i >> 2)) * ldb_t(BN) + c0 + 4 * (i & 3);
    const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s *)p);
    const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s *)(p + 4 * ldb_t(BN)));
    typedef short v8s __attribute__((ext_vector_type(8)));
    const v8s v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(bf16x8_t, v);
  };
  // 2 x 16 of the reduction from one stage: ah.bh + ah.bl (+ al.bh when the
  // A operand has a lo part).
  auto mma = [&](const uint16_t *Ah, const uint16_t *Al, const uint16_t *Bh, const uint16_t *Bl,
                 bool a_lo) {
#pragma unroll
    for (int kk = 0; kk < kBK / 16; ++kk) {
      bf16x8_t ah[TM], al[TM], bh[TN], bl[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        ah[i] = *(const bf16x8_t *)(Ah + sw(wm0 + 32 * i + l32, 2 * kk + h));
        if (a_lo) al[i] = *(const bf16x8_t *)(Al + sw(wm0 + 32 * i + l32, 2 * kk + h));
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        if constexpr (WF == ROWK) {
          bh[j] = *(const bf16x8_t *)(Bh + sw(wn0 + 32 * j + l32, 2 * kk + h));
          bl[j] = *(const bf16x8_t *)(Bl + sw(wn0 + 32 * j + l32, 2 * kk + h));
        } else {
          bh[j] = tr_operand(Bh, 16 * kk + 8 * h, wn0 + 32 * j + 16 * ((lane >> 4) & 1), lane);
          bl[j] = tr_operand(Bl, 16 * kk + 8 * h, wn0 + 32 * j + 16 * ((lane >> 4) & 1), lane);
        }
      }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[i], bh[j], acc[i][j], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[i], bl[j], acc[i][j], 0, 0, 0);
      if (a_lo) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al[i], bh[j], acc[i][j], 0, 0, 0);
      }
    }
  };

  // ---- segment 1: activations x dequantized weight ---------------------------
  using WT = typename std::conditional<WF == ROWK, WTileRow<C, KIND>, WTileKRow<C, KIND>>::type;
  struct Regs {  // one step's loads: KS sub-tiles
    ActTile<XF, C> a[KS];
    WT w[KS];
  };
  // Steps of KS x 32: the forward walks K; the input gradient walks the
  // segments one after the other, each from its first row.
  constexpr int64_t SK = KS * kBK;
  int64_t steps = 0;
  if (WF == ROWK) {
    steps = (g.K + SK - 1) / SK;
  } else {
    for (int i = 0; i < g.nseg; ++i) steps += (g.seg[i].len + SK - 1) / SK;
  }
  const int64_t t0 = steps * z / nz, t1 = steps * (z + 1) / nz;
  auto stage = [&](uint16_t *D, const Regs &R) {
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      uint16_t *E = D + u * SUB;
      R.a[u].store(E, E + A_ELEMS);
      R.w[u].store(E + 2 * A_ELEMS, E + 2 * A_ELEMS + B_ELEMS, lut);
    }
  };
  auto load = [&](Regs &R, int64_t t) {
    if constexpr (WF == ROWK) {
#pragma unroll
      for (int u = 0; u < KS; ++u) {
        const int64_t k = (t * KS + u) * kBK;
        R.a[u].load(g.A, g.lda, m0, g.M, k, g.K);
        R.w[u].load(g.seg[sg].w, n0, k);
      }
    } else {
      int i = 0;
      int64_t tl = t;
      for (; i + 1 < g.nseg; ++i) {
        const int64_t st = (g.seg[i].len + SK - 1) / SK;
        if (tl < st) break;
        tl -= st;
      }
      const Bf16Seg &q = g.seg[i];
#pragma unroll
      for (int u = 0; u < KS; ++u) {
        const int64_t k = (tl * KS + u) * kBK;
        R.a[u].load(q.A, q.lda, m0, g.M, k, q.len);
        R.w[u].load(q.w, n0, k);
      }
    }
  };
  auto mma_stage = [&](const uint16_t *S) {
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      const uint16_t *E = S + u * SUB;
      mma(E, E + A_ELEMS, E + 2 * A_ELEMS, E + 2 * A_ELEMS + B_ELEMS, XF == 1);
    }
  };
  Regs ra;
  if constexpr (C::PP) {
    // Ping-pong: waves 0-3 (group 0) and 4-7 (group 1), one of each per SIMD,
    // take turns: while group 0 runs step t's MFMAs, group 1 dequantizes and
    // writes its half of step t + 1 (A rows BM/2 .., W rows or columns
    // BN/2 ..); after a barrier the roles swap.  So a SIMD keeps one wave on
    // the matrix core while the other does the VALU work.  Two barriers per
    // step; step t + 1's LDS stage is complete (both halves) before either
    // group reads it, and step t's is read by both before step t + 2's
    // writes start.
    using HC = Cfg<C::T / 2, BM / 2, BN / 2>;
    using HW = typename std::conditional<WF == ROWK, WTileRow<HC, KIND>,
                                         WTileKRow<HC, KIND, ldb_t(BN)>>::type;
    struct HRegs {
      ActTile<XF, HC> a;
      HW w;
    };
    const int grp = wave >= C::T / 128 ? 1 : 0;  // wave-uniform
    auto hload = [&](HRegs &R, int64_t t, int hf) {
      const int64_t k = t * kBK, ma = m0 + hf * (BM / 2), nb = n0 + hf * (BN / 2);
      if constexpr (WF == ROWK) {
        R.a.load(g.A, g.lda, ma, g.M, k, g.K);
        R.w.load(g.seg[sg].w, nb, k);
      } else {
        int i = 0;
        int64_t tl = t;
        for (; i + 1 < g.nseg; ++i) {
          const int64_t st = (g.seg[i].len + kBK - 1) / kBK;
          if (tl < st) break;
          tl -= st;
        }
        const Bf16Seg &q = g.seg[i];
        R.a.load(q.A, q.lda, ma, g.M, tl * kBK, q.len);
        R.w.load(q.w, nb, tl * kBK);
      }
    };
    auto hstage = [&](uint16_t *D, const HRegs &R, int hf) {
      const int ao = hf * (BM / 2) * kBK;
      R.a.store(D + ao, D + A_ELEMS + ao);
      const int bo = WF == ROWK ? hf * (BN / 2) * kBK : hf * (BN / 2);
      R.w.store(D + 2 * A_ELEMS + bo, D + 2 * A_ELEMS + B_ELEMS + bo, lut);
    };
    // one copy of the loop per group, its half a constant.  Two register
    // sets per wave: a group's loads for a step go out about three phases
    // before it writes them (group 0 loads step t + 2 as it starts step t's
    // MFMAs, group 1 loads step t + 3 as it starts them), so the staging
    // rarely waits for memory.  The loop runs two steps per turn to keep the
    // sets in fixed registers.
    auto run = [&](auto G) {
      constexpr int gp = decltype(G)::value;
      HRegs ra, rb;
      hload(ra, t0, gp);
      __syncthreads();  // codebook
      hstage(smem, ra, gp);
      if (t0 + 1 < t1) hload(rb, t0 + 1, gp);
      if (gp == 1 && t0 + 2 < t1) hload(ra, t0 + 2, 1);
      __syncthreads();
      // Each step is two phases: group 0 runs step t's MFMAs while group 1
      // writes its half of step t + 1; then group 1 runs step t's MFMAs
      // while group 0 writes its half of step t + 1.  (Each group's loop is
      // straight-line code: with the roles chosen by a branch in one loop the
      // compiler spilled the accumulators.)  `rc` holds step t's loads
      // (already written), `rn` step t + 1's.
      auto step = [&](int64_t t, HRegs &rc, HRegs &rn) {
        uint16_t *cur = smem + ((t - t0) & 1) * STAGE, *nxt = smem + ((t + 1 - t0) & 1) * STAGE;
        if constexpr (gp == 0) {
          if (t + 2 < t1) hload(rc, t + 2, 0);
          mma_stage(cur);
          __syncthreads();
          if (t + 1 < t1) hstage(nxt, rn, 0);
          __syncthreads();
        } else {
          if (t + 1 < t1) hstage(nxt, rn, 1);
          __syncthreads();
          if (t + 3 < t1) hload(rn, t + 3, 1);
          mma_stage(cur);
          __syncthreads();
        }
      };
      for (int64_t t = t0; t < t1; t += 2) {
        step(t, ra, rb);
        if (t + 1 < t1) step(t + 1, rb, ra);
      }
    };
    if (t1 > t0) {
      if (grp == 0) run(std::integral_constant<int, 0>{});
      else run(std::integral_constant<int, 1>{});
    }
  } else if constexpr (C::PF == 1) {
    if (t1 > t0) {
      load(ra, t0);
      __syncthreads();  // codebook
      stage(smem, ra);
      __syncthreads();
      for (int64_t t = t0; t < t1; ++t) {
        const bool more = t + 1 < t1;
        if (more) load(ra, t + 1);
        mma_stage(smem + ((t - t0) & 1) * STAGE);
        if (more) stage(smem + ((t + 1 - t0) & 1) * STAGE, ra);
        __syncthreads();
      }
    }
  } else {
    // Two register sets: at the top of step t the LDS stage of t is full, the
    // loads of step t + 1 are in flight in one set and step t + 2's go out
    // into the other, so each load has two steps of MFMAs to arrive.  The
    // loop runs two steps per turn to keep the sets in fixed registers.
    Regs rb;
    uint16_t *S0 = smem, *S1 = smem + STAGE;
    if (t1 > t0) {
      load(ra, t0);
      if (t0 + 1 < t1) load(rb, t0 + 1);
      __syncthreads();  // codebook
      stage(S0, ra);
      __syncthreads();
      for (int64_t t = t0; t < t1; t += 2) {
        if (t + 2 < t1) load(ra, t + 2);
        mma_stage(S0);
        if (t + 1 < t1) stage(S1, rb);
        __syncthreads();
        if (t + 1 >= t1) break;
        if (t + 3 < t1) load(rb, t + 3);
        mma_stage(S1);
        if (t + 2 < t1) stage(S0, ra);
        __syncthreads();
      }
    }
  }

  // ---- the LoRA terms, three MFMAs per tile ----------------------------------
  if (z == 0) {
    uint16_t *Ah = smem, *Al = smem + A_ELEMS;
    uint16_t *Bh = smem + 2 * A_ELEMS, *Bl = smem + 2 * A_ELEMS + B_ELEMS;
    const int i0 = WF == ROWK ? sg : 0, i1 = WF == ROWK ? sg + 1 : g.nseg;
    for (int i = i0; i < i1; ++i) {
      const Bf16Seg &q = g.seg[i];
      for (int64_t k0 = 0; k0 < q.K2; k0 += kBK) {
        stage_f32_rowk<BM, C::T>(q.A2, q.lda2, m0, g.M, k0, q.K2, 1.0f, Ah, Al);
        if (WF == ROWK)
          stage_f32_rowk<BN, C::T>(q.B2, q.ldb2, n0, n_end, k0, q.K2, q.b2scale, Bh, Bl);
        else
          stage_f32_krow<BN, C::T>(q.B2, q.ldb2, n0, n_end, k0, q.K2, q.b2scale, Bh, Bl);
        __syncthreads();
        mma(Ah, Al, Bh, Bl, true);
        __syncthreads();
      }
    }
  }

  // ---- epilogue ---------------------------------------------------------------
  float *Cz = (WF == ROWK ? g.seg[sg].C : g.C) + (nz > 1 ? (int64_t)z * g.split_stride : 0);
  const int64_t ldc = WF == ROWK ? g.seg[sg].ldc : g.ldc;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int64_t m = m0 + wm0 + 32 * i + 8 * (v / 4) + 4 * h + (v % 4);
        const int64_t n = n0 + wn0 + 32 * j + l32;
        if (m < g.M && n < n_end) {
          const float o = g.alpha * acc[i][j][v];
          Cz[m * ldc + n] = g.beta ? Cz[m * ldc + n] + o : o;
        }
      }
}

template <class C, int WF, int XF, int KIND>
hipError_t run_bf16(const Bf16GemmArgs &g0, int splits, float *partial, hipStream_t s) {
  auto k = k_nf4_bf16<C, WF, XF, KIND>;
  constexpr int b_elems = WF == ROWK ? C::BN * kBK : kBK * ldb_t(C::BN);
  constexpr uint32_t lds = (uint32_t)(2 * C::KS * (2 * C::BM * kBK + 2 * b_elems) * 2 + 16 * 4);
  static bool attr = false;  // per instantiation
  if (!attr) {
    const hipError_t e =
        hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    attr = true;
  }
  Bf16GemmArgs g = g0;
  int tiles_n = 0;
  if (WF == ROWK) {
    for (int i = 0; i < g.nseg; ++i) {
      g.seg[i].tile0 = tiles_n;
      tiles_n += (int)((g.seg[i].len + C::BN - 1) / C::BN);
    }
  } else {
    tiles_n = (int)((g.N + C::BN - 1) / C::BN);
  }
  if (splits > 1) {
    g.beta = 0;  // the partials are written plain; the reduction adds the residual
    if (WF == ROWK) {  // one segment (checked by the caller)
      g.seg[0].C = partial;
      g.seg[0].ldc = g.seg[0].len;
    } else {
      g.C = partial;
      g.ldc = g.N;
    }
    g.split_stride = g.M * g.N;
  }
  const int tiles_m = (int)((g.M + C::BM - 1) / C::BM);
  hipError_t e = qh_launch(k, dim3((unsigned)(tiles_n * tiles_m), (unsigned)splits),
                           dim3(C::T), lds, s, g, tiles_n);
  if (e != hipSuccess || splits <= 1) return e;
  return WF == ROWK ? launch_reduce_splits(partial, splits, g.M, g.N, g0.seg[0].C,
                                           g0.seg[0].ldc, s, g0.beta)
                    : launch_reduce_splits(partial, splits, g.M, g.N, g0.C, g0.ldc, s, g0.beta);
}

// Block shape and reduction splits by problem size.
//  large:  256 x 256 or 256 x 128 tiles, 8 waves, for problems with at least
//          256 tiles of 256 x 256 (MFMA-bound); most of these go through the
//          operand planes of k_plane.hip instead (4096^3 in fp32 400 us here,
//          350 there).  Here come those that planes would not speed up (few
//          columns or rows against the other sizes, K below 512), whose planes
//          pass 2 GiB or cannot have their memory (a full device, a capture
//          before a warm-up), groups, and the allocation-free backward;
//  medium: 128 x 128 tiles, 8 waves, loads two steps ahead, two 32-wide
//          sub-steps per barrier (one when there are more tiles than CUs,
//          so that two blocks share a CU), for 160 or more tiles of
//          128 x 128, or long reductions (24+ steps) over 32+ such tiles;
//  small:  64 x 64 tiles, 4 waves, the same pipelining.
// The medium and small blocks' step loops are latency-bound (about 0.7 us
// per step at C4's shapes), so long reductions are split until the GPU
// holds about one block per CU (four small ones for reductions of 24+
// steps), each split keeping at least 6 steps; at most 8 splits and 64 MB of
// partial sums.
enum Tier { kLarge, kMedium, kSmall };
struct Plan {
  Tier tier;
  int splits;
};
Plan plan_for(int64_t M, int64_t N, int64_t K) {
  const int64_t steps = (K + kBK - 1) / kBK;
  if (M >= 256 && N >= 256 && (M / 256) * (N / 256) >= 256) return Plan{kLarge, 1};
  const int64_t t128 = ((M + 127) / 128) * ((N + 127) / 128);
  int64_t tiles, target;
  Tier tier;
  if (t128 >= 160 || (steps >= 24 && t128 >= 32)) {
    tier = kMedium, tiles = t128, target = 256;
  } else {
    tier = kSmall, tiles = ((M + 63) / 64) * ((N + 63) / 64), target = steps >= 24 ? 1024 : 256;
  }
  int64_t sp = (target + tiles / 2) / (tiles ? tiles : 1);
  if (sp > 8) sp = 8;
  // at least 6 steps per split; a GEMM of at most 16 tiles takes up to 6
  // splits of at least 3 steps (C1's 9 tiles of 18 steps: 6 splits 7.4-7.7
  // us per GEMM against 9.8-10.4 with 3, 2 and 1 slower still)
  const bool few = tiles <= 16;
  if (sp > (few ? steps / 3 : steps / 6)) sp = few ? steps / 3 : steps / 6;
  if (few && sp > 6) sp = 6;
  while (sp > 1 && (size_t)(sp * M * N * 4) > ((size_t)64 << 20)) --sp;
  return Plan{tier, sp < 1 ? 1 : (int)sp};
}

// Large tier: 256 x 256 tiles where they fill at least 3/4 of their rounds of
// 256 workgroups, else 256 x 128.
bool wide_tiles(int64_t M, int64_t N) {
  const int64_t t256 = ((M + 255) / 256) * ((N + 255) / 256), waves = (t256 + 255) / 256;
  return t256 >= 192 && (double)t256 / (double)(waves * 256) >= 0.75;
}

template <int WF, int XF, int KIND>
hipError_t pick(const Bf16GemmArgs &g, int splits, float *partial, hipStream_t s) {
  const Plan pl = plan_for(g.M, g.N, g.K);
  if (pl.tier == kSmall) return run_bf16<CfgS, WF, XF, KIND>(g, splits, partial, s);
  if (pl.tier == kMedium) {
    // more tiles than CUs: one sub-tile per barrier, so two blocks fit a CU
    if (((g.M + 127) / 128) * ((g.N + 127) / 128) > 256)
      return run_bf16<CfgM1, WF, XF, KIND>(g, splits, partial, s);
    return run_bf16<CfgM, WF, XF, KIND>(g, splits, partial, s);
  }
  return wide_tiles(g.M, g.N) ? run_bf16<CfgL256, WF, XF, KIND>(g, 1, nullptr, s)
              : run_bf16<CfgL128, WF, XF, KIND>(g, 1, nullptr, s);
}

template <int WF, int XF>
hipError_t pick_kind(const Bf16GemmArgs &g, int splits, float *partial, hipStream_t s) {
  return g.seg[0].w.kind == 0 ? pick<WF, XF, 0>(g, splits, partial, s)
                              : pick<WF, XF, 1>(g, splits, partial, s);
}

// ---- dense GEMMs on bf16 MFMA: the LoRA-rank products ------------------------
// C = alpha * sum_k A(m, k) B(n, k) with both operands dense fp32 (split into
// bf16 hi + lo) or bf16, each stored either ROWK (row-major along k: staged
// like the activations above) or KROW (k is the row: staged row-major with
// the LDS row stride ldb_t and read by the transpose loads).  Products run
// as ah.bh (+ ah.bl for an fp32 B, + al.bh for an fp32 A).  One output side
// is a LoRA rank (<= 64): 128 x 64 or 64 x 128 tiles, 4 waves, reduction
// split over blocks with partial sums summed in a fixed order.
struct DenseArgs {
  int64_t M, N, K;
  const void *A;  // A(m, k) at A[m lda + k] (ROWK) or A[k lda + m] (KROW)
  int64_t lda;
  const void *B;  // B(n, k) at B[n ldb + k] (ROWK) or B[k ldb + n] (KROW)
  int64_t ldb;
  float *C;
  int64_t ldc;
  float alpha;
  int64_t split_stride;
};

// 32 rows (k) x R columns of a row-major matrix S[k][col] (ld), fp32 (XE = 1,
// split) or bf16, into the transposed LDS layout (row stride ldb_t(R)).
// Thread t (of T) holds EPT consecutive columns of row t / TPR; columns are
// taken in groups of 8 (clim % 8 == 0, 16-byte aligned rows), zeroed at the
// LDS write when out of range.
template <int XE, int T, int R>
struct KTile {
  static constexpr int EPT = R * kBK / T;  // 8 or 16
  static constexpr int TPR = R / EPT;
  static constexpr int NG = EPT / 8;       // groups of 8 columns
  static_assert(EPT == 8 || EPT == 16, "columns per thread");
  static_assert(TPR * kBK == T, "one row per TPR threads");
  float4 f[XE ? 2 * NG : 1];
  uint4 b[XE ? 1 : NG];
  uint32_t okm;
  __device__ __forceinline__ void load(const void *S, int64_t ld, int64_t k0, int64_t klim,
                                       int64_t c0, int64_t clim) {
    const int t = threadIdx.x % T;
    const int64_t k = k0 + t / TPR, c = c0 + (t % TPR) * EPT;
    okm = 0;
#pragma unroll
    for (int q = 0; q < NG; ++q) {
      const bool ok = k < klim && c + 8 * q < clim;
      const int64_t e = ok ? k * ld + c + 8 * q : 0;
      if constexpr (XE) {
        f[2 * q] = *(const float4 *)((const float *)S + e);
        f[2 * q + 1] = *(const float4 *)((const float *)S + e + 4);
      } else {
        b[q] = *(const uint4 *)((const uint16_t *)S + e);
      }
      okm |= (uint32_t)ok << q;
    }
  }
  __device__ __forceinline__ void store(uint16_t *Sh, uint16_t *Sl) const {
    const int t = threadIdx.x % T;
    const int o0 = (t / TPR) * ldb_t(R) + (t % TPR) * EPT;
#pragma unroll
    for (int q = 0; q < NG; ++q) {
      const bool ok = (okm >> q) & 1u;
      if constexpr (XE) {
        const float4 z = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        float4 u0 = f[2 * q], u1 = f[2 * q + 1];
        if (!ok) u0 = z, u1 = z;
        uint32_t h[4], l[4];
        split2(u0.x, u0.y, h[0], l[0]);
        split2(u0.z, u0.w, h[1], l[1]);
        split2(u1.x, u1.y, h[2], l[2]);
        split2(u1.z, u1.w, h[3], l[3]);
        *(uint4 *)(Sh + o0 + 8 * q) = make_uint4(h[0], h[1], h[2], h[3]);
        *(uint4 *)(Sl + o0 + 8 * q) = make_uint4(l[0], l[1], l[2], l[3]);
      } else {
        uint4 v = b[q];
        if (!ok) v = make_uint4(0, 0, 0, 0);
        *(uint4 *)(Sh + o0 + 8 * q) = v;
      }
    }
  }
};

// Elements of one operand stage: ROWK R x 32, KROW 32 x ldb_t(R).
__host__ __device__ constexpr int dense_elems(int form, int R) {
  return form == ROWK ? R * kBK : kBK * ldb_t(R);
}

template <class C, int AF, int BF, int XA, int XB>
__global__ __launch_bounds__(C::T, 2) void k_dense_bf16(DenseArgs g, int tiles_n) {
  constexpr int TM = C::TM, TN = C::TN, BM = C::BM, BN = C::BN;
  constexpr int AE = dense_elems(AF, BM), BE = dense_elems(BF, BN);
  constexpr int STAGE = 2 * AE + 2 * BE;
  extern __shared__ __align__(16) uint16_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, h = lane >> 5;
  const int wm0 = (wave / C::WGN) * C::WTM, wn0 = (wave % C::WGN) * C::WTN;
  const int nb = (int)gridDim.x;
  int tb = (int)blockIdx.x;
  if (nb % 8 == 0) tb = (tb % 8) * (nb / 8) + tb / 8;
  const int64_t m0 = (int64_t)(tb / tiles_n) * BM, n0 = (int64_t)(tb % tiles_n) * BN;
  const int z = (int)blockIdx.y, nz = (int)gridDim.y;

  // operand tiles in registers: ROWK through the activation tile, KROW
  // through KTile
  using CA = Cfg<C::T, BM, 64>;
  using CB = Cfg<C::T, BN, 64>;
  using TA = typename std::conditional<AF == ROWK, ActTile<XA, CA>, KTile<XA, C::T, BM>>::type;
  using TB = typename std::conditional<BF == ROWK, ActTile<XB, CB>, KTile<XB, C::T, BN>>::type;
  struct Regs {
    TA a;
    TB b;
  };
  const int64_t steps = (g.K + kBK - 1) / kBK;
  const int64_t t0 = steps * z / nz, t1 = steps * (z + 1) / nz;
  auto load = [&](Regs &R, int64_t t) {
    const int64_t k = t * kBK;
    if constexpr (AF == ROWK) R.a.load(g.A, g.lda, m0, g.M, k, g.K);
    else R.a.load(g.A, g.lda, k, g.K, m0, g.M);
    if constexpr (BF == ROWK) R.b.load(g.B, g.ldb, n0, g.N, k, g.K);
    else R.b.load(g.B, g.ldb, k, g.K, n0, g.N);
  };
  auto stage = [&](uint16_t *D, const Regs &R) {
    R.a.store(D, D + AE);
    R.b.store(D + 2 * AE, D + 2 * AE + BE);
  };
  typedef short v4s __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) v4s lds_v4s;
  // transposed layout: rows r0 .. r0 + 8 of column c0 + lane % 16 (see mma
  // in k_nf4_bf16)
  auto tr_operand = [&](const uint16_t *B, int ld, int r0, int c0) {
    const int i = lane & 15;
    const uint16_t *p = B + (r0 + (i >> 2)) * ld + c0 + 4 * (i & 3);
    const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s *)p);
    const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s *)(p + 4 * ld));
    typedef short v8s __attribute__((ext_vector_type(8)));
    const v8s v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(bf16x8_t, v);
  };
  auto operand = [&](const uint16_t *S, int form, int ld, int row0, int kk) {
    if (form == ROWK) return *(const bf16x8_t *)(S + sw(row0 + l32, 2 * kk + h));
    return tr_operand(S, ld, 16 * kk + 8 * h, row0 + 16 * ((lane >> 4) & 1));
  };

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;
  auto mma = [&](const uint16_t *D) {
    const uint16_t *Ah = D, *Al = D + AE, *Bh = D + 2 * AE, *Bl = D + 2 * AE + BE;
#pragma unroll
    for (int kk = 0; kk < kBK / 16; ++kk) {
      bf16x8_t ah[TM], al[TM], bh[TN], bl[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        ah[i] = operand(Ah, AF, ldb_t(BM), wm0 + 32 * i, kk);
        if (XA) al[i] = operand(Al, AF, ldb_t(BM), wm0 + 32 * i, kk);
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        bh[j] = operand(Bh, BF, ldb_t(BN), wn0 + 32 * j, kk);
        if (XB) bl[j] = operand(Bl, BF, ldb_t(BN), wn0 + 32 * j, kk);
      }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[i], bh[j], acc[i][j], 0, 0, 0);
          if (XB)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[i], bl[j], acc[i][j], 0, 0, 0);
          if (XA)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al[i], bh[j], acc[i][j], 0, 0, 0);
        }
    }
  };
  if (t1 > t0) {
    Regs R;
    load(R, t0);
    stage(smem, R);
    __syncthreads();
    for (int64_t t = t0; t < t1; ++t) {
      const bool more = t + 1 < t1;
      if (more) load(R, t + 1);
      mma(smem + ((t - t0) & 1) * STAGE);
      if (more) stage(smem + ((t + 1 - t0) & 1) * STAGE, R);
      __syncthreads();
    }
  }
  float *Cz = g.C + (nz > 1 ? (int64_t)z * g.split_stride : 0);
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int64_t m = m0 + wm0 + 32 * i + 8 * (v / 4) + 4 * h + (v % 4);
        const int64_t n = n0 + wn0 + 32 * j + l32;
        if (m < g.M && n < g.N) Cz[m * g.ldc + n] = g.alpha * acc[i][j][v];
      }
}

using CfgD1 = Cfg<256, 128, 64>;  // N is the rank
using CfgD2 = Cfg<256, 64, 128>;  // M is the rank

template <class C, int AF, int BF, int XA, int XB>
hipError_t run_dense(const DenseArgs &g0, int splits, float *partial, hipStream_t s) {
  auto k = k_dense_bf16<C, AF, BF, XA, XB>;
  constexpr uint32_t lds =
      (uint32_t)(2 * (2 * dense_elems(AF, C::BM) + 2 * dense_elems(BF, C::BN)) * 2);
  static bool attr = false;  // per instantiation
  if (!attr) {
    const hipError_t e =
        hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    attr = true;
  }
  DenseArgs g = g0;
  if (splits > 1) {
    g.C = partial;
    g.ldc = g.N;
    g.split_stride = g.M * g.N;
  }
  const int tiles_n = (int)((g.N + C::BN - 1) / C::BN);
  const int tiles_m = (int)((g.M + C::BM - 1) / C::BM);
  hipError_t e = qh_launch(k, dim3((unsigned)(tiles_n * tiles_m), (unsigned)splits),
                           dim3(C::T), lds, s, g, tiles_n);
  if (e != hipSuccess || splits <= 1) return e;
  return launch_reduce_splits(partial, splits, g.M, g.N, g0.C, g0.ldc, s);
}

template <class C, int AF, int BF>
hipError_t dense_types(const DenseArgs &g, int xa, int xb, int splits, float *partial,
                       hipStream_t s) {
  if (xa && xb) return run_dense<C, AF, BF, 1, 1>(g, splits, partial, s);
  if (xa) return run_dense<C, AF, BF, 1, 0>(g, splits, partial, s);
  if (xb) return run_dense<C, AF, BF, 0, 1>(g, splits, partial, s);
  return run_dense<C, AF, BF, 0, 0>(g, splits, partial, s);
}

// Block shape: the rank side gets the 64-wide tile side.
bool dense_rank_n(int64_t M, int64_t N) { return N <= 64 || M > 64; }

int dense_splits_for(int64_t M, int64_t N, int64_t K) {
  const bool rn = dense_rank_n(M, N);
  const int64_t tiles = ((M + (rn ? 127 : 63)) / (rn ? 128 : 64)) *
                        ((N + (rn ? 63 : 127)) / (rn ? 64 : 128));
  const int64_t steps = (K + kBK - 1) / kBK;
  int64_t sp = (768 + tiles - 1) / (tiles ? tiles : 1);
  if (sp > 16) sp = 16;
  if (sp > steps / 8) sp = steps / 8;
  while (sp > 1 && (size_t)(sp * M * N * 4) > ((size_t)64 << 20)) --sp;
  return sp < 1 ? 1 : (int)sp;
}

}  // namespace

// The bf16-MFMA path needs whole 64-element blocks per W row, and activation
// rows it can read as 16-byte vectors (8 elements).
bool bf16_gemm_ok(const DevQW &w, const void *a, int64_t lda, int64_t K) {
  return w.bs == 64 && w.cols % 64 == 0 && lda % 8 == 0 && K % 8 == 0 &&
         (((uintptr_t)a) & 15) == 0;
}

int bf16_gemm_splits(int64_t M, int64_t N, int64_t K) { return plan_for(M, N, K).splits; }

// Fitted to some 2000 forwards and input gradients (16 to 65536 rows and columns, K
// 320 to 11008): within 6 % rms, 3 % above 40 us.  A step of 32 k costs what the
// rounds of workgroups take at full and at partial occupancy (two blocks of the
// medium tier fit a CU where it has more tiles than CUs, four small ones do),
// plus the tiles' share of operand traffic.
double bf16_gemm_us(int64_t M, int64_t N, int64_t K, bool f32, bool split) {
  const Plan p = plan_for(M, N, K);
  const auto up = [](int64_t a, int64_t b) { return (double)((a + b - 1) / b); };
  const int64_t steps = (K + kBK - 1) / kBK;
  const double mn = (double)M * (double)N * 1e-6, mk = (double)M * (double)K * 1e-6;
  if (p.tier == kLarge) {
    const bool wide = wide_tiles(M, N);
    const double t = up(M, 256) * up(N, wide ? 256 : 128), wg = t / 256, R = up((int64_t)t, 256);
    const double s = (double)steps;
    if (wide)
      return f32 ? 0.5 + s * (1.383 * R + 1.204 * wg) + 1.7 * R + 0.55 * mn + 0.19 * mk
                 : 1.8 + s * (1.083 * R + 0.732 * wg) + 4.6 * R + 0.395 * mn + 0.04 * mk;
    return f32 ? 5.3 + s * (1.16 * R + 0.368 * wg) + 3.5 * R + 0.185 * mn + 0.525 * mk
               : 5.4 + s * (0.866 * R + 0.2 * wg) + 6.3 * R - 0.15 * mn + 0.3 * mk;
  }
  const int sp = split ? p.splits : 1;
  const double tile = p.tier == kMedium ? 128 : 64, t = up(M, (int64_t)tile) * up(N, (int64_t)tile);
  const double wg = t * sp / 256, R = up((int64_t)t * sp, 256), ks = up(steps, sp);
  if (p.tier == kSmall)
    return 3.65 + ks * (f32 ? 0.53 + 0.145 * (R - 1) + 0.11 * wg : 0.425 + 0.108 * (R - 1) + 0.083 * wg) +
           (sp > 1 ? 2.1 + 2 * sp * mn : 0);
  if (t <= 256)
    return 5.6 + ks * (f32 ? 0.95 + 0.9 * (R - 1) + 0.09 * wg : 0.8 + 0.72 * (R - 1)) +
           (sp > 1 ? 0.18 + 2.85 * sp * mn : 0) + (f32 ? 0.7 : 0.5) * mn;
  const double R2 = up((int64_t)t * sp, 512);
  return f32 ? 5.8 + ks * (0.277 * R2 + 0.467 * R + 0.285 * wg) + 0.36 * mn + 0.15 * mk
             : 6.2 + ks * (0.258 * R2 + 0.393 * R + 0.126 * wg) + 0.3 * mn + 0.044 * mk;
}

hipError_t launch_gemm_bf16(const Bf16GemmArgs &g, int w_form, int a_f32, int splits,
                            float *partial, hipStream_t s) {
  if (g.M == 0 || g.N == 0) return hipSuccess;
  if (splits < 1 || (splits > 1 && !partial) || g.nseg < 1 || g.nseg > kMaxBf16Segs ||
      (splits > 1 && w_form == ROWK && g.nseg != 1))
    return hipErrorInvalidValue;
  // activation rows are read as 16-byte vectors of 8 elements: row strides
  // and lengths multiples of 8, rows 16-byte aligned
  auto vec_ok = [](const void *a, int64_t lda, int64_t k) {
    return lda % 8 == 0 && k % 8 == 0 && (((uintptr_t)a) & 15) == 0;
  };
  int64_t n_sum = 0;
  for (int i = 0; i < g.nseg; ++i) {
    const Bf16Seg &q = g.seg[i];
    if (q.w.kind != g.seg[0].w.kind) return hipErrorInvalidValue;
    if (w_form == KROW && !vec_ok(q.A, q.lda, q.len)) return hipErrorInvalidValue;
    n_sum += q.len;
  }
  if (w_form == ROWK && (!vec_ok(g.A, g.lda, g.K) || n_sum != g.N)) return hipErrorInvalidValue;
  if (w_form == KROW && n_sum != g.K) return hipErrorInvalidValue;
  if (w_form == ROWK) return a_f32 ? pick_kind<ROWK, 1>(g, splits, partial, s)
                                   : pick_kind<ROWK, 0>(g, splits, partial, s);
  return a_f32 ? pick_kind<KROW, 1>(g, splits, partial, s)
               : pick_kind<KROW, 0>(g, splits, partial, s);
}

// Dense products of the LoRA rank on bf16 MFMA: row strides and the
// contiguous dimensions multiples of 8, operands 16-byte aligned, one side of
// the output at most 64.
bool dense_bf16_ok(int64_t M, int64_t N, int64_t K, int a_form, const void *a, int64_t lda,
                   int b_form, const void *b, int64_t ldb) {
  auto al = [](const void *p) { return (((uintptr_t)p) & 15) == 0; };
  if (M < 1 || N < 1 || K < 1 || (M > 64 && N > 64)) return false;
  if (!al(a) || !al(b) || lda % 8 != 0 || ldb % 8 != 0) return false;
  // the contiguous dimension of each operand is read in groups of 8
  if ((a_form == ROWK ? K : M) % 8 != 0 || (b_form == ROWK ? K : N) % 8 != 0) return false;
  return true;
}

int dense_bf16_splits(int64_t M, int64_t N, int64_t K) { return dense_splits_for(M, N, K); }

hipError_t launch_dense_bf16(const void *a, int a_form, int a_f32, int64_t lda, const void *b,
                             int b_form, int b_f32, int64_t ldb, float *c, int64_t ldc,
                             int64_t M, int64_t N, int64_t K, float alpha, float *partial,
                             hipStream_t s) {
  if (M == 0 || N == 0) return hipSuccess;
  if (!dense_bf16_ok(M, N, K, a_form, a, lda, b_form, b, ldb)) return hipErrorInvalidValue;
  const int splits = dense_splits_for(M, N, K);
  if (splits > 1 && !partial) return hipErrorInvalidValue;
  DenseArgs g{M, N, K, a, lda, b, ldb, c, ldc, alpha, 0};
  const bool rn = dense_rank_n(M, N);
#define QH_DENSE(C_)                                                                       \
  if (a_form == ROWK && b_form == ROWK) return dense_types<C_, ROWK, ROWK>(g, a_f32, b_f32, splits, partial, s); \
  if (a_form == ROWK) return dense_types<C_, ROWK, KROW>(g, a_f32, b_f32, splits, partial, s);                  \
  if (b_form == ROWK) return dense_types<C_, KROW, ROWK>(g, a_f32, b_f32, splits, partial, s);                  \
  return dense_types<C_, KROW, KROW>(g, a_f32, b_f32, splits, partial, s);
  if (rn) {
    QH_DENSE(CfgD1)
  } else {
    QH_DENSE(CfgD2)
  }
#undef QH_DENSE
}

}  // namespace qh
