// k_plane.hip -- the large GEMMs of a QLoRA layer in two passes: the operands
// once into bf16 operand planes, then a GEMM that only moves and multiplies.
//
//   forward  Y = X . W^T + T1 . (s B)^T     (qlora-core/src/qlora.rs:86-107)
//   grad_x   dX = dY . W + Ds . A           (qlora.rs:116-165)
//
// k_nf4_bf16 (k_gemm_bf16.hip) decodes and splits its operands inside the K loop,
// every weight tile once per 256 rows of X and every X tile once per 256
// columns: its phases wait on that work (MFMA busy 0.55 of the cycles).  Here
// k_planes splits X (fp32 into hi + lo) and decodes W (hi + lo) once, in the
// order in which an MFMA operand is read, and k_plane_gemm copies 1 KiB operand
// tiles straight into LDS (global_load_lds, no registers), so its waves do
// nothing but LDS reads and MFMAs: MFMA busy 0.72 (fp32; bf16 0.68), and the card then
// runs at 1.84 GHz instead of 2.4 (the product is bound by power: steps of 32 k
// with half the barriers ran 13 % more cycles at a 7 % higher clock).  The sums are
// those of k_nf4_bf16 without a split reduction, in its order: the same bits.
//
// Measured (fp32 X, r = 64): 4096^3 GEMM 400 -> 309 us + planes 41 us (4.9 TB/s);
// with r = 16, 4096 x 4096 at 2048 tokens 268 -> 209 us forward, 294 -> 234
// backward, 11008 x 4096 at 1536 609 -> 460 / 660 -> 483; bf16 X at 2905 tokens and
// 14336 x 4096 forward + backward 1770 -> 1400 us.
#include <algorithm>
#include <type_traits>

#include "qh_internal.h"
#include "qh_nf4.h"

namespace qh {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;
typedef const __attribute__((address_space(1))) uint8_t glb_u1;
typedef const __attribute__((address_space(1))) void glb_void;

__constant__ float c_lut_pl[17] = QH_NF4_LUT17_INIT;  // the codebook (quant.rs:27-44)

__device__ __forceinline__ uint32_t pk_bf16(float a, float b) {
  const bf16x2_t h = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(uint32_t, h);
}
// hi and lo bf16 parts of two floats (the split of k_gemm_bf16.hip)
__device__ __forceinline__ void split2(float a, float b, uint32_t &hi, uint32_t &lo) {
  hi = pk_bf16(a, b);
  asm("" : "+v"(hi));
  lo = pk_bf16(a - __uint_as_float(hi << 16), b - __uint_as_float(hi & 0xffff0000u));
}
__device__ __forceinline__ float scale_of(const DevQW &w, int64_t blk) {
  if (w.kind == 0) return w.scales[blk];
  // fl(fl(c / 127) * absmax), see k_gemm_bf16.hip
  return (float)((double)(float)(int8_t)w.scale_codes[blk] * (1.0 / 127.0)) * w.absmax[blk >> 8];
}

// ---- operand planes -----------------------------------------------------------
// An operand with rows r and reduction index k is kept as 1 KiB tiles of 32 rows
// x 16 k in MFMA operand order (lane l: row l % 32, k = 8 (l / 32) ... + 8),
// [row tile][k tile][part], parts hi and (P = 2) lo.  k past the reduction is
// zero; rows past the operand are whatever the buffer held (they only reach
// outputs that are not stored).
struct PlaneJob {
  int kind;        // see k_planes
  const void *src; // dense sources
  DevQW w;         // NF4 sources
  uint8_t *dst;
  int64_t ld;
  int rows, K, KT; // KT = ceil(K / 16)
  float scale;
  int wg0;
};
struct PlaneJobs {
  PlaneJob j[4];
  int count;
};
enum PlaneKind {
  kDenseF32,  // src[r * ld + k], fp32: hi, lo (times scale)
  kDenseBf16, // src[r * ld + k], bf16: one part
  kDenseT,    // src[k * ld + r], fp32: hi, lo (times scale)
  kNf4Row,    // W row r, column k
  kNf4Col     // W column r, row k
};

constexpr int kPlThreads = 256;
constexpr int kSpan = 2;  // 64-wide pieces of k a wave takes, all loaded ahead
// Rows x k of a workgroup (4 waves): dense and NF4 rows 32 x 256 kSpan, dense
// columns 32 x 64, NF4 columns 128 columns x 64 kSpan.
int plane_wgs(int kind, int64_t rows, int64_t K) {
  if (kind == kNf4Col) return (int)(((rows + 127) / 128) * ((K + 64 * kSpan - 1) / (64 * kSpan)));
  if (kind == kDenseT) return (int)(((rows + 31) / 32) * ((K + 63) / 64));
  return (int)(((rows + 31) / 32) * ((K + 256 * kSpan - 1) / (256 * kSpan)));
}

// 8 values as hi and lo parts into a tile's 16-byte units
__device__ __forceinline__ void put2(uint8_t *o, const float (&f)[8]) {
  v4u hi, lo;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    uint32_t a, e;
    split2(f[2 * v], f[2 * v + 1], a, e);
    hi[v] = a, lo[v] = e;
  }
  *(v4u *)o = hi;
  *(v4u *)(o + 1024) = lo;
}

__global__ __launch_bounds__(kPlThreads) void k_planes(PlaneJobs A) {
  __shared__ float lut[16];
  __shared__ float scl[64 * kSpan][2];
  int i = 0;
  while (i + 1 < A.count && (int)blockIdx.x >= A.j[i + 1].wg0) ++i;
  const PlaneJob &q = A.j[i];
  const int b = (int)blockIdx.x - q.wg0;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l32 = lane & 31, h = lane >> 5;
  const int K = q.K, KT = q.KT, rows = q.rows;
  if (q.kind == kNf4Col) {
    // 128 W columns x 64 kSpan W rows: the scales of those rows' two blocks,
    // then a lane's column pair (rows % 64 == 0) over 8 W rows at a time
    const int nk = (K + 64 * kSpan - 1) / (64 * kSpan), cg = b / nk;
    const int c0 = 128 * cg, k0 = 64 * kSpan * (b - cg * nk);
    const int c = min(c0 + 2 * lane, rows - 2);
    const uint8_t *src = q.w.codes + ((int64_t)c >> 1);
    uint32_t code[2 * kSpan][8];
#pragma unroll
    for (int p = 0; p < 2 * kSpan; ++p)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        code[p][e] = src[(int64_t)min(k0 + 32 * p + 8 * wave + e, K - 1) * (rows >> 1)];
    if (tid < 16) lut[tid] = c_lut_pl[tid];
    if (tid < 128 * kSpan) {
      const int k = min(k0 + (tid >> 1), K - 1), sc = min(c0 + 64 * (tid & 1), rows - 1);
      scl[tid >> 1][tid & 1] = scale_of(q.w, ((int64_t)k * rows + sc) >> 6);
    }
    __syncthreads();
    if (c0 + 2 * lane >= rows) return;
#pragma unroll
    for (int p = 0; p < 2 * kSpan; ++p) {
      const int kl = 32 * p + 8 * wave;
      if (k0 + kl >= 16 * KT) break;
      float f[2][8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float s = k0 + kl + e < K ? scl[kl + e][lane >> 5] : 0.0f;
        f[0][e] = lut[code[p][e] & 15u] * s;
        f[1][e] = lut[code[p][e] >> 4] * s;
      }
#pragma unroll
      for (int d = 0; d < 2; ++d)
        put2(q.dst + ((int64_t)((c + d) >> 5) * KT + ((k0 + kl) >> 4)) * 2048 +
                 (((kl >> 3) & 1) * 32 + ((c + d) & 31)) * 16,
             f[d]);
    }
    return;
  }
  if (q.kind == kDenseT) {
    // 32 rows x 64 k, a wave 16 k
    const int nk = (K + 63) / 64, rt = b / nk;
    const int kt = 4 * (b - rt * nk) + wave, r = 32 * rt + l32;
    if (kt >= KT) return;
    float f[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int k = 16 * kt + 8 * h + e;
      f[e] = k < K && r < rows ? ((const float *)q.src)[(int64_t)k * q.ld + r] * q.scale : 0.0f;
    }
    put2(q.dst + ((int64_t)rt * KT + kt) * 2048 + lane * 16, f);
    return;
  }
  const int nk = (K + 256 * kSpan - 1) / (256 * kSpan), rt = b / nk;
  const int k0 = 256 * kSpan * (b - rt * nk) + 64 * kSpan * wave, r = 32 * rt + l32;
  const int rc = min(r, rows - 1);
  if (q.kind == kNf4Row) {
    // pieces of 64 k are blocks (K % 64 == 0, 16-byte aligned codes): a lane pair
    // loads its row's 32 code bytes, lane half h decodes dword 2 t + h for k tile t
    v4u c0[kSpan], c1[kSpan];
    float s[kSpan];
#pragma unroll
    for (int p = 0; p < kSpan; ++p) {
      const int64_t e = (int64_t)rc * K + min(k0 + 64 * p, K - 64);
      c0[p] = *(const v4u *)(q.w.codes + (e >> 1));
      c1[p] = *(const v4u *)(q.w.codes + (e >> 1) + 16);
      s[p] = scale_of(q.w, e >> 6);
    }
    if (tid < 16) lut[tid] = c_lut_pl[tid];
    __syncthreads();
#pragma unroll
    for (int p = 0; p < kSpan; ++p) {
      if (k0 + 64 * p >= K) break;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const v4u &cc = t < 2 ? c0[p] : c1[p];
        const uint32_t c = h ? cc[2 * (t & 1) + 1] : cc[2 * (t & 1)];
        float f[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = lut[(c >> (4 * e)) & 15u] * s[p];
        put2(q.dst + ((int64_t)rt * KT + ((k0 + 64 * p) >> 4) + t) * 2048 + lane * 16, f);
      }
    }
    return;
  }
  if (q.kind == kDenseBf16) {  // K % 8 == 0, 16-byte aligned rows
    v4u v[kSpan][4];
#pragma unroll
    for (int p = 0; p < kSpan; ++p)
#pragma unroll
      for (int t = 0; t < 4; ++t)
        v[p][t] = *(const v4u *)((const uint16_t *)q.src + (int64_t)rc * q.ld +
                                 min(k0 + 64 * p + 16 * t + 8 * h, K - 8));
#pragma unroll
    for (int p = 0; p < kSpan; ++p)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int k = k0 + 64 * p + 16 * t + 8 * h, kt = (k0 + 64 * p) / 16 + t;
        if (kt >= KT) break;
        *(v4u *)(q.dst + ((int64_t)rt * KT + kt) * 1024 + lane * 16) =
            k < K ? v[p][t] : v4u{0, 0, 0, 0};
      }
    return;
  }
  const float *src = (const float *)q.src + (int64_t)rc * q.ld;
  const bool vec = q.ld % 4 == 0 && K % 8 == 0 && (((uintptr_t)q.src) & 15) == 0;
  float4 v[kSpan][4][2];
  if (vec) {
#pragma unroll
    for (int p = 0; p < kSpan; ++p)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const float *e = src + min(k0 + 64 * p + 16 * t + 8 * h, K - 8);
        v[p][t][0] = *(const float4 *)e;
        v[p][t][1] = *(const float4 *)(e + 4);
      }
  }
#pragma unroll
  for (int p = 0; p < kSpan; ++p)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int k = k0 + 64 * p + 16 * t + 8 * h, kt = (k0 + 64 * p) / 16 + t;
      if (kt >= KT) break;
      float f[8];
      if (vec) {
        const float4 a = v[p][t][0], c = v[p][t][1];
        f[0] = a.x, f[1] = a.y, f[2] = a.z, f[3] = a.w;
        f[4] = c.x, f[5] = c.y, f[6] = c.z, f[7] = c.w;
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = src[min(k + e, K - 1)];
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = k + e < K ? f[e] * q.scale : 0.0f;
      put2(q.dst + ((int64_t)rt * KT + kt) * 2048 + lane * 16, f);
    }
}

// ---- the GEMM -------------------------------------------------------------------
struct PlaneGemmDev {
  const uint8_t *A, *B;    // planes: M x K (P parts), N x K (2 parts)
  const uint8_t *A2, *B2;  // the LoRA term's planes (2 parts), KT2 k tiles
  float *C;
  int64_t ldc;
  int M, N, KT, KT2, tiles_m, tiles_n, beta;
};

// BM x 256 outputs, 8 waves in a 2 x 4 grid (a wave BM / 2 x 64), P parts of A.
template <int BM_, int P_>
struct Pl {
  static constexpr int BM = BM_, P = P_, BN = 256;
  static constexpr int TM = BM / 64, TN = 2;
  static constexpr int AT = BM / 32 * P, T = AT + BN / 32 * 2;  // tiles of a k tile
  static constexpr int L = (T + 7) / 8;                          // loads a wave
  static constexpr uint32_t SUB = T * 1024u;                     // LDS of a k tile
  static constexpr int NB = 160 * 1024 / SUB < 6 ? 160 * 1024 / SUB : 6;  // ring
  // the LoRA term's k tiles: both parts of A
  static constexpr int AT2 = BM / 32 * 2, T2 = AT2 + BN / 32 * 2, L2 = (T2 + 7) / 8;
  static constexpr uint32_t SUB2 = T2 * 1024u;
  static constexpr int NB2 = 160 * 1024 / SUB2 < 4 ? 160 * 1024 / SUB2 : 4;
  static constexpr uint32_t LDS = NB * SUB > NB2 * SUB2 ? NB * SUB : NB2 * SUB2;
};

constexpr int vmcnt_only(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }

template <class C>
__global__ __launch_bounds__(512, 2) void k_plane_gemm(PlaneGemmDev g) {
  constexpr int TM = C::TM, TN = C::TN, P = C::P, NB = C::NB;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  const int l32 = lane & 31, h = lane >> 5;
  // Blocks go to the 8 XCDs round robin: each gets a contiguous run of tiles,
  // ordered down four rows of tiles at a time, so that a run of 32 covers 4 x 8
  // tiles and its panels meet in one L2.
  const int nb = g.tiles_m * g.tiles_n;
  int tb = (int)blockIdx.x;
  if (nb % 8 == 0) tb = (tb % 8) * (nb / 8) + tb / 8;
  const int width = 4 * g.tiles_n, gr = tb / width, rem = tb - gr * width;
  const int gm = min(g.tiles_m - 4 * gr, 4);
  const int tm = 4 * gr + rem % gm, tn = rem / gm;
  const int m0 = tm * C::BM, n0 = tn * C::BN;

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

  // One k tile's operand tiles into LDS at `base`: A [row tile][part], B [row
  // tile][part], 1 KiB each; wave w copies tiles w, w + 8, ... (the last ones
  // again where the count is uneven, so that every wave issues as many).
  auto copy = [&](const uint8_t *Ap, const uint8_t *Bp, int pa, int KT, int kt, uint32_t base,
                  auto LC, int at, int tt) {
#pragma unroll
    for (int u = 0; u < decltype(LC)::value; ++u) {
      const int t = min(wave + 8 * u, tt - 1);
      const bool isa = t < at;
      const int x = isa ? t : t - at, pp = isa ? pa : 2;
      const int rt = pp == 2 ? x >> 1 : x, part = pp == 2 ? x & 1 : 0;
      const int64_t row = (int64_t)(isa ? m0 : n0) / 32 + rt;
      const uint64_t q = (uint64_t)(isa ? Ap : Bp) + ((row * KT + kt) * pp + part) * 1024;
      const uint64_t p = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(q >> 32)) << 32 |
                         (uint32_t)__builtin_amdgcn_readfirstlane((int)q);
      __builtin_amdgcn_global_load_lds((glb_void *)((glb_u1 *)p + lane * 16u),
                                       (lds_void *)(uintptr_t)(base + (uint32_t)t * 1024u), 16, 0,
                                       0);
    }
  };
  // This wave's operands of the k tile at `base`, complete when it returns
  // (the wait is in the block: the outputs are written by loads).
  v4u a[TM][2], b[TN][2];
  auto read = [&](uint32_t base, auto PC, int at) {
    constexpr int PA = decltype(PC)::value;
    const uint32_t pa = base + (uint32_t)(wm * TM * PA) * 1024u + lane * 16u;
    const uint32_t pb = base + (uint32_t)(at + wn * TN * 2) * 1024u + lane * 16u;
    if constexpr (TM == 4 && PA == 2)
      asm volatile(
          "ds_read_b128 %0, %12\n\tds_read_b128 %8, %13\n\tds_read_b128 %1, %12 offset:1024\n\t"
          "ds_read_b128 %9, %13 offset:1024\n\tds_read_b128 %2, %12 offset:2048\n\t"
          "ds_read_b128 %3, %12 offset:3072\n\tds_read_b128 %4, %12 offset:4096\n\t"
          "ds_read_b128 %5, %12 offset:5120\n\tds_read_b128 %6, %12 offset:6144\n\t"
          "ds_read_b128 %7, %12 offset:7168\n\tds_read_b128 %10, %13 offset:2048\n\t"
          "ds_read_b128 %11, %13 offset:3072\n\ts_waitcnt lgkmcnt(0)"
          : "=&v"(a[0][0]), "=&v"(a[0][1]), "=&v"(a[1][0]), "=&v"(a[1][1]), "=&v"(a[2][0]),
            "=&v"(a[2][1]), "=&v"(a[TM - 1][0]), "=&v"(a[TM - 1][1]), "=&v"(b[0][0]), "=&v"(b[0][1]),
            "=&v"(b[1][0]), "=&v"(b[1][1])
          : "v"(pa), "v"(pb)
          : "memory");
    else if constexpr (TM == 3 && PA == 2)
      asm volatile(
          "ds_read_b128 %0, %10\n\tds_read_b128 %6, %11\n\tds_read_b128 %1, %10 offset:1024\n\t"
          "ds_read_b128 %7, %11 offset:1024\n\tds_read_b128 %2, %10 offset:2048\n\t"
          "ds_read_b128 %3, %10 offset:3072\n\tds_read_b128 %4, %10 offset:4096\n\t"
          "ds_read_b128 %5, %10 offset:5120\n\tds_read_b128 %8, %11 offset:2048\n\t"
          "ds_read_b128 %9, %11 offset:3072\n\ts_waitcnt lgkmcnt(0)"
          : "=&v"(a[0][0]), "=&v"(a[0][1]), "=&v"(a[1][0]), "=&v"(a[1][1]), "=&v"(a[TM - 1][0]),
            "=&v"(a[TM - 1][1]), "=&v"(b[0][0]), "=&v"(b[0][1]), "=&v"(b[1][0]), "=&v"(b[1][1])
          : "v"(pa), "v"(pb)
          : "memory");
    else if constexpr (TM == 2 && PA == 2)
      asm volatile(
          "ds_read_b128 %0, %8\n\tds_read_b128 %4, %9\n\tds_read_b128 %1, %8 offset:1024\n\t"
          "ds_read_b128 %5, %9 offset:1024\n\tds_read_b128 %2, %8 offset:2048\n\t"
          "ds_read_b128 %3, %8 offset:3072\n\tds_read_b128 %6, %9 offset:2048\n\t"
          "ds_read_b128 %7, %9 offset:3072\n\ts_waitcnt lgkmcnt(0)"
          : "=&v"(a[0][0]), "=&v"(a[0][1]), "=&v"(a[1][0]), "=&v"(a[1][1]), "=&v"(b[0][0]),
            "=&v"(b[0][1]), "=&v"(b[1][0]), "=&v"(b[1][1])
          : "v"(pa), "v"(pb)
          : "memory");
    else if constexpr (TM == 4)
      asm volatile(
          "ds_read_b128 %0, %8\n\tds_read_b128 %4, %9\n\tds_read_b128 %1, %8 offset:1024\n\t"
          "ds_read_b128 %5, %9 offset:1024\n\tds_read_b128 %2, %8 offset:2048\n\t"
          "ds_read_b128 %3, %8 offset:3072\n\tds_read_b128 %6, %9 offset:2048\n\t"
          "ds_read_b128 %7, %9 offset:3072\n\ts_waitcnt lgkmcnt(0)"
          : "=&v"(a[0][0]), "=&v"(a[1][0]), "=&v"(a[2][0]), "=&v"(a[TM - 1][0]), "=&v"(b[0][0]),
            "=&v"(b[0][1]), "=&v"(b[1][0]), "=&v"(b[1][1])
          : "v"(pa), "v"(pb)
          : "memory");
    else if constexpr (TM == 3)
      asm volatile(
          "ds_read_b128 %0, %7\n\tds_read_b128 %3, %8\n\tds_read_b128 %1, %7 offset:1024\n\t"
          "ds_read_b128 %4, %8 offset:1024\n\tds_read_b128 %2, %7 offset:2048\n\t"
          "ds_read_b128 %5, %8 offset:2048\n\tds_read_b128 %6, %8 offset:3072\n\t"
          "s_waitcnt lgkmcnt(0)"
          : "=&v"(a[0][0]), "=&v"(a[1][0]), "=&v"(a[TM - 1][0]), "=&v"(b[0][0]), "=&v"(b[0][1]),
            "=&v"(b[1][0]), "=&v"(b[1][1])
          : "v"(pa), "v"(pb)
          : "memory");
    else
      asm volatile(
          "ds_read_b128 %0, %6\n\tds_read_b128 %2, %7\n\tds_read_b128 %1, %6 offset:1024\n\t"
          "ds_read_b128 %3, %7 offset:1024\n\tds_read_b128 %4, %7 offset:2048\n\t"
          "ds_read_b128 %5, %7 offset:3072\n\ts_waitcnt lgkmcnt(0)"
          : "=&v"(a[0][0]), "=&v"(a[1][0]), "=&v"(b[0][0]), "=&v"(b[0][1]), "=&v"(b[1][0]),
            "=&v"(b[1][1])
          : "v"(pa), "v"(pb)
          : "memory");
  };
  auto mf = [](v4u x, v4u y, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, x),
                                                   __builtin_bit_cast(bf16x8_t, y), c, 0, 0, 0);
  };
  // ah.bh + ah.bl (+ al.bh), the order of k_gemm_bf16.hip: the same bits
  auto mma = [&](auto PC) {
#pragma unroll
    for (int q = 0; q < (decltype(PC)::value == 2 ? 3 : 2); ++q)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = mf(a[i][q == 2], b[j][q == 1], acc[i][j]);
  };
  using PC = std::integral_constant<int, P>;
  using LC = std::integral_constant<int, C::L>;
  const int S = g.KT;
  auto load = [&](int s) {
    copy(g.A, g.B, P, S, min(s, S - 1), (uint32_t)(s % NB) * C::SUB, LC{}, C::AT, C::T);
  };

  // Waves 0-3 and 4-7 (one of each per SIMD) take turns on the matrix cores:
  // in phase 2 s the first group reads k tile s's operands from LDS while the
  // second runs tile s - 1's MFMAs, in phase 2 s + 1 they swap.  Tile s + NB - 1 is
  // requested with tile s's reads, into the slot that tile s - 1 left (both
  // groups' reads of it ended a barrier ago), and every wave's copies of
  // tile s + 1 have landed by the barrier that ends phase 2 s + 1: (NB - 2) L
  // younger ones may be in flight.
  constexpr int kYoung = vmcnt_only((NB - 2) * C::L);
  for (int s = 0; s < NB - 1; ++s) load(s);
  __builtin_amdgcn_s_waitcnt(kYoung);
  __builtin_amdgcn_s_barrier();
  if (wm == 0) {
    for (int s = 0; s < S; ++s) {
      read((uint32_t)(s % NB) * C::SUB, PC{}, C::AT);
      load(s + NB - 1);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_s_setprio(1);
      mma(PC{});
      __builtin_amdgcn_s_setprio(0);
      __builtin_amdgcn_s_waitcnt(kYoung);
      __builtin_amdgcn_s_barrier();
    }
    __builtin_amdgcn_s_barrier();
  } else {
    __builtin_amdgcn_s_barrier();
    for (int s = 0; s < S; ++s) {
      read((uint32_t)(s % NB) * C::SUB, PC{}, C::AT);
      load(s + NB - 1);
      __builtin_amdgcn_s_waitcnt(kYoung);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_s_setprio(1);
      mma(PC{});
      __builtin_amdgcn_s_setprio(0);
      __builtin_amdgcn_s_barrier();
    }
  }
  // ---- the LoRA term, NB2 k tiles at a time
  __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
  for (int q0 = 0; q0 < g.KT2; q0 += C::NB2) {
    __builtin_amdgcn_s_barrier();  // every read of the slots is done
    const int nq = min(C::NB2, g.KT2 - q0);
    for (int q = 0; q < nq; ++q)
      copy(g.A2, g.B2, 2, g.KT2, q0 + q, (uint32_t)q * C::SUB2,
           std::integral_constant<int, C::L2>{}, C::AT2, C::T2);
    __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
    __builtin_amdgcn_s_barrier();
    for (int q = 0; q < nq; ++q) {
      read((uint32_t)q * C::SUB2, std::integral_constant<int, 2>{}, C::AT2);
      mma(std::integral_constant<int, 2>{});
    }
  }
  // ---- epilogue
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int m = m0 + wm * (C::BM / 2) + 32 * i + 8 * (v / 4) + 4 * h + (v % 4);
        const int n = n0 + 64 * wn + 32 * j + l32;
        if (m < g.M && n < g.N) {
          float *c = g.C + (int64_t)m * g.ldc + n;
          *c = g.beta ? *c + acc[i][j][v] : acc[i][j][v];
        }
      }
}

template <class C>
hipError_t run_plane(const PlaneGemmDev &g0, hipStream_t st) {
  auto k = k_plane_gemm<C>;
  static bool attr = false;  // per instantiation
  if (!attr) {
    const hipError_t e = hipFuncSetAttribute(
        (const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)C::LDS);
    if (e != hipSuccess) return e;
    attr = true;
  }
  PlaneGemmDev g = g0;
  g.tiles_m = (g.M + C::BM - 1) / C::BM;
  g.tiles_n = (g.N + C::BN - 1) / C::BN;
  return qh_launch(k, dim3((unsigned)(g.tiles_m * g.tiles_n)), dim3(512), C::LDS, st, g);
}

int64_t up(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Tile rows: the count of rounds of 256 workgroups times a tile's time decides: its
// MFMAs plus a fixed part, in fp32 a round's start and end (those of 120000 rows
// over one k: 12 us), in bf16 mostly a k tile's phases (of 80 rows).  Measured over
// 636 calls whose height depends on the fixed part (taken as 12 to 112 rows): within
// 0.2 % of the best height on the mean, at most 4 % in fp32 and 12 in bf16; 24 rows lose
// 5 % in fp32 (up to 24) and 12.5 in bf16 (up to 38), 80 rows 2 % of a 70B-class block in
// fp32, whose long reductions hide a round's ends.
int plane_bm(int64_t M, int64_t N, int64_t K, bool f32) {
  const double fixed = f32 ? 120000.0 / (double)K : 80.0;
  int best = 256;
  double bc = 0;
  for (int bm : {256, 192, 128}) {
    const double c = (double)up(up(M, bm) * up(N, 256), 256) * (bm + fixed);
    if (bc == 0 || c < bc) bc = c, best = bm;
  }
  return best;
}

}  // namespace

// About what the planes and the GEMM take (us): the planes' bytes (dearer past the
// 200 MB that stay in the last-level cache until the GEMM reads them), the rounds of
// tiles, the tiles' operand traffic (less of it where each XCD has its run of tiles)
// and the output.  Fitted to 3000 calls of up to 4e12 products, 3.6 % rms in fp32 and 4.7
// in bf16; the constant is 2 us above the fit, for the calls below 40 us.
double plane_us(int64_t M, int64_t N, int64_t K, bool f32) {
  const int bm = plane_bm(M, N, K, f32);
  const double mk = (double)M * (double)K * 1e-6, nk = (double)N * (double)K * 1e-6;
  const double mn = (double)M * (double)N * 1e-6, k = (double)K * 1e-3;
  const int64_t tiles = up(M, bm) * up(N, 256);
  const double R = (double)up(tiles, 256), rows = (double)tiles * bm * 1e-3;
  const double over = std::max(0.0, (f32 ? 4 : 2) * mk + 4 * nk - 200);
  const bool xcd = tiles % 8 == 0;
  if (f32)
    return 9.2 + 1.09 * mk + 0.81 * nk + 0.123 * over +
           k * (R * (2.5 + 0.0975 * bm) + (xcd ? 0.619 : 0.666) * rows) + 0.16 * mn + 7.9 * R;
  return 9.3 + 0.38 * mk + 0.845 * nk + 0.145 * over +
         k * (R * (8 + 0.0394 * bm) + (xcd ? 0.403 : 0.459) * rows) + 0.255 * mn + 7.7 * R;
}

// Planes where their estimate is not 3 % above that of k_nf4_bf16, in the range measured:
// more than half a round of 128 x 256 tiles and K of 512 or more, at most 2 GiB of
// planes (the LoRA term of rank r included).  The pass over the operands costs
// (8 or 4 bytes) x rows + 4.5 bytes x columns per k, whatever the product, and
// columns are padded to 256, so that narrow outputs and few rows lose: fp32
// 20000 x 192 over 2048 188 us against 150, 64 x 128256 over 4096 888 against 448,
// 2048 x 4096 over 512 39 against 37; they win from about 576 columns and 400 rows
// at K of 1536 (8192 x 576 87 against 97), 1.2 times as fast on the geometric mean
// of the sizes taken here, 1.4 at 1100 x 4096 over 4096.  Of 2572 calls measured,
// fp32 and bf16, forward and input gradient, 2055 are taken, 36 of them slower by
// more than 3 % (17 by more than 6, at most 21); 23 of the others would be faster by
// more than 5 % (if all were taken 402 slower, up to 2.3 times).  Below 288 rows
// forwards with an adapter are slower than estimated (223 x 18032 over 4096 in fp32
// 239 us against 219, 263 x 17416 242 against 229).
// What k_nf4_bf16 splits (at most 128 columns, up to 21760 rows) stays there: its
// bits are those of the allocation-free backward, which takes no planes.
bool plane_ok(int64_t M, int64_t N, int64_t K, int64_t r, bool f32) {
  return M >= 288 && up(M, 128) * up(N, 256) > 128 && K >= 512 && bf16_gemm_splits(M, N, K) == 1 &&
         M < (1 << 24) && N < (1 << 24) && K < (1 << 24) && r < (1 << 24) &&
         plane_a_bytes(M, K, 2) + plane_b_bytes(N, K) + plane_a_bytes(M, r, 2) +
                 plane_b_bytes(N, r) <=
             (size_t)2 << 30 &&
         plane_us(M, N, K, f32) < 1.03 * bf16_gemm_us(M, N, K, f32, true);
}

size_t plane_a_bytes(int64_t M, int64_t K, int parts) {
  return (size_t)(up(M, 768) * 24) * up(K, 16) * 1024 * parts;  // whole tiles of 256, 192, 128 rows
}
size_t plane_b_bytes(int64_t N, int64_t K) { return (size_t)(up(N, 256) * 8) * up(K, 16) * 2048; }

hipError_t launch_planes(const PlaneSrc *src, int count, hipStream_t st) {
  if (count < 1 || count > 4) return hipErrorInvalidValue;
  PlaneJobs A{};
  int wg = 0;
  for (int i = 0; i < count; ++i) {
    const PlaneSrc &s = src[i];
    PlaneJob &q = A.j[A.count++];
    q.kind = s.form == PLANE_NF4_ROW   ? kNf4Row
             : s.form == PLANE_NF4_COL ? kNf4Col
             : s.form == PLANE_KROW    ? kDenseT
             : s.bf16                  ? kDenseBf16
                                       : kDenseF32;
    q.src = s.p;
    q.w = s.w;
    q.dst = (uint8_t *)s.dst;
    q.ld = s.ld;
    q.rows = (int)s.rows;
    q.K = (int)s.K;
    q.KT = (int)up(s.K, 16);
    q.scale = s.scale;
    q.wg0 = wg;
    wg += plane_wgs(q.kind, s.rows, s.K);
  }
  return qh_launch(k_planes, dim3((unsigned)wg), dim3(kPlThreads), 0, st, A);
}

hipError_t launch_plane_gemm(const PlaneGemm &p, hipStream_t st) {
  PlaneGemmDev g{};
  g.A = (const uint8_t *)p.a;
  g.B = (const uint8_t *)p.b;
  g.A2 = (const uint8_t *)p.a2;
  g.B2 = (const uint8_t *)p.b2;
  g.C = p.c;
  g.ldc = p.ldc;
  g.M = (int)p.M;
  g.N = (int)p.N;
  g.KT = (int)up(p.K, 16);
  g.KT2 = (int)up(p.K2, 16);
  g.beta = p.beta;
  const int bm = plane_bm(p.M, p.N, p.K, p.a_parts == 2);
  if (p.a_parts == 2) {
    if (bm == 256) return run_plane<Pl<256, 2>>(g, st);
    if (bm == 192) return run_plane<Pl<192, 2>>(g, st);
    return run_plane<Pl<128, 2>>(g, st);
  }
  if (bm == 256) return run_plane<Pl<256, 1>>(g, st);
  if (bm == 192) return run_plane<Pl<192, 1>>(g, st);
  return run_plane<Pl<128, 1>>(g, st);
}

}  // namespace qh
