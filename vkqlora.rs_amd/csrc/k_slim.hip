// k_slim.hip -- the QLoRA forward for few tokens (17 to some hundreds): serving
// batches past the decode kernels and short prompts.  The forward of
// qlora-wgpu/src/kernels.rs:262-296 (dequant + mm_nt + LoRA mm_nt),
//
//   y[m][n] = sum_b s_{n,b} sum_{k in b} x[m][k] L[c_{n,k}]
//           + (alpha/r) sum_j T1[m][j] B[n][j],      T1 = X A^T,
//
// in two launches for up to four layers: k_slim_prep splits X into bf16 parts
// in MFMA operand order and computes partial T1s; k_slim streams the packed
// weights.
//
// What bounds it.  A 7B-class layer holds 2 to 12 us of work here, so a tiled
// GEMM's chain of dependent K steps and its padding to 128 tokens cost more
// than the work.  k_slim has no barrier between its prologue and its last
// sum: a workgroup owns 16 R weight rows and up to 64 tokens, its 8 waves
// split K, and a wave decodes code bytes straight into MFMA operands through a
// byte-pair table in LDS, with the next two code loads and the next X tiles
// in flight.  Block scales multiply a block's partial sum, once per output.
// Per 128 of K and 48 fp32 tokens the two waves of a SIMD need 1150 cycles per 16
// rows on the matrix cores (36 MFMAs of 16 cycles each) and the CU's eight waves
// 192 KiB of X tiles, 3100 cycles at 64 bytes a cycle from L2, whatever R is, so
// R is as large as the registers allow where that leaves one workgroup per CU.
// The kernel comes to less than half of either: at 37 fp32 tokens 16.3 us for
// 4096 x 4096, 22.4 for 11008 x 4096 (MFMA busy 0.19), 26.4 for 4096 x 11008, of which
// 7.1 to 7.5 are a workgroup's start and end (all of a K of 384), after 6.4 to 8 us of
// preparation.  More tokens take workgroups of their own (the codes
// come from L2 again); K is split over workgroups only where rows are few
// (the last one of a group adds the slices in order).
//
// Measured against the 128 x 128 GEMM tiles and their split reduction, fp32 X
// with r = 16: 4096 x 4096 at 37 tokens 44 -> 24 us, 11008 x 4096 112 -> 29,
// 4096 x 11008 86 -> 34, at 256 tokens 63 -> 57 / 155 -> 130 / 140 -> 115; bf16
// at 256 tokens 55 -> 38 / 125 -> 86 / 112 -> 71.  A 7B-class decoder block's
// seven projections with their norms at 37 tokens: 496 -> 169 us.
#include <algorithm>
#include <cstdint>

#include "decode_common.h"
#include "qh_nf4.h"

namespace qh {
namespace {

constexpr int kWaves = 8;
constexpr int kThreads = kWaves * 64;
constexpr uint32_t kLdsLimit = 160u * 1024u;
constexpr int kUnit = 128;      // elements of a row per code load (64 bytes)
constexpr int kMaxSlices = 16;  // K slices of a layer
constexpr int kMaxNb = 256;     // blocks of a slice: at most two absmax groups a row
constexpr int kMaxT1Parts = 16;

typedef uint32_t v2u __attribute__((ext_vector_type(2)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
// global-memory pointers made from integers (a generic one would load flat)
typedef const __attribute__((address_space(1))) uint8_t glb_u1;
typedef const __attribute__((address_space(1))) v4u glb_u4;
typedef __attribute__((address_space(3))) uint32_t lds_u;
typedef __attribute__((address_space(3))) v2u lds_u2;
typedef __attribute__((address_space(3))) v4u lds_u4;
typedef __attribute__((address_space(3))) float lds_f;
typedef __attribute__((address_space(3))) floatx4 lds_f4;
typedef __attribute__((address_space(3))) int lds_i;
// LDS is addressed by byte offset: the kernel declares no __shared__ object,
// so dynamic LDS starts at 0.
#define LDS_AT(T, off) ((T *)(uintptr_t)(off))

__device__ __forceinline__ uint32_t bf16_pair(float a, float b) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const bf16x2 h = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(uint32_t, h);
}

// The codebook is kept times kAlpha and the block scales divided by it: the
// 16 products kAlpha L round to bf16 hi + lo parts within 3.4e-7 (rms over
// the codes of normal weights) where L itself gives 2.5e-6 (the best of 4
// million factors in [1, 2) tried).
constexpr double kAlpha = 1.3462369441986084;
struct Nibbles {
  uint32_t v[16];  // hi | lo << 16 of kAlpha L
};
constexpr Nibbles make_nibbles() {
  Nibbles t{};
  constexpr float L[17] = QH_NF4_LUT17_INIT;
  for (int c = 0; c < 16; ++c) {
    const float f = (float)(kAlpha * (double)L[c]);
    const uint32_t h = bf16_rne(f);
    t.v[c] = h | (bf16_rne(f - u2f(h << 16)) << 16);
  }
  return t;
}

// Shape of an instantiation: G groups of 16 tokens, X in P bf16 parts (fp32
// hi and lo; bf16 itself), R 16-row tiles of W a wave.  A 16 x 16 x 32 step
// runs as xh.Lh + xh.Ll (+ xl.Lh), leaving out xl.Ll (2^-17 of the product).
template <int G_, int P_, int R_>
struct Slim {
  static constexpr int G = G_, P = P_, R = R_, XT = P * G;
};
// The byte-pair table: entry e holds 32 copies of byte e's hi pair, then 32 of
// its lo pair, so that a lane reads its own bank whatever the codes are.
constexpr int kCopies = 32;
constexpr uint32_t kTabBytes = 256u * kCopies * 8u;

struct SlimSegDev {
  const uint8_t *codes;
  const void *scales;    // kind 0: fp32 scales; kind 1: int8 codes
  const float *absmax;
  const uint8_t *xp;     // operand planes of this segment's X
  const float *t1p, *lb; // nz x M x r partial T1s, N x r (r > 0)
  float *t1;             // M x r: their sum, for the caller (or null)
  float *y;
  float *part;
  unsigned *tick;
  int N, K, kind, r, groups, S, nbp, nz;
  float s_lora;
  int beta;
};
struct SlimArgs {
  SlimSegDev seg[kMaxSlimSegs];
  int M, chunks;
};

// LDS of a workgroup: table, scales and T1 while streaming, then the 8
// waves' sums; a flag word behind both.
uint32_t slim_lds(int G, int R, int nbp, int64_t r) {
  const uint32_t a = kTabBytes + (uint32_t)(16 * R * nbp + 16 * G * r) * 4u;
  const uint32_t b = (uint32_t)(kWaves * R * G) * 1024u;
  return ((a > b ? a : b) + 15u) / 16u * 16u + 16u;
}

// grid (groups of 16 R rows, K slices x token chunks, segments)
template <class C>
__global__ __launch_bounds__(kThreads, 2) void k_slim(SlimArgs A, uint32_t o_flag) {
  constexpr int G = C::G, P = C::P, R = C::R, XT = C::XT;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nl = lane & 15, g = lane >> 4;
  const SlimSegDev &L = A.seg[blockIdx.z];
  const int grp = (int)blockIdx.x;
  const int sl = A.chunks == 1 ? (int)blockIdx.y : (int)blockIdx.y / A.chunks;
  const int chunk = (int)blockIdx.y - sl * A.chunks;
  const int S = L.S;
  if (grp >= L.groups || sl >= S) return;  // the grid covers the largest segment
  const int N = L.N, K = L.K, U = (K + kUnit - 1) / kUnit, KB = K >> 6;
  const int row0 = grp * 16 * R;
  const int us0 = S == 1 ? 0 : U * sl / S, us1 = S == 1 ? U : U * (sl + 1) / S;
  const int nu_s = us1 - us0;
  const int u0 = us0 + nu_s * wave / kWaves;
  const int n = us0 + nu_s * (wave + 1) / kWaves - u0;  // this wave's units

  // ---- loads: lane (nl, g) of tile t reads bytes [16 g, 16 g + 16) of each
  // unit of row row0 + 16 t + nl
  const uint8_t *cbase = L.codes + (int64_t)row0 * (K >> 1);
  uint32_t voff[R];
#pragma unroll
  for (int t = 0; t < R; ++t) {
    const int rl = min(16 * t + nl, N - 1 - row0);
    voff[t] = (uint32_t)rl * (uint32_t)(K >> 1) + 16u * g;
  }
  // the last unit of a K that is an odd number of blocks: the upper half's
  // lanes stay inside the row (their X is zero)
  const int odd_unit = (KB & 1) ? U - 1 : -1;
  const uint32_t odd_back = g >= 2 ? 32u : 0u;
  v4u cc[2][R];
  auto issue_c = [&](int i, v4u (&d)[R]) {
    const int u = u0 + i;
    uint64_t p = (uint64_t)cbase + (uint32_t)u * 64u;
    asm volatile("" : "+s"(p));  // a scalar base: no per-load address in VGPRs
    const uint32_t o = u == odd_unit ? odd_back : 0u;
#pragma unroll
    for (int t = 0; t < R; ++t) d[t] = *(glb_u4 *)((glb_u1 *)p + (voff[t] - o));
  };
  // X planes: [chunk][unit][block 2][step 2][P][G] of 1 KiB operand tiles
  const uint8_t *xb = L.xp + ((int64_t)chunk * U + u0) * (4 * XT * 1024);
  const uint32_t xl = lane * 16;
  v4u xr[2][2][XT];
  auto issue_x = [&](int i, int b, v4u (&d)[2][XT]) {
    uint64_t q = (uint64_t)xb + (uint32_t)(i * 4 + 2 * b) * (XT * 1024u);
#pragma unroll
    for (int v = 0; v < 2 * XT; ++v) {
      if (v % 4 == 0) asm volatile("" : "+s"(q));  // scalar base; offsets below 4 KiB
      d[v / XT][v % XT] = *(glb_u4 *)((glb_u1 *)q + (xl + v % 4 * 1024u));
      if (v % 4 == 3) q += 4096;
    }
  };
  if (n > 0) {
    issue_c(0, cc[0]);
    issue_x(0, 0, xr[0]);
    issue_c(min(1, n - 1), cc[1]);
  }

  // ---- the codebook table, from immediates
  {
    constexpr Nibbles kTab = make_nibbles();
    int nv = 0;
#pragma unroll
    for (int qq = 0; qq < 16; ++qq)
      asm volatile("v_writelane_b32 %0, %1, %2" : "+v"(nv) : "s"((int)kTab.v[qq]), "n"(qq));
    constexpr int TPE = kCopies / 2;    // threads (16-byte stores) per entry
    constexpr int EPP = kThreads / TPE; // entries per pass
#pragma unroll
    for (int i = 0; i < 256 / EPP; ++i) {
      const int e = tid / TPE + EPP * i;
      const uint32_t nlo = (uint32_t)__builtin_amdgcn_ds_bpermute((e & 15) * 4, nv);
      const uint32_t nhi = (uint32_t)__builtin_amdgcn_ds_bpermute((e >> 4) * 4, nv);
      const uint32_t ph = (nlo & 0xffffu) | (nhi << 16), pl = (nlo >> 16) | (nhi & 0xffff0000u);
      const v4u ent = tid % TPE >= TPE / 2 ? v4u{pl, pl, pl, pl} : v4u{ph, ph, ph, ph};
      *LDS_AT(lds_u4, (uint32_t)(e * TPE + tid % TPE) * 16u) = ent;
    }
  }

  // ---- the slice's block scales into LDS: [16 R rows][nbp], the exact fp32 scale
  // times the rounded 1 / kAlpha (one more rounding).
  // TPR threads a row, blocks j, j + TPR, ... of it each.
  const int nb = 2 * nu_s, kb0 = 2 * us0, nbp = L.nbp;
  constexpr uint32_t o_sc = kTabBytes;
  constexpr int TPR = R == 2 ? 16 : 8;
  if (tid < 16 * R * TPR) {
    const int row = tid / TPR, j0 = tid % TPR;
    const int64_t b0 = (int64_t)min(row0 + row, N - 1) * KB + kb0;
    const int nin = min(nb, KB - kb0);  // blocks inside the row
    constexpr int SB = 8;
    for (int jb = 0; jb < nb; jb += TPR * SB) {
      float v[SB];
      if (L.kind == 0) {
#pragma unroll
        for (int q = 0; q < SB; ++q)
          v[q] = ((const float *)L.scales)[b0 + min(jb + j0 + TPR * q, nin - 1)];
      } else {
        int c[SB];
        const float a0 = L.absmax[b0 >> 8], a1 = L.absmax[(b0 + nin - 1) >> 8];
        const int split = 256 - (int)(b0 & 255);  // from here on the second absmax
#pragma unroll
        for (int q = 0; q < SB; ++q)
          c[q] = (int)(int8_t)((const uint8_t *)L.scales)[b0 + min(jb + j0 + TPR * q, nin - 1)];
        // fl(fl(c / 127) * absmax), the quotient as a double product (the
        // IEEE float quotient bit for bit, see k_gemm_bf16.hip)
#pragma unroll
        for (int q = 0; q < SB; ++q)
          v[q] = (float)((double)(float)c[q] * (1.0 / 127.0)) *
                 (jb + j0 + TPR * q < split ? a0 : a1);
      }
#pragma unroll
      for (int q = 0; q < SB; ++q) {
        const int j = jb + j0 + TPR * q;
        if (j < nb) 
          *LDS_AT(lds_f, o_sc + (uint32_t)(row * nbp + j) * 4u) =
              j < nin ? v[q] * (float)(1.0 / kAlpha) : 0.0f;
      }
    }
  }

  // ---- the LoRA operands: T1 (the sum of its partials) into LDS, the wave's
  // share of B into registers.  Wave w takes tile w % R and every KW-th 16
  // ranks (fp32 MFMA; lane (nl, g) supplies ranks 16 j + 4 g + e).
  const int m0 = chunk * 16 * G;
  const int r = sl == 0 ? L.r : 0;
  const uint32_t o_t1 = o_sc + (uint32_t)(16 * R * nbp) * 4u;
  constexpr int KW = kWaves / R < 4 ? kWaves / R : 4;  // waves a tile
  constexpr int JT = (4 + KW - 1) / KW;                // 16-rank steps of a wave
  float bv[JT][4];
  const int lt = wave % R, lk = wave / R;
  if (r > 0) {
    const float *br = L.lb + (int64_t)min(row0 + 16 * lt + nl, N - 1) * r;
#pragma unroll
    for (int q = 0; q < JT; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int j = 16 * (lk + KW * q) + 4 * g + e;
        const float b = br[min(j, r - 1)];
        bv[q][e] = j < r ? b : 0.0f;
      }
    const int mt = min(16 * G, A.M - m0), cnt = mt * r;
    for (int i = tid; i < cnt; i += kThreads) {
      const float *p = L.t1p + (int64_t)m0 * r + i;
      float s = 0.0f;
      for (int z0 = 0; z0 < L.nz; z0 += 8) {
        float v[8];
#pragma unroll
        for (int z = 0; z < 8; ++z) v[z] = p[(int64_t)min(z0 + z, L.nz - 1) * A.M * r];
#pragma unroll
        for (int z = 0; z < 8; ++z) s += z0 + z < L.nz ? v[z] : 0.0f;
      }
      *LDS_AT(lds_f, o_t1 + (uint32_t)i * 4u) = s;
      if (grp == 0 && L.t1) L.t1[(int64_t)m0 * r + i] = s;
    }
  }
  floatx4 acc[R][G];
#pragma unroll
  for (int t = 0; t < R; ++t)
#pragma unroll
    for (int rg = 0; rg < G; ++rg) acc[t][rg] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  __syncthreads();  // table, scales and T1 are in LDS
  if (r > 0 && lk < KW) {
    floatx4 d[G];
#pragma unroll
    for (int rg = 0; rg < G; ++rg) d[rg] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int q = 0; q < JT; ++q) {
      if (16 * (lk + KW * q) >= r) break;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int j = 16 * (lk + KW * q) + 4 * g + e;
#pragma unroll
        for (int rg = 0; rg < G; ++rg) {
          const int ml = min(16 * rg + nl, A.M - m0 - 1);
          const float t = *LDS_AT(const lds_f, o_t1 + (uint32_t)(ml * r + min(j, r - 1)) * 4u);
          d[rg] = __builtin_amdgcn_mfma_f32_16x16x4f32(j < r ? t : 0.0f, bv[q][e], d[rg], 0, 0,
                                                       0);
        }
      }
    }
#pragma unroll
    for (int t = 0; t < R; ++t)
      if (lt == t)
#pragma unroll
        for (int rg = 0; rg < G; ++rg)
#pragma unroll
          for (int v = 0; v < 4; ++v) acc[t][rg][v] = L.s_lora * d[rg][v];
  }

  // ---- the weight stream ----------------------------------------------------
  // byte k of w (two codes) to its table address for this lane's copy
  const uint32_t lo4 = (uint32_t)(lane % kCopies) * 4u;
  auto tab = [&](uint32_t w, int k) {
    return __builtin_amdgcn_perm(w, lo4, 0x0C0C0000u | ((4u + (uint32_t)k) << 8));
  };
  // lane's scale row: LDS address of (row 16 t + nl, block 2 (u0 - us0))
  const uint32_t so = o_sc + ((uint32_t)nl * nbp + 2u * (u0 - us0)) * 4u;
  auto mf = [](v4u a, v4u w, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, w), c, 0, 0, 0);
  };
  auto block = [&](const uint32_t (&sw)[R][4], int b, const v4u (*x)[XT], int i) {
    // tile-steps (t, a) of the block, the next one's lookups requested ahead
    v4u eh[2], el[2];  // B operands: hi and lo parts of 8 codes a lane
    auto fetch = [&](int idx) {
      const uint32_t w = sw[idx / 2][2 * b + idx % 2];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t o = tab(w, k);
        eh[idx & 1][k] = *LDS_AT(const lds_u, o);
        el[idx & 1][k] = *LDS_AT(const lds_u, o + kCopies * 4u);
      }
    };
    float sc[R];
#pragma unroll
    for (int t = 0; t < R; ++t)
      sc[t] = *LDS_AT(const lds_f, so + (uint32_t)(16 * t * nbp + 2 * i + b) * 4u);
    fetch(0);
    // partial sums in flight: two, so that a tile's scaling need not wait for
    // its last MFMA, where the registers hold them
    constexpr int ND = XT >= 6 ? 1 : 2;
    floatx4 d[ND][G];
    auto add = [&](int t) {
#pragma unroll
      for (int rg = 0; rg < G; ++rg)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          acc[t][rg][v] = fmaf(sc[t], d[t % ND][rg][v], acc[t][rg][v]);
    };
#pragma unroll
    for (int idx = 0; idx < 2 * R; ++idx) {
      const int t = idx / 2, a = idx % 2;
      if (idx + 1 < 2 * R) fetch(idx + 1);
      floatx4(&dt)[G] = d[t % ND];
      if (a == 0)
#pragma unroll
        for (int rg = 0; rg < G; ++rg) dt[rg] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int rg = 0; rg < G; ++rg) dt[rg] = mf(x[a][rg], eh[idx & 1], dt[rg]);
#pragma unroll
      for (int rg = 0; rg < G; ++rg) dt[rg] = mf(x[a][rg], el[idx & 1], dt[rg]);
      if constexpr (P == 2)
#pragma unroll
        for (int rg = 0; rg < G; ++rg) dt[rg] = mf(x[a][G + rg], eh[idx & 1], dt[rg]);
      if (ND == 2 && a == 0 && t > 0) add(t - 1);
      if (ND == 1 && a == 1) add(t);
      __builtin_amdgcn_sched_barrier(0);  // keeps later steps' lookups from piling up
    }
    if (ND == 2) add(R - 1);
  };
  // One unit: its codes in set j, its X one block ahead.  The loads are
  // unconditional (past the wave's units they repeat the last one's, from the
  // cache), so that the wait counts are exact; loads return in order, so X
  // goes out before the codes that are needed after it.
  auto unit = [&](int i, auto J) {
    constexpr int j = decltype(J)::value;
    uint32_t sw[R][4];
#pragma unroll
    for (int t = 0; t < R; ++t) {
      auto p = __builtin_amdgcn_permlane32_swap(cc[j][t].x, cc[j][t].y, false, false);
      sw[t][0] = p[0];
      sw[t][2] = p[1];
      p = __builtin_amdgcn_permlane32_swap(cc[j][t].z, cc[j][t].w, false, false);
      sw[t][1] = p[0];
      sw[t][3] = p[1];
    }
    const int i1 = min(i + 1, n - 1), i2 = min(i + 2, n - 1);
    issue_x(i, 1, xr[1]);
    block(sw, 0, xr[0], i);
    issue_x(i1, 0, xr[0]);
    issue_c(i2, cc[j]);
    block(sw, 1, xr[1], i);
  };
  for (int i = 0; i < n; i += 2) {
    unit(i, std::integral_constant<int, 0>{});
    if (i + 1 >= n) break;
    unit(i + 1, std::integral_constant<int, 1>{});
  }

  // ---- the 8 waves' sums in wave order ----------------------------------------
  __syncthreads();  // every read of the table and the scales is done
#pragma unroll
  for (int t = 0; t < R; ++t)
#pragma unroll
    for (int rg = 0; rg < G; ++rg)
      *LDS_AT(lds_f4, (uint32_t)(((wave * R + t) * G + rg) * 64 + lane) * 16u) = acc[t][rg];
  __syncthreads();
  constexpr int O = R * G * 64, KO = (O + kThreads - 1) / kThreads;
  floatx4 out[KO];
#pragma unroll
  for (int k = 0; k < KO; ++k) {
    const int idx = min(tid + k * kThreads, O - 1);
    floatx4 s = *LDS_AT(const lds_f4, (uint32_t)idx * 16u);
#pragma unroll
    for (int w = 1; w < kWaves; ++w) s += *LDS_AT(const lds_f4, (uint32_t)(w * O + idx) * 16u);
    out[k] = s;
  }
  if (S > 1) {
    // this slice's sums out (device-coherent), then the group's ticket; the
    // last slice adds all of them in slice order
    const int64_t gid = (int64_t)chunk * L.groups + grp;
    uint64_t *pp = (uint64_t *)(L.part + (gid * S + sl) * (4 * O));
#pragma unroll
    for (int k = 0; k < KO; ++k) {
      const int idx = tid + k * kThreads;
      if (idx < O) {
        const v4u u = __builtin_bit_cast(v4u, out[k]);
        st_dev64(pp + 2 * idx, (uint64_t)u.y << 32 | u.x);
        st_dev64(pp + 2 * idx + 1, (uint64_t)u.w << 32 | u.z);
      }
    }
    if (!last_arrival(L.tick + gid, (unsigned)S, (int *)LDS_AT(lds_i, o_flag))) return;
    const uint64_t *gp = (const uint64_t *)(L.part + gid * S * (4 * O));
#pragma unroll
    for (int k = 0; k < KO; ++k) {
      const int idx = min(tid + k * kThreads, O - 1);
      floatx4 s = {0.0f, 0.0f, 0.0f, 0.0f};
      for (int s0 = 0; s0 < S; s0 += 4) {
        uint64_t w[4][2];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int64_t o = (int64_t)min(s0 + q, S - 1) * (2 * O) + 2 * idx;
          w[q][0] = ld_dev64(gp + o);
          w[q][1] = ld_dev64(gp + o + 1);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (s0 + q < S) {
            const floatx4 p = __builtin_bit_cast(
                floatx4, v4u{(uint32_t)w[q][0], (uint32_t)(w[q][0] >> 32), (uint32_t)w[q][1],
                             (uint32_t)(w[q][1] >> 32)});
            s = s0 + q == 0 ? p : s + p;
          }
      }
      out[k] = s;
    }
  }
#pragma unroll
  for (int k = 0; k < KO; ++k) {
    const int idx = tid + k * kThreads;
    if (idx >= O) continue;
    const int ol = idx % 64, rg = idx / 64 % G, t = idx / 64 / G;
    const int nn = row0 + 16 * t + (ol & 15);
    if (nn >= N) continue;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int m = m0 + 16 * rg + 4 * (ol >> 4) + v;
      if (m < A.M) {
        float *y = L.y + (int64_t)m * N + nn;
        *y = L.beta ? *y + out[k][v] : out[k][v];
      }
    }
  }
}

// ---- X planes and T1s ---------------------------------------------------------
constexpr int kPrepThreads = 512;
struct PrepX {
  const void *x;
  uint8_t *xp;
  int K, wg0;
  uint32_t units;  // 16-byte units to write
};
struct PrepT1 {
  const void *x;
  const float *a;
  float *t1p;
  int K, r, nz, wg0;
};
struct PrepArgs {
  PrepX x[kMaxSlimSegs];
  PrepT1 t[kMaxSlimSegs];
  int nx, nt, t_wgs, M, G, XT;
};

// Workgroups [0, t_wgs): partial T1 tiles of 16 tokens x 16 ranks over one of
// nz slices of K, 8 waves splitting the slice, on fp32 MFMA (chunk c of 16 k:
// lane quarter g takes k = 16 c + 4 g + e, one float4 of X and of A); the
// rest: X planes, one 16-byte unit a thread.
template <int XB>
__global__ __launch_bounds__(kPrepThreads) void k_slim_prep(PrepArgs A) {
  __shared__ float red[8][16][17];
  const int tid = threadIdx.x, lane = tid & 63;
  const int b = (int)blockIdx.x;
  if (b < A.t_wgs) {
    int i = 0;
    while (i + 1 < A.nt && b >= A.t[i + 1].wg0) ++i;
    const PrepT1 &q = A.t[i];
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, g = lane >> 4;
    const int rt = (q.r + 15) / 16, w = b - q.wg0;
    const int z = w % q.nz, w2 = w / q.nz;
    const int m0 = w2 / rt * 16, j0 = w2 % rt * 16;
    const int64_t K = q.K;
    const int C = q.K / 16, cz0 = C * z / q.nz, cz = C * (z + 1) / q.nz - cz0;
    const int c0 = cz0 + cz * wave / 8, c1 = cz0 + cz * (wave + 1) / 8;
    const float *ar = q.a + (int64_t)min(j0 + l16, q.r - 1) * K + 4 * g;
    const int64_t xo = (int64_t)min(m0 + l16, A.M - 1) * K + 4 * g;
    floatx4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    constexpr int UN = 8;
    for (int c = c0; c < c1; c += UN) {
      float4 xv[UN], av[UN];
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        const int k = 16 * min(c + u, c1 - 1);
        xv[u] = load_x4<XB>(q.x, xo + k);
        av[u] = *(const float4 *)(ar + k);
      }
      __builtin_amdgcn_sched_barrier(0);  // all loads ahead of their uses
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        const bool in = c + u < c1;
        const float4 x = xv[u], a = av[u];
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? x.x : 0.0f, in ? a.x : 0.0f, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? x.y : 0.0f, in ? a.y : 0.0f, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? x.z : 0.0f, in ? a.z : 0.0f, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? x.w : 0.0f, in ? a.w : 0.0f, acc, 0, 0, 0);
      }
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) red[wave][4 * g + v][l16] = acc[v];
    __syncthreads();
    if (tid < 256) {
      const int mm = tid >> 4, j = tid & 15;
      if (m0 + mm < A.M && j0 + j < q.r) {
        float s = red[0][mm][j];
#pragma unroll
        for (int ww = 1; ww < 8; ++ww) s += red[ww][mm][j];
        q.t1p[((int64_t)z * A.M + m0 + mm) * q.r + j0 + j] = s;
      }
    }
    return;
  }
  int i = 0;
  while (i + 1 < A.nx && b >= A.x[i + 1].wg0) ++i;
  const PrepX &q = A.x[i];
  const uint32_t u = (uint32_t)(b - q.wg0) * kPrepThreads + tid;
  if (u >= q.units) return;
  // unit (chunk, unit, step, part, token group, lane); a wave shares all but
  // the lane
  const int ln = (int)(u & 63u), row = ln & 15, g = ln >> 4;
  const uint32_t v = __builtin_amdgcn_readfirstlane(u >> 6);
  const uint32_t w = v / (uint32_t)A.XT;  // ((chunk U) + unit) 4 + step
  const int tl = (int)(v - w * (uint32_t)A.XT), rg = tl >= A.G ? tl - A.G : tl;
  const int s = (int)(w & 3u);
  const uint32_t U = (uint32_t)(q.K + kUnit - 1) / kUnit, cu = w >> 2;
  const int chunk = (int)(cu / U), un = (int)(cu - (uint32_t)chunk * U);
  const int m = (chunk * A.G + rg) * 16 + row;
  const bool low = tl >= A.G;
  const int k = kUnit * un + 64 * (s >> 1) + 32 * (g & 1) + 16 * (s & 1) + 8 * (g >> 1);
  uint4 o = make_uint4(0, 0, 0, 0);
  if (m < A.M && k < q.K) {
    const int64_t e = (int64_t)m * q.K + k;
    if (XB) {
      o = *(const uint4 *)((const uint16_t *)q.x + e);
    } else {
      const float4 a = *(const float4 *)((const float *)q.x + e);
      const float4 c = *(const float4 *)((const float *)q.x + e + 4);
      const float f[8] = {a.x, a.y, a.z, a.w, c.x, c.y, c.z, c.w};
      uint32_t h[4];
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        h[p] = bf16_pair(f[2 * p], f[2 * p + 1]);
        if (low)
          h[p] = bf16_pair(f[2 * p] - __uint_as_float(h[p] << 16),
                           f[2 * p + 1] - __uint_as_float(h[p] & 0xffff0000u));
      }
      o = make_uint4(h[0], h[1], h[2], h[3]);
    }
  }
  *(uint4 *)(q.xp + (size_t)u * 16) = o;
}

// ---- host side --------------------------------------------------------------------
int g_slim_cus[64] = {};
int slim_cus() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  if (g_slim_cus[dev] == 0) {
    int v = 0;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
      return 0;
    g_slim_cus[dev] = v;
  }
  return g_slim_cus[dev];
}

template <class C>
hipError_t run_slim(const SlimArgs &A, dim3 grid, uint32_t lds, hipStream_t st) {
  auto k = k_slim<C>;
  static bool attr = false;  // per instantiation
  if (!attr) {
    const hipError_t e = hipFuncSetAttribute(
        (const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsLimit);
    if (e != hipSuccess) return e;
    attr = true;
  }
  return qh_launch(k, grid, dim3(kThreads), lds, st, A, lds - 16u);
}

}  // namespace

// The forward's calls that this path can take: whole 64-element blocks a row,
// rank at most 64, 16-byte aligned codes, X and A; and the range in which it was
// timed against the GEMM tiles (within it SlimPlan::us decides):
//  * 17 tokens or more (below, the decode kernels),
//  * up to 512 tokens while tokens x rows stay within 3M (fp32) or 6M (bf16), or
//    up to 48 tokens of any row count: 128256 x 4096 at 20 tokens in fp32 161 us
//    against 414, 33000 x 2048 at 48 48 against 112,
//  * with K below 1024 up to 384 tokens; below 768 up to 600k outputs, below 512
//    up to 350k, below 320 none (1752 x 192 14 us against 13 at any count).
bool slim_ok(const DevQW &w, const void *x, int x_bf16, const float *a, int64_t M, int64_t r) {
  auto al = [](const void *p) { return (((uintptr_t)p) & 15) == 0; };
  if (M < 17 || M > (w.cols < 1024 ? 384 : 512) || w.cols < 320) return false;
  const int64_t most = w.cols < 512 ? 350000 : w.cols < 768 ? 600000
                                    : (int64_t)(x_bf16 ? 6 : 3) << 20;
  if (M * w.rows > most && (M > 48 || w.cols < 768)) return false;
  return r >= 0 && r <= 64 && w.bs == 64 && w.rows > 0 && w.cols > 0 && w.cols % 64 == 0 &&
         w.cols < (1 << 24) && w.rows < (1 << 24) && al(w.codes) && al(x) && (r == 0 || al(a));
}

// Token groups: as many as fit (48 fp32 or 64 bf16 tokens a workgroup), evenly
// over the workgroups that share them.  (R, units of K per workgroup): the
// cheapest estimate in cycles of a CU, rounds of one workgroup per CU times
//  * 18000 for a workgroup's start and end (7.1 to 7.5 us measured: arguments,
//    first loads, table, last sum),
//  * per unit of a wave (two waves per SIMD) the larger of its code bytes at
//    the CU's share of HBM and its MFMAs plus its X tiles at 64 bytes a cycle
//    (4 x 16 rows: measured 4200 cycles for R = 2, 6500 for R = 3 at 48
//    fp32 tokens),
// plus 15000 where slices meet (partial sums out, ticket, sums back: 7 us
// measured).  The plan's us is fitted to 3280 calls of one to four layers, r = 0, 8
// and 64 (6 % rms): the rounds, X read and its planes written, the output, the
// codes, and for an adapter T1 and its term; where a group's layers are of
// unequal rows the grid's empty workgroups take slots of full ones (4.5 us once
// they push it past one round).  The runtime takes the plan where us is below
// the tiles' estimate plus 1 us (0.2 without an adapter): 2979 of the 3280, 40 of
// them slower than the tiles by more than 3 %, 8 by more than 6 % (if all were
// taken 255 and 185: 468 tokens of 136 x 2560 without an adapter 20.7 us against
// 13.4, 126 of 13904 x 768 60 against 46, 299 of three layers on 576 26 against 17).
SlimPlan slim_plan(int count, const DevQW *w, const int64_t *r, int64_t M, int x_bf16) {
  SlimPlan p;
  const int cus = slim_cus();
  if (cus <= 0 || count < 1 || count > kMaxSlimSegs || M < 1) return p;
  const int gmax = x_bf16 ? 4 : 3;
  const int64_t gm = (M + 15) / 16;
  p.chunks = (int)((gm + gmax - 1) / gmax);
  p.G = std::max(2, (int)((gm + p.chunks - 1) / p.chunks));
  p.P = x_bf16 ? 1 : 2;
  const double mfma = 128.0 * (p.P + 1) * p.G, xl2 = 512.0 * p.P * p.G;
  int64_t umax = 0, rmax = 0;
  for (int i = 0; i < count; ++i) {
    umax = std::max(umax, (w[i].cols + kUnit - 1) / kUnit);
    rmax = std::max(rmax, r[i]);
  }
  int64_t rows = 0, kmax = 0;
  double code_mb = 0;
  for (int i = 0; i < count; ++i) {
    rows += w[i].rows;
    kmax = std::max(kmax, w[i].cols);
    code_mb += (double)((w[i].cols + kUnit - 1) / kUnit) * (double)w[i].rows * 64e-6;
  }
  const int rhi = p.P * p.G >= 4 && p.G >= 3 ? 3 : 4;  // more spill registers
  double best = 0;
  for (int R = 2; R <= rhi; ++R)
    for (int64_t q = 8; q <= ((umax + 7) / 8) * 8; q += 4) {  // units per workgroup
      int64_t wgs = 0, groups = 0, um = 0;
      int64_t gx = 0;
      int S[kMaxSlimSegs], smax = 1, nbp = 0;
      for (int i = 0; i < count; ++i) {
        const int64_t U = (w[i].cols + kUnit - 1) / kUnit;
        const int64_t T = (w[i].rows + 16 * R - 1) / (16 * R);
        S[i] = (int)((U + q - 1) / q);
        const int64_t us = (U + S[i] - 1) / S[i];
        um = std::max(um, us);
        nbp = std::max(nbp, (int)(2 * us) | 1);
        smax = std::max(smax, S[i]);
        wgs += T * S[i] * p.chunks;
        groups += T * p.chunks;
        gx = std::max(gx, T);
      }
      const uint32_t lds = slim_lds(p.G, R, nbp, rmax);
      if (smax > kMaxSlices || nbp > kMaxNb || groups > kDecodeMaxTiles || lds > kLdsLimit)
        continue;
      const int64_t rounds = (wgs + cus - 1) / cus;
      const double unit = std::max(840.0 * R, mfma * R + xl2);
      const double cost = (double)rounds * (18000.0 + (double)((um + 7) / 8) * unit) +
                          (smax > 1 ? 15000.0 : 0.0);
      if (p.ok && cost >= best) continue;
      best = cost;
      p.ok = true;
      p.R = R;
      p.lds = lds;
      const bool f32 = p.P == 2;
      const double wu = (double)((um + 7) / 8) * unit / 2400.0, occ = (double)wgs / cus;
      const double mk = (double)M * (double)kmax * 1e-6;
      p.us = (f32 ? 3.7 : 3.2) + (double)rounds * (f32 ? 2.5 + 1.13 * wu : 3.2 + 1.06 * wu) +
             occ * (f32 ? -1.3 : -1.3 + 0.15 * wu) + (smax > 1 ? f32 ? 3.4 : 4.3 : 0.0) +
             (f32 ? 5.8 : 2.75) * mk + (f32 ? 8.5 : 5.9) * (double)M * (double)rows * 1e-6 +
             0.175 * code_mb;
      if (rmax > 0)
        p.us += (f32 ? 2.3 : 3.0) +
                (double)((rmax + 15) / 16) * (1.3 * (double)rounds + (f32 ? 0.7 : 1.3) * mk);
      if (count > 1 && wgs <= cus && gx * smax * p.chunks * count > cus) p.us += 4.5;
      for (int i = 0; i < count; ++i) {
        p.S[i] = S[i];
        p.groups[i] = (int)((w[i].rows + 16 * R - 1) / (16 * R));
        p.part_floats[i] =
            S[i] > 1 ? (size_t)p.groups[i] * p.chunks * S[i] * ((size_t)R * p.G * 256) : 0;
        p.xp_bytes[i] =
            (size_t)p.chunks * ((w[i].cols + kUnit - 1) / kUnit) * 4 * p.P * p.G * 1024;
        // K slices of a partial T1: about 1024 elements, so that a wave
        // loads its share at once
        p.nz[i] = (int)std::min<int64_t>(kMaxT1Parts, (w[i].cols + 1023) / 1024);
      }
    }
  return p;
}

hipError_t launch_slim_prep(int count, const SlimIn *in, const SlimPlan &p, int64_t M,
                            int x_bf16, hipStream_t st) {
  PrepArgs A{};
  A.M = (int)M;
  A.G = p.G;
  A.XT = p.P * p.G;
  int wg = 0;
  for (int i = 0; i < count; ++i) {
    if (in[i].r == 0) continue;
    PrepT1 &q = A.t[A.nt++];
    q = PrepT1{in[i].x, in[i].a, in[i].t1p, (int)in[i].w.cols, (int)in[i].r, p.nz[i], wg};
    wg += (int)((M + 15) / 16) * ((q.r + 15) / 16) * q.nz;
  }
  A.t_wgs = wg;
  for (int i = 0; i < count; ++i) {
    bool seen = false;  // segments that read the same X share its planes
    for (int j = 0; j < i; ++j) seen = seen || in[j].xp == in[i].xp;
    if (seen) continue;
    PrepX &q = A.x[A.nx++];
    q = PrepX{in[i].x, (uint8_t *)in[i].xp, (int)in[i].w.cols, wg,
              (uint32_t)(p.xp_bytes[i] / 16)};
    wg += (int)((q.units + kPrepThreads - 1) / kPrepThreads);
  }
  if (x_bf16) return qh_launch(k_slim_prep<1>, dim3(wg), dim3(kPrepThreads), 0, st, A);
  return qh_launch(k_slim_prep<0>, dim3(wg), dim3(kPrepThreads), 0, st, A);
}

hipError_t launch_slim(int count, const SlimIn *in, const SlimPlan &p, int64_t M,
                       unsigned *tickets, hipStream_t st) {
  if (!p.ok || count < 1 || count > kMaxSlimSegs) return hipErrorInvalidValue;
  SlimArgs A{};
  A.M = (int)M;
  A.chunks = p.chunks;
  int gx = 0, gy = 0;
  int64_t used = kDecodeTileCounterBase;
  for (int i = 0; i < count; ++i) {
    const SlimIn &s = in[i];
    SlimSegDev &L = A.seg[i];
    if (p.S[i] > 1 && !s.part) return hipErrorInvalidValue;
    L.codes = s.w.codes;
    L.scales = s.w.kind == 0 ? (const void *)s.w.scales : (const void *)s.w.scale_codes;
    L.absmax = s.w.absmax;
    L.xp = (const uint8_t *)s.xp;
    L.t1p = s.t1p;
    L.t1 = s.t1;
    L.lb = s.lb;
    L.y = s.y;
    L.part = s.part;
    L.tick = tickets + used;
    L.N = (int)s.w.rows;
    L.K = (int)s.w.cols;
    L.kind = s.w.kind;
    L.r = (int)s.r;
    L.nz = p.nz[i];
    L.groups = p.groups[i];
    L.S = p.S[i];
    const int U = (L.K + kUnit - 1) / kUnit;
    L.nbp = (2 * ((U + L.S - 1) / L.S)) | 1;
    L.s_lora = s.s;
    L.beta = s.beta;
    gx = std::max(gx, p.groups[i]);
    gy = std::max(gy, p.S[i]);
    used += (int64_t)p.groups[i] * p.chunks;
  }
  if (used > kTicketWords) return hipErrorInvalidValue;
  const dim3 grid((unsigned)gx, (unsigned)(gy * p.chunks), (unsigned)count);
#define QH_SLIM(G_, P_, R_) \
  if (p.G == G_ && p.P == P_ && p.R == R_) return run_slim<Slim<G_, P_, R_>>(A, grid, p.lds, st);
  QH_SLIM(2, 2, 2)
  QH_SLIM(2, 2, 3)
  QH_SLIM(2, 2, 4)
  QH_SLIM(3, 2, 2)
  QH_SLIM(3, 2, 3)
  QH_SLIM(2, 1, 2)
  QH_SLIM(2, 1, 3)
  QH_SLIM(2, 1, 4)
  QH_SLIM(3, 1, 2)
  QH_SLIM(3, 1, 3)
  QH_SLIM(3, 1, 4)
  QH_SLIM(4, 1, 2)
  QH_SLIM(4, 1, 3)
#undef QH_SLIM
  return hipErrorInvalidValue;
}

}  // namespace qh
