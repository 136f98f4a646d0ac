// "gemm" module, second file: the prefill GEMM on digits, every weight type but Q8_0 (whose int8 kernels
// decode nothing: 4096 x 4096, 300 and 2048 tokens, 28 and 105 us, in two digits 36 and 108).
//
//   C[m][c_off + n] (=, +=, silu(C) *)  sum over 32-blocks b of  (sa[m][b] * ws[n][b]) * J[m][n][b]
//   J[m][n][b] = sum over the block's 32 k of x[m][k] * w[n][k], integers
//
// A kernel on packed weights unpacks them again for every tile of tokens, and the int8 matrix instruction leaves J as
// int32, 16 conversions a lane.  Here both sides come as digits of four bits and a sign, written once per matmul by two
// small kernels: x = 16 x1 + x0 and w = 256 w2 + 16 w1 + w0 (one to three digits, by the type's range).  A digit
// n = 0 .. 15 is the FP6 (E2M3) code n, the number n / 8 (16 is one too, 2.0, the largest top digit);
// v_mfma_scale_f32_32x32x64_f8f6f4 takes 64 of them a row at four times the f16 rate, so a block's 32 k of x0 and of x1
// lie in its two halves with scales 2^3 and 2^7 against the same 32 digits of w in both, and one instruction a weight
// digit gives J: every digit product and every partial sum is an integer below 2^24 (|x| <= 128, |w| <= 4096, 32 of
// them), so the f32 result is exact, as int32 was, and needs no conversion.  What is left to the vector ALU is one fused
// multiply-add per output and block with the scale tile sa x ws, which comes from the outer-product instruction
// (v_mfma_f32_32x32x1_2b_f32: both row tiles at once).
//
// Q6_K and Q3_K, whose sub-scales hold for 16 values, have them folded into w ((q - 32) * sc, three digits; (q - 4) * sc, at
// most 128, two), ws is d; the others' ws is their block scale: Q4_0, MXFP4, IQ3_S, Q4_K and
// Q5_K are one digit, IQ3_XXS, IQ4_XS and IQ4_NL two.
//
// Bound by power: at 17408 x 5120 x 8192 the chip runs this kernel below 1.9 GHz, without its DMA at 2.1, and every part
// that is taken out -- operand reads from LDS, DMA, multiply-adds -- gives back about its share of the energy, not of the
// cycles.  Hence few bytes and few instructions per product: a wave's operands serve 64 x 64 outputs, the addresses of a
// step are six registers and immediate offsets.  Kernel alone, 17408 x 5120 x 8192: one digit 863 TOP/s, two 651, three
// 504 (the int8 kernels on packed weights: Q4_0 and Q3_K at 12288 x 4096 x 4096 650 and 375).
// Q4_K and Q5_K with the min term, 17408 x 5120, us, int8 kernels and this: 8192 tokens Q4_K 2020 / 1850, 2048 544 / 470, Q5_K
// 593 / 472, 300 110 / 100, 143 / 100.
// Matmul with both writing kernels, us, before and now, 12288 x 4096 x 1024: Q4_0 173 / 136, MXFP4 183 / 135, IQ3_S
// 201 / 147, Q3_K 293 / 182, Q6_K 277 / 234; x 4096: Q6_K 1094 / 790, IQ3_XXS 742 / 596.
#include "common.h"
#include <type_traits>

typedef uint32_t u4v __attribute__((ext_vector_type(4)));
typedef uint32_t u2v __attribute__((ext_vector_type(2)));
typedef int i8v __attribute__((ext_vector_type(8)));
typedef int i4v __attribute__((ext_vector_type(4)));
typedef int i2v __attribute__((ext_vector_type(2)));

// LDS by byte offset (the kernel's one shared array begins at 0)
#define LDS_P(T, a) ((__attribute__((address_space(3))) T*)(uint32_t)(a))
// 16 bytes a lane straight into LDS: lane l's land at the wave's base + 16 l
__device__ inline void dma16(const void* src, uint32_t lds_wave_base) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src, LDS_P(void, lds_wave_base), 16, 0, 0);
}

// ---- images, what a work-group's DMA brings as it lies: 128 tokens x one block
//   [4 groups of 32][2 digits][32][16 bytes] the block's first 128 bits, [4][2][32][8 bytes] the other 64, [128] f32 sa
// and 128 weight rows x one block
//   per digit [128][16 bytes], [128][8 bytes]; then [128] f32 ws
// A tile's blocks follow each other.  NB: blocks a step of the GEMM takes; steps are whole KiB.
// Types with a minimum (MN: Q4_K, Q5_K) have behind sa [128][8 bytes] u = sa * S, and behind ws v, of the min term: bf16 pieces
// x1 | x2 << 16, x3 | x3 << 16.
template <int NW, int MN = 0> struct DImg {
  static constexpr int NB = NW == 3 ? 1 : 2;
  static constexpr int R = NB == 2 ? 3 : 4;  // stages in LDS
  static constexpr int T = MN ? 7680 : NB == 2 ? 6656 : 7168, W = NB == 2 ? NW * 3072 + 512 + 1024 * MN : 10240;
  static constexpr int STAGE = NB * (T + W);
  static constexpr int TSA = 6144, TU = 6656, WWS = NW * 3072, WV = WWS + 512;
};

// 16 codes, a byte each, to 96 bits
__device__ inline uint32_t pack4(uint32_t x) {
  const uint32_t a = (x & 0x003F003Fu) | ((x >> 2) & 0x0FC00FC0u);
  return (a & 0xFFFu) | ((a >> 4) & 0xFFF000u);
}
__device__ inline void pack16(const uint32_t* c, uint32_t* o) {
  const uint32_t p0 = pack4(c[0]), p1 = pack4(c[1]), p2 = pack4(c[2]), p3 = pack4(c[3]);
  o[0] = p0 | p1 << 24;
  o[1] = p1 >> 8 | p2 << 16;
  o[2] = p2 >> 16 | p3 << 8;
}
// a block's digit (8 words of codes) of row r of an image
__device__ inline void put_digit(uint8_t* lo, uint8_t* hi, const uint32_t* c) {
  uint32_t o[6];
  pack16(c, o);
  pack16(c + 4, o + 3);
  *(u4v*)lo = (u4v){o[0], o[1], o[2], o[3]};
  *(u2v*)hi = (u2v){o[4], o[5]};
}
// four int8 values: sign bits at bit 0 of each byte, magnitudes
__device__ inline void sign_mag(uint32_t v, uint32_t& s, uint32_t& a) {
  s = (v >> 7) & 0x01010101u;
  a = (v ^ ((s << 8) - s)) + s;
}

// act_digits: aq [M][K], asc [K/32][M], absum [K/16][M] -> token images xt of img bytes, 7680: with u.  Rows past M are
// zeros.  A thread: two blocks of a row.  grid (K / 256, 2 * token tiles), local 256.
extern "C" __global__ __launch_bounds__(256) void act_digits(const signed char* __restrict__ aq, const float* __restrict__ asc,
                                                             const short* __restrict__ absum, int M, int K, int img,
                                                             uint8_t* __restrict__ xt) {
  const int s = blockIdx.x, r = (blockIdx.y & 1) * 64 + (threadIdx.x & 63), q = threadIdx.x >> 6, m = (blockIdx.y >> 1) * 128 + r;
  uint8_t* dst = xt + ((size_t)(blockIdx.y >> 1) * (K >> 5) + s * 8 + 2 * q) * img;
  u4v x[4] = {};
  if (m < M)
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = *(const u4v*)(aq + (size_t)m * K + s * 256 + q * 64 + i * 16);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    uint32_t lo[8], hi[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      uint32_t sg, a;
      sign_mag(x[2 * i + (k >> 2)][k & 3], sg, a);
      lo[k] = (a & 0x0F0F0F0Fu) | sg << 5;
      hi[k] = ((a >> 4) & 0x0F0F0F0Fu) | sg << 5;
    }
    uint8_t* p = dst + i * img + (r >> 5) * 1024 + (r & 31) * 16;
    uint8_t* p8 = dst + i * img + 4096 + (r >> 5) * 512 + (r & 31) * 8;
    put_digit(p, p8, lo);
    put_digit(p + 512, p8 + 256, hi);
    const int b = s * 8 + 2 * q + i;
    const float sa = m < M ? asc[(size_t)b * M + m] : 0.0f;
    *(float*)(dst + i * img + 6144 + r * 4) = sa;
    if (img == DImg<1, 1>::T) {
      uint32_t w0, w1;
      split3(m < M ? sa * (float)((int)absum[(size_t)(2 * b) * M + m] + (int)absum[(size_t)(2 * b + 1) * M + m]) : 0.0f, w0, w1);
      *(u2v*)(dst + i * img + DImg<1, 1>::TU + r * 8) = (u2v){w0, w1 | w1 << 16};
    }
  }
}

// ---- the rows.  A thread: two blocks b[0], b[1] of row n; v[i]: their values as int8, four a word, or, with the sub-scales
// folded in (Q6_K, Q3_K), signs and the products of the magnitudes.
template <int QT> struct DType { enum { NW = 1, MN = 0 }; };
template <> struct DType<QT_Q6_K> { enum { NW = 3, MN = 0 }; };
template <> struct DType<QT_Q3_K> { enum { NW = 2, MN = 0 }; };
template <> struct DType<QT_IQ3_XXS> { enum { NW = 2, MN = 0 }; };
template <> struct DType<QT_IQ4_XS> { enum { NW = 2, MN = 0 }; };
template <> struct DType<QT_IQ4_NL> { enum { NW = 2, MN = 0 }; };
template <> struct DType<QT_Q4_K> { enum { NW = 1, MN = 1 }; };
template <> struct DType<QT_Q5_K> { enum { NW = 1, MN = 1 }; };

// int8 values of eight words -> NW digits' codes
template <int NW> __device__ inline void codes_i8(const uint32_t* v, uint32_t (*c)[8]) {
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    uint32_t sg, a;
    sign_mag(v[k], sg, a);
    if constexpr (NW == 1) {
      c[0][k] = a | sg << 5;
    } else {
      c[0][k] = (a & 0x0F0F0F0Fu) | sg << 5;
      c[1][k] = ((a >> 4) & 0x0F0F0F0Fu) | sg << 5;
    }
  }
}
// the same times a sub-scale of each half
template <int NW> __device__ inline void codes_scaled(const uint32_t* v, int sc0, int sc1, uint32_t (*c)[8]) {
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int sc = k < 4 ? sc0 : sc1;
    const uint32_t asc = (uint32_t)abs(sc);
    uint32_t sg, a;
    sign_mag(v[k], sg, a);
    sg = (sg ^ (sc < 0 ? 0x01010101u : 0u)) << 5;
    // (two 16-bit products in one 32-bit multiply: each is at most 4096)
    const uint32_t e = (a & 0x00FF00FFu) * asc, o = ((a >> 8) & 0x00FF00FFu) * asc;
    c[0][k] = (e & 0x000F000Fu) | (o & 0x000F000Fu) << 8 | sg;
    c[1][k] = ((e >> 4) & 0x000F000Fu) | ((o << 4) & 0x0F000F00u) | sg;
    if constexpr (NW == 3) c[2][k] = ((e >> 8) & 0x001F001Fu) | (o & 0x1F001F00u) | sg;
  }
}

// row_digits__QT: the raw planes' rows n0 .. n0 + gridDim.y * 64 (those past N as zeros) -> row images wt.
// grid (K / 256, 2 * row tiles), local 256.  (tabs: the codebooks)
template <int QT>
__device__ inline void row_digits(const uint8_t* __restrict__ raw, const uint32_t* __restrict__ tabs, int N, int nsb, int n0,
                                  uint8_t* __restrict__ wt) {
  constexpr int NW = DType<QT>::NW, MN = DType<QT>::MN;
  using I = DImg<NW, MN>;
  const int s = blockIdx.x, r = (blockIdx.y & 1) * 64 + (threadIdx.x & 63), q = threadIdx.x >> 6, n = n0 + (blockIdx.y >> 1) * 128 + r;
  const bool in = n < N;
  const size_t u = (size_t)(in ? n : 0) * nsb + s;  // the row's superblock in every plane
  int b[2] = {2 * q, 2 * q + 1};
  uint32_t c[2][NW][8];
  float ws[2], mv[2] = {};  // (mv: the min term's row factor)
  if constexpr (QT == QT_Q6_K) {
    // blocks 4 n2 + c and 4 n2 + c + 2: low and high nibbles of ql bytes 64 n2 + 32 c + 0..31, bits 2 c + 4 i of qh bytes 32 n2 + 0..31
    const PlanesQ6K pl = planes_q6k((size_t)N, nsb);
    const int n2 = q >> 1, c1 = q & 1;
    b[0] = 4 * n2 + c1;
    b[1] = b[0] + 2;
    const u4v L[2] = {*(const u4v*)(raw + pl.ql + u * 128 + 64 * n2 + 32 * c1), *(const u4v*)(raw + pl.ql + u * 128 + 64 * n2 + 32 * c1 + 16)};
    const u4v H[2] = {*(const u4v*)(raw + pl.qh + u * 64 + 32 * n2), *(const u4v*)(raw + pl.qh + u * 64 + 32 * n2 + 16)};
    const signed char* sc = (const signed char*)(raw + pl.sc + u * 16);
    ws[0] = ws[1] = f16_bits_to_f32(*(const unsigned short*)(raw + pl.d + u * 2));
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      uint32_t v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const uint32_t l = (L[k >> 2][k & 3] >> (4 * i)) & 0x0F0F0F0Fu, h = (H[k >> 2][k & 3] >> (2 * c1 + 4 * i)) & 0x03030303u;
        v[k] = ((l | h << 4) + 0x60606060u) ^ 0x80808080u;  // q - 32
      }
      codes_scaled<3>(v, sc[2 * b[i]], sc[2 * b[i] + 1], c[i]);
    }
  } else if constexpr (QT == QT_Q4_K || QT == QT_Q5_K) {
    // blocks 2 q and 2 q + 1: the low and high nibbles of bytes 32 q .. 32 q + 31.  The values are taken around their middle
    // h = 8 or 16, which makes Q5_K's one digit (-16 is one) and leaves less to cancel between products and min term, v: d sc
    // q - dmin mn = d sc (q - h) + (h d sc - dmin mn).  Off by, against 64 bits, K = 5120 and 17408, of the result's norm: Q4_K
    // 1.2e-7 and 1.7e-7 (int8 kernels 1.6e-7, 2.4e-7), tokens with a mean of half their deviation 2.3e-7 and 3.8e-7 (2.8e-7,
    // 3.3e-7; with the values as they are 9.7e-7, 1.8e-6), Q5_K 1.6e-7 and 2.5e-7.
    const PlanesQ4K pl = planes_q4k((size_t)N, nsb);
    const u4v L[2] = {*(const u4v*)(raw + pl.qs + u * 128 + 32 * q), *(const u4v*)(raw + pl.qs + u * 128 + 32 * q + 16)};
    const u4v h = *(const u4v*)(raw + pl.hdr + u * 16);
    u2v H = {0, 0};
    if constexpr (QT == QT_Q5_K) H = *(const u2v*)(raw + pl.qh + u * 32 + 8 * q);
    const float d = f16_bits_to_f32(h[0]), dmin = f16_bits_to_f32(h[0] >> 16);
    int sc[2], mn[2];
    q4k_scales_pair(h[1], h[2], h[3], q, sc[0], sc[1], mn[0], mn[1]);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      uint32_t v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const uint32_t w = L[k >> 2][k & 3];
        if constexpr (QT == QT_Q4_K) v[k] = q40_vals(w >> (4 * i));  // q - 8
        else v[k] = ((i ? q5k_hi(w, H[k >> 2], k & 3) : q5k_lo(w, H[k >> 2], k & 3)) + 0x70707070u) ^ 0x80808080u;  // q - 16
      }
      codes_i8<1>(v, c[i]);
      ws[i] = d * (float)sc[i];
      mv[i] = (QT == QT_Q4_K ? 8.0f : 16.0f) * ws[i] - dmin * (float)mn[i];
    }
  } else if constexpr (QT == QT_Q3_K) {
    const PlanesIQ3S pl = planes_iq3s((size_t)N, nsb);
    const uint32_t* h = (const uint32_t*)(raw + pl.hd + u * 12);
    ws[0] = ws[1] = f16_bits_to_f32(*(const unsigned short*)(raw + pl.d + u * 2));
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const u2v D = *(const u2v*)(raw + pl.qs + u * 64 + b[i] * 8);
      const uint32_t H = *(const uint32_t*)(raw + pl.sg + u * 32 + b[i] * 4);
      uint32_t v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = q3k_vals(D[k >> 2], H, k);
      int sc0, sc1;
      q3k_scales(h[0], h[1], h[2], b[i], sc0, sc1);
      codes_scaled<2>(v, sc0, sc1, c[i]);
    }
  } else if constexpr (QT == QT_IQ4_XS) {
    const u2v h = *(const u2v*)(raw + planes_iq4xs((size_t)N, nsb).hdr + u * 8);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const u4v w = *(const u4v*)(raw + u * 128 + 16 * b[i]);
      uint32_t v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = iq4_lookup(k < 4 ? w[k] : w[k - 4] >> 4);
      codes_i8<2>(v, c[i]);
      ws[i] = f16_bits_to_f32(h[0]) * (float)((int)(((h[1] >> (4 * b[i])) & 15u) | ((h[0] >> (16 + 2 * b[i])) & 3u) << 4) - 32);
    }
  } else if constexpr (QT == QT_Q4_0 || QT == QT_MXFP4 || QT == QT_IQ4_NL) {
    // block b: 16 bytes, low nibbles values 0..15, high nibbles 16..31
    const uint32_t h = QT == QT_MXFP4 ? *(const unsigned short*)(raw + planes_mxfp4((size_t)N, nsb).e + u * 8 + 2 * q)
                                      : *(const uint32_t*)(raw + planes_q40((size_t)N, nsb).d + u * 16 + 4 * q);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const u4v w = *(const u4v*)(raw + u * 128 + 16 * b[i]);
      uint32_t v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const uint32_t x = k < 4 ? w[k] : w[k - 4] >> 4;
        v[k] = nib_vals<QT>(x);
      }
      codes_i8<NW>(v, c[i]);
      ws[i] = QT == QT_MXFP4 ? e8m0_half(h >> (8 * i)) : f16_bits_to_f32(i ? h >> 16 : h);
    }
  } else if constexpr (QT == QT_IQ3_S) {
    const PlanesIQ3S pl = planes_iq3s((size_t)N, nsb);
    const uint32_t* h = (const uint32_t*)(raw + pl.hd + u * 12);
    const float d = f16_bits_to_f32(*(const unsigned short*)(raw + pl.d + u * 2));
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const u2v D = *(const u2v*)(raw + pl.qs + u * 64 + b[i] * 8);
      const uint32_t S = *(const uint32_t*)(raw + pl.sg + u * 32 + b[i] * 4), h9 = h[b[i] >> 2] >> (8 * (b[i] & 3));
      uint32_t v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const uint32_t idx = ((D[k >> 2] >> (8 * (k & 3))) & 0xFFu) | ((h9 >> k) & 1u) << 8;
        v[k] = iq3s_signed4(tabs[idx], (S >> (4 * k)) & 0xFu);
      }
      codes_i8<1>(v, c[i]);
      ws[i] = d * (float)(1 + 2 * (int)((h[2] >> (4 * b[i])) & 0xFu));
    }
  } else {  // IQ3_XXS
    const PlanesIQ3XXS pl = planes_iq3xxs((size_t)N, nsb);
    const float d = 0.25f * f16_bits_to_f32(*(const unsigned short*)(raw + pl.d + u * 2));
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const u2v D = *(const u2v*)(raw + pl.qs + u * 64 + b[i] * 8);
      const uint32_t a = *(const uint32_t*)(raw + pl.ss + u * 32 + b[i] * 4);
      uint32_t v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k)
        v[k] = iq3s_signed4(tabs[512 + ((D[k >> 2] >> (8 * (k & 3))) & 0xFFu)], (iq3xxs_signs8(a, k >> 1) >> (4 * (k & 1))) & 0xFu);
      codes_i8<2>(v, c[i]);
      ws[i] = d * (float)(1 + 2 * (int)(a >> 28));
    }
  }
  uint8_t* dst = wt + ((size_t)(blockIdx.y >> 1) * nsb + s) * 8 * I::W;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    uint8_t* img = dst + b[i] * I::W;
#pragma unroll
    for (int d = 0; d < NW; ++d) {
      if (!in)
#pragma unroll
        for (int k = 0; k < 8; ++k) c[i][d][k] = 0;
      put_digit(img + d * 3072 + r * 16, img + d * 3072 + 2048 + r * 8, c[i][d]);
    }
    *(float*)(img + I::WWS + r * 4) = in ? ws[i] : 0.0f;
    if (!in) mv[i] = 0.0f;
    if constexpr (MN) {
      uint32_t w0, w1;
      split3(mv[i], w0, w1);
      *(u2v*)(img + I::WV + r * 8) = (u2v){w0, w1 | w1 << 16};
    }
  }
}
#define ROW_DIGITS(QT)                                                                                                  \
  extern "C" __global__ __launch_bounds__(256) void row_digits__QTYPE##QT(const uint8_t* raw, const uint32_t* tabs, int N, \
                                                                          int nsb, int n0, uint8_t* wt) {               \
    row_digits<QT>(raw, tabs, N, nsb, n0, wt);                                                                          \
  }
ROW_DIGITS(12) ROW_DIGITS(13) ROW_DIGITS(14) ROW_DIGITS(2) ROW_DIGITS(20) ROW_DIGITS(23) ROW_DIGITS(39) ROW_DIGITS(11) ROW_DIGITS(21) ROW_DIGITS(18)

// ---- gemm_d: 128 tokens x 128 rows in four waves of 64 x 64, two work-groups a compute unit.  Blocks [b0, b1), an even number.
// (Eight waves of 32 x 64, four a SIMD, hide more waits and read each row digit from LDS twice as often: 5 - 6 % slower, at
// 17408 x 5120 x 8192 812 against 863 TOP/s with one digit, 632 / 651 with two, 476 / 504 with three.)
template <int NW, int MN>
__device__ __forceinline__ void gemm_d_body(uint8_t* lds_base, const uint8_t* __restrict__ xt, const uint8_t* __restrict__ wt,
                                            float* __restrict__ C, int M, int N, int ldc, int c_off, int accumulate, int m0,
                                            int n0, int nblk, int b0, int b1) {
  // (every access below is by offset; the array itself has to stay)
  asm volatile("" :: "v"((__attribute__((address_space(3))) uint8_t*)lds_base) : "memory");
  using I = DImg<NW, MN>;
  constexpr int NB = I::NB, R = I::R, STAGE = I::STAGE, TS = NB * I::T, WS = NB * I::W;
  constexpr int TKB = TS / 1024, KB = STAGE / 1024, ND = (KB + 3) / 4;
  const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave & 1, wn = wave >> 1;
  const int steps = (b1 - b0) / NB;
  const uint8_t* tsrc = xt + ((size_t)(m0 >> 7) * nblk + b0) * I::T + wave * 1024;
  const uint8_t* wsrc = wt + ((size_t)(n0 >> 7) * nblk + b0) * I::W + wave * 1024 - TS;
  uint32_t lane16 = lane * 16;
  // piece i of a step's DMA for this wave: KiB wave + 4 i of the stage, tokens then rows
  auto dma = [&](const uint8_t* ts, const uint8_t* ws, uint32_t stage, int i) {
    if (4 * i + 4 > KB && wave >= (KB & 3)) return;
    const uint8_t* src = 4 * i + 4 <= TKB || (4 * i < TKB && wave + 4 * i < TKB) ? ts : ws;
    asm volatile("" : "+v"(lane16));
    dma16(src + i * 4096 + lane16, stage + wave * 1024 + i * 4096);
  };
  struct F6 { u4v lo; u2v hi; };
  F6 A[2], W[2][NW];
  float saop[2], wsop;
  // addresses of the step the loads are in: token digits, their second part, sa; row digits, second part, ws; the min term's
  const uint32_t oA16 = wm * 2048 + lane * 16, oA8 = 4096 + wm * 1024 + lane * 8;
  const uint32_t oW16 = TS + (wn * 64 + l32) * 16, oW8 = TS + 2048 + (wn * 64 + l32) * 8;
  const uint32_t oSA = I::TSA + (wm * 64 + l32) * 4, oWS = TS + I::WWS + (wn * 64 + lane) * 4;
  const uint32_t oU = I::TU + g * I::T + (wm * 64 + l32) * 8, oV = TS + I::WV + g * I::W + (wn * 64 + l32) * 8;
  uint32_t pA16, pA8, pW16, pW8, pSA, pWS, pU = 0, pV = 0;
  auto at = [&](uint32_t stage) {
    pA16 = oA16 + stage; pA8 = oA8 + stage; pW16 = oW16 + stage; pW8 = oW8 + stage; pSA = oSA + stage; pWS = oWS + stage;
    asm volatile("" : "+v"(pA16), "+v"(pA8), "+v"(pW16), "+v"(pW8), "+v"(pSA), "+v"(pWS));
    if constexpr (MN) {
      pU = oU + stage; pV = oV + stage;
      asm volatile("" : "+v"(pU), "+v"(pV));
    }
  };
  auto ldA = [&](int ms, int blk) {
    A[ms].lo = *LDS_P(const u4v, pA16 + (NB == 2 ? blk : 0) * I::T + ms * 1024);
    A[ms].hi = *LDS_P(const volatile u2v, pA8 + (NB == 2 ? blk : 0) * I::T + ms * 512);
  };
  auto ldW = [&](int ns, int blk) {
#pragma unroll
    for (int d = 0; d < NW; ++d) {
      W[ns][d].lo = *LDS_P(const u4v, pW16 + (NB == 2 ? blk : 0) * I::W + d * 3072 + ns * 512);
      W[ns][d].hi = *LDS_P(const volatile u2v, pW8 + (NB == 2 ? blk : 0) * I::W + d * 3072 + ns * 256);
    }
  };
  auto ldSA = [&](int ms, int blk) { saop[ms] = *LDS_P(const float, pSA + (NB == 2 ? blk : 0) * I::T + ms * 128); };
  auto ldWS = [&](int blk) { wsop = *LDS_P(const float, pWS + (NB == 2 ? blk : 0) * I::W); };
  auto six = [](const F6& f) {
    const i4v a = __builtin_bit_cast(i4v, f.lo);
    const i2v b = __builtin_bit_cast(i2v, f.hi);
    return (i8v){a[0], a[1], a[2], a[3], b[0], b[1], 0, 0};
  };
  const int sca = g ? 134 : 130, scb = 0x008A8682;  // token digit g 2^3 or 2^7; row digit d 2^3, 2^7, 2^11, a byte each

  v16f res[2][2], J[2];
  v32f P[2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) res[i][0][e] = res[i][1][e] = J[i][e] = 0.0f;
#pragma unroll
  for (int e = 0; e < 32; ++e) P[0][e] = P[1][e] = 0.0f;
  auto mfma_p = [&](int ms) {
    v32f z;
#pragma unroll
    for (int e = 0; e < 32; ++e) z[e] = 0.0f;
    P[ms] = __builtin_amdgcn_mfma_f32_32x32x1f32(saop[ms], wsop, z, 0, 0, 0);
  };
  // The min term, u x v of both blocks of a step in one bf16 instruction, added straight to the results: a lane half takes a
  // block, its eight k are the products of the pieces but u3 v3 (2^-32 of the whole).
  u2v U[2], V[2];
  auto ldU = [&](int ms) { U[ms] = *LDS_P(const u2v, pU + ms * 256); };
  auto ldV = [&](int ns) { V[ns] = *LDS_P(const u2v, pV + ns * 256); };
  auto mfma_min = [&](int ms, int ns) {
    typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
    const uint32_t v11 = __builtin_amdgcn_perm(V[ns][0], V[ns][0], 0x01000100u), v22 = __builtin_amdgcn_perm(V[ns][0], V[ns][0], 0x03020302u);
    const u4v a = {U[ms][0], U[ms][0], U[ms][0], U[ms][1]}, b = {v11, v22, V[ns][1], V[ns][0]};
    res[ms][ns] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf8, a), __builtin_bit_cast(bf8, b), res[ms][ns], 0, 0, 0);
  };
  // ---- prologue: the first R - 1 steps on their way, the first block's operands
#pragma unroll
  for (int q = 0; q < R - 1; ++q)
#pragma unroll
    for (int i = 0; i < ND; ++i) dma(tsrc + (size_t)min(q, steps - 1) * TS, wsrc + (size_t)min(q, steps - 1) * WS, q * STAGE, i);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  at(0);
  ldA(0, 0); ldSA(0, 0);
  ldW(0, 0); ldWS(0);
  mfma_p(0);
  ldSA(1, 0);
  uint32_t st = 0;
  int step = 0;
  uint32_t stf = (R - 2) * STAGE;  // (the first turn's first pieces: of a step that the prologue brought, once more)
  const uint8_t *tf = tsrc + (size_t)min(R - 2, steps - 1) * TS, *wf = wsrc + (size_t)min(R - 2, steps - 1) * WS;
  // Two blocks a turn, four products a block: tiles (0,0) (0,1) (1,1) (1,0), then (0,1) (0,0) (1,0) (1,1), so that the operands
  // that come free first are those the next block begins with.  A product's values are added while the next one runs; a
  // slot also carries a piece of the loads.  The stage of the step R - 1 on is refilled behind the meeting, when no wave
  // reads the step before any more.
#pragma unroll 1
  for (int b = b0; b < b1; b += 2) {
#pragma unroll
    for (int p = 0; p < 8; ++p) {
      const int blk = p >> 2, q = p & 3, ms = q >> 1, ns = blk ? (q == 0 || q == 3) : (q == 1 || q == 2);
      // -- the product
      {
        v16f z;
#pragma unroll
        for (int e = 0; e < 16; ++e) z[e] = 0.0f;
        v16f& j = J[p & 1];
        j = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(six(A[ms]), six(W[ns][0]), z, 2, 2, 0, sca, 0, scb);
        if constexpr (NW > 1) j = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(six(A[ms]), six(W[ns][1]), j, 2, 2, 0, sca, 1, scb);
        if constexpr (NW > 2) j = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(six(A[ms]), six(W[ns][2]), j, 2, 2, 0, sca, 2, scb);
      }
      if (q == 1) mfma_p(1);
      if (q == 3) mfma_p(0);
      if constexpr (MN) {  // (each tile between two of its multiply-adds)
        if (p == 2) mfma_min(0, 0);
        if (p == 3) mfma_min(0, 1);
        if (p == 4) mfma_min(1, 1);
        if (p == 5) mfma_min(1, 0);
      }
      // -- the step's meeting: what the waves brought for the next step lies in LDS, the step before is read
      if (NB == 2 ? p == 6 : q == 2) {
        __builtin_amdgcn_sched_barrier(0);
        if (NB == 2) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        else if (wave < (KB & 3)) asm volatile("s_waitcnt vmcnt(5)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        stf = st == 0 ? (R - 1) * STAGE : st - STAGE;
        st = st + STAGE == R * STAGE ? 0 : st + STAGE;
        at(st);
        const int nf = min(step + R - 1, steps - 1);
        tf = tsrc + (size_t)nf * TS; wf = wsrc + (size_t)nf * WS;
        ++step;
      }
      // -- loads for later
      const int nb = (p + 2) >> 2 & 1;  // (block of the loads below: from p == 2 the second, from 6 the next step's first)
      if (q == 0) { ldW(blk ? 0 : 1, blk); ldA(1, blk); }
      if (q == 2) { ldA(0, nb); ldSA(0, nb); ldWS(nb); }
      if (q == 3) { ldW(blk ? 0 : 1, nb); ldSA(1, nb); }
      if constexpr (MN) {
        if (p == 0) { ldU(0); ldV(0); ldV(1); }
        if (p == 1) ldU(1);
      }
      {
        // (two blocks a step: two pieces a slot, 6, 7 and, one turn on, 0, 1; one: three and two)
        const int f = NB == 2 ? (p + 2 & 7) * 2 : q == 2 ? 0 : q == 3 ? 3 : ND;
        if (f < ND) dma(tf, wf, stf, f);
        if (f + 1 < ND) dma(tf, wf, stf, f + 1);
        if (NB == 1 && q == 2) dma(tf, wf, stf, 2);
      }
      __builtin_amdgcn_sched_barrier(0);
      // -- the values of the product before
      {
        const int pb = (p + 7) & 7, blp = pb >> 2, qp = pb & 3, mp = qp >> 1, np = blp ? (qp == 0 || qp == 3) : (qp == 1 || qp == 2);
#pragma unroll
        for (int e = 0; e < 16; ++e) res[mp][np][e] = __builtin_fmaf(P[mp][16 * np + e], J[pb & 1][e], res[mp][np][e]);
        asm volatile("" : "+v"(res[mp][np]));
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  // the last product: tile (1, 1) of the second block
#pragma unroll
  for (int e = 0; e < 16; ++e) res[1][1][e] = __builtin_fmaf(P[1][16 + e], J[1][e], res[1][1][e]);

  // ---- epilogue: lane = weight row n, accumulator i = token row 8 * (i / 4) + 4 * g + i % 4
#pragma unroll
  for (int ms = 0; ms < 2; ++ms)
#pragma unroll
    for (int ns = 0; ns < 2; ++ns) {
      const int n = n0 + wn * 64 + ns * 32 + l32, m = m0 + wm * 64 + ms * 32 + 4 * g;
      if (n >= N || m >= M) continue;
      store16<true>(res[ms][ns], C + (size_t)m * ldc + c_off + n, ldc, M - m, accumulate, [](float v, int) { return v; });
    }
}

// Work-groups go to the eight chiplets in turn: chiplet x takes the x-th eighth of a list of n, so that neighbours in it
// share an L2 (chiplet y has n / 8, one more if y < n % 8).
__device__ inline int d_list_of(int id, int n) {
  const int x = id & 7;
  return x * (n >> 3) + min(x, n & 7) + (id >> 3);
}
// Tile L of the list of mt token tiles x nt row tiles: panels of eight token tiles, row tile by row tile.
__device__ inline void d_tile_of(int L, int mt, int nt, int& tm, int& tn) {
  const int panel = L / (8 * nt), rem = L - panel * 8 * nt, pw = min(8, mt - panel * 8);
  tn = rem / pw;
  tm = panel * 8 + rem - tn * pw;
}

// gemm_d__NW: rows [n0, n0 + 128 ..) of an N-row matrix, nt row tiles of them in wt.  The list's first `whole` tiles take a
// work-group each; each of the others is shared out over `pieces`, superblocks by superblocks, which leave their sums in ws
// [tile][piece][128][128] for d_reduce: a launch's last round, of a few tiles, would take as long as a full one (17408 x 5120,
// Q4_0: 512 tokens are 544 tiles on 512 places, 139 us, with the last 32 in 10 pieces 109).  grid (whole + (tiles - whole) *
// pieces).
#define GEMM_D(NAME, ...)                                                                                               \
  extern "C" __global__ __launch_bounds__(256, 2) void gemm_d__##NAME(                                                  \
      const uint8_t* xt, const uint8_t* wt, float* C, int M, int N, int K, int ldc, int c_off, int accumulate, int n0, int nt, \
      int whole, int pieces, float* ws) {                                                                               \
    using I = DImg<__VA_ARGS__>;                                                                                        \
    __shared__ __attribute__((aligned(1024))) uint8_t lds[I::R * I::STAGE];                                             \
    const int mt = (M + 127) / 128, tail = mt * nt - whole, nsb = K >> 8;                                               \
    int L, y = 0, ny = 1;                                                                                               \
    if ((int)blockIdx.x < whole) {                                                                                      \
      L = d_list_of(blockIdx.x, whole);                                                                                 \
    } else {                                                                                                            \
      const int q = blockIdx.x - whole;                                                                                 \
      y = q / tail;                                                                                                     \
      ny = pieces;                                                                                                      \
      L = whole + d_list_of(q - y * tail, tail);                                                                        \
    }                                                                                                                   \
    int tm, tn;                                                                                                         \
    d_tile_of(L, mt, nt, tm, tn);                                                                                       \
    const int m0 = tm * 128, r0 = n0 + tn * 128;                                                                        \
    if (ny > 1) {                                                                                                       \
      C = ws + (ptrdiff_t)((L - whole) * ny + y) * 16384 - (ptrdiff_t)(m0 * 128 + r0);                                  \
      ldc = 128;                                                                                                        \
      c_off = accumulate = 0;                                                                                           \
    }                                                                                                                   \
    gemm_d_body<__VA_ARGS__>(lds, xt, wt - (size_t)(n0 >> 7) * (K >> 5) * I::W, C, M, N, ldc, c_off, accumulate, m0, r0, \
                             K >> 5, nsb * y / ny * 8, nsb * (y + 1) / ny * 8);                                         \
  }
GEMM_D(NW1, 1, 0) GEMM_D(NW2, 2, 0) GEMM_D(NW3, 3, 0) GEMM_D(NW1_MN1, 1, 1)

// d_reduce: the pieces' sums of the tiles from `whole` on, added in their order, out to C.  wide: rows of whole vectors.
// grid (tiles, 16), local 256: eight rows of a tile; eight planes are loaded before the first is added.
extern "C" __global__ __launch_bounds__(256) void d_reduce(const float* __restrict__ ws, float* __restrict__ C, int M, int N, int ldc,
                                                           int c_off, int accumulate, int wide, int n0, int nt, int whole,
                                                           int pieces) {
  int tm, tn;
  d_tile_of(whole + blockIdx.x, (M + 127) / 128, nt, tm, tn);
  const int r = blockIdx.y * 8 + (threadIdx.x >> 5), m = tm * 128 + r, c = threadIdx.x & 31;
  if (m >= M) return;
  // (a thread: four columns next to each other, or, where a row's vectors would not be whole, 32 apart)
  const float* p = ws + (size_t)blockIdx.x * pieces * 16384 + r * 128;
  const int nb = n0 + tn * 128;
  v4f s = {0.0f, 0.0f, 0.0f, 0.0f};
  auto plane = [&](int y) {
    const float* q = p + (size_t)y * 16384;
    return wide ? *(const v4f*)(q + 4 * c) : (v4f){q[c], q[c + 32], q[c + 64], q[c + 96]};
  };
  for (int y = 0; y < pieces; y += 8) {
    v4f a[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) a[i] = plane(min(y + i, pieces - 1));
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (y + i < pieces) s += a[i];
  }
  float* cr = C + (size_t)m * ldc + c_off + nb;
  auto out = [&](float v, float old) { return accumulate == 1 ? v + old : accumulate == 2 ? v * (old / (1.0f + __expf(-old))) : v; };
  if (wide) {
    if (nb + 4 * c >= N) return;
    v4f* o = (v4f*)(cr + 4 * c);
    const v4f old = accumulate ? *o : s;
    *o = (v4f){out(s[0], old[0]), out(s[1], old[1]), out(s[2], old[2]), out(s[3], old[3])};
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int n = c + 32 * i;
    if (nb + n < N) cr[n] = out(s[i], accumulate ? cr[n] : 0.0f);
  }
}
