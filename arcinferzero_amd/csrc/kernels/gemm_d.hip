// "gemm" module, second file: the prefill GEMM on digits (Q4_0, MXFP4, IQ3_S, IQ3_XXS, Q3_K, Q6_K; long chunks).
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
// most 128, two), ws is d; the others' ws is their block scale: Q4_0, MXFP4 and IQ3_S are one digit, IQ3_XXS two.
//
// Bound by power: at 17408 x 5120 x 8192 the chip runs this kernel at 1.85 GHz, without its DMA at 2.1, and every part that
// is taken out -- operand reads from LDS, DMA, multiply-adds -- gives back about its share of the energy, not of the
// cycles.  Hence few bytes per product (the digits of a row are read once for two tiles, a type of fewer digits is
// faster), and four waves a SIMD rather than two with twice the tile.  Kernel alone, 17408 x 5120 x 4096: one digit 765 -
// 800 TOP/s, two 595, three 465 (the int8 kernels on packed weights: Q4_0 and Q3_K at 12288 x 4096 x 4096 650 and 375).
// Matmul with both writing kernels, us, before and now, 12288 x 4096 x 1024: Q4_0 173 / 149, MXFP4 183 / 147, IQ3_S
// 201 / 160, Q3_K 293 / 203; x 4096: Q6_K 1094 / 901, IQ3_XXS 742 / 671.
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
template <int NW> struct DImg {
  static constexpr int NB = NW == 3 ? 1 : 2;
  static constexpr int R = NB == 2 ? 3 : 4;  // stages in LDS
  static constexpr int T = NB == 2 ? 6656 : 7168, W = NB == 2 ? NW * 3072 + 512 : 10240;
  static constexpr int STAGE = NB * (T + W);
  static constexpr int TSA = 6144, WWS = NW * 3072;
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

// act_digits: aq [M][K], asc [K/32][M] -> token images xt of img bytes.  Rows past M are zeros.  A thread: two blocks of a
// row.  grid (K / 256, 2 * token tiles), local 256.
extern "C" __global__ __launch_bounds__(256) void act_digits(const signed char* __restrict__ aq, const float* __restrict__ asc,
                                                             int M, int K, int img, uint8_t* __restrict__ xt) {
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
  }
}

// ---- the rows.  A thread: two blocks b[0], b[1] of row n; v[i]: their values as int8, four a word, or, with the sub-scales
// folded in (Q6_K, Q3_K), signs and the products of the magnitudes.
template <int QT> struct DType;
template <> struct DType<QT_Q6_K> { enum { NW = 3 }; };
template <> struct DType<QT_Q4_0> { enum { NW = 1 }; };
template <> struct DType<QT_MXFP4> { enum { NW = 1 }; };
template <> struct DType<QT_Q3_K> { enum { NW = 2 }; };
template <> struct DType<QT_IQ3_S> { enum { NW = 1 }; };
template <> struct DType<QT_IQ3_XXS> { enum { NW = 2 }; };

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
  constexpr int NW = DType<QT>::NW;
  using I = DImg<NW>;
  const int s = blockIdx.x, r = (blockIdx.y & 1) * 64 + (threadIdx.x & 63), q = threadIdx.x >> 6, n = n0 + (blockIdx.y >> 1) * 128 + r;
  const bool in = n < N;
  const size_t u = (size_t)(in ? n : 0) * nsb + s;  // the row's superblock in every plane
  int b[2] = {2 * q, 2 * q + 1};
  uint32_t c[2][NW][8];
  float ws[2];
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
  } else if constexpr (QT == QT_Q4_0 || QT == QT_MXFP4) {
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
        v[k] = QT == QT_MXFP4 ? mxfp4_lookup(x) : nib_vals<QT>(x);
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
  }
}
#define ROW_DIGITS(QT)                                                                                                  \
  extern "C" __global__ __launch_bounds__(256) void row_digits__QTYPE##QT(const uint8_t* raw, const uint32_t* tabs, int N, \
                                                                          int nsb, int n0, uint8_t* wt) {               \
    row_digits<QT>(raw, tabs, N, nsb, n0, wt);                                                                          \
  }
ROW_DIGITS(14) ROW_DIGITS(2) ROW_DIGITS(39) ROW_DIGITS(11) ROW_DIGITS(21) ROW_DIGITS(18)

// A result leaves for good: stored past the caches, which keep the operands of the neighbouring tiles.
__device__ inline void st_stream(float* p, float v) { __builtin_nontemporal_store(v, p); }

// ---- gemm_d: 128 tokens x 128 rows in eight waves of 32 x 64, two work-groups a compute unit: four waves a SIMD, in 128
// registers, so that a wave's waits -- for a product, for the next operands -- lie under the others' work.  Blocks [b0, b1),
// an even number.
template <int NW>
__device__ __forceinline__ void gemm_d_body(uint8_t* lds_base, const uint8_t* __restrict__ xt, const uint8_t* __restrict__ wt,
                                            float* __restrict__ C, int M, int N, int ldc, int c_off, int accumulate, int m0,
                                            int n0, int nblk, int b0, int b1) {
  // (every access below is by offset; the array itself has to stay)
  asm volatile("" :: "v"((__attribute__((address_space(3))) uint8_t*)lds_base) : "memory");
  using I = DImg<NW>;
  constexpr int NB = I::NB, R = I::R, STAGE = I::STAGE, KB = STAGE / 1024, TKB = NB * I::T / 1024, ND = (KB + 7) / 8;
  const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave & 3, wn = wave >> 2;
  const int steps = (b1 - b0) / NB;
  const uint8_t* tsrc = xt + ((size_t)(m0 >> 7) * nblk + b0) * I::T;
  const uint8_t* wsrc = wt + ((size_t)(n0 >> 7) * nblk + b0) * I::W;
  uint32_t lane16 = lane * 16;
  // piece i of a step's DMA for this wave: KiB wave + 8 i of the stage
  auto dma = [&](int step, uint32_t stage, int i) {
    const int k = wave + 8 * i;
    if (8 * i + 8 > KB && k >= KB) return;
    const size_t off = k < TKB ? (size_t)(tsrc - xt) + (size_t)step * (NB * I::T) + k * 1024 : (size_t)step * (NB * I::W) + (k - TKB) * 1024;
    const uint8_t* src = (k < TKB ? xt : wsrc) + off;
    asm volatile("" : "+v"(lane16));
    dma16(src + lane16, stage + k * 1024);
  };
  struct F6 { u4v lo; u2v hi; };
  F6 A, W[NW];
  float saop, wsop;
  // (two lane offsets, the others formed where they are used: registers are the scarce thing)
  auto low16 = [&]() { uint32_t r; asm volatile("v_and_b32 %0, 0x1f0, %1" : "=v"(r) : "v"(lane16)); return r; };  // 16 l32
  auto shr = [](uint32_t o, auto n) { uint32_t r; asm volatile("v_lshrrev_b32 %0, %1, %2" : "=v"(r) : "i"(decltype(n)::value), "v"(o)); return r; };
  constexpr std::integral_constant<int, 1> by2{};
  constexpr std::integral_constant<int, 2> by4{};
  const uint32_t tw = wm * 1024, rw = wn * 1024;
  auto ldA = [&](uint32_t tb) {
    A.lo = *LDS_P(const u4v, lane16 + (tb + tw));
    A.hi = *LDS_P(const volatile u2v, shr(lane16, by2) + (tb + 4096 + tw / 2));
    saop = *LDS_P(const float, shr(low16(), by4) + (tb + I::TSA + tw / 8));
  };
  auto ldW = [&](int ns, uint32_t wb) {
    const uint32_t l16 = low16(), o8 = shr(l16, by2) + (wb + rw / 2);
#pragma unroll
    for (int d = 0; d < NW; ++d) {
      W[d].lo = *LDS_P(const u4v, l16 + (wb + rw) + d * 3072 + ns * 512);
      W[d].hi = *LDS_P(const volatile u2v, o8 + d * 3072 + 2048 + ns * 256);
    }
    if (ns == 0) wsop = *LDS_P(const float, shr(lane16, by4) + (wb + I::WWS + rw / 4));
  };
  auto six = [](const F6& f) {
    const i4v a = __builtin_bit_cast(i4v, f.lo);
    const i2v b = __builtin_bit_cast(i2v, f.hi);
    return (i8v){a[0], a[1], a[2], a[3], b[0], b[1], 0, 0};
  };
  // the scales: token digit g 2^3 or 2^7 (three digits: formed where they are used), row digit d 2^3, 2^7, 2^11, a byte each
  auto scale_a = [&]() {
    int v = g ? 134 : 130;
    if constexpr (NW == 3) asm volatile("v_bfe_u32 %0, %1, 9, 1\n\tv_lshl_or_b32 %0, %0, 2, %2" : "=&v"(v) : "v"(lane16), "s"(130));
    return v;
  };
  auto scale_b = []() {
    int v = 0x008A8682;
    if constexpr (NW == 3) asm volatile("v_mov_b32 %0, %1" : "=v"(v) : "i"(0x008A8682));
    return v;
  };
  v16f res[2];
#pragma unroll
  for (int e = 0; e < 16; ++e) res[0][e] = res[1][e] = 0.0f;
  auto product = [&]() {
    v16f J;
#pragma unroll
    for (int e = 0; e < 16; ++e) J[e] = 0.0f;
    const int sca = scale_a(), scb = scale_b();
    J = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(six(A), six(W[0]), J, 2, 2, 0, sca, 0, scb);
    if constexpr (NW > 1) J = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(six(A), six(W[1]), J, 2, 2, 0, sca, 1, scb);
    if constexpr (NW > 2) J = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(six(A), six(W[2]), J, 2, 2, 0, sca, 2, scb);
    return J;
  };

  // ---- prologue: the first R - 1 steps on their way, the first block's operands
#pragma unroll
  for (int q = 0; q < R - 1; ++q)
#pragma unroll
    for (int i = 0; i < ND; ++i) dma(min(q, steps - 1), q * STAGE, i);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  auto tok_of = [&](uint32_t stage, int blk) { return NB == 2 ? stage + blk * I::T : stage; };
  auto row_of = [&](uint32_t stage, int blk) { return NB == 2 ? stage + NB * I::T + blk * I::W : stage + I::T; };
  ldA(0); ldW(0, row_of(0, 0));
  uint32_t st = 0;  // the step's stage
  int step = 0;

#pragma unroll 1
  for (int b = b0; b < b1; b += 2) {
#pragma unroll
    for (int blk = 0; blk < 2; ++blk) {
      const uint32_t st1 = st + STAGE == R * STAGE ? 0 : st + STAGE;  // the next step's stage
      const uint32_t stf = st == 0 ? (R - 1) * STAGE : st - STAGE;    // the stage of step R - 1 from here, which nobody reads any more
      const bool last = NB == 1 || blk == 1;                          // the step's last block
      const uint32_t cur_t = tok_of(st, blk), cur_w = row_of(st, blk);
      const uint32_t nxt_t = last ? st1 : tok_of(st, 1), nxt_w = last ? row_of(st1, 0) : row_of(st, 1);
      v32f P;
#pragma unroll
      for (int e = 0; e < 32; ++e) P[e] = 0.0f;
      P = __builtin_amdgcn_mfma_f32_32x32x1f32(saop, wsop, P, 0, 0, 0);
      v16f J = product();
      __builtin_amdgcn_sched_barrier(0);
      ldW(1, cur_w);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int e = 0; e < 16; ++e) res[0][e] = __builtin_fmaf(P[e], J[e], res[0][e]);
      asm volatile("" : "+v"(res[0]));
      __builtin_amdgcn_sched_barrier(0);
      J = product();
      __builtin_amdgcn_sched_barrier(0);
      if (last) {  // the meeting: what the waves brought for the next step lies in LDS, and the step before is read
        if (NB == 2) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        else if (ND == 3 && wave < (KB & 7)) asm volatile("s_waitcnt vmcnt(3)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
      }
      ldA(nxt_t); ldW(0, nxt_w);
      if (last) {
#pragma unroll
        for (int i = 0; i < ND; ++i) dma(min(step + R - 1, steps - 1), stf, i);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int e = 0; e < 16; ++e) res[1][e] = __builtin_fmaf(P[16 + e], J[e], res[1][e]);
      asm volatile("" : "+v"(res[1]));
      __builtin_amdgcn_sched_barrier(0);
      if (last) { st = st1; ++step; }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // ---- epilogue (its lane index from the one offset that was kept): lane = weight row n, accumulator i = token row 8 * (i / 4) + 4 * g + i % 4
#pragma unroll
  for (int ns = 0; ns < 2; ++ns) {
    const int el = (int)(lane16 >> 4), n = n0 + wn * 64 + ns * 32 + (el & 31);
    if (n >= N) continue;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int m = m0 + wm * 32 + 8 * (i >> 2) + 4 * (el >> 5) + (i & 3);
      if (m >= M) continue;
      float v = res[ns][i];
      float* cp = C + (size_t)m * ldc + c_off + n;
      if (accumulate == 1) {
        v += *cp;
      } else if (accumulate == 2) {
        const float gt = *cp;
        v *= gt / (1.0f + __expf(-gt));
      }
      st_stream(cp, v);
    }
  }
}

// Tile L of mt token tiles x nt row tiles: work-groups go to the eight chiplets in turn, so chiplet x takes the x-th eighth of
// a list of tiles in panels of eight token tiles, row tile by row tile -- neighbours in one L2 share rows and tokens.
__device__ inline void d_tile_of(int id, int mt, int nt, int& tm, int& tn) {
  const int total = mt * nt, x = id & 7, j = id >> 3;
  const int L = x * (total >> 3) + min(x, total & 7) + j;  // (chiplet y has total / 8 tiles, one more if y < total % 8)
  const int panel = L / (8 * nt), rem = L - panel * 8 * nt, pw = min(8, mt - panel * 8);
  tn = rem / pw;
  tm = panel * 8 + rem - tn * pw;
}

// gemm_d__NW: rows [n0, n0 + 128 ..) of an N-row matrix, nt row tiles of them in wt.  grid (ceil(M / 128) * nt, ny); ny > 1:
// the superblocks shared out, plane y of C (here a workspace [ny][M][ldc]) the y-th piece's sums.
#define GEMM_D(NWV)                                                                                                     \
  extern "C" __global__ __launch_bounds__(512, 4) void gemm_d__NW##NWV(                                                 \
      const uint8_t* xt, const uint8_t* wt, float* C, int M, int N, int K, int ldc, int c_off, int accumulate, int n0, int nt) { \
    __shared__ __attribute__((aligned(1024))) uint8_t lds[DImg<NWV>::R * DImg<NWV>::STAGE];                             \
    int tm, tn;                                                                                                         \
    d_tile_of(blockIdx.x, (M + 127) / 128, nt, tm, tn);                                                                 \
    const int y = blockIdx.y, ny = gridDim.y, nsb = K >> 8;                                                             \
    gemm_d_body<NWV>(lds, xt, wt - (size_t)(n0 >> 7) * (K >> 5) * DImg<NWV>::W, C + (size_t)y * M * ldc, M, N, ldc, c_off, \
                     accumulate, tm * 128, n0 + tn * 128, K >> 5, nsb * y / ny * 8, nsb * (y + 1) / ny * 8);            \
  }
GEMM_D(1) GEMM_D(2) GEMM_D(3)
