// The GEMM on digits, what its kernels share (gemm_d.hip: dense matrices; moe_d.hip: expert tiles): images and digits, the rows'
// decoding, the loop.
#pragma once
#include "digit_pack.h"

typedef int i8v __attribute__((ext_vector_type(8)));
typedef int i4v __attribute__((ext_vector_type(4)));
typedef int i2v __attribute__((ext_vector_type(2)));

// LDS by byte offset (the kernel's one shared array begins at 0)
#define LDS_P(T, a) ((__attribute__((address_space(3))) T*)(uint32_t)(a))
// 16 bytes a lane straight into LDS: lane l's land at the wave's base + 16 l.  From a buffer: a base and an offset in scalar
// registers and the lane's own offset, so that a step's pieces take no vector instruction.  (As 64-bit addresses they took ten a
// turn of the loop.  us before / now: Q4_K 17408 x 5120, 8192 tokens 1827 / 1772, the 300-token block 381 / 364, the 4096-token
// layer 622 / 613, the 1000-token block of Q3_K 499 / 493.)
typedef __amdgpu_buffer_rsrc_t d_buf;
__device__ __forceinline__ d_buf d_buffer(const void* p, size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ void dma16(d_buf b, uint32_t lane_off, uint32_t off, uint32_t lds_wave_base) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(b, LDS_P(void, lds_wave_base), 16, lane_off, off, 0, 0);
}

// a block's digit (8 words of codes) of row r of an image
__device__ inline void put_digit(uint8_t* lo, uint8_t* hi, const uint32_t* c) {
  uint32_t o[6];
  pack16(c, o);
  pack16(c + 4, o + 3);
  *(u4v*)lo = (u4v){o[0], o[1], o[2], o[3]};
  *(u2v*)hi = (u2v){o[4], o[5]};
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

// Row digits of superblock u (row * superblocks a row + superblock, of rows_total rows) as thread q of its four has them: blocks
// b[0], b[1], their digits' codes, scales and, with a minimum, the min term's factors.
template <int QT> struct RowDigits {
  static constexpr int NW = DType<QT>::NW, MN = DType<QT>::MN;
  int b[2];
  uint32_t c[2][NW][8];
  float ws[2], mv[2];
};
template <int QT>
__device__ inline void row_decode(const uint8_t* __restrict__ raw, const uint32_t* __restrict__ tabs, size_t rows_total, int nsb, size_t u, int q,
                                  RowDigits<QT>& out) {
  constexpr int NW = DType<QT>::NW;
  auto& b = out.b;
  auto& c = out.c;
  auto& ws = out.ws;
  auto& mv = out.mv;
  mv[0] = mv[1] = 0.0f;
  b[0] = 2 * q;
  b[1] = 2 * q + 1;
  if constexpr (QT == QT_Q6_K) {
    // blocks 4 n2 + c and 4 n2 + c + 2: low and high nibbles of ql bytes 64 n2 + 32 c + 0..31, bits 2 c + 4 i of qh bytes 32 n2 + 0..31
    const PlanesQ6K pl = planes_q6k(rows_total, nsb);
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
    // q - dmin mn = d sc (q - h) + (h d sc - dmin mn).  Off by, against 64 bits, 300 tokens x 2048 rows, K = 5120 and 17408 (in
    // pieces), of the result's norm: Q4_K 1.2e-7 and 1.9e-7 (int8 kernels 1.6e-7, 2.4e-7), tokens with a mean of half their
    // deviation 1.3e-7 and 1.9e-7 (2.7e-7, 3.2e-7); Q5_K the same.
    const PlanesQ4K pl = planes_q4k(rows_total, nsb);
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
    const PlanesIQ3S pl = planes_iq3s(rows_total, nsb);
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
    const u2v h = *(const u2v*)(raw + planes_iq4xs(rows_total, nsb).hdr + u * 8);
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
    const uint32_t h = QT == QT_MXFP4 ? *(const unsigned short*)(raw + planes_mxfp4(rows_total, nsb).e + u * 8 + 2 * q)
                                      : *(const uint32_t*)(raw + planes_q40(rows_total, nsb).d + u * 16 + 4 * q);
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
    const PlanesIQ3S pl = planes_iq3s(rows_total, nsb);
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
    const PlanesIQ3XXS pl = planes_iq3xxs(rows_total, nsb);
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
}

// ---- the loop: a wave's 64 x 64 outputs over `blocks` blocks, an even number, in a work-group of four waves.  I: the stages and the
// strides within them, of the second token tile (A_MS, A8_MS, S_MS, U_MS), of a further row digit (DIG), of a step's second block
// (T, W); o: the lane's addresses of the first.  dma.at(step), dma(stage, i): where piece i of a step, KiB wave + 4 i of its
// stage, comes from.  Every wave is behind its last reads of LDS when it returns, its last pieces have landed.
struct DAddr { uint32_t A16, A8, SA, U, W16, W8, WS, V; };
// Waits for a wave's pieces of stages of KB KiB but those of the last `later` steps: KB / 4 a step.  (The first waves have one more
// where KB / 4 is not whole, and wait for as many of the last step's too: a branch on the wave costs more, 64-token tiles of
// Q4_K, 300 tokens x 17408 rows, 111 -> 118 us.  EXACT: by the wave, where the last step's pieces were asked for just before.)
template <int KB, int later, bool EXACT> __device__ __forceinline__ void d_wait_but(int wave) {
  if (EXACT && later && KB % 4 && wave < KB % 4) asm volatile("s_waitcnt vmcnt(%0)" :: "n"(later * (KB / 4 + 1)) : "memory");
  else asm volatile("s_waitcnt vmcnt(%0)" :: "n"(later * (KB / 4)) : "memory");
}
// The work-group's waves meet; nothing but the wait before it is waited for
__device__ __forceinline__ void d_meet() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
// Brings the first AHEAD steps (the last step in the place of those past it) and waits for the first of them -- for all, if these are
// R - 1: 300 tokens x 17408 rows, 340 work-groups, otherwise 1 % slower.
template <class I, class DMA> __device__ __forceinline__ void d_prologue(DMA& dma, int steps) {
  constexpr int KB = I::STAGE / 1024, FIRST = I::R - 1;
#pragma unroll
  for (int q = 0; q < I::AHEAD; ++q) {
    if (q == FIRST) {  // (a stage each is on its way; the last is asked for when the first is there)
      d_wait_but<KB, FIRST - 1, false>(0);
      d_meet();
    }
    dma.at(min(q, steps - 1));
#pragma unroll
    for (int i = 0; i < (KB + 3) / 4; ++i) dma(q * I::STAGE, i);
  }
  if (I::AHEAD == FIRST) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  }
}
template <int NW, int MN, class I, class DMA>
__device__ __forceinline__ void d_loop(const DAddr& o, DMA& dma, int blocks, v16f (&res)[2][2]) {
  constexpr int NB = I::NB, R = I::R, STAGE = I::STAGE, KB = STAGE / 1024, ND = (KB + 3) / 4;
  static_assert(ND <= (NB == 2 ? 8 : 6), "the slots below carry that many pieces");
  const int lane = threadIdx.x & 63, g = lane >> 5, steps = blocks / NB;
  struct F6 { u4v lo; u2v hi; };
  F6 A[2], W[2][NW];
  float saop[2], wsop;
  // the lane's addresses in the first stage; st, the stage that the loads are in, and what else a place adds are immediate offsets
  uint32_t pA16 = o.A16, pA8 = o.A8, pW16 = o.W16, pW8 = o.W8, pSA = o.SA, pWS = o.WS, pU = o.U, pV = o.V;
  asm volatile("" : "+v"(pA16), "+v"(pA8), "+v"(pW16), "+v"(pW8), "+v"(pSA), "+v"(pWS));
  if constexpr (MN) asm volatile("" : "+v"(pU), "+v"(pV));
  static_assert((R - 1) * STAGE + (NB - 1) * I::W + (NW - 1) * I::DIG + 512 < 65536 && (R - 1) * STAGE + (NB - 1) * I::T + 2 * I::A_MS < 65536, "16 bits");
  int st = 0;
  auto ldA = [&](int ms, int blk) {
    A[ms].lo = *LDS_P(const u4v, pA16 + st * STAGE + (NB == 2 ? blk : 0) * I::T + ms * I::A_MS);
    A[ms].hi = *LDS_P(const volatile u2v, pA8 + st * STAGE + (NB == 2 ? blk : 0) * I::T + ms * I::A8_MS);
  };
  auto ldW = [&](int ns, int blk) {
#pragma unroll
    for (int d = 0; d < NW; ++d) {
      W[ns][d].lo = *LDS_P(const u4v, pW16 + st * STAGE + (NB == 2 ? blk : 0) * I::W + d * I::DIG + ns * 512);
      W[ns][d].hi = *LDS_P(const volatile u2v, pW8 + st * STAGE + (NB == 2 ? blk : 0) * I::W + d * I::DIG + ns * 256);
    }
  };
  auto ldSA = [&](int ms, int blk) { saop[ms] = *LDS_P(const float, pSA + st * STAGE + (NB == 2 ? blk : 0) * I::T + ms * I::S_MS); };
  auto ldWS = [&](int blk) { wsop = *LDS_P(const float, pWS + st * STAGE + (NB == 2 ? blk : 0) * I::W); };
  auto six = [](const F6& f) {
    const i4v a = __builtin_bit_cast(i4v, f.lo);
    const i2v b = __builtin_bit_cast(i2v, f.hi);
    return (i8v){a[0], a[1], a[2], a[3], b[0], b[1], 0, 0};
  };
  const int sca = g ? 134 : 130, scb = 0x008A8682;  // token digit g 2^3 or 2^7; row digit d 2^3, 2^7, 2^11, a byte each

  v16f J[2];
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
  auto ldU = [&](int ms) { U[ms] = *LDS_P(const u2v, pU + st * STAGE + ms * I::U_MS); };
  auto ldV = [&](int ns) { V[ns] = *LDS_P(const u2v, pV + st * STAGE + ns * 256); };
  auto mfma_min = [&](int ms, int ns) {
    typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
    const uint32_t v11 = __builtin_amdgcn_perm(V[ns][1], V[ns][1], 0x01000100u), v22 = __builtin_amdgcn_perm(V[ns][1], V[ns][1], 0x03020302u);
    const u4v a = {U[ms][0], U[ms][0], U[ms][0], U[ms][1]}, b = {v11, v22, V[ns][0], V[ns][1]};
    res[ms][ns] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf8, a), __builtin_bit_cast(bf8, b), res[ms][ns], 0, 0, 0);
  };
  // ---- prologue: the first R steps on their way (the last of them behind the first one's arrival), the first block's operands
  d_prologue<I>(dma, steps);
  ldA(0, 0); ldSA(0, 0);
  ldW(0, 0); ldWS(0);
  mfma_p(0);
  ldSA(1, 0);
  int step = 0;
  // Two blocks a turn, four products a block: tiles (0,0) (0,1) (1,1) (1,0), then (0,1) (0,0) (1,0) (1,1), so that the operands
  // that come free first are those the next block begins with.  A product's values are added while the next one runs; a
  // slot also carries a piece of the loads.  Behind a step's meeting the stage of that very step is refilled, with the step R on
  // (AHEAD = R: the products issued before the meeting wait for the last of the step's operands, no wave reads them any
  // more), so that pieces have R - 1 steps to arrive; or (AHEAD = R - 1) the stage of the step before.  us with the first, before in
  // the second way: Q4_K 17408 x 5120, 8192 tokens 1847 -> 1827, the 4096-token layer of Q4_K experts 631 -> 619, the 1000-token block
  // of Q3_K 506 -> 498; but 300 tokens of Q4_K on gemm_d64 374 -> 382.
  // Turn u of as many as bring the stages round, so that every place in LDS is a constant (with the stage in registers, eight more
  // vector instructions a turn.  us: Q4_K 17408 x 5120, 8192 tokens 1713 -> 1686, the 4096-token layer 595 -> 586, the 1000-token block of
  // Q3_K 476 -> 467.)
  auto turn = [&](auto u_) {
    constexpr int u = decltype(u_)::value;
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
        d_wait_but<KB, I::AHEAD - 2, (I::AHEAD < R)>(dma.wave);
        d_meet();
        __builtin_amdgcn_sched_barrier(0);
        dma.at(min(step + I::AHEAD, steps - 1));
        ++step;
      }
      // -- loads for later
      st = (NB == 2 ? u + (p >= 6) : 2 * u + (p >= 2) + (p >= 6)) % R;
      const int nb = (p + 2) >> 2 & 1;  // (block of the loads below: from p == 2 the second, from 6 the next step's first)
      if (q == 0) { ldW(blk ? 0 : 1, blk); ldA(1, blk); }
      if (q == 2) { ldA(0, nb); ldSA(0, nb); ldWS(nb); }
      if (q == 3) { ldW(blk ? 0 : 1, nb); ldSA(1, nb); }
      if constexpr (MN) {
        if (p == 0) { ldU(0); ldV(0); ldV(1); }
        if (p == 1) ldU(1);
      }
      {
        // (two blocks a step: two pieces a slot, 6, 7 and, one turn on, 0, 1; one: three each)
        const int f = NB == 2 ? (p + 2 & 7) * 2 : q == 2 ? 0 : q == 3 ? 3 : ND;
        // (the first turn's first pieces are of a step that the prologue brought, once more)
        const int met = NB == 2 ? u + R - (p < 6) : 2 * u + blk, stf = (I::AHEAD == R ? met : met + R - 1) % R * STAGE;
        if (f < ND) dma(stf, f);
        if (f + 1 < ND) dma(stf, f + 1);
        if (NB == 1 && f + 2 < ND) dma(stf, f + 2);
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
  };
  constexpr int TURNS = NB == 2 ? R : R % 2 ? R : R / 2;
  int b = 0;
#pragma unroll 1
  for (; b + 2 * TURNS <= blocks; b += 2 * TURNS) {
    turn(std::integral_constant<int, 0>());
    turn(std::integral_constant<int, 1>());
    if constexpr (TURNS > 2) turn(std::integral_constant<int, 2>());
  }
  if (b < blocks) {
    turn(std::integral_constant<int, 0>());
    if constexpr (TURNS > 2)
      if (b + 2 < blocks) turn(std::integral_constant<int, 1>());
  }
  static_assert(TURNS == 2 || TURNS == 3, "the turns above");
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  // the last product: tile (1, 1) of the second block
#pragma unroll
  for (int e = 0; e < 16; ++e) res[1][1][e] = __builtin_fmaf(P[1][16 + e], J[1][e], res[1][1][e]);
}

// The same for 32 tokens: an expert's tile of at most 32 slots.  Both row tiles of a block one after the other, the next block's
// operands read before the products.
template <int NW, int MN, class I, class DMA>
__device__ __forceinline__ void d_loop32(const DAddr& o, DMA& dma, int blocks, v16f (&res)[2]) {
  constexpr int NB = I::NB, R = I::R, STAGE = I::STAGE, KB = STAGE / 1024, ND = (KB + 3) / 4;
  const int g = (threadIdx.x & 63) >> 5, steps = blocks / NB;
  struct F6 { u4v lo; u2v hi; };
  F6 A[2], W[2][2][NW];
  float saop[2], wsop[2];
  u2v U, V[2];
  uint32_t st = 0;
  auto load = [&](int k, int blk) {
    const uint32_t t = st + (NB == 2 ? blk : 0) * I::T, w = st + (NB == 2 ? blk : 0) * I::W;
    A[k].lo = *LDS_P(const u4v, o.A16 + t);
    A[k].hi = *LDS_P(const u2v, o.A8 + t);
#pragma unroll
    for (int ns = 0; ns < 2; ++ns)
#pragma unroll
      for (int d = 0; d < NW; ++d) {
        W[k][ns][d].lo = *LDS_P(const u4v, o.W16 + w + d * I::DIG + ns * 512);
        W[k][ns][d].hi = *LDS_P(const u2v, o.W8 + w + d * I::DIG + ns * 256);
      }
    saop[k] = *LDS_P(const float, o.SA + t);
    wsop[k] = *LDS_P(const float, o.WS + w);
    if constexpr (MN)
      if (blk == 0) {
        U = *LDS_P(const u2v, o.U + st);
        V[0] = *LDS_P(const u2v, o.V + st);
        V[1] = *LDS_P(const u2v, o.V + st + 256);
      }
  };
  auto six = [](const F6& f) {
    const i4v a = __builtin_bit_cast(i4v, f.lo);
    const i2v b = __builtin_bit_cast(i2v, f.hi);
    return (i8v){a[0], a[1], a[2], a[3], b[0], b[1], 0, 0};
  };
  const int sca = g ? 134 : 130, scb = 0x008A8682;
#pragma unroll
  for (int e = 0; e < 16; ++e) res[0][e] = res[1][e] = 0.0f;
  d_prologue<I>(dma, steps);
  load(0, 0);
  int step = 0;
#pragma unroll 1
  for (int b = 0; b < blocks; b += 2) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      if constexpr (MN)
        if (k == 0) {
          typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
          const u4v a = {U[0], U[0], U[0], U[1]};
#pragma unroll
          for (int ns = 0; ns < 2; ++ns) {
            const u4v v = {__builtin_amdgcn_perm(V[ns][1], V[ns][1], 0x01000100u), __builtin_amdgcn_perm(V[ns][1], V[ns][1], 0x03020302u), V[ns][0], V[ns][1]};
            res[ns] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf8, a), __builtin_bit_cast(bf8, v), res[ns], 0, 0, 0);
          }
        }
      if (NB == 1 || k == 1) {  // (the step's meeting, as in d_loop)
        __builtin_amdgcn_sched_barrier(0);
        if (I::AHEAD == R) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (the step's last operands: its stage is refilled)
        d_wait_but<KB, I::AHEAD - 2, (I::AHEAD < R)>(dma.wave);
        d_meet();
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t stf = I::AHEAD == R ? st : st == 0 ? (R - 1) * STAGE : st - STAGE;
        st = st + STAGE == R * STAGE ? 0 : st + STAGE;
        dma.at(min(step + I::AHEAD, steps - 1));
        ++step;
        load(1 - k, 0);
#pragma unroll
        for (int i = 0; i < ND; ++i) dma(stf, i);
      } else {
        load(1 - k, 1);
      }
      v16f z, J[2];
      v32f zp;
#pragma unroll
      for (int e = 0; e < 16; ++e) z[e] = 0.0f;
#pragma unroll
      for (int e = 0; e < 32; ++e) zp[e] = 0.0f;
      const v32f P = __builtin_amdgcn_mfma_f32_32x32x1f32(saop[k], wsop[k], zp, 0, 0, 0);
#pragma unroll
      for (int ns = 0; ns < 2; ++ns) {
        J[ns] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(six(A[k]), six(W[k][ns][0]), z, 2, 2, 0, sca, 0, scb);
        if constexpr (NW > 1) J[ns] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(six(A[k]), six(W[k][ns][1]), J[ns], 2, 2, 0, sca, 1, scb);
        if constexpr (NW > 2) J[ns] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(six(A[k]), six(W[k][ns][2]), J[ns], 2, 2, 0, sca, 2, scb);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ns = 0; ns < 2; ++ns)
#pragma unroll
        for (int e = 0; e < 16; ++e) res[ns][e] = __builtin_fmaf(P[16 * ns + e], J[ns][e], res[ns][e]);
      asm volatile("" : "+v"(res[0]), "+v"(res[1]));
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}
