// int8 values as FP6 digits: the codes and their packing (digits.h has what they are for).
#pragma once
#include "common.h"

typedef uint32_t u4v __attribute__((ext_vector_type(4)));
typedef uint32_t u2v __attribute__((ext_vector_type(2)));

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
// four int8 values: sign bits at bit 0 of each byte, magnitudes
__device__ inline void sign_mag(uint32_t v, uint32_t& s, uint32_t& a) {
  s = (v >> 7) & 0x01010101u;
  a = (v ^ ((s << 8) - s)) + s;
}
// ... and the codes of their two digits
__device__ inline void digits_i8(uint32_t v, uint32_t& lo, uint32_t& hi) {
  uint32_t sg, a;
  sign_mag(v, sg, a);
  lo = (a & 0x0F0F0F0Fu) | sg << 5;
  hi = ((a >> 4) & 0x0F0F0F0Fu) | sg << 5;
}

// Tokens as records of digits (moe_d.hip): aq [M][K], asc [K/32][M], absum [K/16][M] -> rec [rows][K/32][64 bytes].  64 rows x a superblock a work-group, the
// eight lanes of a row next to each other (its 256 values in, its 512 bytes out; a row a lane, 16 bytes each of 64 lines, took
// 20 us for 4096 x 2048, now 9); the scales and sums, a row of which is a block's, come through LDS.
// A work-group of 256: superblock s, rows 64 y ..
__device__ __forceinline__ void act_records_body(const signed char* __restrict__ aq, const float* __restrict__ asc, const short* __restrict__ absum, int M,
                                                 int K, int rows, uint8_t* __restrict__ rec, int s, int y) {
  __shared__ float lsa[8][65];
  __shared__ int ls[8][65];
  const int m0 = y * 64, t = threadIdx.x;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int b = (t >> 6) + 4 * i, r = t & 63, m = m0 + r;
    if (m >= rows) continue;
    const size_t at = (size_t)(s * 8 + b);
    lsa[b][r] = asc[at * M + m];
    ls[b][r] = (int)absum[2 * at * M + m] + (int)absum[(2 * at + 1) * M + m];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int b = t & 7, r = (t >> 3) + 32 * i, m = m0 + r;
    if (m >= rows) continue;
    const u4v* src = (const u4v*)(aq + (size_t)m * K + s * 256 + b * 32);
    const u4v x[2] = {src[0], src[1]};
    uint32_t c[2][8], o[2][6], w0, w1;
#pragma unroll
    for (int k = 0; k < 8; ++k) digits_i8(x[k >> 2][k & 3], c[0][k], c[1][k]);
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      pack16(c[d], o[d]);
      pack16(c[d] + 4, o[d] + 3);
    }
    const float sa = lsa[b][r];
    split3(sa * (float)ls[b][r], w0, w1);
    u4v* to = (u4v*)(rec + ((size_t)m * (K >> 5) + s * 8 + b) * 64);
    to[0] = (u4v){o[0][0], o[0][1], o[0][2], o[0][3]};
    to[1] = (u4v){o[1][0], o[1][1], o[1][2], o[1][3]};
    to[2] = (u4v){o[0][4], o[0][5], o[1][4], o[1][5]};
    to[3] = (u4v){w0, w1 | w1 << 16, __float_as_uint(sa), 0u};
  }
}
