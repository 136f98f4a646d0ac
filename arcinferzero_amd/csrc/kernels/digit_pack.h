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
