// "gemm" module, second file: the prefill GEMM on digits, every weight type but Q8_0 (whose int8 kernels
// decode nothing: 4096 x 4096, 300 and 2048 tokens, 28 and 105 us, in two digits 36 and 108).
//
//   C[m][c_off + n] (=, +=, silu(C) *)  sum over 32-blocks b of  (sa[m][b] * ws[n][b]) * J[m][n][b]
//   J[m][n][b] = sum over the block's 32 k of x[m][k] * w[n][k], integers
//
// A kernel on packed weights unpacks them again for every tile of tokens, and the int8 matrix instruction leaves J as
// int32, 16 conversions a lane.  Here both sides come as digits of four bits and a sign, written by two small kernels, the
// tokens' once per matmul, the rows' when the weight is uploaded (or per matmul, where they are not kept): x = 16 x1 + x0 and w = 256 w2 + 16 w1 + w0 (one to three digits, by the type's range).  A digit
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
// Bound by the matrix and the vector unit, which run beside each other only in part.  At 17408 x 5120 x 8192 a 32 x 32 x 32
// block-tile takes a SIMD 131, 162, 207 cycles with one, two, three digits and 148 with one and a minimum, at 2.0, 1.8, 1.8
// and 1.9 GHz, which is what the power limit leaves; the matrix unit is busy 64, 96, 128, 80 of them, vector instructions are
// 76, 84, 93, 83, and waves wait 45 - 50 % of their cycles.  The loop's arithmetic alone, out of registers, takes 120 of the 148
// at 2.3 GHz (product 33, scale tile 32, multiply-adds 50, min term 17: the f32 scale tile adds to the multiply-adds in full);
// the rest are operand reads from LDS, DMA and the meeting.  Hence few bytes and few instructions per product: a wave's operands
// serve 64 x 64 outputs, the addresses of a step are six registers and immediate offsets, its pieces' are scalars.  (Before the
// latter, with the stage in registers: 151, 185, 233, 170 cycles at 2.2, 1.9, 1.9, 2.0 GHz.)  Kernel alone, 17408 x 5120 x 8192:
// one digit 1014 TOP/s, two 751, three 578, one and a minimum 859 (the int8 kernels on packed weights: Q4_0 and Q3_K at 12288 x
// 4096 x 4096 650 and 375).
// Q4_K and Q5_K with the min term, 17408 x 5120, us, int8 kernels and this: 8192 tokens Q4_K 2020 / 1700, 2048 544 / 470, Q5_K
// 593 / 472, 300 115 / 93, 143 / 93 (weights from memory, 64-token tiles).
// Matmul with both writing kernels, us, before and now, 12288 x 4096 x 1024: Q4_0 173 / 136, MXFP4 183 / 135, IQ3_S
// 201 / 147, Q3_K 293 / 182, Q6_K 277 / 234; x 4096: Q6_K 1094 / 790, IQ3_XXS 742 / 596.
#include "digits.h"

// ---- images, what a work-group's DMA brings as it lies: 128 tokens x one block
//   [4 groups of 32][2 digits][32][16 bytes] the block's first 128 bits, [4][2][32][8 bytes] the other 64, [128] f32 sa
// and 128 weight rows x one block
//   per digit [128][16 bytes], [128][8 bytes]; then [128] f32 ws
// A tile's blocks follow each other.  NB: blocks a step of the GEMM takes; steps are whole KiB.
// Types with a minimum (MN: Q4_K, Q5_K) have behind sa [128][8 bytes] u = sa * S, and behind ws v, of the min term: bf16 pieces
// u1 | u2 << 16, u3 | u3 << 16 and v3 | v3 << 16, v1 | v2 << 16 (so that both lie as the products take them).
template <int NW, int MN = 0> struct DImg {
  static constexpr int NB = NW == 3 ? 1 : 2;
  static constexpr int R = NB == 2 ? 3 : 4, AHEAD = R;  // stages in LDS, steps on their way
  static constexpr int T = MN ? 7680 : NB == 2 ? 6656 : 7168, W = NB == 2 ? NW * 3072 + 512 + 1024 * MN : 10240;
  static constexpr int STAGE = NB * (T + W);
  static constexpr int TSA = 6144, TU = 6656, WWS = NW * 3072, WV = WWS + 512;
  static constexpr int A_MS = 1024, A8_MS = 512, S_MS = 128, U_MS = 256, DIG = 3072;
};

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
    for (int k = 0; k < 8; ++k) digits_i8(x[2 * i + (k >> 2)][k & 3], lo[k], hi[k]);
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
  RowDigits<QT> d;
  row_decode<QT>(raw, tabs, (size_t)N, nsb, u, q, d);
  uint8_t* dst = wt + ((size_t)(blockIdx.y >> 1) * nsb + s) * 8 * I::W;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    uint8_t* img = dst + d.b[i] * I::W;
#pragma unroll
    for (int j = 0; j < NW; ++j) {
      if (!in)
#pragma unroll
        for (int k = 0; k < 8; ++k) d.c[i][j][k] = 0;
      put_digit(img + j * 3072 + r * 16, img + j * 3072 + 2048 + r * 8, d.c[i][j]);
    }
    *(float*)(img + I::WWS + r * 4) = in ? d.ws[i] : 0.0f;
    if constexpr (MN) {
      uint32_t w0, w1;
      split3(in ? d.mv[i] : 0.0f, w0, w1);
      *(u2v*)(img + I::WV + r * 8) = (u2v){w1 | w1 << 16, w0};
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
// (Eight waves of 32 x 64, four a SIMD, hide more waits and read each row digit from LDS twice as often: 5 - 6 % slower, before
// the rows' digits were kept, at 17408 x 5120 x 8192 812 against 863 TOP/s with one digit, 632 / 651 with two, 476 / 504 with
// three.)
template <int NW, int MN>
__device__ __forceinline__ void gemm_d_body(uint8_t* lds_base, const uint8_t* __restrict__ xt, const uint8_t* __restrict__ wt,
                                            float* __restrict__ C, int M, int N, int ldc, int c_off, int accumulate, int m0,
                                            int n0, int nblk, int b0, int b1) {
  // (every access below is by offset; the array itself has to stay)
  asm volatile("" :: "v"((__attribute__((address_space(3))) uint8_t*)lds_base) : "memory");
  using I = DImg<NW, MN>;
  static constexpr int TS = I::NB * I::T, WS = I::NB * I::W, TKB = TS / 1024, KB = I::STAGE / 1024;
  const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave & 1, wn = wave >> 1;
  struct {
    d_buf t, w;
    uint32_t lane16, to, wo;
    int wave;
    __device__ void at(int step) {
      to = step * TS + wave * 1024;
      wo = step * WS + wave * 1024 - TS;
    }
    __device__ void operator()(uint32_t stage, int i) {  // (tokens, then rows)
      if (4 * i + 4 > KB && wave >= (KB & 3)) return;
      const uint32_t lds = stage + wave * 1024 + i * 4096;
      if (4 * i + 4 <= TKB || (4 * i < TKB && wave + 4 * i < TKB)) dma16(t, lane16, to + i * 4096, lds);
      else dma16(w, lane16, wo + i * 4096, lds);
    }
  } dma = {d_buffer(xt + ((size_t)(m0 >> 7) * nblk + b0) * I::T, (size_t)(b1 - b0) * I::T),
           d_buffer(wt + ((size_t)(n0 >> 7) * nblk + b0) * I::W, (size_t)(b1 - b0) * I::W), (uint32_t)lane * 16, 0u, 0u, wave};
  const DAddr o = {wm * 2048u + lane * 16u, 4096u + wm * 1024u + lane * 8u, I::TSA + (wm * 64u + l32) * 4u, I::TU + g * I::T + (wm * 64u + l32) * 8u,
                   TS + (wn * 64u + l32) * 16u, TS + 2048u + (wn * 64u + l32) * 8u, TS + I::WWS + (wn * 64u + lane) * 4u,
                   TS + I::WV + g * I::W + (wn * 64u + l32) * 8u};
  v16f res[2][2];
  d_loop<NW, MN, I>(o, dma, b1 - b0, res);

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

// ---- gemm_d64: 64 tokens x 256 rows, the same loop and the same images: half a token tile's, two row tiles'.  Where its tiles are
// fewer: 300 tokens are five token tiles of 64 instead of three of 128, with 17408 rows 340 tiles of the same work instead of
// 408 (Q4_K, K = 5120, 101 -> 95 us).  A tile of at most 32 tokens takes the loop for those.
template <int NW, int MN> struct HImg {
  using D = DImg<NW, MN>;
  static constexpr int NB = NW == 1 ? 2 : 1, R = NW == 2 ? 4 : 3, AHEAD = R - 1;  // (AHEAD = R: slower, digits.h)
  static constexpr int T = 4096, W = D::W, STAGE = NB * (T + 2 * W);  // (a block's tokens: 2 KiB, 1 KiB; sa, u)
  static constexpr int A_MS = 1024, A8_MS = 512, S_MS = 128, U_MS = 256, DIG = 3072;
};
template <int NW, int MN>
__device__ __forceinline__ void gemm_d64_body(uint8_t* lds_base, const uint8_t* __restrict__ xt, const uint8_t* __restrict__ wt,
                                              float* __restrict__ C, int M, int N, int ldc, int c_off, int accumulate, int m0,
                                              int n0, int valid, int nblk, int b0, int b1) {
  asm volatile("" :: "v"((__attribute__((address_space(3))) uint8_t*)lds_base) : "memory");
  using I = HImg<NW, MN>;
  using D = DImg<NW, MN>;
  static constexpr int TS = I::NB * I::T, WS = I::NB * I::W, KB = I::STAGE / 1024;
  const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = (m0 >> 6) & 1;
  struct {
    d_buf t, w;
    uint32_t toff, lane16, split, gap, to, wo;  // (gap: from a step's end in the first row tile's image to its start in the second's)
    int wave;
    __device__ void at(int step) {
      to = step * I::NB * D::T;
      wo = step * WS + wave * 1024;
    }
    __device__ void operator()(uint32_t stage, int i) {
      if (4 * i + 4 > KB && wave >= (KB & 3)) return;
      const uint32_t lds = stage + wave * 1024 + i * 4096;
      if (i < I::NB) {
        dma16(t, toff, to + i * D::T, lds);
      } else {
        const int j = wave + 4 * (i - I::NB);  // (KiB j of the rows' part; the one that holds both tiles': its lanes differ)
        dma16(w, WS % 1024 != 0 && i - I::NB == WS / 4096 ? split : lane16, wo + (i - I::NB) * 4096 + (j * 1024 >= WS ? gap : 0), lds);
      }
    }
  } dma = {d_buffer(xt + ((size_t)(m0 >> 7) * nblk + b0) * D::T, (size_t)(b1 - b0) * D::T),
           d_buffer(wt + ((size_t)(n0 >> 7) * nblk + b0) * D::W, (size_t)(nblk + b1 - b0) * D::W),
           // a wave's KiB of a block's tokens: both groups of 32's first 16 bytes, their other 8, sa and u
           wave < 2 ? half * 2048 + wave * 1024 + lane * 16u : wave == 2 ? 4096 + half * 1024 + lane * 16u
           : MN && lane >= 16 && lane < 48 ? D::TU + half * 512 + (lane - 16) * 16u : D::TSA + half * 256 + (lane & 15) * 16u,
           (uint32_t)lane * 16, 0u, (uint32_t)(nblk * D::W - WS), 0u, 0u, wave};
  // (NW = 2: KiB WS / 1024, a wave's, is the first tile's up to byte WS)
  dma.split = lane * 16u + (wave == (WS / 1024 & 3) && WS / 1024 * 1024 + lane * 16 >= WS ? dma.gap : 0u);
  const uint32_t row = TS + (wave >> 1) * WS, r = (wave & 1) * 64;
  const DAddr o = {lane * 16u, 2048u + lane * 8u, 3072u + l32 * 4u, 3328u + g * I::T + l32 * 8u, row + (r + l32) * 16u, row + 2048u + (r + l32) * 8u,
                   row + D::WWS + (r + lane) * 4u, row + D::WV + g * I::W + (r + l32) * 8u};
  v16f res[2][2];
  if (valid - m0 <= 32) {
    d_loop32<NW, MN, I>(o, dma, b1 - b0, res[0]);
#pragma unroll
    for (int i = 0; i < 16; ++i) res[1][0][i] = res[1][1][i] = 0.0f;
  } else {
    d_loop<NW, MN, I>(o, dma, b1 - b0, res);
  }
#pragma unroll
  for (int ms = 0; ms < 2; ++ms)
#pragma unroll
    for (int ns = 0; ns < 2; ++ns) {
      const int n = n0 + wave * 64 + ns * 32 + l32, m = m0 + ms * 32 + 4 * g;
      if (n >= N || m >= M) continue;
      store16<true>(res[ms][ns], C + (size_t)m * ldc + c_off + n, ldc, M - m, accumulate, [](float v, int) { return v; });
    }
}
// The padding rows [m, M) of 256 columns: products of zeros
__device__ inline void d_zero_rows(float* C, int m, int M, int N, int ldc, int c_off, int accumulate, int n0) {
  const int n = n0 + threadIdx.x;
  if (accumulate == 1 || n >= N) return;
  for (; m < M; ++m) C[(size_t)m * ldc + c_off + n] = 0.0f;
}
// gemm_d64__NW: arguments as gemm_d's, and the rows that are not padding; token tiles that hold padding alone are left out, the last
// one's work-groups write their zeros.
#define GEMM_D64(NAME, ...)                                                                                             \
  extern "C" __global__ __launch_bounds__(256, 2) void gemm_d64__##NAME(                                                \
      const uint8_t* xt, const uint8_t* wt, float* C, int M, int N, int K, int ldc, int c_off, int accumulate, int valid, \
      int whole, int pieces, float* ws) {                                                                               \
    using I = HImg<__VA_ARGS__>;                                                                                        \
    __shared__ __attribute__((aligned(1024))) uint8_t lds[I::R * I::STAGE];                                             \
    const int mt = (valid + 63) / 64, nt = (N + 255) / 256, tail = mt * nt - whole, nsb = K >> 8;                       \
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
    const int m0 = tm * 64, r0 = tn * 256;                                                                              \
    if (ny == 1 && tm == mt - 1) d_zero_rows(C, mt * 64, M, N, ldc, c_off, accumulate, r0);                             \
    if (ny > 1) {                                                                                                       \
      C = ws + (ptrdiff_t)((L - whole) * ny + y) * 16384 - (ptrdiff_t)(m0 * 256 + r0);                                  \
      ldc = 256;                                                                                                        \
      c_off = accumulate = 0;                                                                                           \
    }                                                                                                                   \
    gemm_d64_body<__VA_ARGS__>(lds, xt, wt, C, M, N, ldc, c_off, accumulate, m0, r0, valid, K >> 5, nsb * y / ny * 8,   \
                               nsb * (y + 1) / ny * 8);                                                                 \
  }
GEMM_D64(NW1, 1, 0) GEMM_D64(NW2, 2, 0) GEMM_D64(NW3, 3, 0) GEMM_D64(NW1_MN1, 1, 1)

// d_reduce: the pieces' sums of the tiles from `whole` on, added in their order, out to C.  wide: rows of whole vectors.  th: a
// tile's token rows, 128 or 64 (of `valid` rows, padding rows as gemm_d64 writes them).  grid (tiles, 16), local 256: a sixteenth of a
// tile; eight planes are loaded before the first is added.
extern "C" __global__ __launch_bounds__(256) void d_reduce(const float* __restrict__ ws, float* __restrict__ C, int M, int N, int ldc,
                                                           int c_off, int accumulate, int wide, int n0, int nt, int whole,
                                                           int pieces, int th, int valid) {
  const int cols = 16384 / th, vecs = cols >> 2, mt = th == 64 ? (valid + 63) / 64 : (M + 127) / 128;
  int tm, tn;
  d_tile_of(whole + blockIdx.x, mt, nt, tm, tn);
  const int nb = n0 + tn * cols;
  if (th == 64 && blockIdx.y == 0 && tm == mt - 1) d_zero_rows(C, mt * 64, M, N, ldc, c_off, accumulate, nb);
  const int r = blockIdx.y * (th >> 4) + (threadIdx.x / vecs), m = tm * th + r, c = threadIdx.x & (vecs - 1);
  if (m >= M) return;
  // (a thread: four columns next to each other, or, where a row's vectors would not be whole, a quarter of the row apart)
  const float* p = ws + (size_t)blockIdx.x * pieces * 16384 + r * cols;
  v4f s = {0.0f, 0.0f, 0.0f, 0.0f};
  auto plane = [&](int y) {
    const float* q = p + (size_t)y * 16384;
    return wide ? *(const v4f*)(q + 4 * c) : (v4f){q[c], q[c + vecs], q[c + 2 * vecs], q[c + 3 * vecs]};
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
    const int n = c + vecs * i;
    if (nb + n < N) cr[n] = out(s[i], accumulate ? cr[n] : 0.0f);
  }
}
