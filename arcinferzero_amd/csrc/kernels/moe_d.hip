// "gemm" module, third file: the expert tiles of the GEMM on digits, 64 slots x 256 rows in four waves of 64 x 64.
//
// An expert's rows are kept as digits with the layer (row_digits_e), the tokens' are written once per pass as records
// (act_records) that a tile's DMA gathers by its slots: a record is a block's 64 bytes
//   x0's first 16 bytes, x1's, the other 8 of both, u | u | sa | 0 (u = sa * S in bf16 pieces, for the min term)
// and lies in LDS as 64 bytes a slot, its four pieces rotated among the slots so that a wave's reads touch every bank.  A tile's
// 256 rows go to the waves in pairs of 32: rows 32 w .. of gate and of up, so that silu(gate) * up meets in a lane; of the down
// projection rows 32 w .. of the tile's first and of its second half.
// Image of a tile and block: per digit [256][16 bytes], [256][8 bytes]; [256] f32 ws; with a minimum [256][8 bytes] v.
#include "digits.h"
#include "tile64.h"

template <int NW, int MN> struct EImg {
  static constexpr int NB = NW == 1 ? 2 : 1, R = NW == 2 ? 4 : 3, AHEAD = R;
  static constexpr int T = 4096, W = NW * 6144 + 1024 + 2048 * MN;
  static constexpr int STAGE = NB * (T + W);
  static constexpr int WWS = NW * 6144, WV = WWS + 1024;
  static constexpr int A_MS = 2048, A8_MS = 2048, S_MS = 2048, U_MS = 2048, DIG = 6144;
  static constexpr int LDS = R * STAGE;
  static_assert(LDS >= 36352 && 2 * LDS <= 160 * 1024, "the epilogues' array; two work-groups a compute unit");
};

// act_records (digit_pack.h): grid (K / 256, ceil(rows / 64)), local 256.
extern "C" __global__ __launch_bounds__(256) void act_records(const signed char* __restrict__ aq, const float* __restrict__ asc,
                                                              const short* __restrict__ absum, int M, int K, int rows,
                                                              uint8_t* __restrict__ rec) {
  act_records_body(aq, asc, absum, M, K, rows, rec, blockIdx.x, blockIdx.y);
}

// row_digits_e__QT: tiles of an expert tensor.  Tile i: rows i * step .. + 127 of raw0 for the waves' first 32 rows, i * step + second ..
// of raw1 for the others (gate and up: 128, 0; down: 256, 128 of the same planes).  grid (K / 256, 4 * tiles), local 256.
template <int QT>
__device__ inline void row_digits_e(const uint8_t* __restrict__ raw0, const uint8_t* __restrict__ raw1, const uint32_t* __restrict__ tabs,
                                    size_t rows_total, int nsb, int step, int second, uint8_t* __restrict__ wt) {
  constexpr int NW = DType<QT>::NW, MN = DType<QT>::MN;
  using I = EImg<NW, MN>;
  const int s = blockIdx.x, pos = (blockIdx.y & 3) * 64 + (threadIdx.x & 63), q = threadIdx.x >> 6, tile = blockIdx.y >> 2;
  const int ns = (pos >> 5) & 1;
  const size_t row = (size_t)tile * step + (ns ? second : 0) + (pos >> 6) * 32 + (pos & 31);
  RowDigits<QT> d;
  row_decode<QT>(ns ? raw1 : raw0, tabs, rows_total, nsb, row * nsb + s, q, d);
  uint8_t* dst = wt + ((size_t)tile * nsb + s) * 8 * I::W;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    uint8_t* img = dst + d.b[i] * I::W;
#pragma unroll
    for (int j = 0; j < NW; ++j) put_digit(img + j * 6144 + pos * 16, img + j * 6144 + 4096 + pos * 8, d.c[i][j]);
    *(float*)(img + I::WWS + pos * 4) = d.ws[i];
    if constexpr (MN) {
      uint32_t w0, w1;
      split3(d.mv[i], w0, w1);
      *(u2v*)(img + I::WV + pos * 8) = (u2v){w1 | w1 << 16, w0};
    }
  }
}
#define ROW_DIGITS_E(QT)                                                                                                \
  extern "C" __global__ __launch_bounds__(256) void row_digits_e__QTYPE##QT(                                            \
      const uint8_t* raw0, const uint8_t* raw1, const uint32_t* tabs, size_t rows_total, int nsb, int step, int second, uint8_t* wt) { \
    row_digits_e<QT>(raw0, raw1, tabs, rows_total, nsb, step, second, wt);                                              \
  }
ROW_DIGITS_E(12) ROW_DIGITS_E(13) ROW_DIGITS_E(14) ROW_DIGITS_E(2) ROW_DIGITS_E(20) ROW_DIGITS_E(23) ROW_DIGITS_E(39) ROW_DIGITS_E(11)
ROW_DIGITS_E(21) ROW_DIGITS_E(18)

// A tile's sums: slot r of it is record map[m0 + r] (or m0 + r), the rows' image wt.  true: at most 32 slots, res[1] is not set.
template <int NW, int MN>
__device__ __forceinline__ bool tile_d_sums(uint8_t* lds_base, const uint8_t* __restrict__ rec, const int* __restrict__ map,
                                            const uint8_t* __restrict__ wt, int nblk, int m0, int rows_valid, v16f (&res)[2][2]) {
  asm volatile("" :: "v"((__attribute__((address_space(3))) uint8_t*)lds_base) : "memory");
  using I = EImg<NW, MN>;
  static constexpr int TS = I::NB * I::T, WS = I::NB * I::W, KB = I::STAGE / 1024;
  const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  struct {
    d_buf t, w;
    uint32_t lane16, toff, to, wo;
    int wave;
    __device__ void at(int step) {
      to = step * I::NB * 64;
      wo = step * WS + wave * 1024 - TS;
    }
    __device__ void operator()(uint32_t stage, int i) {  // (a block's 64 slots are four KiB)
      if (4 * i + 4 > KB && wave >= (KB & 3)) return;
      const uint32_t lds = stage + wave * 1024 + i * 4096;
      if (i < I::NB) dma16(t, toff, to + i * 64, lds);
      else dma16(w, lane16, wo + i * 4096, lds);
    }
  } dma;
  {
    // (the slot's records: 64 bytes a block; a pass's are below 4 GiB, the engine sees to it)
    const int r = 16 * wave + (lane >> 2), rr = r < rows_valid ? r : 0;  // (slots past the tile read its first)
    dma = {d_buffer(rec, 0xFFFFFFFFu), d_buffer(wt, (size_t)nblk * I::W), (uint32_t)lane * 16,
           (uint32_t)(map ? map[m0 + rr] : m0 + rr) * (uint32_t)nblk * 64u + 16u * ((lane & 3) ^ ((r >> 2) & 3)), 0u, 0u, wave};
  }
  const uint32_t sw = (l32 >> 2) & 3, t = l32 * 64u;  // (piece p of slot r at 16 (p ^ r / 4 % 4))
  const DAddr o = {t + ((g ^ sw) << 4), t + ((2 ^ sw) << 4) + g * 8u, t + ((3 ^ sw) << 4) + 8u, g * I::T + t + ((3 ^ sw) << 4),
                   TS + (wave * 64u + l32) * 16u, TS + 4096u + (wave * 64u + l32) * 8u, TS + I::WWS + (wave * 64u + lane) * 4u,
                   TS + I::WV + g * I::W + (wave * 64u + l32) * 8u};
  const bool few = rows_valid <= 32;
  if (few) d_loop32<NW, MN, I>(o, dma, nblk, res[0]);
  else d_loop<NW, MN, I>(o, dma, nblk, res);
  __syncthreads();  // (the stages are the epilogue's)
  return few;
}

// moe_gu_d__NW: h = silu(gate) * up of a tile's slots and 128 rows, its int8 form and the records of that (tile64.h).  moe_down_d__NW: 256 rows of y, times the
// slots' weights.  tiles, stok, swt as the int8 tile kernels take them; grid (row tiles * 256, tile work-groups: a multiple of 8).
#define MOE_D(NAME, ...)                                                                                                \
  extern "C" __global__ __launch_bounds__(256, 2) void moe_gu_d__##NAME(                                                \
      const uint8_t* rec, const uint8_t* wt, int F, int K, const int* tiles, const int* stok, float* h, int S, signed char* hq, \
      float* hsc, short* hbs, uint8_t* hrec) {                                                                          \
    __shared__ __attribute__((aligned(1024))) uint8_t lds[EImg<__VA_ARGS__>::LDS];                                      \
    int ti, chunk;                                                                                                      \
    if (!moe_tile_of(tiles[0], gridDim.x, ti, chunk)) return;                                                           \
    const int e = tiles[1 + 3 * ti], r0 = tiles[2 + 3 * ti], nr = min(tiles[3 + 3 * ti], 64), nblk = K >> 5;            \
    v16f res[2][2], hv[2];                                                                                              \
    const bool few = tile_d_sums<__VA_ARGS__>(                                                                          \
        lds, rec, stok, wt + ((size_t)e * gridDim.x + chunk) * nblk * EImg<__VA_ARGS__>::W, nblk, r0, nr, res);         \
    _Pragma("unroll") for (int ms = 0; ms < 2; ++ms)                                                                    \
      _Pragma("unroll") for (int i = 0; i < 16; ++i) {                                                                  \
        const float gt = ms && few ? 0.0f : few ? res[0][0][i] : res[ms][0][i], up = ms && few ? 0.0f : few ? res[0][1][i] : res[ms][1][i]; \
        hv[ms][i] = up * (gt / (1.0f + __expf(-gt)));                                                                   \
      }                                                                                                                 \
    store_tile64_quant<true>(lds, hv, h, F, r0, nr, chunk * 128, S, hq, hsc, hbs, nullptr, hrec);                       \
  }                                                                                                                     \
  extern "C" __global__ __launch_bounds__(256, 2) void moe_down_d__##NAME(                                              \
      const uint8_t* rec, const uint8_t* wt, int N, int K, const int* tiles, const float* swt, float* y) {              \
    __shared__ __attribute__((aligned(1024))) uint8_t lds[EImg<__VA_ARGS__>::LDS];                                      \
    int ti, chunk;                                                                                                      \
    if (!moe_tile_of(tiles[0], gridDim.x, ti, chunk)) return;                                                           \
    const int e = tiles[1 + 3 * ti], r0 = tiles[2 + 3 * ti], nr = min(tiles[3 + 3 * ti], 64), nblk = K >> 5;            \
    v16f res[2][2];                                                                                                     \
    const bool few = tile_d_sums<__VA_ARGS__>(                                                                          \
        lds, rec, nullptr, wt + ((size_t)e * gridDim.x + chunk) * nblk * EImg<__VA_ARGS__>::W, nblk, r0, nr, res);      \
    _Pragma("unroll") for (int ns = 0; ns < 2; ++ns) {                                                                  \
      v16f v[2];                                                                                                        \
      _Pragma("unroll") for (int i = 0; i < 16; ++i) {                                                                  \
        v[0][i] = res[0][ns][i];                                                                  \
        v[1][i] = few ? 0.0f : res[1][ns][i];                                                                           \
      }                                                                                                                 \
      store_tile64(lds, v, y, N, 0, 0, r0, nr, chunk * 256 + ns * 128, N, swt, 1);                                      \
      __syncthreads();                                                                                                  \
    }                                                                                                                   \
  }
MOE_D(NW1, 1, 0) MOE_D(NW2, 2, 0) MOE_D(NW3, 3, 0) MOE_D(NW1_MN1, 1, 1)
