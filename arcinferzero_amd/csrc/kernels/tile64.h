// What the kernels over expert tiles of 64 slots share: which tile a work-group takes, and the epilogues of a wave that holds
// all 64 slots of 32 rows.
#pragma once
#include "common.h"
#include "digit_pack.h"
#include "quant.h"

// The (tile, row chunk) a work-group of a tile kernel takes, nc row chunks a tile, grid (nc, tile work-groups) with the
// tile work-groups at least the tiles there are, and a multiple of 8.  The XCDs take work-groups in turn (linear id % 8) and each has its own L2, so the
// tile list, which is sorted by expert, is cut into 8 runs, one per XCD, and the work-groups of an XCD walk their run
// in groups of 4 tiles, row chunk by row chunk: four neighbours read the same rows of an expert (mostly: an expert of
// 256 slots has 4 or 5 tiles), and the 4 nc work-groups of a group the same slots' activations, out of one L2.  Every
// tile and chunk is taken exactly once; work-groups beyond their XCD's run do nothing (false).
__device__ inline bool moe_tile_of(int nt, int nc, int& ti, int& chunk) {
  if (gridDim.y & 7) {  // (a launch of another shape: work-group (x, y) takes chunk x of tile y)
    ti = blockIdx.y;
    chunk = blockIdx.x;
    return ti < nt;
  }
  const int id = blockIdx.x + gridDim.x * blockIdx.y, x = id & 7, j = id >> 3;
  const int t0 = (int)(((long long)nt * x) >> 3), t1 = (int)(((long long)nt * (x + 1)) >> 3);  // this XCD's tiles
  if (j >= (t1 - t0) * nc) return false;
  const int grp = j / (4 * nc), first = t0 + 4 * grp, in_grp = min(4, t1 - first);  // (the run's last group may be short)
  const int r = j - grp * 4 * nc;
  chunk = r / in_grp;
  ti = first + r - chunk * in_grp;
  return true;
}

// Epilogue of the 64-slot bodies (a wave holds all 64 slots of its 32 weight rows: lane = row, accumulator i of tile ms
// = slot 32 ms + 8 (i / 4) + 4 g + i % 4) for a whole tile of 128 rows whose output rows are 16-byte aligned: the sums
// go through LDS (the stages are free: every wave is past the last step's barrier), slot r at 528 r bytes behind the
// slots' scales -- 16 bytes of padding keep the two lane halves, four slots apart, on different banks -- so that a
// thread writes 16 bytes and a wave two whole 512-byte rows of the tile: 8 store instructions a lane instead of 32,
// each over half as many lines.  What the accumulate modes read of C is loaded for all 8 before the first store, and
// the slots' scales come from LDS: loads between the stores would each wait for the stores before them (one counter
// orders both), 32 round trips to memory in a row.  false: not such a tile, nothing done (the caller's scalar path).
__device__ __forceinline__ bool store_tile64(uint8_t* lds, const v16f (&res)[2], float* __restrict__ C, int ldc, int c_off,
                                             int accumulate, int m0, int rows_valid, int n0, int N,
                                             const float* __restrict__ rowscale, int use_scale) {
  if (n0 + 128 > N || ((ldc | c_off) & 3) != 0 || ((uintptr_t)C & 15) != 0) return false;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), l32 = lane & 31, g = lane >> 5;
  float* rs = (float*)lds;
  uint8_t* tl = lds + 256;
  if (use_scale && t < 64) rs[t] = t < rows_valid ? rowscale[m0 + t] : 0.0f;
#pragma unroll
  for (int ms = 0; ms < 2; ++ms)
#pragma unroll
    for (int i = 0; i < 16; ++i)
      *(float*)(tl + (ms * 32 + 8 * (i >> 2) + 4 * g + (i & 3)) * 528 + (wave * 32 + l32) * 4) = res[ms][i];
  const int c4 = t & 31, rr = t >> 5;
  float* cp = C + (size_t)(m0 + rr) * ldc + c_off + n0 + 4 * c4;
  float4 cv[8];
  if (accumulate != 0) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      cv[i] = rr + 8 * i < rows_valid ? *(const float4*)(cp + (size_t)8 * i * ldc) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int r = rr + 8 * i;
    if (r >= rows_valid) continue;
    float4 v = *(const float4*)(tl + r * 528 + c4 * 16);
    if (use_scale) {
      const float sc = rs[r];
      v.x *= sc; v.y *= sc; v.z *= sc; v.w *= sc;
    }
    if (accumulate == 1) {
      v.x += cv[i].x; v.y += cv[i].y; v.z += cv[i].z; v.w += cv[i].w;
    } else if (accumulate == 2) {  // fused SwiGLU: C holds the gate projection, v the up projection
      v.x *= cv[i].x / (1.0f + __expf(-cv[i].x));
      v.y *= cv[i].y / (1.0f + __expf(-cv[i].y));
      v.z *= cv[i].z / (1.0f + __expf(-cv[i].z));
      v.w *= cv[i].w / (1.0f + __expf(-cv[i].w));
    }
    *(float4*)(cp + (size_t)8 * i * ldc) = v;
  }
  return true;
}

// The gate/up tile's h = silu(gate) * up, stored as store_tile64 stores it, and quantized on the way out as the expert
// inputs' quantizer does (moe_quant_sums in moe.hip: per 32 values amax, q = rte(v * (127 / amax)), scale amax / 127,
// the sums of 16 -- the same helper, the same bits): the tile lies in LDS slot-major for the stores, a thread takes
// two half blocks of 16 values (neighbouring lanes the two halves of a block), writes their int8 values, and the
// scales and sums leave through LDS in rows of 64 slots.  hq [S][F], hsc [F/32][S], hbs [F/16][S].  Whole tiles of 128
// rows only (F a multiple of 128).  REC: also as the records [S][F/32][64 bytes] that the down projection's tiles on digits gather
// (moe_d.hip); the two threads of a block put its four pieces together.
template <bool REC = false>
__device__ __forceinline__ void store_tile64_quant(uint8_t* lds, const v16f (&hv)[2], float* __restrict__ H, int F, int m0,
                                                   int rows_valid, int n0, int S, signed char* __restrict__ hq,
                                                   float* __restrict__ hsc, short* __restrict__ hbs,
                                                   float* __restrict__ hu = nullptr, uint8_t* __restrict__ rec = nullptr) {
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), l32 = lane & 31, g = lane >> 5;
  uint8_t* tl = lds + 256;
  float* lasc = (float*)(lds + 256 + 64 * 528);       // [4][64]
  short* lsum = (short*)(lds + 256 + 64 * 528 + 1024);  // [8][64]
#pragma unroll
  for (int ms = 0; ms < 2; ++ms)
#pragma unroll
    for (int i = 0; i < 16; ++i)
      *(float*)(tl + (ms * 32 + 8 * (i >> 2) + 4 * g + (i & 3)) * 528 + (wave * 32 + l32) * 4) = hv[ms][i];
  __syncthreads();
  const int c4 = t & 31, rr = t >> 5;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int r = rr + 8 * i;
    if (r < rows_valid) *(float4*)(H + (size_t)(m0 + r) * F + n0 + 4 * c4) = *(const float4*)(tl + r * 528 + c4 * 16);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int idx = t + 256 * i, hb = idx & 7, r = idx >> 3;
    float v[16];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4 f = *(const float4*)(tl + r * 528 + hb * 64 + q * 16);
      v[4 * q] = f.x; v[4 * q + 1] = f.y; v[4 * q + 2] = f.z; v[4 * q + 3] = f.w;
    }
    const float amax = block_amax(v, 1);
    uint4 pk;
    int sum;
    quant16(v, amax, pk, sum);
    if (r < rows_valid) *(uint4*)(hq + (size_t)(m0 + r) * F + n0 + hb * 16) = pk;
    if ((hb & 1) == 0) lasc[(hb >> 1) * 64 + r] = amax / 127.0f;
    lsum[hb * 64 + r] = (short)sum;
    if constexpr (REC) {
      const uint32_t w[4] = {pk.x, pk.y, pk.z, pk.w};
      uint32_t c[2][4], o[2][3], w0, w1;
#pragma unroll
      for (int q = 0; q < 4; ++q) digits_i8(w[q], c[0][q], c[1][q]);
      pack16(c[0], o[0]);
      pack16(c[1], o[1]);
      const uint32_t p0 = __shfl_xor(o[0][0], 1, 64), p1 = __shfl_xor(o[1][0], 1, 64);
      const float sc = amax / 127.0f;
      split3(sc * (float)(sum + __shfl_xor(sum, 1, 64)), w0, w1);
      u4v* to = (u4v*)(rec + ((size_t)(m0 + r) * (F >> 5) + (n0 >> 5) + (hb >> 1)) * 64 + (hb & 1) * 32);
      if (r < rows_valid) {
        to[0] = hb & 1 ? (u4v){o[0][1], o[0][2], o[1][1], o[1][2]} : (u4v){o[0][0], o[0][1], o[0][2], p0};
        to[1] = hb & 1 ? (u4v){w0, w1 | w1 << 16, __float_as_uint(sc), 0u} : (u4v){o[1][0], o[1][1], o[1][2], p1};
      }
    }
  }
  __syncthreads();
  {
    const int b = t >> 6, r = t & 63;
    if (r < rows_valid) hsc[((size_t)(n0 >> 5) + b) * S + m0 + r] = lasc[b * 64 + r];
    // (hu [F/32][S]: scale times the block's sum, what act_usum would make of hsc and hbs, for the down kernel's PRE form)
    if (hu && r < rows_valid)
      hu[((size_t)(n0 >> 5) + b) * S + m0 + r] = lasc[b * 64 + r] * (float)((int)lsum[2 * b * 64 + r] + (int)lsum[(2 * b + 1) * 64 + r]);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int hb = b + 4 * i;
      if (r < rows_valid) hbs[((size_t)(n0 >> 4) + hb) * S + m0 + r] = lsum[hb * 64 + r];
    }
  }
}
