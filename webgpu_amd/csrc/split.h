// split.h — the prompt GEMM's activation format: scaled f16 (hi, lo) pairs in MFMA fragment
// order.
//
// f16 keeps 11 significant bits, so a value is carried as v = s * (hi + lo) with
// hi = RN_f16(v / s) and lo = RN_f16(v / s - hi): about 22 bits together. s is a power of two
// per token and 128 columns that puts their largest magnitude into [2^14, 2^15), so nothing
// overflows. The pair's last place is 2^-24 s, at most 2^-38 of the largest: a value below 2^-24 of it
// keeps fewer than the 16 bits that a bf16 pair kept at any magnitude, and below about 2^-39 becomes zero.
// Beside the largest one's product that is less than f32's rounding; it counts only where that
// column's weight is zero. The activations [batch][cols] are stored as blocks of 16 tokens x 128 columns,
// block (token / 16, k / 128) of SPLIT_BLOCK bytes:
//   [hl][j][g][c][8] f16: token c's columns 32 g + 8 j .. + 8 of the hi (hl = 0) or lo part, in
//     the order 0 2 1 3 4 6 5 7: lane 16 g + c of a v_mfma_f32_16x16x32_f16 takes the 16 bytes
//     at fragment (hl, j) + 16 * lane. The order inside the eight is the one in which a
//     dword of packed quants unpacks into f16 pairs (bytes 0 and 2, then 1 and 3);
//   [g][c] f32: the sum of token c's columns 32 g .. + 32 over s (the min term of the K-quants: over s,
//     because 32 columns of 2^123 or more would overflow, whose products with the weights need not);
//   [c] f32: token c's s.
// Producers that already hold a batch of activations (RMSNorm, the GLU) write this form
// beside their f32 output so the GEMMs that read it need no split pass of their own.
#pragma once
#include "internal.h"

namespace wgd {

constexpr uint32_t SPLIT_N = 16, SPLIT_K = 128;
constexpr uint32_t SPLIT_COLS = 64;  // widths are whole multiples of this
constexpr uint32_t SPLIT_LO = 4096, SPLIT_SUM = 8192, SPLIT_SCALE = SPLIT_SUM + 256;  // byte offsets in a block
constexpr uint32_t SPLIT_BLOCK = SPLIT_SCALE + 64;
constexpr uint32_t SPLIT_TOK = 128;  // tokens whose blocks of one k are adjacent
// Byte offset of the block of tokens 16 b .. + 16 and columns 128 kb .. + 128, of kbs blocks of columns.
__host__ __device__ constexpr uint64_t split_block_at(uint32_t b, uint32_t kb, uint32_t kbs) {
  constexpr uint32_t per = SPLIT_TOK / SPLIT_N;
  return (((uint64_t)(b / per) * kbs + kb) * per + b % per) * SPLIT_BLOCK;
}
__host__ __device__ constexpr uint32_t split_kblocks(uint32_t cols) { return (cols + SPLIT_K - 1) / SPLIT_K; }

#ifdef __HIPCC__
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

// The gate activations of the GLU: SiLU (act 0) and tanh-approximated GELU (act 1).
__device__ __forceinline__ float glu_act(float x, int act) {
  if (!act) return x / (1.f + expf(-x));
  return 0.5f * x * (1.f + tanhf(0.7978845608f * (x + 0.044715f * x * x * x)));
}

// The value of another lane of this lane's row of 16 (this lane's own where that lane is off).
template <int CTRL> __device__ __forceinline__ uint32_t row_other(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, 0xf, 0xf, false);
}

// Two scaled floats -> (hi, lo) f16 pairs.
__device__ __forceinline__ void split2(float a, float b, uint32_t &hi, uint32_t &lo) {
  const f32x2 v = {a, b};
  const f16x2 h = __builtin_convertvector(v, f16x2);
  hi = __builtin_bit_cast(uint32_t, h);
  lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(v - __builtin_convertvector(h, f32x2), f16x2));
}

// Columns k..k+7 (k % 8 == 0) of token tok. The 16 lanes of a row together hold 128 columns:
// lane % 16 == (k / 8) % 16, with the lanes of columns past `cols` (a multiple of 64) off. The
// largest magnitude goes over those lanes as exponent bits. An infinity's lo part is NaN (inf - inf), so its
// token's products are NaN; a NaN stays one.
__device__ __forceinline__ void split_store8(uint8_t *xs, uint32_t cols, uint32_t tok, uint32_t k, float4 a, float4 b) {
  uint32_t m = 0;
  const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
  for (int e = 0; e < 8; e++) m = max(m, __float_as_uint(v[e]) & 0x7FFFFFFFu);
  m = max(m, row_other<0xB1>(m));   // quad_perm [1,0,3,2]
  m = max(m, row_other<0x4E>(m));   // quad_perm [2,3,0,1]
  m = max(m, row_other<0x141>(m));  // row_half_mirror
  m = max(m, row_other<0x140>(m));  // row_mirror
  // s = 2^(E - 127 - 14) for the biased exponent E, bounded so that s and 1 / s are normal
  const uint32_t E = min(max(m >> 23, 16u), 254u);
  const float s = __uint_as_float((E - 14u) << 23), inv = __uint_as_float((254u + 14u - E) << 23);
  a.x *= inv; a.y *= inv; a.z *= inv; a.w *= inv;
  b.x *= inv; b.y *= inv; b.z *= inv; b.w *= inv;
  float sum = ((a.x + a.y) + (a.z + a.w)) + ((b.x + b.y) + (b.z + b.w));
  sum += __uint_as_float(row_other<0xB1>(__float_as_uint(sum)));
  sum += __uint_as_float(row_other<0x4E>(__float_as_uint(sum)));
  uint32_t h[4], l[4];
  split2(a.x, a.z, h[0], l[0]);
  split2(a.y, a.w, h[1], l[1]);
  split2(b.x, b.z, h[2], l[2]);
  split2(b.y, b.w, h[3], l[3]);
  const uint32_t c = tok % SPLIT_N, kk = k % SPLIT_K, g = kk / 32, j = (kk % 32) / 8;
  uint8_t *t = xs + split_block_at(tok / SPLIT_N, k / SPLIT_K, split_kblocks(cols));
  uint8_t *f = t + ((j * 4 + g) * 16 + c) * 16;
  *(uint4 *)f = make_uint4(h[0], h[1], h[2], h[3]);
  *(uint4 *)(f + SPLIT_LO) = make_uint4(l[0], l[1], l[2], l[3]);
  if (j == 0) *(float *)(t + SPLIT_SUM + (g * 16 + c) * 4) = sum;
  if (kk == 0) *(float *)(t + SPLIT_SCALE + c * 4) = s;
}
#endif

}  // namespace wgd
