// gemm.hip — prompt-batch dequant-GEMM on the matrix cores (gfx950).
//
// The batched form of matmulShader (src/core/shaders.ts:39-54, dispatched with
// batch = prompt chunk by engine.ts:130): y[b*stride + rowBase + r] = sum_c W[r][c] x[b+off][c].
// It is a real dense contraction, so it runs on MFMA. 16-bit operands alone would break the
// 1e-3 logits bound, so operands are split into (hi, lo) pairs.
//
// k_gemm (GGUF-layout weights, F16, F32) splits both sides into bf16 pairs, hi = RN_bf16(v),
// lo = RN_bf16(v - hi), and sums hi*hi + hi*lo + lo*hi in f32 (relative error ~2^-16). A
// workgroup (4 wavefronts) owns 64 rows x 64 tokens; each wavefront owns 16 rows x 64
// tokens = four 16x16 accumulator tiles; K advances 32 per MFMA step and 64 per LDS tile.
// k_gemm_q (planar weights) is described at its definition below.
#include "internal.h"
#include "decode.h"
#include "split.h"

namespace wgd {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Round-to-nearest-even f32 -> bf16 bits (finite inputs).
__device__ __forceinline__ uint32_t bf16_rne(float v) {
  uint32_t b = __float_as_uint(v);
  return (b + 0x7FFFu + ((b >> 16) & 1u)) >> 16;
}
__device__ __forceinline__ void split8(const float *v, uint4 &hi, uint4 &lo) {
  uint32_t h[8], l[8];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    h[i] = bf16_rne(v[i]);
    l[i] = bf16_rne(v[i] - __uint_as_float(h[i] << 16));
  }
  hi = make_uint4(h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16), h[6] | (h[7] << 16));
  lo = make_uint4(l[0] | (l[1] << 16), l[2] | (l[3] << 16), l[4] | (l[5] << 16), l[6] | (l[7] << 16));
}

struct GemmArgs {
  const uint8_t *w; int type, layout;
  uint64_t rb, nbt; uint32_t bpr;
  const float *x; float *y;
  uint32_t cols, rows, stride, row_base, input_offset, batch;
};

// Eight consecutive weights w[row][k .. k+8) (k % 8 == 0) as f32.
__device__ __forceinline__ void load_a8(const GemmArgs &a, uint32_t row, uint32_t k, float *o) {
  if (a.type == Q4_K && a.layout == LAYOUT_GGUF) {
    const uint8_t *blk = a.w + (uint64_t)row * a.rb + (uint64_t)(k >> 8) * 144;
    uint32_t j = k & 255, s = j >> 5, l0 = j & 31;
    uint4 h = *(const uint4 *)blk;
    uint2 qv = *(const uint2 *)(blk + 16 + (s >> 1) * 32 + l0);
    uint32_t A = h.y, B = h.z, C = h.w, sh = 8 * (s & 3), sc, m;
    if (s < 4) { sc = (A >> sh) & 63u; m = (B >> sh) & 63u; }
    else { sc = ((C >> sh) & 15u) | (((A >> sh) >> 6 & 3u) << 4); m = ((C >> sh) >> 4 & 15u) | (((B >> sh) >> 6 & 3u) << 4); }
    float dsc = half_bits(h.x & 0xFFFFu) * (float)sc, dmm = half_bits(h.x >> 16) * (float)m;
    uint32_t sq = 4 * (s & 1);
#pragma unroll
    for (int i = 0; i < 8; i++) {
      uint32_t byte = ((i < 4 ? qv.x : qv.y) >> (8 * (i & 3))) & 0xFFu;
      o[i] = dsc * (float)((byte >> sq) & 15u) - dmm;
    }
    return;
  }
  if (a.type == Q4_K && a.layout == LAYOUT_PLANAR) {
    const Q4Planes p = q4_planes(a.nbt);
    const uint32_t j = k & 255, s = j >> 5, e0 = k & 31;
    uint4 h = *(const uint4 *)(a.w + p.hdr + tiled(row, k >> 8, a.bpr) * 16);
    // chunk k / 32, bytes e0 % 16 .. +8, nibble e0 / 16
    uint2 qv = *(const uint2 *)(a.w + p.qs + tiled(row, k >> 5, a.bpr * 8) * 16 + (e0 & 15));
    uint32_t A = h.y, B = h.z, C = h.w, sh = 8 * (s & 3), sc, m;
    if (s < 4) { sc = (A >> sh) & 63u; m = (B >> sh) & 63u; }
    else { sc = ((C >> sh) & 15u) | (((A >> sh) >> 6 & 3u) << 4); m = ((C >> sh) >> 4 & 15u) | (((B >> sh) >> 6 & 3u) << 4); }
    float dsc = half_bits(h.x & 0xFFFFu) * (float)sc, dmm = half_bits(h.x >> 16) * (float)m;
    uint32_t sq = 4 * (e0 >> 4);
#pragma unroll
    for (int i = 0; i < 8; i++) {
      uint32_t byte = ((i < 4 ? qv.x : qv.y) >> (8 * (i & 3))) & 0xFFu;
      o[i] = dsc * (float)((byte >> sq) & 15u) - dmm;
    }
    return;
  }
  if (a.type == Q6_K && a.layout == LAYOUT_PLANAR) {
    const Q6Planes p = q6_planes(a.nbt);
    const uint32_t e0 = k & 31, h = e0 >> 4;
    const uint64_t ci = tiled(row, k >> 5, a.bpr * 8);
    uint2 lo = *(const uint2 *)(a.w + p.ql + ci * 16 + (e0 & 15));
    // high bits of elements e0 .. e0+7: qh dword (e0 % 16) / 8, byte i % 4, bit 4 * (i / 4) + 2h
    uint32_t hq = *(const uint32_t *)(a.w + p.qh + ci * 8 + 4 * ((e0 & 15) >> 3));
    float sc = (float)(int8_t)a.w[p.sc + ci * 2 + h];
    float d = half_bits(*(const uint16_t *)(a.w + p.d + tiled(row, k >> 8, a.bpr) * 2)) * sc;
    uint32_t ls = 4 * h;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      uint32_t lb = ((i < 4 ? lo.x : lo.y) >> (8 * (i & 3))) & 0xFFu;
      uint32_t hb = (hq >> (8 * (i & 3) + 4 * (i >> 2) + 2 * h)) & 3u;
      o[i] = d * (float)((int)(((lb >> ls) & 15u) | (hb << 4)) - 32);
    }
    return;
  }
  if (a.type == Q5_K && a.layout == LAYOUT_PLANAR) {
    const Q5Planes p = q5_planes(a.nbt);
    const uint32_t j = k & 255, s = j >> 5, e0 = k & 31;
    uint4 h = *(const uint4 *)(a.w + p.hdr + tiled(row, k >> 8, a.bpr) * 16);
    uint2 qv = *(const uint2 *)(a.w + p.qs + tiled(row, k >> 5, a.bpr * 8) * 16 + (e0 & 15));
    const uint32_t hb = *(const uint32_t *)(a.w + p.qh + tiled(row, k >> 5, a.bpr * 8) * 4);
    uint32_t A = h.y, B = h.z, C = h.w, sh = 8 * (s & 3), sc, m;
    if (s < 4) { sc = (A >> sh) & 63u; m = (B >> sh) & 63u; }
    else { sc = ((C >> sh) & 15u) | (((A >> sh) >> 6 & 3u) << 4); m = ((C >> sh) >> 4 & 15u) | (((B >> sh) >> 6 & 3u) << 4); }
    float dsc = half_bits(h.x & 0xFFFFu) * (float)sc, dmm = half_bits(h.x >> 16) * (float)m;
    uint32_t sq = 4 * (e0 >> 4);
#pragma unroll
    for (int i = 0; i < 8; i++) {
      // fifth bit of chunk element e: byte e % 4, bit e / 4 (e < 16) or 4 + (e - 16) / 4
      const uint32_t e = e0 + i, pos = 8 * (e & 3) + (e < 16 ? e / 4 : 4 + (e - 16) / 4);
      uint32_t byte = ((i < 4 ? qv.x : qv.y) >> (8 * (i & 3))) & 0xFFu;
      o[i] = dsc * (float)(((byte >> sq) & 15u) | (((hb >> pos) & 1u) << 4)) - dmm;
    }
    return;
  }
  if (a.type == Q4_0 && a.layout == LAYOUT_PLANAR) {
    const Q40Planes p = q40_planes(a.nbt);
    const uint32_t e0 = k & 31;
    uint2 qv = *(const uint2 *)(a.w + p.qs + tiled(row, k >> 5, a.bpr) * 16 + (e0 & 15));
    float d = half_bits(*(const uint16_t *)(a.w + p.d + tiled(row, k >> 5, a.bpr) * 2));
    uint32_t sq = 4 * (e0 >> 4);
#pragma unroll
    for (int i = 0; i < 8; i++) {
      uint32_t byte = ((i < 4 ? qv.x : qv.y) >> (8 * (i & 3))) & 0xFFu;
      o[i] = d * (float)((int)((byte >> sq) & 15u) - 8);
    }
    return;
  }
  if (a.type == Q8_0 && a.layout == LAYOUT_PLANAR) {
    const Q8Planes p = q8_planes(a.nbt);
    uint2 q = *(const uint2 *)(a.w + p.qs + tiled(row, k >> 4, a.bpr * 2) * 16 + (k & 15));
    float d = half_bits(*(const uint16_t *)(a.w + p.d + tiled(row, k >> 5, a.bpr) * 2));
#pragma unroll
    for (int i = 0; i < 8; i++) o[i] = d * (float)(int8_t)(((i < 4 ? q.x : q.y) >> (8 * (i & 3))) & 0xFFu);
    return;
  }
  const uint8_t *r = a.w + (uint64_t)row * a.rb;
  if (a.type == F16 && (a.rb & 15) == 0) {
    // eight halves in one 16-byte load (rows stay 16-byte aligned for K % 8 == 0)
    const uint4 v = *(const uint4 *)(r + 2 * (uint64_t)k);
    const uint32_t h[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
      o[2 * i] = half_bits(h[i] & 0xFFFFu);
      o[2 * i + 1] = half_bits(h[i] >> 16);
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < 8; i++) o[i] = deq_elem(a.type, r, k + i);
}

constexpr int KT = 64;              // K per LDS tile
constexpr int NT = 64;              // tokens per workgroup
constexpr int XPITCH = KT + 8;      // bf16 elements per LDS row (16-byte pad)

__global__ __launch_bounds__(256) void k_gemm(GemmArgs a) {
  __shared__ __attribute__((aligned(16))) uint16_t xh[NT * XPITCH];
  __shared__ __attribute__((aligned(16))) uint16_t xl[NT * XPITCH];
  const uint32_t tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const uint32_t m0 = blockIdx.x * 64 + wv * 16, n0 = blockIdx.y * NT;
  const uint32_t arow = m0 + (lane & 15), kg = 8 * (lane >> 4);
  f32x4 acc[4];
#pragma unroll
  for (int t = 0; t < 4; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (uint32_t k0 = 0; k0 < a.cols; k0 += KT) {
    // Stage x[n0 .. n0+64)[k0 .. k0+64) as split bf16: 256 threads x 16 elements.
    {
      uint32_t n = tid >> 2, kk = (tid & 3) * 16;
      float v[16];
      if (n0 + n < a.batch && k0 + kk < a.cols) {
        const float4 *src = (const float4 *)(a.x + (uint64_t)(n0 + n + a.input_offset) * a.cols + k0 + kk);
#pragma unroll
        for (int i = 0; i < 4; i++) { float4 t = src[i]; v[4 * i] = t.x; v[4 * i + 1] = t.y; v[4 * i + 2] = t.z; v[4 * i + 3] = t.w; }
      } else {
#pragma unroll
        for (int i = 0; i < 16; i++) v[i] = 0.f;
      }
      uint4 h0, l0, h1, l1;
      split8(v, h0, l0); split8(v + 8, h1, l1);
      *(uint4 *)&xh[n * XPITCH + kk] = h0; *(uint4 *)&xh[n * XPITCH + kk + 8] = h1;
      *(uint4 *)&xl[n * XPITCH + kk] = l0; *(uint4 *)&xl[n * XPITCH + kk + 8] = l1;
    }
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < KT; ks += 32) {
      float wv8[8];
      if (arow < a.rows) load_a8(a, arow, k0 + ks + kg, wv8);
      else {
#pragma unroll
        for (int i = 0; i < 8; i++) wv8[i] = 0.f;
      }
      uint4 ah, al;
      split8(wv8, ah, al);
      bf16x8 Ah = __builtin_bit_cast(bf16x8, ah), Al = __builtin_bit_cast(bf16x8, al);
#pragma unroll
      for (int t = 0; t < 4; t++) {
        uint32_t n = t * 16 + (lane & 15);
        bf16x8 Bh = __builtin_bit_cast(bf16x8, *(const uint4 *)&xh[n * XPITCH + ks + kg]);
        bf16x8 Bl = __builtin_bit_cast(bf16x8, *(const uint4 *)&xl[n * XPITCH + ks + kg]);
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(Ah, Bh, acc[t], 0, 0, 0);
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(Ah, Bl, acc[t], 0, 0, 0);
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(Al, Bh, acc[t], 0, 0, 0);
      }
    }
    __syncthreads();
  }
  // D layout: lane holds rows 4*(lane/16)+i, token column lane%16 of each 16x16 tile.
#pragma unroll
  for (int t = 0; t < 4; t++) {
    uint32_t tok = n0 + t * 16 + (lane & 15);
    if (tok >= a.batch) continue;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      uint32_t row = m0 + 4 * (lane >> 4) + i;
      if (row < a.rows) a.y[(uint64_t)tok * a.stride + a.row_base + row] = acc[t][i];
    }
  }
}

// ------------------------------------------------------------------ planar quant GEMM
//
// The prompt GEMM of the planar layouts (Q4_K, Q5_K, Q6_K, Q8_0, Q4_0; the decode matvec's
// weights). A workgroup owns 128 weight rows x 16 TT tokens (256 x 128: TT = 8) and a K span (split-K when
// the rows alone give too few workgroups; partial sums are added in split order by the
// finishes, so results do not depend on timing).
//
// Every weight is unpacked once per workgroup, in registers, by the one wavefront that uses
// it: lane 16 g + c loads the 32-element chunk g of row c of a 128-column unit (1 KB of
// contiguous bytes a wavefront), and its four groups of eight are the B operands of four
// v_mfma_f32_16x16x32_f16, each summing over one group of every chunk. The weights enter as exact
// f16 integers: sc * q <= 63 * 31 for Q4_K and Q5_K, q for Q8_0 and Q4_0, and sc * (q - 32)
// as an exact (hi, lo) pair for Q6_K. The activations are split.h's (hi, lo) pairs: two
// MFMAs per product (three for Q6_K; its lo * lo part is below 2^-22 of the product). A unit's
// sums are scaled by the row's d in f32, the K-quants' min terms, -dmin * m times the sums of x over
// the token's scale, come from one f32 MFMA (16x16x4: its four K entries are the unit's four chunks) and are added, and
// the token's scale comes last. The worst errors against float64 are those of f32 sums (mlp of Q6_K 4096 x
// 14336, 32 tokens: 2.8e-7 relative; bf16 pairs of both operands gave 6.9e-6).
//
// The activations go through two LDS buffers of S units: the next S units are loaded into
// registers while the current ones are used, one barrier per S units. D units of weights are
// in flight per row tile. No load has a branch around it (past the span it reads through an empty
// resource), so each wait counts exactly the loads behind it; only the products of a unit past the span are
// skipped.
//
// What it replaces: bf16 pairs of dequantized weights in LDS, always 128 tokens wide, three
// MFMAs per product and about 210 VALU instructions per 32 weights against about 70. Kernel times
// of the 8B shape in the model, Q4_K: 16 tokens, gate + up (28672 x 4096) 86 -> 21 us (3.1 TB/s of weights), down
// 47 -> 14, a prompt of 250 tokens in 16s over 4 layers 12.8 -> 5.7 ms; 128 tokens, gate + up 88 ->
// 79 us (0.76 PFLOP/s of f16 products), down 47 -> 41. By its counters, gate + up at 16 tokens spends 41% of
// a wavefront's life on loads, 32% waiting for an issue slot and 27% issuing, with the matrix cores busy for
// 18% of the launch; at 128 tokens 33%, 40% and 27%, the matrix cores 38%. 128 tokens need 33 us of LDS
// reads and 20 us of VALU issue beside 30 us of MFMAs; they add up to the launch rather than overlap.
constexpr uint32_t QG_M = 128, QG_K = 64;
constexpr uint32_t QG_U = SPLIT_K;   // columns of a unit

// One weight matrix of a grouped launch: its planar geometry, the row-tile count, and where
// its rows go (y, or rows [row0, row0 + rows) of the group's split-K partial sums).
struct QJob {
  const uint8_t *w; uint32_t wbytes;
  uint32_t C, bpr, nbp;  // chunk columns, blocks per row, blocks of the padded matrix
  uint32_t rows, tiles, kind, row0, off;  // off: the launch's tiles before this matrix's, mod 8
  float *y; uint32_t stride, row_base;
};
constexpr uint32_t QG_MAX_JOBS = 3;
// Matrices that read the same activations, launched together: workgroups (tile, split)
// over the concatenated row tiles; kind 0 / 1 selects the launch's first / second type.
struct QGemm {
  QJob job[QG_MAX_JOBS]; uint32_t njobs;
  const uint8_t *xs; float *part;
  uint32_t cols, batch, kspan, rows_total, accumulate;  // kspan: a multiple of QG_U
};

// Activations [batch][cols] f32 -> the split form (split.h): one thread per eight
// consecutive columns of a token, 16 threads per 128 columns.
__global__ __launch_bounds__(256) void k_gemm_split(const float *x, uint8_t *xs, uint32_t cols, uint32_t count) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x, c8 = split_kblocks(cols) * 16, tok = i / c8, k = (i % c8) * 8;
  if (i >= count || k >= cols) return;
  const float4 *p = (const float4 *)(x + (uint64_t)tok * cols + k);
  split_store8(xs, cols, tok, k, p[0], p[1]);
}

typedef __amdgpu_buffer_rsrc_t QRsrc;
__device__ __forceinline__ uint4 qld16(QRsrc r, uint32_t off) {
  typedef unsigned int u4 __attribute__((ext_vector_type(4)));
  const u4 v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
  return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ uint2 qld8(QRsrc r, uint32_t off) {
  typedef unsigned int u2 __attribute__((ext_vector_type(2)));
  const u2 v = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0);
  return make_uint2(v.x, v.y);
}
__device__ __forceinline__ uint32_t qld2(QRsrc r, uint32_t off) { return __builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0); }

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ f16x2 h2(uint32_t v) { return __builtin_bit_cast(f16x2, v); }
__device__ __forceinline__ uint32_t u32(f16x2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ f16x2 both(_Float16 v) { return f16x2{v, v}; }
__device__ __forceinline__ float f16_lo(uint32_t v) { return (float)__builtin_bit_cast(_Float16, (uint16_t)v); }
// Bytes 0 and 2, and bytes 1 and 3, of a dword as 1024 + byte in f16 (the byte in the mantissa's
// low bits): one byte permute each.
__device__ __forceinline__ f16x2 bytes02(uint32_t v) { return h2(__builtin_amdgcn_perm(0x64646464u, v, 0x04020400u)); }
__device__ __forceinline__ f16x2 bytes13(uint32_t v) { return h2(__builtin_amdgcn_perm(0x64646464u, v, 0x04030401u)); }
// (v & mask) | bits as one instruction (the compiler keeps two where both are literals).
__device__ __forceinline__ uint32_t and_or(uint32_t v, uint32_t mask, uint32_t bits) {
  asm("" : "+s"(mask));
  asm("" : "+v"(bits));
  return (v & mask) | bits;
}
__device__ __forceinline__ f16x2 fma2(f16x2 a, f16x2 b, f16x2 c) { return __builtin_elementwise_fma(a, b, c); }
__device__ __forceinline__ f16x8 oct(f16x2 a, f16x2 b, f16x2 c, f16x2 d) {
  return __builtin_bit_cast(f16x8, make_uint4(u32(a), u32(b), u32(c), u32(d)));
}
// The 6-bit scale and min of chunk g of a unit, the first (odd = 0) or second of its block
// (quant.ts:9-12).
__device__ __forceinline__ void scale_min(const uint4 &h, uint32_t odd, uint32_t g, uint32_t &sc, uint32_t &m) {
  const uint32_t sh = 8 * g, A = h.y >> sh, B = h.z >> sh, C = h.w >> sh;
  sc = odd ? (C & 15u) | ((A >> 2) & 48u) : A & 63u;
  m = odd ? ((C >> 4) & 15u) | ((B >> 2) & 48u) : B & 63u;
}

// A lane's weights of 16 rows x one 128-column unit. fetch() loads them; unpack() leaves the MFMA
// operands w[j] (wl[j]: their lo parts, LO types), for the types of whole 256-column blocks the row's d in d[0] and
// the chunk's -dmin * m in mn (MIN types), for the 32-column block types block j's d in d[j].
// CHUNK types: operand j holds elements 8 j .. + 8 of chunk g; else elements 8 g .. + 8 of block j.
template <int TYPE> struct QUnit;
template <> struct QUnit<Q4_K> {
  static constexpr bool CHUNK = true, LO = false, MIN = true;
  uint4 q, h;
  __device__ void fetch(const QJob &a, QRsrc rw, uint32_t T, uint32_t u, uint32_t g, uint32_t c) {
    q = qld16(rw, ((T * a.C + 4 * u + g) * 16 + c) * 16);
    h = qld16(rw, a.nbp * 128 + ((T * a.bpr + u / 2) * 16 + c) * 16);
  }
  __device__ void unpack(uint32_t odd, uint32_t g, f16x8 *w, f16x8 *, float *d, float &mn) const {
    uint32_t sc, m;
    scale_min(h, odd, g, sc, m);
    d[0] = f16_lo(h.x);
    mn = -f16_lo(h.x >> 16) * (float)m;
    // low nibbles as 1024 + q, high nibbles (bits 4-7 of the mantissa, in units of 1/16 at 64) as 64 + q:
    // sc * (1024 + q) - 1024 sc and sc * (64 + q) - 64 sc are exact, 1024 sc <= 64512
    const f16x2 s = both((_Float16)(uint16_t)sc), bl = s * both((_Float16)-1024.f), bh = s * both((_Float16)-64.f);
    auto lo = [&](uint32_t v) { return fma2(h2(and_or(v, 0x000F000Fu, 0x64006400u)), s, bl); };
    auto hi = [&](uint32_t v) { return fma2(h2(and_or(v, 0x00F000F0u, 0x54005400u)), s, bh); };
    const uint32_t x = q.x >> 8, y = q.y >> 8, z = q.z >> 8, t = q.w >> 8;
    w[0] = oct(lo(q.x), lo(x), lo(q.y), lo(y));
    w[1] = oct(lo(q.z), lo(z), lo(q.w), lo(t));
    w[2] = oct(hi(q.x), hi(x), hi(q.y), hi(y));
    w[3] = oct(hi(q.z), hi(z), hi(q.w), hi(t));
  }
};
// Q5_K: Q4_K's chunk and header planes (the header after the fifth-bit plane) and the
// chunk's dword of fifth bits, moved to bit 4 of each quant byte.
template <> struct QUnit<Q5_K> {
  static constexpr bool CHUNK = true, LO = false, MIN = true;
  uint4 q, h; uint32_t b;
  __device__ void fetch(const QJob &a, QRsrc rw, uint32_t T, uint32_t u, uint32_t g, uint32_t c) {
    const uint32_t tc = (T * a.C + 4 * u + g) * 16 + c;
    q = qld16(rw, tc * 16);
    b = __builtin_amdgcn_raw_buffer_load_b32(rw, a.nbp * 128 + tc * 4, 0, 0);
    h = qld16(rw, a.nbp * 160 + ((T * a.bpr + u / 2) * 16 + c) * 16);
  }
  __device__ void unpack(uint32_t odd, uint32_t g, f16x8 *w, f16x8 *, float *d, float &mn) const {
    uint32_t sc, m;
    scale_min(h, odd, g, sc, m);
    d[0] = f16_lo(h.x);
    mn = -f16_lo(h.x >> 16) * (float)m;
    const f16x2 s = both((_Float16)(uint16_t)sc), bl = s * both((_Float16)-1024.f);
    const uint32_t qw[4] = {q.x, q.y, q.z, q.w};
    f16x2 v[16];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const uint32_t lo = (qw[k] & 0x0F0F0F0Fu) | ((b << (4 - k)) & 0x10101010u);
      const uint32_t hi = ((qw[k] >> 4) & 0x0F0F0F0Fu) | ((b >> k) & 0x10101010u);
      v[2 * k] = fma2(bytes02(lo), s, bl);
      v[2 * k + 1] = fma2(bytes13(lo), s, bl);
      v[8 + 2 * k] = fma2(bytes02(hi), s, bl);
      v[8 + 2 * k + 1] = fma2(bytes13(hi), s, bl);
    }
#pragma unroll
    for (int j = 0; j < 4; j++) w[j] = oct(v[4 * j], v[4 * j + 1], v[4 * j + 2], v[4 * j + 3]);
  }
};
// Q6_K: sc * (q - 32) has up to 12 bits; hi = RN_f16, lo = the exact rest.
template <> struct QUnit<Q6_K> {
  static constexpr bool CHUNK = true, LO = true, MIN = false;
  uint4 q; uint2 qh; uint32_t sc, dd;
  __device__ void fetch(const QJob &a, QRsrc rw, uint32_t T, uint32_t u, uint32_t g, uint32_t c) {
    const uint32_t tc = (T * a.C + 4 * u + g) * 16 + c;
    q = qld16(rw, tc * 16);
    qh = qld8(rw, a.nbp * 128 + tc * 8);
    sc = qld2(rw, a.nbp * 192 + tc * 2);
    dd = qld2(rw, a.nbp * 208 + ((T * a.bpr + u / 2) * 16 + c) * 2);
  }
  __device__ void unpack(uint32_t, uint32_t, f16x8 *w, f16x8 *wl, float *d, float &) const {
    d[0] = f16_lo(dd);
    const f16x2 s0 = both((_Float16)(int16_t)(int8_t)sc), s1 = both((_Float16)(int16_t)(int8_t)(sc >> 8));
    const f16x2 off = both((_Float16)-1056.f);
    const uint32_t qw[4] = {q.x, q.y, q.z, q.w};
    f16x2 v[16], r[16];
    auto put = [&](int i, f16x2 n, f16x2 s) {
      n += off;
      v[i] = n * s;
      r[i] = fma2(n, s, -v[i]);
    };
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const uint32_t Q = (k < 2 ? qh.x : qh.y) >> (4 * (k & 1));
      const uint32_t lo = (qw[k] & 0x0F0F0F0Fu) | ((Q << 4) & 0x30303030u);
      const uint32_t hi = ((qw[k] >> 4) & 0x0F0F0F0Fu) | ((Q << 2) & 0x30303030u);
      put(2 * k, bytes02(lo), s0);
      put(2 * k + 1, bytes13(lo), s0);
      put(8 + 2 * k, bytes02(hi), s1);
      put(8 + 2 * k + 1, bytes13(hi), s1);
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
      w[j] = oct(v[4 * j], v[4 * j + 1], v[4 * j + 2], v[4 * j + 3]);
      wl[j] = oct(r[4 * j], r[4 * j + 1], r[4 * j + 2], r[4 * j + 3]);
    }
  }
};
// Q8_0: block j of the unit is chunks 2 j, 2 j + 1 of 16 bytes; a lane takes eight of its bytes.
template <> struct QUnit<Q8_0> {
  static constexpr bool CHUNK = false, LO = false, MIN = false;
  uint2 q[4]; uint32_t dd[4];
  __device__ void fetch(const QJob &a, QRsrc rw, uint32_t T, uint32_t u, uint32_t g, uint32_t c) {
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) {
      q[j] = qld8(rw, ((T * a.C + 8 * u + 2 * j + (g >> 1)) * 16 + c) * 16 + 8 * (g & 1));
      dd[j] = qld2(rw, a.nbp * 32 + ((T * a.bpr + 4 * u + j) * 16 + c) * 2);
    }
  }
  __device__ void unpack(uint32_t, uint32_t, f16x8 *w, f16x8 *, float *d, float &) const {
    const f16x2 off = both((_Float16)-1152.f);  // the sign bit flipped: byte + 128
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const uint32_t x = q[j].x ^ 0x80808080u, y = q[j].y ^ 0x80808080u;
      w[j] = oct(bytes02(x) + off, bytes13(x) + off, bytes02(y) + off, bytes13(y) + off);
      d[j] = f16_lo(dd[j]);
    }
  }
};
// Q4_0: block j is one chunk; lane group g takes bytes 8 (g % 2) .. + 8, nibble g / 2.
template <> struct QUnit<Q4_0> {
  static constexpr bool CHUNK = false, LO = false, MIN = false;
  uint2 q[4]; uint32_t dd[4];
  __device__ void fetch(const QJob &a, QRsrc rw, uint32_t T, uint32_t u, uint32_t g, uint32_t c) {
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) {
      const uint32_t tc = (T * a.C + 4 * u + j) * 16 + c;
      q[j] = qld8(rw, tc * 16 + 8 * (g & 1));
      dd[j] = qld2(rw, a.nbp * 16 + tc * 2);
    }
  }
  __device__ void unpack(uint32_t, uint32_t g, f16x8 *w, f16x8 *, float *d, float &) const {
    const f16x2 off = both((_Float16)-1032.f);
    const uint32_t sh = 4 * (g >> 1);
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const uint32_t x = (q[j].x >> sh) & 0x0F0F0F0Fu, y = (q[j].y >> sh) & 0x0F0F0F0Fu;
      w[j] = oct(bytes02(x) + off, bytes13(x) + off, bytes02(y) + off, bytes13(y) + off);
      d[j] = f16_lo(dd[j]);
    }
  }
};

// Row tiles per wavefront. Up to 32 tokens the weight stream is the bound, and eight
// wavefronts of one row tile (84 to 119 registers, so four or five per SIMD; 120 to 140 and three with two
// types at 32 tokens) hide its latency better
// than four of two (8B prompt in 16s 6.22 against 6.34 ms); for 64 tokens two row tiles halve
// the LDS reads of the activations per MFMA.
constexpr uint32_t qg_rt(uint32_t tt) { return tt <= 2 ? 1 : 2; }
// Rows per workgroup: 128, and 256 (eight wavefronts) where it takes 128 tokens.
constexpr uint32_t qg_rows(uint32_t tt) { return tt == 8 ? 2 * QG_M : QG_M; }
constexpr uint32_t qg_threads(uint32_t tt) { return qg_rows(tt) / 16 / qg_rt(tt) * 64; }
// Units of weights in flight per row tile (registers), and units of activations per LDS buffer (17
// KB at 16 tokens, 34 at 32 and 64, 68 at 128, where the two buffers leave room for one workgroup per CU).
// Two units suffice with eight wavefronts or more a CU; four and eight were slower
// (28672 x 4096 Q4_K, 16 tokens: 20.5, 21.5 and 28.8 us), their registers and prologue cost more.
// Past 32 tokens the registers are full, and some kernels spill outside their inner products: Q4_K or
// Q5_K with Q6_K (Q, K and V of the usual mixes) 68 bytes a lane, Q5_K and Q6_K at 128 tokens 16. One
// unit of Q6_K in flight at 64 tokens spills nothing (208 registers) and is slower: Q, K and V of the 8B
// widths, 128 tokens, 29.2 against 27.9 us.
constexpr uint32_t qg_depth(int type, uint32_t tt) { return tt == 8 || (tt == 4 && (type == Q8_0 || type == Q4_0)) ? 1 : 2; }
constexpr uint32_t qg_stage(int type, uint32_t tt) { return tt >= 4 ? 1 : qg_depth(type, tt); }

template <int TYPE, uint32_t TT>
__device__ __forceinline__ void gemm_tile(const QGemm &a, const QJob &jb, uint32_t mt, uint8_t *lds) {
  constexpr uint32_t RT = qg_rt(TT), D = qg_depth(TYPE, TT), S = qg_stage(TYPE, TT), UB = TT * SPLIT_BLOCK, NT = qg_threads(TT);
  typedef QUnit<TYPE> W;
  const uint32_t tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, g = lane >> 4, c = lane & 15;
  uint32_t m0 = mt * QG_M + wv * 16 * RT;
  if constexpr (qg_rows(TT) == 2 * QG_M) {
    // Two runs of 128 rows. The finishes expect run r on XCD r % 8 (as 128-row tiles put it), so of every
    // eight whole tiles, on XCDs off, off + 1, ..., tile t takes the runs r and r + 8 with r = t's XCD.
    const uint32_t half = wv >> 2, t8 = mt / 8 * 8;
    const uint32_t run = t8 + 8 <= jb.tiles ? 2 * t8 + (mt + jb.off) % 8 + 8 * half : 2 * mt + half;
    m0 = run * QG_M + (wv & 3) * 16 * RT;
  }
  const uint32_t b0 = blockIdx.y * TT, z = blockIdx.z;
  const uint32_t kbs = split_kblocks(a.cols);
  const uint32_t u0 = z * (a.kspan / QG_U), ue = u0 + a.kspan / QG_U, u1 = ue < kbs ? ue : kbs;
  const uint32_t T0 = m0 / 16;
  f32x4 acc[RT][TT];
#pragma unroll
  for (uint32_t r = 0; r < RT; r++)
#pragma unroll
    for (uint32_t t = 0; t < TT; t++) acc[r][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  W buf[D][RT];
  // Units past the span read zeros (a resource of no bytes) and no memory: the loop below has
  // no branch around a load or its use, so the waits count exactly the loads behind them.
  auto fetch = [&](uint32_t d, uint32_t u) {
    const QRsrc rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(jb.w), 0, u < u1 ? (int)jb.wbytes : 0, 0x00020000);
#pragma unroll
    for (uint32_t r = 0; r < RT; r++) buf[d][r].fetch(jb, rw, T0 + r, u, g, c);
  };
  // units [u, u + S) of the split input (those inside the span; zeros past it): TT blocks a
  // unit, contiguous, loaded into registers and stored into one of the two LDS buffers
  constexpr uint32_t STEP = (SPLIT_TOK / SPLIT_N) * SPLIT_BLOCK, P = S * UB / 16, PN = (P + NT - 1) / NT;
  uint4 sv[PN];
  auto stage_load = [&](uint32_t u) {
    const uint32_t nu = u >= u1 ? 0 : u1 - u < S ? u1 - u : S;
    const QRsrc rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(a.xs + split_block_at(b0, u, kbs)), 0,
                                                       nu ? (int)((nu - 1) * STEP + UB) : 0, 0x00020000);
#pragma unroll
    for (uint32_t k = 0; k < PN; k++) {
      const uint32_t i = tid + k * NT;
      sv[k] = qld16(rx, (i / (UB / 16)) * STEP + (i % (UB / 16)) * 16);
    }
  };
  auto stage_store = [&](uint32_t u) {
    uint8_t *dst = lds + (((u - u0) / S) & 1) * (S * UB);
#pragma unroll
    for (uint32_t k = 0; k < PN; k++)
      if ((k + 1) * NT <= P || tid + k * NT < P) *(uint4 *)(dst + (tid + k * NT) * 16) = sv[k];
  };
  auto compute = [&](uint32_t d, uint32_t u) {
    const uint8_t *xl = lds + ((u - u0) % (2 * S)) * UB;
    // the last unit of a width of 64 (mod 128) columns: its first two blocks
    const bool half = !W::CHUNK && a.cols - u * QG_U < QG_U;
    f16x8 w[RT][4], wl[RT][W::LO ? 4 : 1];
    float dr[RT][W::CHUNK ? 1 : 4], mn[RT];
#pragma unroll
    for (uint32_t r = 0; r < RT; r++) buf[d][r].unpack(D > 1 ? d % 2 : u % 2, g, w[r], wl[r], dr[r], mn[r]);
#pragma unroll
    for (uint32_t t = 0; t < TT; t++) {
      const uint8_t *xb = xl + t * SPLIT_BLOCK;
      const f32x4 s = *(const f32x4 *)(xb + SPLIT_SCALE + 16 * g);
      f16x8 xh[4], xo[4];
#pragma unroll
      for (uint32_t j = 0; j < 4; j++) {
        const uint32_t at = W::CHUNK ? (j * 64 + lane) * 16 : ((g * 4 + j) * 16 + c) * 16;
        xh[j] = *(const f16x8 *)(xb + at);
        xo[j] = *(const f16x8 *)(xb + at + SPLIT_LO);
      }
      const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
      if constexpr (W::CHUNK) {
        f32x4 p[RT];
#pragma unroll
        for (uint32_t j = 0; j < 4; j++) {
#pragma unroll
          for (uint32_t r = 0; r < RT; r++)
            p[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[j], w[r][j], j ? p[r] : zero, 0, 0, 0);
#pragma unroll
          for (uint32_t r = 0; r < RT; r++) p[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xo[j], w[r][j], p[r], 0, 0, 0);
          if constexpr (W::LO) {
#pragma unroll
            for (uint32_t r = 0; r < RT; r++) p[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[j], wl[r][j], p[r], 0, 0, 0);
          }
        }
        const float xsum = W::MIN ? *(const float *)(xb + SPLIT_SUM + 4 * lane) : 0.f;
#pragma unroll
        for (uint32_t r = 0; r < RT; r++) {
          if constexpr (W::MIN && TT <= 2) {  // the min terms beside the products: a shorter chain, four registers more
            const f32x4 m = __builtin_amdgcn_mfma_f32_16x16x4f32(xsum, mn[r], zero, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; i++) p[r][i] = fmaf(p[r][i], dr[r][0], m[i]);
          } else {
#pragma unroll
            for (int i = 0; i < 4; i++) p[r][i] *= dr[r][0];
            if constexpr (W::MIN) p[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(xsum, mn[r], p[r], 0, 0, 0);
          }
#pragma unroll
          for (int i = 0; i < 4; i++) acc[r][t][i] = fmaf(p[r][i], s[i], acc[r][t][i]);
        }
      } else {
        f32x4 q[RT];
#pragma unroll
        for (uint32_t j = 0; j < 4; j++) {
          if (half && j >= 2) break;
          f32x4 p[RT];
#pragma unroll
          for (uint32_t r = 0; r < RT; r++) p[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[j], w[r][j], zero, 0, 0, 0);
#pragma unroll
          for (uint32_t r = 0; r < RT; r++) p[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xo[j], w[r][j], p[r], 0, 0, 0);
#pragma unroll
          for (uint32_t r = 0; r < RT; r++)
#pragma unroll
            for (int i = 0; i < 4; i++) q[r][i] = j ? fmaf(p[r][i], dr[r][j], q[r][i]) : p[r][i] * dr[r][j];
        }
#pragma unroll
        for (uint32_t r = 0; r < RT; r++)
#pragma unroll
          for (int i = 0; i < 4; i++) acc[r][t][i] = fmaf(q[r][i], s[i], acc[r][t][i]);
      }
    }
  };
  stage_load(u0);
#pragma unroll
  for (uint32_t d = 0; d < D; d++) fetch(d, u0 + d);
  stage_store(u0);
  __syncthreads();
  for (uint32_t ub = u0; ub < u1; ub += D) {
#pragma unroll
    for (uint32_t d = 0; d < D; d++) {
      const uint32_t u = ub + d;
      if (d % S == 0) stage_load(u + S);
      if (u < u1) compute(d, u);
      fetch(d, u + D);
      if (d % S == S - 1) {
        stage_store(u + 1);
        __syncthreads();
      }
    }
  }
  // The products are formed as X W^T, so lane (g, c) of tile (r, t) holds tokens 16 t + 4 g + i
  // of row 16 r + c: each store writes 16 consecutive rows of four tokens.
  float *out = a.part ? a.part + (uint64_t)z * a.batch * a.rows_total + jb.row0 : jb.y + jb.row_base;
  const uint32_t stride = a.part ? a.rows_total : jb.stride;
  const bool add = a.accumulate && !a.part;  // partials are added by their finish
#pragma unroll
  for (uint32_t r = 0; r < RT; r++) {
    const uint32_t row = m0 + 16 * r + c;
    if (row >= jb.rows) continue;
#pragma unroll
    for (uint32_t t = 0; t < TT; t++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const uint32_t tok = (b0 + t) * 16 + 4 * g + i;
        if (tok >= a.batch) continue;
        float *py = out + (uint64_t)tok * stride + row;
        *py = add ? *py + acc[r][t][i] : acc[r][t][i];
      }
  }
}

// blockIdx.x walks the jobs' row tiles in order; a job of kind 1 runs the second type.
template <int T0, int T1, uint32_t TT>
__global__ __launch_bounds__(qg_threads(TT), 2) void k_gemm_q(QGemm a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t qlds[];
  uint32_t t = blockIdx.x, j = 0;
  while (j + 1 < a.njobs && t >= a.job[j].tiles) { t -= a.job[j].tiles; j++; }
  const QJob &jb = a.job[j];
  if (T0 == T1 || jb.kind == 0) gemm_tile<T0, TT>(a, jb, t, qlds);
  else gemm_tile<T1, TT>(a, jb, t, qlds);
}

// Sum of the split-K partials part[z][tok][rows_total] in split order into each job's rows
// (accumulate: added to y).
template <uint32_t S>
__global__ __launch_bounds__(256) void k_gemm_reduce(QGemm a, uint32_t splits) {
  const uint64_t n = (uint64_t)a.rows_total * a.batch;
  const __amdgpu_buffer_rsrc_t rp = split_rsrc(a.part, splits, n);
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256) {
    const float v = split_sum<S>(rp, splits, (uint32_t)(4 * n), (uint32_t)(4 * i));
    const uint32_t tok = (uint32_t)(i / a.rows_total);
    uint32_t r = (uint32_t)(i % a.rows_total), j = 0;
    while (j + 1 < a.njobs && r >= a.job[j].rows) { r -= a.job[j].rows; j++; }
    float *py = a.job[j].y + (uint64_t)tok * a.job[j].stride + a.job[j].row_base + r;
    *py = a.accumulate ? *py + v : v;
  }
}

// The GLU finish (k_glu_reduce) of columns k .. k + 7 of token tok.
template <uint32_t S>
__device__ __forceinline__ void glu_finish8(const float *part, uint32_t splits, uint32_t R, uint32_t batch, float *y,
                                            uint8_t *xs, int act, const DeferredNorm &dn, uint32_t tok, uint32_t k) {
  const uint64_t n = (uint64_t)2 * R * batch, row = (uint64_t)tok * 2 * R;
  const __amdgpu_buffer_rsrc_t rp = split_rsrc(part, splits, n);
  const uint32_t sb = (uint32_t)(4 * n), og = (uint32_t)(4 * (row + k)), ou = og + 4 * R;
  const float4 g0 = split_sum4<S>(rp, splits, sb, og), g1 = split_sum4<S>(rp, splits, sb, og + 16);
  const float4 u0 = split_sum4<S>(rp, splits, sb, ou), u1 = split_sum4<S>(rp, splits, sb, ou + 16);
  float g[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
  float u[8] = {u0.x, u0.y, u0.z, u0.w, u1.x, u1.y, u1.z, u1.w};
  if (dn.sq) {
    const float xinv = deferred_inv(dn, tok);
#pragma unroll
    for (int e = 0; e < 8; e++) { g[e] *= xinv; u[e] *= xinv; }
  }
  float v[8];
#pragma unroll
  for (int e = 0; e < 8; e++) v[e] = glu_act(g[e], act) * u[e];
  const float4 a = make_float4(v[0], v[1], v[2], v[3]), b = make_float4(v[4], v[5], v[6], v[7]);
  if (y) {
    *(float4 *)(y + (uint64_t)tok * R + k) = a;
    *(float4 *)(y + (uint64_t)tok * R + k + 4) = b;
  }
  split_store8(xs, R, tok, k, a, b);
}

// gate (rows [0, R)) and up (rows [R, 2R)) from the split-K partials, then act(gate) * up
// into y [batch][R] and its split form for the down GEMM: one thread per eight columns of a
// token. S >= splits.
//
// The GEMM's 128-row tile t ran on XCD t % 8 (its grid's first dimension, the tile count, is
// a multiple of 8, and workgroups go to the XCDs round-robin), and with R a multiple of 1024
// the up tile of a column has the gate tile's residue. (Of 256-row workgroups gemm_tile places whole groups
// of eight per matrix so; the runs of a last group of fewer, 8 of 168 at R = 21504, are read from other
// XCDs' partials.) Then (by_xcd) workgroup w, on XCD
// w % 8, takes token w / 8 and the columns of the tiles t = w (mod 8), reading only
// partials its XCD wrote: each 128-row run of the scratch stays with one XCD, and the next
// GEMM's writes to it take no coherence probes. Otherwise workgroup w takes 256
// consecutive column groups.
template <uint32_t S>
__global__ __launch_bounds__(256) void k_glu_reduce(const float *part, uint32_t splits, uint32_t R, uint32_t batch,
                                                    float *y, uint8_t *xs, int act, DeferredNorm dn, uint32_t by_xcd) {
  if (!by_xcd) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x, c8 = split_kblocks(R) * 16, tok = i / c8, k = (i % c8) * 8;
    if (tok < batch && k < R) glu_finish8<S>(part, splits, R, batch, y, xs, act, dn, tok, k);
    return;
  }
  const uint32_t x = blockIdx.x % 8, tok = blockIdx.x / 8;
  for (uint32_t j = threadIdx.x; j < R / 64; j += 256)
    glu_finish8<S>(part, splits, R, batch, y, xs, act, dn, tok, (x + 8 * (j / 16)) * 128 + (j % 16) * 8);
}

static bool qgemm_supported(const Matrix &w) {
  if (w.layout != LAYOUT_PLANAR) return false;
  if (w.type == Q4_K || w.type == Q5_K || w.type == Q6_K) return w.cols % 256 == 0;
  return (w.type == Q8_0 || w.type == Q4_0) && w.cols % QG_K == 0;
}

// The type pairs (t0 <= t1) with a grouped kernel: every type alone, and the mixes of real
// checkpoints (K-quant projections beside Q6_K or Q8_0 ones).
static bool qgemm_pair(int a, int b) {
  if (a == b) return true;
  return (a == Q4_K && b == Q6_K) || (a == Q8_0 && b == Q4_K) || (a == Q8_0 && b == Q6_K) ||
         (a == Q4_K && b == Q5_K) || (a == Q5_K && b == Q6_K);
}

// The launch's two weight types (t[0] <= t[1]); false for more than two.
static bool group_types(const GemmGroup &g, int t[2]) {
  t[0] = t[1] = -1;
  for (uint32_t j = 0; j < g.n; j++) {
    const int ty = g.job[j].w->type;
    if (ty == t[0] || ty == t[1]) continue;
    if (t[0] < 0) t[0] = ty;
    else if (t[1] < 0) t[1] = ty;
    else return false;
  }
  if (t[1] < 0) t[1] = t[0];
  if (t[0] > t[1]) std::swap(t[0], t[1]);
  return true;
}

bool gemm_group_ok(const GemmGroup &g, uint32_t batch) {
  if (!g.n || g.n > QG_MAX_JOBS || !batch) return false;
  for (uint32_t j = 0; j < g.n; j++)
    if (!g.job[j].w || !g.job[j].w->data || !qgemm_supported(*g.job[j].w) || g.job[j].w->cols != g.job[0].w->cols)
      return false;
  if (g.glu_out && (g.n != 2 || g.job[0].w->rows != g.job[1].w->rows || g.job[0].w->rows % QG_K)) return false;
  int t[2];
  return group_types(g, t) && qgemm_pair(t[0], t[1]);
}

// 16-token blocks of a workgroup: the smallest of 1, 2, 4 that covers the batch; past 64 tokens
// workgroups of 64 each. K-quant groups of one type whose 128-row tiles fill half the CUs or
// more take 8: workgroups of 256 rows x 128 tokens, which unpack each weight once (28672 x 4096 as one
// wgd_matmul over several matrices, 128 tokens: Q4_K 93.7 -> 88.2 us, Q6_K 131.5 -> 111.8; the model's
// gate + up 79). Shorter matrices need the smaller
// workgroups (4096 x 4096: 18.4 against 22.3), and the 32-column types the registers (Q8_0
// 100 against 122.5). Q6_K, whose two lo halves cost the most to unpack, takes 8 for shorter matrices
// too where their columns keep five units or more per workgroup: 100 tokens, 5376 x 21504 117 -> 94,
// 4096 x 14336 72 -> 62 (with 64 tokens both were slower than the former bf16 kernel's 111 and 70); at 5376 x
// 5376 (3.4 units) 39.7 against 38.7, at 4096 x 4096 (two) 28.9 against 30.8.
static uint32_t token_blocks(const GemmGroup &g, uint32_t batch) {
  if (batch <= 16) return 1;
  if (batch <= 64) return batch <= 32 ? 2 : 4;
  uint32_t tiles = 0, tall = 0;  // of 128 and of 256 rows
  const Matrix &w = *g.job[0].w;
  for (uint32_t j = 0; j < g.n; j++) {
    const int t = g.job[j].w->type;
    if (t != w.type || t == Q8_0 || t == Q4_0) return 4;
    tiles += (g.job[j].w->rows + QG_M - 1) / QG_M;
    tall += (g.job[j].w->rows + 2 * QG_M - 1) / (2 * QG_M);
  }
  const uint32_t cus = (uint32_t)device_cu_count();
  if (2 * tiles >= cus) return 8;
  return w.type == Q6_K && (uint64_t)tall * split_kblocks(w.cols) >= 5 * cus ? 8 : 4;
}

// K span per workgroup: splits until the launch fills its workgroup slots, each at least two units, and
// no more partial sums than the scratch holds.
static uint32_t group_kspan(const GemmGroup &g, uint32_t batch, uint64_t scratch_floats, uint32_t *rows_total) {
  // splits end on pairs of units, a K-quant's block, so the kernel knows at compile time which half
  // of a block a unit is
  const uint32_t align = 2 * QG_U, tb = token_blocks(g, batch);
  uint32_t tiles = 0, rows = 0;
  for (uint32_t j = 0; j < g.n; j++) {
    const Matrix &w = *g.job[j].w;
    tiles += (w.rows + qg_rows(tb) - 1) / qg_rows(tb);
    rows += w.rows;
  }
  tiles *= (batch + 16 * tb - 1) / (16 * tb);
  *rows_total = rows;
  // Up to 32 tokens, where the rows give at most half a workgroup per CU, the splits stop at one
  // workgroup (eight wavefronts) per CU: fewer partial sums, the same or less time (16 tokens: 4096 x
  // 4096 7.9 -> 7.0 us, 6144 x 4096 10.1 -> 8.8, 4096 x 14336 13.9 -> 13.6). Taller matrices would be left
  // with one long split (28672 x 4096: 22.2 us against 20.5 in two), 64 tokens with less to
  // overlap (4096 x 14336 31.8 against 28.8).
  const uint32_t cus = (uint32_t)device_cu_count(), cols = g.job[0].w->cols;
  const uint32_t target = tb == 8 || (tb <= 2 && 2 * tiles <= cus) ? cus : 2 * cus;  // 8: one fits a CU
  uint32_t splits = tiles >= target ? 1 : target / tiles;
  const uint32_t units = (cols + align - 1) / align;
  if (splits > units) splits = units;
  if (splits > 16) splits = 16;
  // The workgroups run in rounds of `target` slots, and a short last round leaves CUs idle
  // (336 gate/up tiles in one split fill 66% of one round). Up to twice the splits are
  // considered, and one that fills its rounds at least 10 points better is taken: 336 tiles
  // then run in 3 splits, 1008 workgroups in two rounds at 98%. The split count is
  // ceil(units / per) for the span per = ceil(units / s).
  auto workgroups = [&](uint32_t s) {
    const uint32_t per = (units + s - 1) / s;
    return (uint64_t)tiles * ((units + per - 1) / per);
  };
  auto rounds = [&](uint64_t wg) { return (wg + target - 1) / target; };
  uint64_t bw = workgroups(splits);
  const uint32_t s0 = splits;
  for (uint32_t s = s0 + 1; s <= 2 * s0 + 1 && s <= units && s <= 16; s++) {
    const uint64_t w = workgroups(s);
    // w / (rounds(w) T) > bw / (rounds(bw) T) + 0.1, times 10 rounds(w) rounds(bw) T
    if (10 * w * rounds(bw) > 10 * bw * rounds(w) + rounds(w) * rounds(bw) * target) { splits = s; bw = w; }
  }
  while (splits > 1 && (uint64_t)splits * batch * rows > scratch_floats) splits--;
  const uint32_t per = (units + splits - 1) / splits;
  return per * align;
}

uint64_t gemm_group_split_floats(const GemmGroup &g, uint32_t batch) {
  if (!gemm_group_ok(g, batch)) return 0;
  uint32_t rows = 0;
  const uint32_t kspan = group_kspan(g, batch, ~0ull, &rows);
  const uint32_t splits = (g.job[0].w->cols + kspan - 1) / kspan;
  // the GLU finish and a kept group read their partials whole, so they always have room
  return splits > 1 || g.glu_out || g.keep_partials ? (uint64_t)splits * batch * rows : 0;
}

uint64_t gemm_split_floats(const Matrix &w, uint32_t batch) {
  GemmGroup g;
  g.job[0].w = &w; g.n = 1;
  return gemm_group_split_floats(g, batch);
}

uint64_t gemm_input_bytes(uint32_t cols, uint32_t batch) {
  return (uint64_t)(batch + SPLIT_TOK - 1) / SPLIT_TOK * split_kblocks(cols) * (SPLIT_TOK / SPLIT_N) * SPLIT_BLOCK;
}

bool gemm_splits_input(const Matrix &w, const GemmScratch *scratch, uint32_t batch) {
  return qgemm_supported(w) && scratch && scratch->xs && scratch->xs_bytes >= gemm_input_bytes(w.cols, batch);
}

template <int T0, int T1, uint32_t TT>
static void launch_qgemm_tt(hipStream_t s, dim3 grid, const QGemm &q) {
  constexpr uint32_t S = qg_stage(T0, TT) > qg_stage(T1, TT) ? qg_stage(T0, TT) : qg_stage(T1, TT);
  constexpr uint32_t lds = 2 * S * TT * SPLIT_BLOCK;
  if (lds > 65536) lds_opt_in((const void *)k_gemm_q<T0, T1, TT>);
  hipLaunchKernelGGL((k_gemm_q<T0, T1, TT>), grid, dim3(qg_threads(TT)), lds, s, q);
}
template <int T0, int T1>
static void launch_qgemm(hipStream_t s, dim3 grid, uint32_t tb, const QGemm &q) {
  if constexpr (T0 == T1 && T0 != Q8_0 && T0 != Q4_0)
    if (tb == 8) return launch_qgemm_tt<T0, T1, 8>(s, grid, q);
  switch (tb) {
    case 1: return launch_qgemm_tt<T0, T1, 1>(s, grid, q);
    case 2: return launch_qgemm_tt<T0, T1, 2>(s, grid, q);
    default: return launch_qgemm_tt<T0, T1, 4>(s, grid, q);
  }
}

hipError_t gemm_group(hipStream_t s, const GemmGroup &g, const float *x, uint32_t batch, GemmScratch *scratch) {
  if (!batch) return hipSuccess;
  const uint32_t cols = g.job[0].w->cols;
  if (!gemm_group_ok(g, batch) || !scratch || !scratch->xs || scratch->xs_bytes < gemm_input_bytes(cols, batch) ||
      (uintptr_t)x % 16)
    return hipErrorInvalidValue;
  if (g.glu_out && (scratch->xs_bytes < gemm_input_bytes(g.job[0].w->rows, batch) || (uintptr_t)g.glu_out % 16))
    return hipErrorInvalidValue;
  if (scratch->xs_of != x || scratch->xs_cols != cols || scratch->xs_batch != batch) {
    const uint32_t count = batch * split_kblocks(cols) * 16;
    hipLaunchKernelGGL(k_gemm_split, dim3((count + 255) / 256), dim3(256), 0, s, x, scratch->xs, cols, count);
    WGD_HIP(hipGetLastError());
    scratch->xs_of = x; scratch->xs_cols = cols; scratch->xs_batch = batch;
  }
  int types[2];
  group_types(g, types);
  const uint32_t tb = token_blocks(g, batch);
  QGemm q{};
  q.njobs = g.n; q.xs = scratch->xs; q.cols = cols; q.batch = batch; q.accumulate = g.accumulate ? 1u : 0u;
  uint32_t tiles = 0, row0 = 0;
  for (uint32_t j = 0; j < g.n; j++) {
    const Matrix &w = *g.job[j].w;
    const uint64_t wbytes = planar_bytes(w.type, w.cols, w.rows);
    if (wbytes >= (1ull << 31)) return hipErrorInvalidValue;
    QJob &jb = q.job[j];
    jb.w = w.data; jb.wbytes = (uint32_t)wbytes;
    jb.C = w.cols / chunk_elems(w.type); jb.bpr = w.cols / block_size(w.type); jb.nbp = jb.bpr * (uint32_t)tile_rows(w.rows);
    jb.rows = w.rows; jb.tiles = (w.rows + qg_rows(tb) - 1) / qg_rows(tb); jb.off = tiles % 8; jb.kind = w.type == types[0] ? 0u : 1u; jb.row0 = row0;
    jb.y = g.job[j].y; jb.stride = g.job[j].stride; jb.row_base = g.job[j].row_base;
    tiles += jb.tiles; row0 += w.rows;
  }
  q.kspan = group_kspan(g, batch, scratch->p ? scratch->floats : 0, &q.rows_total);
  const uint32_t splits = (cols + q.kspan - 1) / q.kspan;
  // the GLU finish and a kept group always reduce from the partials (a single split too)
  const bool partials = splits > 1 || g.glu_out || g.keep_partials;
  if (partials && (!scratch->p || (uint64_t)splits * batch * q.rows_total > scratch->floats)) return hipErrorInvalidValue;
  // the finishes read the partials through 32-bit buffer offsets
  if (partials && (splits > MAX_SPLITS || (uint64_t)splits * batch * q.rows_total * 4 >= (1ull << 31)))
    return hipErrorInvalidValue;
  q.part = partials ? scratch->p : nullptr;
  const dim3 grid(tiles, (batch + 16 * tb - 1) / (16 * tb), splits);
  const int a = types[0], b = types[1];
  if (a == Q4_K && b == Q4_K) launch_qgemm<Q4_K, Q4_K>(s, grid, tb, q);
  else if (a == Q6_K && b == Q6_K) launch_qgemm<Q6_K, Q6_K>(s, grid, tb, q);
  else if (a == Q8_0 && b == Q8_0) launch_qgemm<Q8_0, Q8_0>(s, grid, tb, q);
  else if (a == Q4_K && b == Q6_K) launch_qgemm<Q4_K, Q6_K>(s, grid, tb, q);
  else if (a == Q8_0 && b == Q4_K) launch_qgemm<Q8_0, Q4_K>(s, grid, tb, q);
  else if (a == Q8_0 && b == Q6_K) launch_qgemm<Q8_0, Q6_K>(s, grid, tb, q);
  else if (a == Q5_K && b == Q5_K) launch_qgemm<Q5_K, Q5_K>(s, grid, tb, q);
  else if (a == Q4_0 && b == Q4_0) launch_qgemm<Q4_0, Q4_0>(s, grid, tb, q);
  else if (a == Q4_K && b == Q5_K) launch_qgemm<Q4_K, Q5_K>(s, grid, tb, q);
  else if (a == Q5_K && b == Q6_K) launch_qgemm<Q5_K, Q6_K>(s, grid, tb, q);
  else return hipErrorInvalidValue;
  WGD_HIP(hipGetLastError());
  if (g.glu_out) {
    const uint32_t R = g.job[0].w->rows, count = batch * split_kblocks(R) * 16;
    const uint32_t by_xcd = R % 1024 == 0 && tiles % 8 == 0 ? 1u : 0u;
    const dim3 grid(by_xcd ? batch * 8 : (count + 255) / 256);
    const float *part = q.part;
    float *y = g.glu_f32 ? g.glu_out : nullptr;
    if (splits <= 2)
      hipLaunchKernelGGL(k_glu_reduce<2>, grid, dim3(256), 0, s, part, splits, R, batch, y, scratch->xs, g.glu_act,
                         g.glu_norm, by_xcd);
    else if (splits <= 4)
      hipLaunchKernelGGL(k_glu_reduce<4>, grid, dim3(256), 0, s, part, splits, R, batch, y, scratch->xs, g.glu_act,
                         g.glu_norm, by_xcd);
    else
      hipLaunchKernelGGL(k_glu_reduce<MAX_SPLITS>, grid, dim3(256), 0, s, part, splits, R, batch, y, scratch->xs,
                         g.glu_act, g.glu_norm, by_xcd);
    WGD_HIP(hipGetLastError());
    scratch->xs_of = g.glu_out; scratch->xs_cols = R; scratch->xs_batch = batch;
  } else if (g.keep_partials) {
    if (g.splits) *g.splits = splits;
  } else if (splits > 1) {
    const uint64_t n = (uint64_t)q.rows_total * batch;
    uint32_t blocks = (uint32_t)((n + 255) / 256);
    if (blocks > 4096) blocks = 4096;
    if (splits <= 4) hipLaunchKernelGGL(k_gemm_reduce<4>, dim3(blocks), dim3(256), 0, s, q, splits);
    else hipLaunchKernelGGL(k_gemm_reduce<MAX_SPLITS>, dim3(blocks), dim3(256), 0, s, q, splits);
  }
  return hipGetLastError();
}

hipError_t gemm(hipStream_t s, const Matrix &w, const float *x, float *y, uint32_t stride,
                uint32_t row_base, uint32_t input_offset, uint32_t batch, GemmScratch *scratch, bool accumulate) {
  if (!w.rows || !batch) return hipSuccess;
  const float *xb = x + (uint64_t)input_offset * w.cols;
  if (gemm_splits_input(w, scratch, batch) && (uintptr_t)xb % 16 == 0) {
    GemmGroup g;
    g.job[0] = GemmJob{&w, y, stride, row_base};
    g.n = 1; g.accumulate = accumulate;
    return gemm_group(s, g, xb, batch, scratch);
  }
  if (accumulate) return hipErrorInvalidValue;  // only the planar-weight GEMM adds into y
  if (w.cols % KT) return hipErrorInvalidValue;
  GemmArgs a;
  a.w = w.data; a.type = w.type; a.layout = w.layout;
  a.rb = row_bytes(w.type, w.cols); a.bpr = w.cols / block_size(w.type);
  a.nbt = (uint64_t)a.bpr * (w.layout == LAYOUT_PLANAR ? tile_rows(w.rows) : w.rows);
  a.x = x; a.y = y; a.cols = w.cols; a.rows = w.rows; a.stride = stride; a.row_base = row_base;
  a.input_offset = input_offset; a.batch = batch;
  dim3 grid((w.rows + 63) / 64, (batch + NT - 1) / NT);
  hipLaunchKernelGGL(k_gemm, grid, dim3(256), 0, s, a);
  return hipGetLastError();
}

}  // namespace wgd
