// matmul's row path (quant.cpp:171-191 vec_dot, 330-351 matmul): the reference evaluates every output as one weight
// row (GGUF bytes, not repacked) dotted with one activation row. It runs for F32 / F16 / BF16 weights (they have no
// panels) and, with MALKIN_NO_PACK, for the quantized types too. Its arithmetic differs from the panel kernels, so it
// has its own kernel here, bit-identical to the AVX-512 row kernels (kernels_avx512.cpp:31-171):
//   a 16-lane group of a wave plays one 512-bit accumulator: lane l holds lane l of the reference's register and
//   runs its fma chain; the halving tree of _mm512_reduce_add_ps then combines the 16 lanes (shuffles 8, 4, 2, 1
//   apart); lane 0 finishes the scalar parts (the F types' k % 16 tail, Q8_0's odd last block, the K-quants' mins /
//   bias chains).
// A wave holds four groups, a workgroup sixteen: one weight row per group, NT tokens of it at once so that a row is read
// once per token tile. F32 / F16 / BF16 rows go to the matrix cores instead (k_rows_mfma) unless they are unaligned.
#include <algorithm>
#include <utility>

#include "ctx.h"
#include "ops.h"

namespace mk {
namespace {

constexpr int kRowsThreads = 256;
constexpr int kRowsNT = 8;  // tokens per group pass

__device__ __forceinline__ float bf16_to_float(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

__device__ __forceinline__ uint16_t ld_u16(const uint8_t* p) { return (uint16_t)(p[0] | (p[1] << 8)); }

// Four bytes at any alignment, as the little-endian int of four int8 values.
__device__ __forceinline__ int ld_i8x4(const uint8_t* p) {
  return (int)((uint32_t)p[0] | ((uint32_t)p[1] << 8) | ((uint32_t)p[2] << 16) | ((uint32_t)p[3] << 24));
}

// Sum over the 16 lanes of a group in the order of _mm512_reduce_add_ps (pairs 8, 4, 2, 1 apart); lane 0 holds it.
__device__ __forceinline__ float tree16(float v) {
  v = v + __shfl_down(v, 8, 16);
  v = v + __shfl_down(v, 4, 16);
  v = v + __shfl_down(v, 2, 16);
  v = v + __shfl_down(v, 1, 16);
  return v;
}

// kernels.h:18-26: the 6-bit scale and min of sub-block j from the 12 packed bytes.
__device__ __forceinline__ void scale_min_k4(int j, const uint8_t* q, int& sc, int& m) {
  if (j < 4) {
    sc = q[j] & 63;
    m = q[j + 4] & 63;
  } else {
    sc = (q[j + 4] & 0xF) | ((q[j - 4] >> 6) << 4);
    m = (q[j + 4] >> 4) | ((q[j] >> 6) << 4);
  }
}

__device__ __forceinline__ int xq_word(const BlockQ8& b, int g) { return reinterpret_cast<const int*>(b.qs)[g]; }

template <int TYPE>
__global__ __launch_bounds__(kRowsThreads) void k_rows(const uint8_t* __restrict__ W, size_t row_bytes, int64_t rows,
                                                       int64_t cols, const float* __restrict__ x, int64_t xs,
                                                       const BlockQ8* __restrict__ xq, int n, float* __restrict__ y,
                                                       int64_t ys, int accumulate) {
  const int lane = threadIdx.x & 15;
  const int64_t r = (int64_t)blockIdx.x * (kRowsThreads / 16) + threadIdx.x / 16;
  const int t0 = blockIdx.y * kRowsNT;
  if (r >= rows) return;  // a whole group leaves together: the shuffles below stay within live groups
  const int nt = min(kRowsNT, n - t0);
  const uint8_t* w = W + (size_t)r * row_bytes;
  const int64_t nb = cols / 32;
  float acc[kRowsNT], tail[kRowsNT];
#pragma unroll
  for (int t = 0; t < kRowsNT; ++t) acc[t] = 0.0f, tail[t] = 0.0f;

  if constexpr (TYPE == kF32 || TYPE == kF16 || TYPE == kBF16) {
    // kernels_avx512.cpp:82-107: lane l accumulates elements 16 i + l, then the tree, then the scalar tail.
    const int64_t full = cols / 16 * 16;
    for (int64_t i = lane; i < full; i += 16) {
      float wv;
      if constexpr (TYPE == kF32)
        wv = reinterpret_cast<const float*>(w)[i];
      else if constexpr (TYPE == kF16)
        wv = half_to_float(reinterpret_cast<const uint16_t*>(w)[i]);
      else
        wv = bf16_to_float(reinterpret_cast<const uint16_t*>(w)[i]);
#pragma unroll
      for (int t = 0; t < kRowsNT; ++t)
        if (t < nt) acc[t] = fma_(wv, x[(int64_t)(t0 + t) * xs + i], acc[t]);
    }
#pragma unroll
    for (int t = 0; t < kRowsNT; ++t) acc[t] = tree16(acc[t]);
    if (lane == 0)
      for (int64_t i = full; i < cols; ++i) {
        float wv;
        if constexpr (TYPE == kF32)
          wv = reinterpret_cast<const float*>(w)[i];
        else if constexpr (TYPE == kF16)
          wv = half_to_float(reinterpret_cast<const uint16_t*>(w)[i]);
        else
          wv = bf16_to_float(reinterpret_cast<const uint16_t*>(w)[i]);
#pragma unroll
        for (int t = 0; t < kRowsNT; ++t)
          if (t < nt) acc[t] = fma_(wv, x[(int64_t)(t0 + t) * xs + i], acc[t]);
      }
  } else if constexpr (TYPE == kQ8_0) {
    // kernels_avx512.cpp:110-137: block pairs, lane l = 4-byte group l % 8 of block 2p + l / 8.
    const int g = lane & 7;
    for (int64_t b0 = 0; b0 + 2 <= nb; b0 += 2) {
      const int64_t b = b0 + lane / 8;
      const uint8_t* blk = w + b * 34;
      const int wq = ld_i8x4(blk + 2 + 4 * g);
      const float dw = half_to_float(ld_u16(blk));
#pragma unroll
      for (int t = 0; t < kRowsNT; ++t)
        if (t < nt) {
          const BlockQ8& xb = xq[(int64_t)(t0 + t) * nb + b];
          acc[t] = fma_((float)dot4(wq, xq_word(xb, g), 0), dw * xb.d, acc[t]);
        }
    }
#pragma unroll
    for (int t = 0; t < kRowsNT; ++t) acc[t] = tree16(acc[t]);
    if ((nb & 1) && lane == 0) {
      const int64_t b = nb - 1;
      const uint8_t* blk = w + b * 34;
      const float dw = half_to_float(ld_u16(blk));
#pragma unroll
      for (int t = 0; t < kRowsNT; ++t)
        if (t < nt) {
          const BlockQ8& xb = xq[(int64_t)(t0 + t) * nb + b];
          int dp = 0;
          for (int e = 0; e < 8; ++e) dp = dot4(ld_i8x4(blk + 2 + 4 * e), xq_word(xb, e), dp);
          acc[t] = fma_((float)dp * dw, xb.d, acc[t]);
        }
    }
  } else if constexpr (TYPE == kQ4_K || TYPE == kQ5_K) {
    // kernels_avx512.cpp:31-64: per sub-block pair j, lanes 0-7 the 4-value groups of sub-block 2j (low nibbles),
    // lanes 8-15 those of 2j + 1 (high nibbles); Q5_K adds each value's high bit.
    constexpr bool kHigh = TYPE == kQ5_K;
    constexpr int kBytes = kHigh ? 176 : 144;
    const int hi = lane >> 3, g = lane & 7;
    for (int64_t sb = 0; sb < cols / 256; ++sb) {
      const uint8_t* s = w + sb * kBytes;
      const float d = half_to_float(ld_u16(s)), dmin = half_to_float(ld_u16(s + 2));
      const uint8_t* qh = s + 16;
      const uint8_t* q = s + (kHigh ? 48 : 16);
      for (int j = 0; j < 4; ++j, q += 32) {
        int s0, m0, s1, m1;
        scale_min_k4(2 * j, s + 4, s0, m0);
        scale_min_k4(2 * j + 1, s + 4, s1, m1);
        const uint32_t qw = (uint32_t)ld_i8x4(q + 4 * g);
        uint32_t v = hi ? (qw >> 4) & 0x0F0F0F0Fu : qw & 0x0F0F0F0Fu;
        if constexpr (kHigh) v |= (((uint32_t)ld_i8x4(qh + 4 * g) >> (2 * j + hi)) & 0x01010101u) << 4;
#pragma unroll
        for (int t = 0; t < kRowsNT; ++t)
          if (t < nt) {
            const BlockQ8* xb = xq + (int64_t)(t0 + t) * nb + sb * 8 + 2 * j;
            const BlockQ8& xh = xb[hi];
            const float sc = d * (float)(hi ? s1 : s0) * xh.d;
            acc[t] = fma_((float)dot4((int)v, xq_word(xh, g), 0), sc, acc[t]);
            // mins = fma(dmin, fma(m0 * dx0, S0, (m1 * dx1) * S1), mins): lane 0's copy is the one used
            const float in = fma_((float)m0 * xb[0].d, (float)(xb[0].s[0] + xb[0].s[1]),
                                  ((float)m1 * xb[1].d) * (float)(xb[1].s[0] + xb[1].s[1]));
            tail[t] = fma_(dmin, in, tail[t]);
          }
      }
    }
#pragma unroll
    for (int t = 0; t < kRowsNT; ++t) acc[t] = tree16(acc[t]) - tail[t];
  } else {  // kQ6_K
    // kernels_avx512.cpp:142-171: per 128-value half, two passes; in pass p lane l takes the 4-value group l % 8 of
    // the half's 32-value group 2 p + l / 8 (unsigned q) times sub-block scale 4 p + l / 4; bias restores q - 32.
    const int g = lane & 7;
    for (int64_t sb = 0; sb < cols / 256; ++sb) {
      const uint8_t* s = w + sb * 210;
      const float d = half_to_float(ld_u16(s + 208));
      for (int hf = 0; hf < 2; ++hf) {
        const uint8_t* ql = s + 64 * hf;
        const uint8_t* qh = s + 128 + 32 * hf;
        const int8_t* sc = reinterpret_cast<const int8_t*>(s + 192 + 8 * hf);
        const uint32_t l0 = (uint32_t)ld_i8x4(ql + 4 * g), l1 = (uint32_t)ld_i8x4(ql + 32 + 4 * g);
        const uint32_t hb = (uint32_t)ld_i8x4(qh + 4 * g);
        // 32-value groups 0..3 of the half: low nibbles of bytes 0-31 / 32-63, then their high nibbles
        const uint32_t q0 = (l0 & 0x0F0F0F0Fu) | ((hb & 0x03030303u) << 4);
        const uint32_t q1 = (l1 & 0x0F0F0F0Fu) | (((hb >> 2) & 0x03030303u) << 4);
        const uint32_t q2 = ((l0 >> 4) & 0x0F0F0F0Fu) | (((hb >> 4) & 0x03030303u) << 4);
        const uint32_t q3 = ((l1 >> 4) & 0x0F0F0F0Fu) | (((hb >> 6) & 0x03030303u) << 4);
        const int up = lane >> 3;  // 0: first 32-value group of the pass, 1: second
#pragma unroll
        for (int t = 0; t < kRowsNT; ++t)
          if (t < nt) {
            const BlockQ8* xb = xq + (int64_t)(t0 + t) * nb + sb * 8 + 4 * hf;
#pragma unroll
            for (int p = 0; p < 2; ++p) {
              const int grp = 2 * p + up;
              const uint32_t qv = p == 0 ? (up ? q1 : q0) : (up ? q3 : q2);
              const int dp = dot4((int)qv, xq_word(xb[grp], g), 0) * (int)sc[4 * p + lane / 4];
              acc[t] = fma_((float)dp, d * xb[grp].d, acc[t]);
            }
#pragma unroll
            for (int k = 0; k < 4; ++k)
              tail[t] = fma_(d * xb[k].d * 32.0f,
                             (float)((int)sc[2 * k] * xb[k].s[0] + (int)sc[2 * k + 1] * xb[k].s[1]), tail[t]);
          }
      }
    }
#pragma unroll
    for (int t = 0; t < kRowsNT; ++t) acc[t] = tree16(acc[t]) - tail[t];
  }
  if (lane == 0)
#pragma unroll
    for (int t = 0; t < kRowsNT; ++t)
      if (t < nt) {
        float* o = y + (int64_t)(t0 + t) * ys + r;
        *o = accumulate ? *o + acc[t] : acc[t];
      }
}

// The panel kernels' arithmetic for Q4_K / Q5_K (gemm_avx512.cpp:104-155 compact, 217-266 wide: the same sequence)
// read straight from GGUF rows: per output, per 32-value sub-block j in order, acc = fma(float(int dot), (d * sc) * dx,
// acc), then acc = fma(-(dmin * m), dx * (s0 + s1), acc). An 8-lane group owns one row: lane g takes the 4-value
// group g of each sub-block, the exact int dot is summed over the group (butterfly), and every lane keeps the same
// chain. Q5_K weights have no CDNA layout and are read this way; rows that are not 16-byte aligned take this kernel, all
// others the two below it (k_gguf45_gemv, and gemm_kq.hip's Q5_K form).
template <bool kHigh>
__global__ __launch_bounds__(kRowsThreads) void k_gguf45(const uint8_t* __restrict__ W, size_t row_bytes, int64_t rows,
                                                         int64_t cols, const BlockQ8* __restrict__ xq, int n,
                                                         float* __restrict__ y, int64_t ys, int accumulate) {
  constexpr int kBytes = kHigh ? 176 : 144;
  const int g = threadIdx.x & 7;
  const int64_t r = (int64_t)blockIdx.x * (kRowsThreads / 8) + threadIdx.x / 8;
  const int t0 = blockIdx.y * kRowsNT;
  if (r >= rows) return;  // whole 8-lane groups leave together
  const int nt = min(kRowsNT, n - t0);
  const uint8_t* w = W + (size_t)r * row_bytes;
  const int64_t nb = cols / 32;
  float acc[kRowsNT];
#pragma unroll
  for (int t = 0; t < kRowsNT; ++t) acc[t] = 0.0f;
  for (int64_t sb = 0; sb < cols / 256; ++sb) {
    const uint8_t* s = w + sb * kBytes;
    const float d = half_to_float(ld_u16(s)), dmin = half_to_float(ld_u16(s + 2));
    const uint32_t qh = kHigh ? (uint32_t)ld_i8x4(s + 16 + 4 * g) : 0u;
    for (int j = 0; j < 8; ++j) {
      int sc, m;
      scale_min_k4(j, s + 4, sc, m);
      const float fsc = d * (float)sc, fmn = dmin * (float)m;
      const uint32_t qw = (uint32_t)ld_i8x4(s + (kHigh ? 48 : 16) + 32 * (j / 2) + 4 * g);
      uint32_t v = (j & 1) ? (qw >> 4) & 0x0F0F0F0Fu : qw & 0x0F0F0F0Fu;
      if constexpr (kHigh) v |= ((qh >> j) & 0x01010101u) << 4;
#pragma unroll
      for (int t = 0; t < kRowsNT; ++t)
        if (t < nt) {
          const BlockQ8& xb = xq[(int64_t)(t0 + t) * nb + sb * 8 + j];
          int ai = dot4((int)v, xq_word(xb, g), 0);
          ai += __shfl_xor(ai, 1, 8);
          ai += __shfl_xor(ai, 2, 8);
          ai += __shfl_xor(ai, 4, 8);
          const float dsx = xb.d * (float)(xb.s[0] + xb.s[1]);
          acc[t] = fma_((float)ai, fsc * xb.d, acc[t]);
          acc[t] = fma_(-fmn, dsx, acc[t]);
        }
    }
  }
  if (g == 0)
#pragma unroll
    for (int t = 0; t < kRowsNT; ++t)
      if (t < nt) {
        float* o = y + (int64_t)(t0 + t) * ys + r;
        *o = accumulate ? *o + acc[t] : acc[t];
      }
}

// The same arithmetic for up to NT tokens per pass with 16 lanes per row: lane l takes sub-block l % 8 of super-block
// 2 p + l / 8 whole (16-byte loads, its exact int dot in one lane), so a pass forms the terms of 16 consecutive
// sub-blocks and the row's chain then runs through them in order, every lane alike, one operand broadcast by the fma's
// DPP. The next pass's row bytes and activations are loaded while this one runs. What bounds it: the vector work of a
// pass (about 150 instructions per 4 rows x 512 weights, 1408 bytes) and, with few rows, the chain's 32 dependent
// fmas. Measured against the byte-wise kernel above (8 lanes per row, the dot summed across lanes per sub-block): Q5_K
// 2560 x 9728 at one token 141 -> 9.7 us, 19456 x 2560 71 -> 10.9 (weights in the Infinity Cache; 10.8 and 12.0 between a
// layer's other matmuls); 2560 x 9728 at 4 tokens 342 -> 26. Q4_K takes it at any count of
// tokens: 1024 x 3072 at one 44 -> 3.8 us, at 300 218 -> 92, at 512 293 -> 148; 2560 x 9728 at 300 1572 -> 609; 19456 x 2560 at
// 128 1072 -> 589.
template <bool kHigh, int NT>
__global__ __launch_bounds__(kRowsThreads) void k_gguf45_gemv(const uint8_t* __restrict__ W, size_t row_bytes,
                                                              int64_t rows, int64_t cols,
                                                              const BlockQ8* __restrict__ xq, int n,
                                                              float* __restrict__ y, int64_t ys, int accumulate) {
  constexpr int kBytes = kHigh ? 176 : 144;
  const int l = threadIdx.x & 15, j = l & 7;
  const int64_t r = (int64_t)blockIdx.x * (kRowsThreads / 16) + threadIdx.x / 16;
  const int t0 = blockIdx.y * NT;
  const int nsb = (int)(cols / 256), passes = (nsb + 1) / 2;
  const uint8_t* w = W + (size_t)min(r, rows - 1) * row_bytes;
  const int64_t nb = cols / 32;
  struct Pass {
    uint4 hd, qh[kHigh ? 2 : 1], qs[2];
    uint2 x[NT][5];
  };
  // Never predicated: past the last super-block (or token) the last one again, unused.
  auto load = [&](Pass& P, int p) __attribute__((always_inline)) {
    const int sb = min(2 * p + (l >> 3), nsb - 1);
    const uint8_t* s = w + (size_t)sb * kBytes;
    P.hd = *reinterpret_cast<const uint4*>(s);
    if constexpr (kHigh) {
      P.qh[0] = *reinterpret_cast<const uint4*>(s + 16);
      P.qh[1] = *reinterpret_cast<const uint4*>(s + 32);
    }
    const uint8_t* q = s + (kHigh ? 48 : 16) + 32 * (j >> 1);
    P.qs[0] = *reinterpret_cast<const uint4*>(q);
    P.qs[1] = *reinterpret_cast<const uint4*>(q + 16);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const uint2* xb = reinterpret_cast<const uint2*>(xq + (int64_t)min(t0 + t, n - 1) * nb + (int64_t)sb * 8 + j);
#pragma unroll
      for (int k = 0; k < 5; ++k) P.x[t][k] = xb[k];
    }
  };
  float acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = 0.0f;
  auto run = [&](const Pass& P, bool second) __attribute__((always_inline)) {
    const float d = half_to_float((uint16_t)(P.hd.x & 0xFFFF)), dmin = half_to_float((uint16_t)(P.hd.x >> 16));
    // scale_min_k4 of sub-block j: the low four take 6 bits of words 1 and 2, the high four nibbles of word 3 and the
    // top bits of those
    const int sh = 8 * (j & 3);
    const uint32_t b1 = P.hd.y >> sh, b2 = P.hd.z >> sh, b3 = P.hd.w >> sh;
    const uint32_t sc = j < 4 ? b1 & 63u : (b3 & 15u) | ((b1 >> 2) & 0x30u);
    const uint32_t mn = j < 4 ? b2 & 63u : ((b3 >> 4) & 15u) | ((b2 >> 2) & 0x30u);
    const float fsc = d * (float)sc, nmn = -(dmin * (float)mn);
    const uint32_t q[8] = {P.qs[0].x, P.qs[0].y, P.qs[0].z, P.qs[0].w, P.qs[1].x, P.qs[1].y, P.qs[1].z, P.qs[1].w};
    int v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      v[k] = (int)((q[k] >> (4 * (j & 1))) & 0x0F0F0F0Fu);
      if constexpr (kHigh) {
        const uint32_t hb = k < 4 ? (&P.qh[0].x)[k] : (&P.qh[1].x)[k - 4];
        v[k] |= (int)(((hb >> j) & 0x01010101u) << 4);
      }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      int ai = 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        ai = dot4(v[2 * k], (int)P.x[t][k + 1].x, ai);
        ai = dot4(v[2 * k + 1], (int)P.x[t][k + 1].y, ai);
      }
      const float dx = __uint_as_float(P.x[t][0].x);
      const uint32_t sw = P.x[t][0].y;
      const float e0 = (float)ai, e1 = fsc * dx, e3 = dx * (float)((int)(int16_t)(sw & 0xFFFF) + (int)(int16_t)(sw >> 16));
      [&]<int... K>(std::integer_sequence<int, K...>) __attribute__((always_inline)) {
        ((acc[t] = fma_bcast16<K>(e0, bcast16(e1, K), acc[t]), acc[t] = fma_bcast16<K>(nmn, bcast16(e3, K), acc[t])), ...);
        if (second)
          ((acc[t] = fma_bcast16<K + 8>(e0, bcast16(e1, K + 8), acc[t]),
            acc[t] = fma_bcast16<K + 8>(nmn, bcast16(e3, K + 8), acc[t])),
           ...);
      }(std::make_integer_sequence<int, 8>{});
    }
  };
  Pass A, B;
  load(A, 0);
  for (int p = 0; p < passes; p += 2) {
    load(B, min(p + 1, passes - 1));
    run(A, 2 * p + 1 < nsb);
    if (p + 1 >= passes) break;
    load(A, min(p + 2, passes - 1));
    run(B, 2 * p + 3 < nsb);
  }
  if (l == 0 && r < rows)
#pragma unroll
    for (int t = 0; t < NT; ++t)
      if (t0 + t < n) {
        float* o = y + (int64_t)(t0 + t) * ys + r;
        *o = accumulate ? *o + acc[t] : acc[t];
      }
}

// F32 / F16 / BF16 rows on the matrix cores. v_mfma_f32_16x16x4_f32 runs each output element as four fmas in
// ascending k, each rounded once (measured bit for bit against fmaf over normal, denormal, infinite and signed-zero
// operands), so one instruction advances a lane chain of kernels_avx512.cpp:82-107 by four steps for 16 rows x 16
// tokens. Chain l takes elements 16 c + l: MFMA k index q is chunk c + q, so a lane that reads four consecutive values
// of chunk c + lane / 16 holds the operands of four chains.
//
// A workgroup owns 16 RT rows by 16 TT tokens and walks K in stages of KS steps of 64 columns, held in a ring of NS LDS
// buffers that direct global -> LDS copies fill NS - 1 stages ahead (16-byte pieces: lanes reading their operands
// straight from global memory touch 64 separate 64-byte segments per load, which bound the kernel at 60 TFLOP/s).
// Wave w runs chains 4 w .. 4 w + 3 of all the outputs; the halving tree then joins the waves' chains through LDS.
// The pieces of a row are stored rotated (xor) so that the 16 rows of a read fall on different banks.
// What bounds it: for prompts the fp32 matrix rate (153 TFLOP/s measured on a large product), for a few tokens the
// stream of weights. Measured in
// BF16, one 16-lane group per row with scalar loads (k_rows) -> this: 19456 x 2560 at 256 tokens 4858 -> 291 us, at one
// 110 -> 23; 1024 x 3072 at 96 166 -> 14.
typedef float f4 __attribute__((ext_vector_type(4)));

template <int TYPE>
__device__ __forceinline__ void row_floats(const uint8_t* p, float (&v)[4]) {  // four consecutive weights
  if constexpr (TYPE == kF32) {
    const float4 f = *reinterpret_cast<const float4*>(p);
    v[0] = f.x, v[1] = f.y, v[2] = f.z, v[3] = f.w;
  } else {
    const uint2 u = *reinterpret_cast<const uint2*>(p);
    if constexpr (TYPE == kF16) {
      v[0] = half_to_float((uint16_t)(u.x & 0xFFFF)), v[1] = half_to_float((uint16_t)(u.x >> 16));
      v[2] = half_to_float((uint16_t)(u.y & 0xFFFF)), v[3] = half_to_float((uint16_t)(u.y >> 16));
    } else {
      v[0] = __uint_as_float(u.x << 16), v[1] = __uint_as_float(u.x & 0xFFFF0000u);
      v[2] = __uint_as_float(u.y << 16), v[3] = __uint_as_float(u.y & 0xFFFF0000u);
    }
  }
}
template <int TYPE>
__device__ __forceinline__ float row_value(const uint8_t* w, int64_t i) {
  if constexpr (TYPE == kF32)
    return reinterpret_cast<const float*>(w)[i];
  else if constexpr (TYPE == kF16)
    return half_to_float(reinterpret_cast<const uint16_t*>(w)[i]);
  else
    return bf16_to_float(reinterpret_cast<const uint16_t*>(w)[i]);
}

// TN: tokens staged per token tile (fewer than 16 for a few tokens; lanes past them repeat them, unused).
template <int TYPE, int RT, int TT, int TN, int KS, int NS>
struct RowTile {
  static constexpr int elem = TYPE == kF32 ? 4 : 2;
  static constexpr int wp = 64 * elem / 16;            // 16-byte pieces of a row per step
  static constexpr int toks = TN * TT;
  static constexpr int xpieces = toks * 16, pieces = xpieces + 16 * RT * wp;  // per step: x, then weights
  static constexpr int loads = KS * pieces / 256;      // copies per wave and stage
  static_assert(KS * pieces % 256 == 0 && xpieces % 64 == 0 && (TN == 16 || TT == 1), "whole copies per wave");
  static constexpr int stage = KS * pieces * 16;       // bytes
  static constexpr int part = 2 * 4 * RT * TT * 64 * 16;  // the tree's exchange, after the last stage
  static constexpr int lds = NS * stage > part ? NS * stage : part;
};

template <int TYPE, int RT, int TT, int TN, int KS, int NS>
__global__ __launch_bounds__(kRowsThreads) __attribute__((amdgpu_waves_per_eu(RT * TT == 4 ? 3 : 4))) void k_rows_mfma(const uint8_t* W, size_t row_bytes, int64_t rows,
                                                            int64_t cols, const float* x, int64_t xs, int n,
                                                            float* __restrict__ y, int64_t ys, int accumulate,
                                                            int n_tt, int tiles) {
  using T = RowTile<TYPE, RT, TT, TN, KS, NS>;
  extern __shared__ __align__(16) uint8_t smem[];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), i = lane & 15, q = lane >> 4;
  const int tile = xcd_run((int)blockIdx.x, tiles);  // token tiles of a row tile on one XCD: its rows are read once
  const int64_t r0 = (int64_t)(tile / n_tt) * (16 * RT);
  const int t0 = (tile % n_tt) * (16 * TT);
  const int chunks = (int)(cols / 16), nstages = (chunks + 4 * KS - 1) / (4 * KS);

  // This lane's copies: piece g of the stage comes from chunk cc[j] of the stage (clamped to the last chunk), at
  // src[j] plus whole chunks.
  const uint8_t* src[T::loads];
  int cc[T::loads];
#pragma unroll
  for (int j = 0; j < T::loads; ++j) {
    const int g0 = (w * T::loads + j) * 64, ks = g0 / T::pieces, g = g0 % T::pieces + lane;
    if (g0 % T::pieces < T::xpieces) {
      const int tok = g / 16, p = (g % 16) ^ (tok & 15);
      cc[j] = 4 * ks + p / 4;
      src[j] = reinterpret_cast<const uint8_t*>(x + (int64_t)min(t0 + tok, n - 1) * xs) + 16 * (p % 4);
    } else {
      const int h = g - T::xpieces, row = h / T::wp;
      const int p = (h % T::wp) ^ (T::wp == 16 ? row & 15 : (row >> 1) & 7);
      constexpr int pc = T::wp / 4;  // pieces per chunk
      cc[j] = 4 * ks + p / pc;
      src[j] = W + (size_t)min(r0 + row, rows - 1) * row_bytes + 16 * (p % pc);
    }
  }
  auto issue = [&](int st, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < T::loads; ++j) {
      const int g0 = (w * T::loads + j) * 64;
      const int bytes = g0 % T::pieces < T::xpieces ? 64 : 16 * T::elem;  // per chunk
      lds_copy16(src[j] + (size_t)min(4 * KS * st + cc[j], chunks - 1) * bytes, smem + buf * T::stage + g0 * 16);
    }
  };
  f4 acc[4][RT][TT];
#pragma unroll
  for (int e = 0; e < 4; ++e)
#pragma unroll
    for (int a = 0; a < RT; ++a)
#pragma unroll
      for (int b = 0; b < TT; ++b) acc[e][a][b] = f4{0.0f, 0.0f, 0.0f, 0.0f};
  auto step = [&](const uint8_t* sp, int s) __attribute__((always_inline)) {
    float wv[RT][4], xv[TT][4];
#pragma unroll
    for (int b = 0; b < TT; ++b) {
      const int tok = 16 * b + i % TN;
      const float4 f = *reinterpret_cast<const float4*>(sp + (tok * 16 + ((4 * q + w) ^ (tok & 15))) * 16);
      xv[b][0] = f.x, xv[b][1] = f.y, xv[b][2] = f.z, xv[b][3] = f.w;
    }
#pragma unroll
    for (int a = 0; a < RT; ++a) {
      const int row = 16 * a + i;
      const uint8_t* wr = sp + (T::xpieces + row * T::wp) * 16;
      if constexpr (T::wp == 16)
        row_floats<TYPE>(wr + ((4 * q + w) ^ (row & 15)) * 16, wv[a]);
      else
        row_floats<TYPE>(wr + ((2 * q + (w >> 1)) ^ ((row >> 1) & 7)) * 16 + 8 * (w & 1), wv[a]);
    }
    if (4 * s + 4 > chunks) {  // chunks past the last: fma(-0, 0, acc) == acc for every acc, -0 too
      const bool in = 4 * s + q < chunks;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
#pragma unroll
        for (int a = 0; a < RT; ++a) wv[a][e] = in ? wv[a][e] : 0.0f;
#pragma unroll
        for (int b = 0; b < TT; ++b) xv[b][e] = in ? xv[b][e] : -0.0f;
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int a = 0; a < RT; ++a)
#pragma unroll
        for (int b = 0; b < TT; ++b)
          acc[e][a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[b][e], wv[a][e], acc[e][a][b], 0, 0, 0);
  };
  for (int st = 0; st < NS - 1 && st < nstages; ++st) issue(st, st);
  int buf = 0;
  for (int st = 0; st < nstages; ++st) {
    // Stage st has landed once at most the copies of the stages after it are outstanding; the buffer that stage
    // st + NS - 1 goes into was read in stage st - 1, finished by every wave before this barrier.
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    wait_vm_stages<T::loads, NS - 2>(min(NS - 2, nstages - 1 - st));
    ring_barrier();
    if (st + NS - 1 < nstages) issue(st + NS - 1, buf == 0 ? NS - 1 : buf - 1);
    const uint8_t* sp = smem + buf * T::stage;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) step(sp + ks * T::pieces * 16, KS * st + ks);
    buf = buf == NS - 1 ? 0 : buf + 1;
  }
  __syncthreads();  // the ring becomes the tree's exchange
  f4(*part)[4][RT * TT][64] = reinterpret_cast<f4(*)[4][RT * TT][64]>(smem);

  // The halving tree over chains 4 w + e: pairs 8 apart are waves w and w + 2, pairs 4 apart waves 0 and 1, pairs 2 and
  // 1 apart chains of one wave.
  auto put = [&](int slot) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int a = 0; a < RT; ++a)
#pragma unroll
        for (int b = 0; b < TT; ++b) part[slot][e][a * TT + b][lane] = acc[e][a][b];
  };
  auto add = [&](int slot) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int a = 0; a < RT; ++a)
#pragma unroll
        for (int b = 0; b < TT; ++b) acc[e][a][b] = acc[e][a][b] + part[slot][e][a * TT + b][lane];
  };
  if (w >= 2) put(w - 2);
  __syncthreads();
  if (w < 2) add(w);
  if (w == 1) put(1);  // this wave's own slot, which only it has read
  __syncthreads();
  if (w != 0) return;
  add(1);
#pragma unroll
  for (int a = 0; a < RT; ++a)
#pragma unroll
    for (int b = 0; b < TT; ++b) {
      const int64_t r = r0 + 16 * a + i;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int t = t0 + 16 * b + 4 * q + j;
        if (r >= rows || t >= n) continue;
        float v = (acc[0][a][b][j] + acc[2][a][b][j]) + (acc[1][a][b][j] + acc[3][a][b][j]);
        for (int64_t k = 16 * (int64_t)chunks; k < cols; ++k)  // the scalar tail of k % 16 columns
          v = fma_(row_value<TYPE>(W + (size_t)r * row_bytes, k), x[(int64_t)t * xs + k], v);
        float* o = y + (int64_t)t * ys + r;
        *o = accumulate ? *o + v : v;
      }
    }
}

// Tile rule: the largest tile that still gives the chip enough workgroups (a 32 x 32 tile runs at 75-88 TFLOP/s from
// about four workgroups per CU, but at 12-30 below one). Measured in BF16, 16x16 / 16 rows x 32 tokens / 32x32, us:
// 19456 x 2560 at 256 tokens 368 / 321 / 291 (4864 32 x 32 tiles), 6144 x 1024 at 96 22.6 / 21.3 / 22.6 (576), 2560 x 9728
// at 96 72 / 67 / 67 (240; 480 tiles of 16 x 32), at 48 38 / 63 / 65 (160; 320), 1024 x 3072 at 96 14 / 16 / 23 (96).
// Up to 4 tokens only 4 token rows are staged: 19456 x 2560 at one token 38 (16 rows staged) -> 23 us, 4.4 TB/s; with
// no more workgroups than CUs stages twice as long (2560 x 9728: 21.9 -> 18.9 us).
template <int TYPE>
void launch_rows_mfma(hipStream_t s, const uint8_t* w, size_t row_bytes, int64_t rows, int64_t cols, const float* x,
                      int64_t xs, int n, float* y, int64_t ys, bool accumulate) {
  auto tiles = [&](int rt, int tt) { return (rows + 16 * rt - 1) / (16 * rt) * ((n + 16 * tt - 1) / (16 * tt)); };
  auto go = [&]<int RT, int TT, int TN, int KS, int NS>() {
    constexpr int lds = RowTile<TYPE, RT, TT, TN, KS, NS>::lds;
    static_assert(lds <= 65536, "dynamic LDS without an attribute");
    hipLaunchKernelGGL((k_rows_mfma<TYPE, RT, TT, TN, KS, NS>), dim3((unsigned)tiles(RT, TT)), dim3(kRowsThreads), lds, s,
                       w, row_bytes, rows, cols, x, xs, n, y, ys, accumulate ? 1 : 0, (n + 16 * TT - 1) / (16 * TT),
                       (int)tiles(RT, TT));
  };
  constexpr bool f32 = TYPE == kF32;
  const int64_t cus = device_cus();
  if (n <= 4) {
    if (tiles(1, 1) > cus)
      go.template operator()<1, 1, 4, 4, 2>();
    else if constexpr (f32)
      go.template operator()<1, 1, 4, 4, 3>();
    else
      go.template operator()<1, 1, 4, 8, 2>();
  } else if (n > 16 && tiles(2, 2) >= 4 * cus) {
    go.template operator()<2, 2, 16, 2, 2>();
  } else if (n > 16 && 4 * tiles(1, 2) >= 7 * cus) {
    go.template operator()<1, 2, 16, 2, 2>();
  } else {
    go.template operator()<1, 1, 16, 4, 2>();
  }
}

// The MFMA form's copies: whole 16-byte pieces of aligned rows; at least one 16-value chunk.
bool rows_mfma_ok(int type, const void* w, size_t row_bytes, int64_t rows, int64_t cols, const float* x, int64_t xs,
                  int n) {
  return (type == kF32 || type == kF16 || type == kBF16) && cols >= 16 && (uintptr_t)w % 16 == 0 &&
         row_bytes % 16 == 0 && (uintptr_t)x % 16 == 0 && xs % 4 == 0 &&
         (rows + 15) / 16 * ((n + 15) / 16) < INT32_MAX;
}

}  // namespace

bool rows_supported(int type, int64_t cols) {
  switch (type) {
    case kF32:
    case kF16:
    case kBF16:
      return cols > 0;
    case kQ8_0:
      return cols > 0 && cols % 32 == 0;
    case kQ4_K:
    case kQ5_K:
    case kQ6_K:
      return cols > 0 && cols % 256 == 0;
    default:
      return false;
  }
}

void matmul_rows(hipStream_t s, int type, const void* w, size_t row_bytes, int64_t rows, int64_t cols, const float* x,
                 int64_t xs, const BlockQ8* xq, int n, float* y, int64_t ys, bool accumulate) {
  require(rows_supported(type, cols), "matmul_rows: type / width without a row kernel");
  if (rows <= 0 || n <= 0) return;
  const bool f = type == kF32 || type == kF16 || type == kBF16;
  require(f ? x != nullptr : xq != nullptr, "matmul_rows: missing activations (fp32 for F32/F16/BF16, BlockQ8 else)");
  if (rows_mfma_ok(type, w, row_bytes, rows, cols, x, xs, n)) {
    // A launch has less than 2^32 threads, 2^24 workgroups here; a batch that large runs in 32 x 32 tiles.
    const int64_t most = ((int64_t)1 << 24) - 1, row_tiles = (rows + 31) / 32, per = 32 * std::max<int64_t>(1, most / row_tiles);
    if (n > per) {
      matmul_rows(s, type, w, row_bytes, rows, cols, x, xs, xq, (int)per, y, ys, accumulate);
      matmul_rows(s, type, w, row_bytes, rows, cols, x + per * xs, xs, xq, n - (int)per, y + per * ys, ys, accumulate);
      return;
    }
    auto* wb = static_cast<const uint8_t*>(w);
    if (type == kF32)
      launch_rows_mfma<kF32>(s, wb, row_bytes, rows, cols, x, xs, n, y, ys, accumulate);
    else if (type == kF16)
      launch_rows_mfma<kF16>(s, wb, row_bytes, rows, cols, x, xs, n, y, ys, accumulate);
    else
      launch_rows_mfma<kBF16>(s, wb, row_bytes, rows, cols, x, xs, n, y, ys, accumulate);
    check_launch("matmul_rows");
    return;
  }
  const dim3 grid((unsigned)((rows + kRowsThreads / 16 - 1) / (kRowsThreads / 16)), (unsigned)((n + kRowsNT - 1) / kRowsNT));
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, dim3(kRowsThreads), 0, s, static_cast<const uint8_t*>(w), row_bytes, rows, cols, x,
                       xs, xq, n, y, ys, accumulate ? 1 : 0);
  };
  switch (type) {
    case kF32: go(k_rows<kF32>); break;
    case kF16: go(k_rows<kF16>); break;
    case kBF16: go(k_rows<kBF16>); break;
    case kQ8_0: go(k_rows<kQ8_0>); break;
    case kQ4_K: go(k_rows<kQ4_K>); break;
    case kQ5_K: go(k_rows<kQ5_K>); break;
    default: go(k_rows<kQ6_K>); break;
  }
  check_launch("matmul_rows");
}

void matmul_gguf(hipStream_t s, int type, const void* w, size_t row_bytes, int64_t rows, int64_t cols,
                 const BlockQ8* xq, int n, float* y, int64_t ys, bool accumulate) {
  require((type == kQ4_K || type == kQ5_K) && cols > 0 && cols % 256 == 0,
          "matmul_gguf: Q4_K / Q5_K rows of a multiple of 256 values");
  require(xq != nullptr, "matmul_gguf: missing activations");
  if (rows <= 0 || n <= 0) return;
  if (const int most = 1 << 17; n > most) {  // a grid has at most 65536 groups of tokens
    matmul_gguf(s, type, w, row_bytes, rows, cols, xq, most, y, ys, accumulate);
    matmul_gguf(s, type, w, row_bytes, rows, cols, xq + most * (cols / 32), n - most, y + most * ys, ys, accumulate);
    return;
  }
  if (row_bytes % 16 == 0 && (uintptr_t)w % 16 == 0) {
    // Q5_K batches: the GEMV's waves (4 rows each, a group of 4 tokens) cost about 0.85 us per pass of 512 columns and
    // wave of a SIMD, the MFMA kernel about 3.1 us per 512 columns whatever the batch (up to 32 tokens), so it takes
    // over past 3.6 waves per SIMD, i.e. 58 rows x groups per CU. Measured, GEMV / MFMA: 2560 x 9728 at 16 tokens 52 / 60
    // us, at 24 68 / 68; 19456 x 2560 at 2 tokens 16 / 19, at 4 27 / 19; 5120 x 13824 at 8 70 / 79, at 12 95 / 82;
    // 1024 x 3072 at 32 15 / 25, at 64 27 / 25; 27648 x 5120 at one token 28 / 35.
    if (type == kQ5_K && n > 2 && rows * ((n + 3) / 4) > 58 * (int64_t)device_cus()) {
      gemm_q5_gguf(s, w, row_bytes, rows, cols, xq, n, y, ys, accumulate);
      return;
    }
    auto gemv = [&](auto kern, int nt) {
      const dim3 grid((unsigned)((rows + kRowsThreads / 16 - 1) / (kRowsThreads / 16)), (unsigned)((n + nt - 1) / nt));
      hipLaunchKernelGGL(kern, grid, dim3(kRowsThreads), 0, s, static_cast<const uint8_t*>(w), row_bytes, rows, cols,
                         xq, n, y, ys, accumulate ? 1 : 0);
    };
    if (n == 1)
      type == kQ5_K ? gemv(k_gguf45_gemv<true, 1>, 1) : gemv(k_gguf45_gemv<false, 1>, 1);
    else if (n == 2)
      type == kQ5_K ? gemv(k_gguf45_gemv<true, 2>, 2) : gemv(k_gguf45_gemv<false, 2>, 2);
    else
      type == kQ5_K ? gemv(k_gguf45_gemv<true, 4>, 4) : gemv(k_gguf45_gemv<false, 4>, 4);
    check_launch("matmul_gguf");
    return;
  }
  const dim3 grid((unsigned)((rows + kRowsThreads / 8 - 1) / (kRowsThreads / 8)), (unsigned)((n + kRowsNT - 1) / kRowsNT));
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, dim3(kRowsThreads), 0, s, static_cast<const uint8_t*>(w), row_bytes, rows, cols, xq,
                       n, y, ys, accumulate ? 1 : 0);
  };
  if (type == kQ5_K)
    go(k_gguf45<true>);
  else
    go(k_gguf45<false>);
  check_launch("matmul_gguf");
}

}  // namespace mk
