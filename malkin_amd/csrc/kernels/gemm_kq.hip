// Prefill / batch GEMM for K-quant weights (Q4_K, Q6_K, and Q5_K from its GGUF rows) on int8 MFMA, bit-identical to the reference's panel kernels:
//   Q4_K, Q5_K (gemm_avx512.cpp:104-155, the wide panels use the same arithmetic), per 32-weight sub-block j in order:
//     acc = fma(float(sum q4 x), (d sc_j) dx, acc);  acc = fma(-(dmin m_j), dx (s0 + s1), acc)
//   Q6_K compact (gemm_avx512.cpp:157-205), per 16-value half h in order:
//     acc = fma(float(sum (q6 - 32) x), (d sc_h) dx, acc)
//   Q6_K wide (gemm_avx512.cpp:268-316; n > 16 unless MALKIN_NO_WIDE), per 32-weight block b in order:
//     s = fma(float(ai1), d sc_2b+1, float(ai0) (d sc_2b));  acc = fma(s, dx, acc)
// Every integer dot is exact (MFMA int32); every fp32 operation is the reference's, in its order.
//
// Roles are swapped against the Q8_0 kernel: the MFMA's A operand is the activations (tokens) and B the weights, so an
// accumulator element of lane l is (token 8 (i / 4) + 4 (l / 32) + i % 4, weight row l % 32) and every per-row scale
// (d sc, dmin m) is one register per lane; per-token values (dx, dx (s0 + s1)) come from LDS as 16 registers. The
// rank-1 products (d sc_h) dx and (d sc_j) dx run on the matrix cores (v_mfma_f32_32x32x1_2b_f32, one block per half
// or per sub-block), int -> float conversions as in the Q8_0 kernel (0x4B400000 accumulator start, then an fp32
// outer product adding -12582912; |dot| <= 32 * 128 * 128 < 2^22). The weights are unpacked from the CDNA planes of
// layout.h into int8 in registers: Q4_K nibbles 0..15; Q6_K q - 32 per byte as ((q | 0x80) - 0x20) ^ 0x80, which
// never borrows across bytes for q < 64.
//
// What bounds it: one wave per SIMD is a serial chain of LDS reads, an MFMA, its conversion and 32 (Q4_K) or 48 (Q6_K wide)
// vector fmas per unit, about 600 cycles where the fmas alone take 130-190. So a unit's dots and products are issued
// on the matrix pipe while the unit before it runs its epilogue on the vector pipe, its operands are read one unit
// ahead, and a stage's last unit finishes in the next stage. Q4_K 2560 x 9728 at 203 tokens 86 -> 70 us, 5120 x 17408 at
// 100 150 -> 122; Q6_K 2560 x 9728 at 203 96 -> 86, 19456 x 2560 at 512 200 -> 187, 34816 x 5120 at 17 60 -> 58.
//
// A workgroup (4 waves) owns a 128-row x 32-token tile (or a 32-row tail tile), 32 rows per wave, and walks K in
// stages of half a super-block (4 units of 32 weights) held in a ring of NS LDS buffers filled by direct global -> LDS
// loads NS - 1 stages ahead.
#include <utility>

#include "ctx.h"
#include "ops.h"

namespace mk {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v32f __attribute__((ext_vector_type(32)));
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) void glb_void;

constexpr int kThreads = 256;
constexpr int kRowsT = 128, kTokT = 32;  // workgroup tile
constexpr int kKB = 4;                   // 32-weight units per stage (half a super-block)
constexpr int kMagic = 0x4B400000;       // bits of 12582912.0f
constexpr float kMagicF = 12582912.0f;

template <int TYPE>
struct KqLds;
template <>
struct KqLds<kQ6_K> {
  static constexpr int a = 0;                    // [4 units][16 groups][192 B]: nib plane 8 x 16 B, hbit plane 8 x 8 B
  static constexpr int sc = a + 4 * 16 * 192;    // [16 groups][8 rows][16 int8] (the whole super-block)
  static constexpr int d = sc + 16 * 128;        // [16 groups][8 rows] f16
  static constexpr int x = d + 16 * 16;          // [4 units][32 tok][32 B] BlockQ8 qs
  static constexpr int dx = x + 4 * 32 * 32;     // [4 units][32 tok] f32
  static constexpr int bytes = dx + 4 * 32 * 4;  // 19200
  static constexpr int loads = 6;                // global -> LDS loads per wave per stage
  static constexpr int tail_loads = 4;           // ... in a 32-row tail tile
};
template <>
struct KqLds<kQ4_K> {
  static constexpr int a = 0;                       // [2 chunks][16 groups][256 B]: lo plane 8 x 16 B, hi plane 8 x 16 B
  static constexpr int hdr = a + 2 * 16 * 256;      // [16 groups][8 rows][16 B] GGUF header (d, dmin, scales)
  static constexpr int x = hdr + 16 * 128;          // [4 units][32 tok][32 B]
  static constexpr int dx = x + 4 * 32 * 32;        // [4 units][32 tok] f32
  static constexpr int s = dx + 4 * 32 * 4;         // [4 units][32 tok] int16 pair (s0, s1)
  static constexpr int dsx = s + 4 * 32 * 4;        // [4 waves][4 units][32 tok] f32: dx (s0 + s1), one copy per wave
  static constexpr int bytes = dsx + 4 * 4 * 32 * 4;  // 17408
  static constexpr int loads = 5;
};

// Q5_K rows stay GGUF rows (mk_matmul_gguf): per row of a stage 7 pieces of 16 bytes, the header (d, dmin, scales), the
// super-block's 32 high-bit bytes and the half's 64 nibble bytes, in consecutive lanes' copies (whole 48- and 64-byte
// runs of a row) and in LDS row after row: a 112-byte row stride puts 16 rows' pieces on different banks.
template <>
struct KqLds<kQ5_K> {
  static constexpr int piece = 7;
  static constexpr int a = 0;                         // [4 waves][32 rows][7][16 B], 4096 B per wave
  static constexpr int x = a + 4 * 4096;              // [4 units][32 tok][32 B]
  static constexpr int dx = x + 4 * 32 * 32;          // [4 units][32 tok] f32
  static constexpr int s = dx + 4 * 32 * 4;           // [4 units][32 tok] int16 pair (s0, s1)
  static constexpr int dsx = s + 4 * 32 * 4;          // [4 waves][4 units][32 tok] f32
  static constexpr int bytes = dsx + 4 * 4 * 32 * 4;  // 23552
  static constexpr int loads = 6;
};

__device__ __forceinline__ void load_lds16(const void* g, uint8_t* l) { lds_copy16(g, l); }
__device__ __forceinline__ void load_lds4(const void* g, uint8_t* l) { lds_copy4(g, l); }
// float(int8 byte K of v)
template <int K>
__device__ __forceinline__ float sbyte_f(uint32_t v) {
  return (float)(int8_t)((v >> (8 * K)) & 0xFF);
}

__device__ __forceinline__ v16f conv(v16i c) {
  return __builtin_amdgcn_mfma_f32_16x16x1f32(-kMagicF, 1.0f, __builtin_bit_cast(v16f, c), 0, 0, 0);
}

// q - 32 per byte for bytes q < 64.
__device__ __forceinline__ uint32_t minus32(uint32_t q) { return ((q | 0x80808080u) - 0x20202020u) ^ 0x80808080u; }

// NS: stages in the LDS ring, NS - 1 of them in flight. 3 when the grid takes several workgroups per CU (prefill);
// deeper rings when few row tiles cover the matrix (short batches), where the stream is latency-bound otherwise.
// NE: accumulator elements with a live token. Element i holds tokens 8 (i / 4) + i % 4 and 8 (i / 4) + 4 + i % 4 of
// the tile, so for a batch of at most 17 tokens (config 5's tree verification) elements 9..15 hold only padding
// tokens in every lane: NE = 9 skips their epilogue (their MFMA results are computed and dropped).
template <int TYPE, bool WIDE, int NS, int NE>
__global__ __launch_bounds__(kThreads) void k_gemm_kq(const uint8_t* W, int64_t rows, int64_t cols,
                                                      const BlockQ8* x, int n, float* __restrict__ y, int64_t ys,
                                                      int accumulate, int n_rt, int n_tt, int n_big, size_t row_bytes) {
  using S = KqLds<TYPE>;
  // Q4_K on large grids runs three waves per SIMD, which cover each other's latency; the pipeline's second register set
  // would leave two (19456 x 2560 at 512 tokens 135 us without it, 144 with it; 5120 x 17408 268 and 286).
  constexpr bool kPipe = !(TYPE == kQ4_K && NS == 3);
  extern __shared__ __align__(16) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wu = __builtin_amdgcn_readfirstlane(w);
  // Workgroup -> (row tile, token tile): tiles numbered row-major, each XCD a contiguous run of them (token tiles of a
  // row tile on one XCD, rows read once into its L2).
  // With 32-row tail tiles (n_big < n_rt, one token tile): tiles in launch order, so the n_big = CU count full tiles
  // take one CU each and the tail tiles a second slot on CUs of every XCD.
  const int tile = n_big < n_rt ? (int)blockIdx.x : xcd_run((int)blockIdx.x, n_rt * n_tt);
  const int rt = tile / n_tt, tt = tile % n_tt;
  const int nb = (int)(cols / 32), nsb = (int)(cols / 256);
  const int64_t r0 = rt < n_big ? (int64_t)rt * kRowsT : (int64_t)n_big * kRowsT + (int64_t)(rt - n_big) * 32;
  const int64_t g0 = r0 / 8;
  const int ngroups = (int)min<int64_t>(rt < n_big ? kRowsT / 8 : 4, rows / 8 - g0);  // 4 .. 16 (rows % 32 == 0)
  // this wave's 32 rows hold a row of the matrix (else: copies only)
  const bool live = TYPE == kQ5_K ? r0 + 32 * wu < rows : 32 * wu < 8 * ngroups;
  const int t0 = tt * kTokT;
  const int nstages = nb / kKB;  // cols % 256 == 0: whole stages

  // Activation copies, per lane: X (wave w: unit w; lane -> token lane / 2, 16-byte half lane % 2); per-token words
  // (unit = 2 c + lane / 32, token lane % 32).
  const uint8_t* x_base = reinterpret_cast<const uint8_t*>(x + (int64_t)t0 * nb);
  const int tx = min(t0 + (lane >> 1), n - 1) - t0, tw = min(t0 + (lane & 31), n - 1) - t0;
  const uint32_t x_off = (uint32_t)(tx * nb * 40 + 8 + 16 * (lane & 1));
  const uint32_t tw_off = (uint32_t)(tw * nb * 40 + (lane >> 5) * 40);  // + 80 c for unit 2 c + lane / 32

  // Weight copies: every piece is 16 (or 4) bytes of a packed (group, unit) record, LDS destinations lane-linear.
  uint32_t a_off[3], m_off = 0, t_off = 0;
  const uint8_t *a_base = W, *m_base = nullptr, *d_base = nullptr;
  const uint8_t* q_src[4];  // Q5_K: this lane's four pieces, at super-block 0 and half 0
  uint32_t q_half[4];       // and their step to half 1
  uint32_t d_off = 0;
  if constexpr (TYPE == kQ6_K) {
    const PackedQ6_K L{rows, nsb};
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const int p = 64 * (3 * w + c) + lane, u = p / 192, q = p % 192;
      const int gi = min(q / 12, ngroups - 1);
      a_off[c] = (uint32_t)((gi * nsb * 8 + u) * 192 + 16 * (q % 12));
    }
    a_base = W + L.quants(g0, 0, 0);
    {
      const int p = 64 * (w & 1) + lane, gi = min(p / 8, ngroups - 1);
      m_off = (uint32_t)(gi * nsb * 128 + 16 * (p % 8));
      m_base = W + L.scales(g0, 0);
    }
    d_off = (uint32_t)(min(lane / 4, ngroups - 1) * nsb * 16 + 4 * (lane % 4));
    d_base = W + L.dscale(g0, 0);
    // Tail tile (4 groups): wave w copies unit w of the stage, lanes 0..47 its 4 x 12 pieces; lanes 48..63 re-read
    // group 3 into the unused group 4-5 slots.
    t_off = (uint32_t)((min(lane / 12, ngroups - 1) * nsb * 8 + w) * 192 + 16 * (lane % 12));
  } else if constexpr (TYPE == kQ5_K) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int g = min(64 * c + lane, 32 * S::piece - 1), p = g % S::piece;
      q_src[c] = W + (size_t)min(r0 + 32 * w + g / S::piece, rows - 1) * row_bytes + 16 * p;
      q_half[c] = p < 3 ? 0u : 64u;
    }
  } else {
    const PackedQ4_K L{rows, nsb};
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int p = 64 * (2 * w + c) + lane, cc = p / 256, q = p % 256;
      const int gi = min(q / 16, ngroups - 1);
      a_off[c] = (uint32_t)((gi * nsb * 4 + cc) * 256 + 16 * (q % 16));
    }
    a_off[2] = 0;
    a_base = W + L.quants(g0, 0, 0);
    {
      const int p = 64 * (w & 1) + lane, gi = min(p / 8, ngroups - 1);
      m_off = (uint32_t)(gi * nsb * 128 + 16 * (p % 8));
      m_base = W + L.headers(g0, 0);
    }
  }

  // Stage sn (units 4 sn .. 4 sn + 3: super-block sn / 2, half sn % 2) into buffer BUF. Every wave issues S::loads
  // loads (a wave with fewer repeats its activation copy), so one wait count fits all; Q6_K tail tiles (TAIL) copy
  // only the 4 groups' quants and scales, S::tail_loads per wave.
  auto issue = [&]<int BUF, bool TAIL>(int sn) __attribute__((always_inline)) {
    uint8_t* st = smem + BUF * S::bytes;
    const int sb = sn >> 1, hf = sn & 1;
    const uint8_t* xb = x_base + (size_t)(4 * sn) * 40;
    if constexpr (TYPE == kQ6_K && TAIL) {
      using T = KqLds<kQ6_K>;
      const uint8_t* ab = a_base + ((size_t)sb * 8 + 4 * hf) * 192;
      load_lds16(ab + t_off, st + T::a + 3072 * wu);
      if (wu == 0)
        load_lds16(m_base + (size_t)sb * 128 + m_off, st + T::sc);
      else if (wu == 1)
        load_lds16(xb + (size_t)wu * 40 + x_off, st + T::x + 1024 * wu);
      else if (wu == 2)
        load_lds4(d_base + (size_t)sb * 16 + d_off, st + T::d);
      else
        load_lds4(xb + tw_off, st + T::dx);
      if (wu == 3)
        load_lds4(xb + 80 + tw_off, st + T::dx + 256);
      else
        load_lds16(xb + (size_t)wu * 40 + x_off, st + T::x + 1024 * wu);
      load_lds16(xb + (size_t)wu * 40 + x_off, st + T::x + 1024 * wu);
    } else if constexpr (TYPE == kQ6_K) {
      const uint8_t* ab = a_base + ((size_t)sb * 8 + 4 * hf) * 192;
#pragma unroll
      for (int c = 0; c < 3; ++c) load_lds16(ab + a_off[c], st + S::a + 1024 * (3 * wu + c));
      if (wu < 2) {
        load_lds16(m_base + (size_t)sb * 128 + m_off, st + S::sc + 1024 * wu);
      } else if (wu == 2) {
        load_lds4(d_base + (size_t)sb * 16 + d_off, st + S::d);
      } else {
        load_lds4(xb + tw_off, st + S::dx);
        load_lds4(xb + 80 + tw_off, st + S::dx + 256);
      }
      load_lds16(xb + (size_t)wu * 40 + x_off, st + S::x + 1024 * wu);
      if (wu != 3) load_lds16(xb + (size_t)wu * 40 + x_off, st + S::x + 1024 * wu);
    } else if constexpr (TYPE == kQ5_K) {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        load_lds16(q_src[c] + (size_t)sb * 176 + (hf ? q_half[c] : 0u), st + S::a + 4096 * wu + 1024 * c);
      load_lds4(xb + 4 * (wu >> 1) + 80 * (wu & 1) + tw_off, st + (wu < 2 ? S::dx : S::s) + 256 * (wu & 1));
      load_lds16(xb + (size_t)wu * 40 + x_off, st + S::x + 1024 * wu);
    } else {
      const uint8_t* ab = a_base + ((size_t)sb * 4 + 2 * hf) * 256;
#pragma unroll
      for (int c = 0; c < 2; ++c) load_lds16(ab + a_off[c], st + S::a + 1024 * (2 * wu + c));
      if (wu < 2) {
        load_lds16(m_base + (size_t)sb * 128 + m_off, st + S::hdr + 1024 * wu);
        load_lds16(xb + (size_t)wu * 40 + x_off, st + S::x + 1024 * wu);
      } else if (wu == 2) {
        load_lds4(xb + tw_off, st + S::dx);
        load_lds4(xb + 80 + tw_off, st + S::dx + 256);
      } else {
        load_lds4(xb + 4 + tw_off, st + S::s);
        load_lds4(xb + 84 + tw_off, st + S::s + 256);
      }
      load_lds16(xb + (size_t)wu * 40 + x_off, st + S::x + 1024 * wu);
    }
  };

  v16f acc = {};
  v16i magic;
#pragma unroll
  for (int i = 0; i < 16; ++i) magic[i] = kMagic;
  asm volatile("" : "+v"(magic));  // keep it in VGPRs: as a uniform value it would be copied from SGPRs per MFMA
  const v32f zero = {};
  const int li = lane & 31, h = lane >> 5;
  const int gi = 4 * w + (li >> 3), r8 = li & 7;  // this lane's weight row: group gi, row r8 of it
  const int tok_i = 4 * h;                         // tokens of element i: 8 (i / 4) + 4 h + i % 4

  // 16 per-token floats of element i from a [32 tok] f32 array: tokens 8 q + 4 h .. + 3 for q = 0..3.
  auto tok16 = [&](const uint8_t* p) __attribute__((always_inline)) {
    v16f v;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4 f = *reinterpret_cast<const float4*>(p + 4 * (8 * q + tok_i));
      v[4 * q] = f.x, v[4 * q + 1] = f.y, v[4 * q + 2] = f.z, v[4 * q + 3] = f.w;
    }
    return v;
  };

  // One unit in the pipeline: its MFMA results and the operands of its epilogue. Q4_K: f0 = float(dot), p2 (below), b =
  // dx (s0 + s1) per token, s0 = -(dmin m). Q6_K: f0 / f1 = the halves' float(dot); wide: b = dx per token, s0 / s1 = d
  // sc of the halves; compact: p = (d sc_h) dx, halves 0 and 1.
  struct Unit {
    v16f f0, f1, b;
    v32f p;
    float s0 = 0.0f, s1 = 0.0f;
  };
  Unit U[2];
  v16i i0 = magic, i1 = magic;  // the next unit's int dots, between its two steps
  v32f p2 = zero;               // Q4_K: (d sc_j) dx of the unit pair
  U[1].f0 = U[1].f1 = U[1].b = v16f{};
  U[1].p = v32f{};

  // The first and second half of a unit's epilogue, in the reference's order.
  auto epi_a = [&](const Unit& u, int odd) __attribute__((always_inline)) {
    if constexpr (TYPE == kQ6_K && WIDE) {
#pragma unroll
      for (int i = 0; i < NE / 2; ++i) acc[i] = fma_(fma_(u.f1[i], u.s1, u.f0[i] * u.s0), u.b[i], acc[i]);
    } else if constexpr (TYPE == kQ6_K) {
#pragma unroll
      for (int i = 0; i < NE; ++i) acc[i] = fma_(u.f0[i], u.p[i], acc[i]);
    } else {
#pragma unroll
      for (int i = 0; i < NE; ++i) acc[i] = fma_(u.f0[i], p2[16 * odd + i], acc[i]);
    }
  };
  auto epi_b = [&](const Unit& u) __attribute__((always_inline)) {
    if constexpr (TYPE == kQ6_K && WIDE) {
#pragma unroll
      for (int i = NE / 2; i < NE; ++i) acc[i] = fma_(fma_(u.f1[i], u.s1, u.f0[i] * u.s0), u.b[i], acc[i]);
    } else if constexpr (TYPE == kQ6_K) {
#pragma unroll
      for (int i = 0; i < NE; ++i) acc[i] = fma_(u.f1[i], u.p[16 + i], acc[i]);
    } else {
#pragma unroll
      for (int i = 0; i < NE; ++i) acc[i] = fma_(u.s0, u.b[i], acc[i]);
    }
  };

  auto stage = [&]<int BUF, bool TAIL>(int s) __attribute__((always_inline)) {
    // Stage s has landed once at most the loads of the stages issued after it (s + 1 .. s + NS - 2, fewer at the
    // end) are outstanding; the buffer stage s + NS - 1 goes into was read in stage s - 1, finished by every wave
    // before this barrier.
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    if constexpr (TAIL)
      wait_vm_stages<KqLds<kQ6_K>::tail_loads, NS - 2>(min(NS - 2, nstages - 1 - s));
    else
      wait_vm_stages<S::loads, NS - 2>(min(NS - 2, nstages - 1 - s));
    ring_barrier();
    if (s + NS - 1 < nstages) issue.template operator()<(BUF + NS - 1) % NS, TAIL>(s + NS - 1);
    if (!live) return;
    uint8_t* st = smem + BUF * S::bytes;
    const int hf = s & 1;
    // The lane's weight scales for the stage, then per unit: `begin` reads its operands and issues the int dots,
    // `mid` converts them and issues the scale products.
    float sca[kKB], scb[kKB];
    uint4 raw[2], qh;
    if constexpr (TYPE == kQ6_K) {
      const float d = half_to_float(*reinterpret_cast<const uint16_t*>(st + S::d + gi * 16 + r8 * 2));
      const uint2 scw = *reinterpret_cast<const uint2*>(st + S::sc + gi * 128 + r8 * 16 + 8 * hf);
#pragma unroll
      for (int u = 0; u < kKB; ++u) {
        const uint32_t sw = u < 2 ? scw.x : scw.y;
        sca[u] = d * sbyte_f<0>(sw >> (16 * (u & 1)));
        scb[u] = d * sbyte_f<1>(sw >> (16 * (u & 1)));
      }
    } else {
      // dx (s0 + s1) of the stage's 4 units x 32 tokens, into this wave's own copy
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int p = 64 * c + lane;
        const float dxv = *reinterpret_cast<const float*>(st + S::dx + 4 * p);
        const uint32_t sv = *reinterpret_cast<const uint32_t*>(st + S::s + 4 * p);
        const int ss = (int)(int16_t)(sv & 0xFFFF) + (int)(int16_t)(sv >> 16);
        *reinterpret_cast<float*>(st + S::dsx + w * 512 + 4 * p) = dxv * (float)ss;
      }
      uint4 hd;
      if constexpr (TYPE == kQ5_K) {
        const uint8_t* row = st + S::a + 4096 * w + 16 * S::piece * li;
        hd = *reinterpret_cast<const uint4*>(row);
        qh = *reinterpret_cast<const uint4*>(row + 16 + 16 * h);
#pragma unroll
        for (int cc = 0; cc < 2; ++cc) raw[cc] = *reinterpret_cast<const uint4*>(row + 48 + 32 * cc + 16 * h);
      } else {
#pragma unroll
        for (int cc = 0; cc < 2; ++cc)
          raw[cc] = *reinterpret_cast<const uint4*>(st + S::a + cc * 4096 + gi * 256 + h * 128 + r8 * 16);
        hd = *reinterpret_cast<const uint4*>(st + S::hdr + gi * 128 + r8 * 16);
      }
      const float d = half_to_float((uint16_t)(hd.x & 0xFFFF)), dmin = half_to_float((uint16_t)(hd.x >> 16));
      // scale_min_k4 (the reference's kernels.h:18-26) of sub-blocks 4 hf + 0..3, byte u of each word (hd.y, hd.z, hd.w: the 12 packed bytes): the low
      // half of a super-block takes 6 bits of hd.y / hd.z, the high half nibbles of hd.w and the top bits of those.
      const uint32_t sc4 = hf ? (hd.w & 0x0F0F0F0Fu) | ((hd.y >> 2) & 0x30303030u) : hd.y & 0x3F3F3F3Fu;
      const uint32_t mn4 = hf ? ((hd.w >> 4) & 0x0F0F0F0Fu) | ((hd.z >> 2) & 0x30303030u) : hd.z & 0x3F3F3F3Fu;
#pragma unroll
      for (int u = 0; u < kKB; ++u) {
        sca[u] = d * (float)((sc4 >> (8 * u)) & 0xFFu);
        scb[u] = -(dmin * (float)((mn4 >> (8 * u)) & 0xFFu));
      }
    }
    if constexpr (!kPipe) {
#pragma unroll
      for (int cc = 0; cc < 2; ++cc) {
        // (d sc_j) dx for units 2 cc and 2 cc + 1: block h takes unit 2 cc + h
        const float dxl = *reinterpret_cast<const float*>(st + S::dx + (2 * cc + h) * 128 + li * 4);
        const v32f p = __builtin_amdgcn_mfma_f32_32x32x1f32(dxl, h ? sca[2 * cc + 1] : sca[2 * cc], zero, 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const int u = 2 * cc + e;
          const v4i wq = {(int)((raw[cc].x >> (4 * e)) & 0x0F0F0F0Fu), (int)((raw[cc].y >> (4 * e)) & 0x0F0F0F0Fu),
                          (int)((raw[cc].z >> (4 * e)) & 0x0F0F0F0Fu), (int)((raw[cc].w >> (4 * e)) & 0x0F0F0F0Fu)};
          const v4i xa = *reinterpret_cast<const v4i*>(st + S::x + u * 1024 + li * 32 + 16 * h);
          const v16f f = conv(__builtin_amdgcn_mfma_i32_32x32x32_i8(xa, wq, magic, 0, 0, 0));
          const v16f dsx = tok16(st + S::dsx + w * 512 + u * 128);
#pragma unroll
          for (int i = 0; i < NE; ++i) {
            acc[i] = fma_(f[i], p[16 * e + i], acc[i]);
            acc[i] = fma_(scb[u], dsx[i], acc[i]);
          }
        }
      }
      return;
    }
    // A unit's operands, read one unit ahead of its dots (Q4_K: x; Q6_K: nibbles, high bits, the halves of x).
    struct Ops {
      v4i xa;
      uint2 nib, hb;
      long xa0, xa1;
    } ops[2];
    auto read = [&](int u) __attribute__((always_inline)) {
      Ops& o = ops[u & 1];
      if constexpr (TYPE == kQ6_K) {
        const uint8_t* au = st + S::a + u * 3072 + gi * 192;
        o.nib = *reinterpret_cast<const uint2*>(au + r8 * 16 + 8 * h);
        o.hb = *reinterpret_cast<const uint2*>(au + 128 + r8 * 8);
        const uint8_t* xu = st + S::x + u * 1024 + li * 32 + 8 * h;
        o.xa0 = *reinterpret_cast<const long*>(xu);
        o.xa1 = *reinterpret_cast<const long*>(xu + 16);
      } else {
        o.xa = *reinterpret_cast<const v4i*>(st + S::x + u * 1024 + li * 32 + 16 * h);
      }
    };
    // The unit's int dots; its per-token operands are read behind them.
    float dxl = 0.0f;
    auto begin = [&](Unit& n, int u) __attribute__((always_inline)) {
      const Ops& o = ops[u & 1];
      if constexpr (TYPE == kQ6_K) {
        // half hw: bytes r = 0..7 are q[16 hw + 8 h + r]
        long wq[2];
#pragma unroll
        for (int hw = 0; hw < 2; ++hw) {
          const uint32_t hv = (hw ? o.hb.y : o.hb.x) >> (4 * h);
          const uint32_t q0 = ((o.nib.x >> (4 * hw)) & 0x0F0F0F0Fu) | ((hv & 0x03030303u) << 4);
          const uint32_t q1 = ((o.nib.y >> (4 * hw)) & 0x0F0F0F0Fu) | (((hv >> 2) & 0x03030303u) << 4);
          wq[hw] = (long)(((uint64_t)minus32(q1) << 32) | minus32(q0));
        }
        i0 = __builtin_amdgcn_mfma_i32_32x32x16_i8(o.xa0, wq[0], magic, 0, 0, 0);
        i1 = __builtin_amdgcn_mfma_i32_32x32x16_i8(o.xa1, wq[1], magic, 0, 0, 0);
        if constexpr (WIDE)
          n.b = tok16(st + S::dx + u * 128);
        else
          dxl = *reinterpret_cast<const float*>(st + S::dx + u * 128 + li * 4);
      } else {
        const uint4 r = raw[u >> 1];
        const int sh = 4 * (u & 1);
        v4i wq = {(int)((r.x >> sh) & 0x0F0F0F0Fu), (int)((r.y >> sh) & 0x0F0F0F0Fu),
                  (int)((r.z >> sh) & 0x0F0F0F0Fu), (int)((r.w >> sh) & 0x0F0F0F0Fu)};
        if constexpr (TYPE == kQ5_K) {
          const int j = 4 * hf + u;  // the sub-block's bit of the high-bit bytes
          wq |= v4i{(int)(((qh.x >> j) & 0x01010101u) << 4), (int)(((qh.y >> j) & 0x01010101u) << 4),
                    (int)(((qh.z >> j) & 0x01010101u) << 4), (int)(((qh.w >> j) & 0x01010101u) << 4)};
        }
        i0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(o.xa, wq, magic, 0, 0, 0);
        n.b = tok16(st + S::dsx + w * 512 + u * 128);
        if (u % 2 == 0) dxl = *reinterpret_cast<const float*>(st + S::dx + (u + h) * 128 + li * 4);
      }
      if (u + 1 < kKB) read(u + 1);
    };
    // Its float dots and scale products.
    auto mid = [&](Unit& n, int u) __attribute__((always_inline)) {
      n.f0 = conv(i0);
      if constexpr (TYPE == kQ6_K) {
        n.f1 = conv(i1);
        n.s0 = sca[u];
        n.s1 = scb[u];
        // compact: (d sc_h) dx for both halves: block h of the outer product takes dx (A) and d sc_h (B)
        if constexpr (!WIDE) n.p = __builtin_amdgcn_mfma_f32_32x32x1f32(dxl, h ? scb[u] : sca[u], zero, 0, 0, 0);
      } else {
        n.s0 = scb[u];
        // (d sc_j) dx for units u and u + 1: block h takes unit u + h
        if (u % 2 == 0) p2 = __builtin_amdgcn_mfma_f32_32x32x1f32(dxl, h ? sca[u + 1] : sca[u], zero, 0, 0, 0);
      }
    };
    // While a unit's epilogue runs on the vector pipe, the next unit's dots and products run on the matrix pipe; the
    // stage's last unit finishes in the next stage (whose first operands are read behind its epilogue's first half).
    // The scheduling barriers keep the two interleaved.
    read(0);
    __builtin_amdgcn_sched_barrier(0);
    epi_a(U[1], 1);
    __builtin_amdgcn_sched_barrier(0);
    begin(U[0], 0);
    __builtin_amdgcn_sched_barrier(0);
    epi_b(U[1]);
    __builtin_amdgcn_sched_barrier(0);
    mid(U[0], 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 1; u < kKB; ++u) {
      Unit &cur = U[(u + 1) & 1], &nxt = U[u & 1];
      begin(nxt, u);
      __builtin_amdgcn_sched_barrier(0);
      epi_a(cur, (u + 1) & 1);
      __builtin_amdgcn_sched_barrier(0);
      mid(nxt, u);
      __builtin_amdgcn_sched_barrier(0);
      epi_b(cur);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  auto run = [&]<bool TAIL>() __attribute__((always_inline)) {
    [&]<int... B>(std::integer_sequence<int, B...>) __attribute__((always_inline)) {
      ((B < nstages ? issue.template operator()<B, TAIL>(B) : void()), ...);
    }(std::make_integer_sequence<int, NS - 1>{});
    for (int s = 0; s < nstages; s += NS) {
      [&]<int... B>(std::integer_sequence<int, B...>) __attribute__((always_inline)) {
        ((s + B < nstages ? stage.template operator()<B, TAIL>(s + B) : void()), ...);
      }(std::make_integer_sequence<int, NS>{});
    }
  };
  if constexpr (TYPE == kQ6_K) {
    if (rt >= n_big)
      run.template operator()<true>();
    else
      run.template operator()<false>();
  } else {
    run.template operator()<false>();
  }

  // Element i: token t0 + 8 (i / 4) + 4 h + i % 4, row 128 rt + 32 w + li.
  if (live) {
    if constexpr (kPipe) {
      epi_a(U[1], 1);
      epi_b(U[1]);
    }
    float* yr = y + r0 + 32 * w + li;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int t = t0 + 8 * (i / 4) + tok_i + i % 4;
      if (t < n && (TYPE != kQ5_K || r0 + 32 * w + li < rows)) {
        float* o = yr + (int64_t)t * ys;
        *o = accumulate ? *o + acc[i] : acc[i];
      }
    }
  }
}

template <int TYPE, bool WIDE, int NS, int NE>
void launch_kq_ns(hipStream_t s, const void* w, int64_t rows, int64_t cols, const BlockQ8* x, int n, float* y,
                  int64_t ys, bool accumulate, int n_rt, int n_tt, int n_big, size_t row_bytes = 0) {
  const size_t lds = NS * (size_t)KqLds<TYPE>::bytes;
  static bool attr = false;  // per instantiation: rings past 64 KB of dynamic LDS
  if (!attr) {
    check(hipFuncSetAttribute(reinterpret_cast<const void*>(k_gemm_kq<TYPE, WIDE, NS, NE>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds),
          "hipFuncSetAttribute");
    attr = true;
  }
  hipLaunchKernelGGL((k_gemm_kq<TYPE, WIDE, NS, NE>), dim3((unsigned)((int64_t)n_rt * n_tt)), dim3(kThreads), lds, s,
                     static_cast<const uint8_t*>(w), rows, cols, x, n, y, ys, accumulate ? 1 : 0, n_rt, n_tt, n_big,
                     row_bytes);
}

// Ring depth by grid size: one workgroup per CU takes an 8-stage ring (7 stages, about 130 KB, in flight), two per CU
// a 4-stage ring; larger grids (prefill) keep 3 stages and several workgroups per CU.
template <int TYPE, bool WIDE>
void launch_kq(hipStream_t s, const void* w, int64_t rows, int64_t cols, const BlockQ8* x, int n, float* y, int64_t ys,
               bool accumulate) {
  int n_rt = (int)((rows + kRowsT - 1) / kRowsT), n_big = n_rt;
  const int n_tt = (n + kTokT - 1) / kTokT;
  const int64_t cus = device_cus();
  // A short batch over slightly more than one 128-row tile per CU (the 14B gate|up, 34816 rows: 272 tiles) takes one
  // full tile per CU and covers the rest with 32-row tiles (one live wave), so that no CU runs two full tiles.
  // Measured at 17 tokens (bit-identical): Q6_K 34816 x 5120 65.3 -> 62.3 us, 40960 x 5120 66.4 -> 63.6, Q4_K
  // 34816 x 5120 50.5 -> 48.4; at 24 tokens Q6_K 34816 x 5120 78.2 -> 75.6. Q6_K tail tiles copying only their
  // 4 groups' quants and scales (4 instead of 6 copies per wave and stage): 61.9 -> 60.9 us, at 24 tokens 73.3 -> 70.8.
  if (n_tt == 1 && n_rt > cus && rows <= (kRowsT + 32) * cus) {
    n_big = (int)cus;
    n_rt = n_big + (int)((rows - kRowsT * cus) / 32);
  }
  const int64_t wgs = (int64_t)n_rt * n_tt;
  if (wgs <= cus)
    n <= 17 ? launch_kq_ns<TYPE, WIDE, 8, 9>(s, w, rows, cols, x, n, y, ys, accumulate, n_rt, n_tt, n_big)
            : launch_kq_ns<TYPE, WIDE, 8, 16>(s, w, rows, cols, x, n, y, ys, accumulate, n_rt, n_tt, n_big);
  else if (wgs <= 2 * cus)
    n <= 17 ? launch_kq_ns<TYPE, WIDE, 4, 9>(s, w, rows, cols, x, n, y, ys, accumulate, n_rt, n_tt, n_big)
            : launch_kq_ns<TYPE, WIDE, 4, 16>(s, w, rows, cols, x, n, y, ys, accumulate, n_rt, n_tt, n_big);
  else
    launch_kq_ns<TYPE, WIDE, 3, 16>(s, w, rows, cols, x, n, y, ys, accumulate, n_rt, n_tt, n_big);
}

// Q5_K: rings of 6 stages (138 KB) where the grid fits the CUs once, 3 (two workgroups per CU) past that; elements of
// tokens past n are skipped in whole quarters (element i holds tokens 8 (i / 4) + 0..7). Measured against the
// byte-wise kernel of rowpath.hip: 19456 x 2560 at 32 tokens 382 -> 23 us, at 256 2252 -> 87; 2560 x 9728 at 128 769 -> 72.
void launch_q5(hipStream_t s, const void* w, size_t row_bytes, int64_t rows, int64_t cols, const BlockQ8* x, int n,
               float* y, int64_t ys, bool accumulate) {
  const int n_rt = (int)((rows + kRowsT - 1) / kRowsT), n_tt = (n + kTokT - 1) / kTokT;
  auto go = [&]<int NE>() {
    if ((int64_t)n_rt * n_tt <= device_cus())
      launch_kq_ns<kQ5_K, false, 6, NE>(s, w, rows, cols, x, n, y, ys, accumulate, n_rt, n_tt, n_rt, row_bytes);
    else
      launch_kq_ns<kQ5_K, false, 3, NE>(s, w, rows, cols, x, n, y, ys, accumulate, n_rt, n_tt, n_rt, row_bytes);
  };
  if (n <= 8)
    go.template operator()<4>();
  else if (n <= 16)
    go.template operator()<8>();
  else
    go.template operator()<16>();
}

}  // namespace

void gemm_q5_gguf(hipStream_t s, const void* w, size_t row_bytes, int64_t rows, int64_t cols, const BlockQ8* x, int n,
                  float* y, int64_t ys, bool accumulate) {
  require(cols % 256 == 0 && rows > 0 && n > 0 && row_bytes % 16 == 0 && (uintptr_t)w % 16 == 0,
          "gemm_q5_gguf: 16-byte aligned rows of a multiple of 256 values");
  launch_q5(s, w, row_bytes, rows, cols, x, n, y, ys, accumulate);
  check_launch("gemm_q5_gguf");
}

bool gemm_kq_supported(int type, int64_t rows, int64_t cols, int n) {
  return (type == kQ4_K || type == kQ6_K) && rows % 32 == 0 && cols % 256 == 0 && n > 8;
}

void gemm_kq(hipStream_t s, int type, bool wide, const void* w, int64_t rows, int64_t cols, const BlockQ8* x, int n,
             float* y, int64_t ys, bool accumulate) {
  require(gemm_kq_supported(type, rows, cols, n), "gemm_kq: Q4_K/Q6_K, rows a multiple of 32, cols of 256, n > 8");
  if (type == kQ4_K)
    launch_kq<kQ4_K, false>(s, w, rows, cols, x, n, y, ys, accumulate);
  else if (wide && n > 16)
    launch_kq<kQ6_K, true>(s, w, rows, cols, x, n, y, ys, accumulate);
  else
    launch_kq<kQ6_K, false>(s, w, rows, cols, x, n, y, ys, accumulate);
  check_launch("gemm_kq");
}

}  // namespace mk
