// Attention of many query rows at once (prompt chunks and other long plain batches) on the fp32 matrix cores, attend_t
// semantics (kernels_avx512.cpp:228-267) for head_dim 128 over the permuted device cache, G <= 16 query heads per KV
// head, bit-identical to the reference. v_mfma_f32_16x16x4_f32 runs every output element as four correctly rounded fmas
// in ascending k, so both the scores' lane chains and P.V's sequential chain over the keys run on it in the
// reference's order, at twice the vector unit's non-packed fp32 rate.
//
// A workgroup of 8 waves takes the 16 / G consecutive tokens of one token block and the G query heads of one KV group:
// up to 16 query rows that share every K and V row they read.
//   scores  a wave takes 16 keys at a time. Chain l of attend_t is sum over c of q[16 c + l] k[16 c + l], c = 0..7: two
//           MFMAs (A: the rows' q, resident; B: the keys), started from -0 so that the first fma is the reference's
//           multiply. A permuted K row holds a chain's eight values in two dwords; MFMA k index q is c = q (+ 4), so
//           lane (key, q) needs byte q of every dword (transpose_rows). The halving tree over the 16 chains is 15 adds of 4 registers;
//   softmax e = exp512(s - max) with 32 threads per row (the exact max was kept beside the scores), and the 16
//           sequential lane sums and their halving tree; the row's P.V coefficient e * v_scale replaces the score;
//   P.V     a wave owns 16 of the 128 values of every row: one MFMA per 4 keys, A = the coefficients, B = V, whose int8
//           rows come through a ring of LDS stages filled by direct copies; a stage's operands are read into registers
//           while the stage before it runs. Keys past a row's end have coefficient 0 and fma(0, v, acc) == acc.
// Scores and v scales of a 16-key group lie in LDS in the order lane q of the P.V reads them (key 4 s + q at 4 q + s).
// Rows longer than LDS holds (LONG) take two passes: the maxima first, then the scores again, kChunk keys at a time, each
// chunk's sums and P.V continuing the last one's. Tokens of a block that belong to different sequences are handled
// one sequence at a time, each in a walk over that sequence's keys.
//
// What bounds it: fp32 MFMAs and vector instructions share a SIMD's issue (measured: they do not overlap), so a 16-key
// score tile costs 32 x 32 cycles of MFMA and about 150 vector instructions (transpose, conversions, the trees), and
// P.V 32 cycles per 4 keys and wave. 512 tokens of 32 heads over 8 KV heads (16-row workgroups, one per CU past 704
// keys), us against the vector kernel this replaced (one key per thread, fp32 V tiles): first chunk 81 -> 58, behind 512
// tokens 320 -> 122, behind 1024 506 -> 184. With one scalar byte read of V per value instead of the transposing LDS
// read, and the K loads left to the compiler's order (behind half of the tile's MFMAs): 134 instead of 122.
#include <algorithm>

#include "attn_dec.h"
#include "ctx.h"
#include "ops.h"

namespace mk {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) v2i lds_v2i;

constexpr int kD = 128;
constexpr int kThreads = 512, kWaves = 8;
constexpr int kRows = 16;                 // query rows per workgroup
constexpr int kVKeys = 64, kVStages = 4;  // keys per V stage (one 1 KB copy per wave), ring depth
constexpr int kVBytes = kVKeys * kD;
constexpr int kChunk = 512;               // keys per pass of LONG rows
static_assert(kVBytes == 1024 * kWaves && kVStages * kVBytes >= kRows * (kD + 4) * 4, "ring");

// Position of key j's entry in its 16-key group.
__device__ __forceinline__ int key_pos(int j) { return (j & ~15) | ((j & 3) << 2) | ((j >> 2) & 3); }

__host__ __device__ constexpr int sc_stride(int nk_pad) { return nk_pad + 4; }
__host__ __device__ constexpr int pad64(int nk) { return (nk + 63) & ~63; }  // whole V stages
__host__ __device__ constexpr size_t mma_lds_bytes(int nk_pad) {
  return (size_t)kVStages * kVBytes + 4 * ((size_t)kRows * sc_stride(nk_pad) + nk_pad);
}

// r[p] of lane row q (16 lanes) = byte-transposed t[q] of row p: the four rows hold 16 consecutive bytes each of a
// permuted K row's 64 (dwords t[0..3]); row q ends with byte q of every dword, r[p] byte j that of row p's dword j. In a
// lane a 4 x 4 byte transpose (8 v_perm), between the rows a 4 x 4 dword transpose (4 permlane swaps): the wave then
// loads every byte of its 16 K rows once instead of each lane row loading all of them.
__device__ __forceinline__ void transpose_rows(const v4i& t, uint32_t (&r)[4]) {
  const uint32_t a = __builtin_amdgcn_perm((uint32_t)t[1], (uint32_t)t[0], 0x05010400u);  // b0 b0 b1 b1 of t0, t1
  const uint32_t b = __builtin_amdgcn_perm((uint32_t)t[3], (uint32_t)t[2], 0x05010400u);
  const uint32_t c = __builtin_amdgcn_perm((uint32_t)t[1], (uint32_t)t[0], 0x07030602u);  // b2 b2 b3 b3
  const uint32_t d = __builtin_amdgcn_perm((uint32_t)t[3], (uint32_t)t[2], 0x07030602u);
  const uint32_t t0 = __builtin_amdgcn_perm(b, a, 0x05040100u), t1 = __builtin_amdgcn_perm(b, a, 0x07060302u);
  const uint32_t t2 = __builtin_amdgcn_perm(d, c, 0x05040100u), t3 = __builtin_amdgcn_perm(d, c, 0x07060302u);
  const auto x = __builtin_amdgcn_permlane16_swap(t0, t1, false, false);
  const auto y = __builtin_amdgcn_permlane16_swap(t2, t3, false, false);
  const auto u = __builtin_amdgcn_permlane32_swap(x[0], y[0], false, false);
  const auto v = __builtin_amdgcn_permlane32_swap(x[1], y[1], false, false);
  r[0] = u[0], r[2] = u[1], r[1] = v[0], r[3] = v[1];
}

template <bool LONG>
__global__ __launch_bounds__(kThreads) void k_attention_mma(const float* __restrict__ q, int64_t q_stride,
                                                            float* __restrict__ out, int64_t out_stride, int G,
                                                            float scale, AttnAddr a, const int32_t* __restrict__ seqs,
                                                            const int32_t* __restrict__ n_keys, int n, int KV,
                                                            int max_pad, BlockQ8* __restrict__ xq, int64_t xq_stride,
                                                            const int32_t* __restrict__ route) {
  if (LONG && route && *route != kRouteMma) return;
  const int nk_pad = LONG ? kChunk : max_pad;  // keys held in LDS
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lq = lane >> 4;
  const int TQ = kRows / G, nblk = (n + TQ - 1) / TQ;
  // Workgroup -> (KV group, token block): each XCD a contiguous run of pairs, so a group's K/V rows are read into one
  // L2; within a group the blocks with the most keys start first.
  const int pair = xcd_run((int)blockIdx.x, nblk * KV), g = pair / nblk, blk = nblk - 1 - pair % nblk;
  const int t0 = blk * TQ, tq = min(TQ, n - t0), R = tq * G;
  extern __shared__ __align__(16) uint8_t smem[];
  const int S = sc_stride(nk_pad);
  float* sc = reinterpret_cast<float*>(smem + kVStages * kVBytes);  // [16][S]: scores, then e
  float* vsc = sc + kRows * S;                                      // [nk_pad]: v scales
  __shared__ int seq_s[kRows], nk_s[kRows];
  __shared__ float inv_s[kRows], max_s[kWaves][kRows];
  // Row r: token t0 + r / G, query head g * G + r % G.
  if (tid < kRows) {
    const int t = t0 + min(tid / G, tq - 1);
    const int sv = seqs[t], kv = n_keys[t];
    seq_s[tid] = tid < R ? sv : -1;
    nk_s[tid] = tid < R ? kv : 0;
  }
  // The A operand of the scores: q of row li, qa[l][hf] = q[16 (4 hf + lq) + l].
  float qa[16][2];
  {
    const int r = min(li, R - 1);
    const float* qr = q + (int64_t)(t0 + r / G) * q_stride + (int64_t)(g * G + r % G) * kD;
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
#pragma unroll
        for (int k = 0; k < 4; ++k) qa[4 * u + k][hf] = qr[16 * (4 * hf + lq) + 4 * u + k];
      }
  }
  __syncthreads();
  const uint32_t all = (1u << R) - 1;
  uint32_t done = 0;
  while (done != all) {
    // The pass's sequence: that of the first row not done; its rows and their longest key range.
    const int s = __builtin_amdgcn_readfirstlane(seq_s[__builtin_ctz(~done)]);
    uint32_t act = 0;
    int nkb = 1;
    for (int r = 0; r < R; ++r) {
      const int sr = __builtin_amdgcn_readfirstlane(seq_s[r]);
      if (sr == s) {
        act |= 1u << r;
        nkb = max(nkb, __builtin_amdgcn_readfirstlane(nk_s[r]));
      }
    }
    nkb = min(nkb, max_pad);  // max_pad covers max_keys, which bounds every token's keys
    const int tiles = (nkb + 15) / 16;
    const int8_t* kb = a.k + (int64_t)s * a.k_seq + g * a.k_head;
    const int8_t* vb = a.v + (int64_t)s * a.k_seq + g * a.k_head;
    const char* ksb = a.ks + (int64_t)s * a.s_seq + g * a.s_head;
    const char* vsb = a.vs + (int64_t)s * a.s_seq + g * a.s_head;

    // V stage c: keys 64 c .. (past the last key it again), 16-byte pieces p of key k at slot p ^ ((k / 2) % 8): a P.V
    // read's four keys then lie on different banks.
    const int nst = (nkb + kVKeys - 1) / kVKeys;
    auto v_issue = [&](int c) __attribute__((always_inline)) {
      const int g0 = 64 * w + lane, k = g0 >> 3, p = (g0 & 7) ^ ((k >> 1) & 7);
      const int j = min(c * kVKeys + k, nkb - 1);
      lds_copy16(vb + (int64_t)j * a.k_row + 16 * p, smem + (c % kVStages) * kVBytes + 1024 * w);
    };

    // Scores (kernels_avx512.cpp:234-244) of tiles kt0 .. kt1 - 1 into LDS (STORE), and the maximum of this lane's keys
    // in each of its rows. Loads are never predicated: past the last key they re-read it, unused.
    int nk4[4];
    float m4[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      nk4[i] = min(nk_s[4 * lq + i], nkb);
      m4[i] = -INFINITY;
    }
    auto scores = [&]<bool STORE>(int kt0, int kt1) __attribute__((always_inline)) {
      struct Tile {
        v4i k[2];  // bytes 32 lq .. 32 lq + 31 of the key's row
        float ks, vs;
      };
      auto load = [&](Tile& T, int kt) __attribute__((always_inline)) {
        const int j = min(16 * kt + li, nkb - 1);
#pragma unroll
        for (int u = 0; u < 2; ++u)
          T.k[u] = *reinterpret_cast<const v4i*>(kb + (int64_t)j * a.k_row + 32 * lq + 16 * u);
        T.ks = *reinterpret_cast<const float*>(ksb + (int64_t)j * a.s_row);
        if constexpr (STORE) T.vs = *reinterpret_cast<const float*>(vsb + (int64_t)j * a.s_row);
      };
      const v4f mzero = {-0.0f, -0.0f, -0.0f, -0.0f};
      auto score = [&](const Tile& T, int kt) __attribute__((always_inline)) {
        uint32_t x[2][4];  // byte 2 (l % 2) + hf of x[l / 2 % 2][l / 4]: the key's value of chain l at c = 4 hf + lq
#pragma unroll
        for (int u = 0; u < 2; ++u) transpose_rows(T.k[u], x[u]);
        // Chains o, o + 8, o + 4, o + 12, whose results make one value of the tree's third level. Converted by the
        // compiler, not by i8_to_f32: an MFMA reads a register that a vector instruction wrote only after some wait
        // states, which the compiler does not place behind inline assembly.
        auto chains = [&](v4f(&r)[4], int o) __attribute__((always_inline)) {
          float k0[4], k1[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int l = o + 4 * i;
            const uint32_t d = x[(l >> 1) & 1][l >> 2];
            k0[i] = (float)(int8_t)(d >> (16 * (l & 1)));
            k1[i] = (float)(int8_t)(d >> (16 * (l & 1) + 8));
          }
#pragma unroll
          for (int i = 0; i < 4; ++i)
            r[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[o + 4 * i][0], k0[i], mzero, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; ++i) r[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[o + 4 * i][1], k1[i], r[i], 0, 0, 0);
        };
        auto tree = [](const v4f(&r)[4]) __attribute__((always_inline)) { return (r[0] + r[2]) + (r[1] + r[3]); };
        // Two groups in flight: a group's adds come after the next group's MFMAs, so that none waits for its result.
        v4f X[4], Y[4];
        chains(X, 0);
        chains(Y, 2);
        __builtin_amdgcn_sched_barrier(0);
        const v4f b0 = tree(X);
        __builtin_amdgcn_sched_barrier(0);
        chains(X, 1);
        __builtin_amdgcn_sched_barrier(0);
        const v4f c0 = b0 + tree(Y);
        __builtin_amdgcn_sched_barrier(0);
        chains(Y, 3);
        __builtin_amdgcn_sched_barrier(0);
        const v4f b1 = tree(X);
        const v4f c1 = b1 + tree(Y);
        const v4f sm = c0 + c1;
        const float kss = T.ks * scale;
        const int j = 16 * kt + li, at = key_pos(j - 16 * kt0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float v = sm[i] * kss;
          if constexpr (STORE) sc[(4 * lq + i) * S + at] = v;
          m4[i] = fmaxf(m4[i], j < nk4[i] ? v : -INFINITY);
        }
        if constexpr (STORE)
          if (lq == 0) vsc[at] = T.vs;
      };
      Tile A, B;
      if (kt0 + w < kt1) load(A, kt0 + w);
      for (int kt = kt0 + w; kt < kt1; kt += 2 * kWaves) {
        load(B, min(kt + kWaves, kt1 - 1));
        __builtin_amdgcn_sched_barrier(0);  // the loads stay ahead of the tile's arithmetic
        score(A, kt);
        if (kt + kWaves >= kt1) break;
        load(A, min(kt + 2 * kWaves, kt1 - 1));
        __builtin_amdgcn_sched_barrier(0);
        score(B, kt + kWaves);
      }
    };
    auto put_max = [&] {  // this wave's maxima; a row's is then the largest of the waves'
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int off = 8; off > 0; off >>= 1) m4[i] = fmaxf(m4[i], __shfl_xor(m4[i], off, 16));
        if (li == 0) max_s[w][4 * lq + i] = m4[i];
      }
    };
    if constexpr (LONG) {
      scores.template operator()<false>(0, tiles);
      put_max();
    }
    const int sr = tid >> 5, sx = tid & 31;  // softmax: threads 32 r .. 32 r + 31 of row r
    const int nkr = sr < R && ((act >> sr) & 1) ? min(nk_s[sr], nkb) : 0;
    float lane_sum = 0.0f;  // threads x < 16 of a row: lane x's sequential sum
    v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};  // P.V: values 16 w + li of rows 4 lq + i
    for (int k0 = 0; k0 < nkb; k0 += nk_pad) {
      const int tl = min(tiles, (k0 + nk_pad) / 16), st0 = k0 / kVKeys, st1 = min(nst, (k0 + nk_pad) / kVKeys);
      const int held = (st1 - st0) * kVKeys;  // keys in LDS, whole V stages
      scores.template operator()<true>(k0 / 16, tl);
      if constexpr (!LONG) put_max();
      __syncthreads();
      for (int c = st0; c < st0 + kVStages - 1 && c < st1; ++c) v_issue(c);  // in flight during the softmax

      // softmax_inplace (kernels_avx512.cpp:205-226): two keys, 16 apart, on lanes x and x + 16 per 32 keys, added in
      // that order by lane x. Past the row's end e = +0, which leaves the sum unchanged, and so is the coefficient,
      // whatever the scales of keys that only other rows have (0 * inf).
      {
        float m = max_s[0][sr];
#pragma unroll
        for (int i = 1; i < kWaves; ++i) m = fmaxf(m, max_s[i][sr]);
        float* srow = sc + sr * S;
        auto one = [&](int j) __attribute__((always_inline)) {
          const int at = key_pos(j);
          const bool in = k0 + j < nkr;
          const float e = in ? exp512(srow[at] - m) : 0.0f;
          srow[at] = in ? e * vsc[at] : 0.0f;
          return e;
        };
        for (int j = sx; j < held; j += 64) {
          const float e0 = one(j), e1 = one(j + 32);
          const float f0 = __shfl_down(e0, 16, 32), f1 = __shfl_down(e1, 16, 32);
          lane_sum = (((lane_sum + e0) + f0) + e1) + f1;
        }
      }
      lds_barrier();

      // P.V (kernels_avx512.cpp:247-265).
      struct Ops {
        float4 p[4];
        v2i v[2];  // byte s of v[h]: V of key 32 h + 4 s + lq
      } A, B;
      auto read = [&](Ops& o, int c) __attribute__((always_inline)) {
        const uint8_t* vt = smem + (c % kVStages) * kVBytes;
#pragma unroll
        for (int gk = 0; gk < 4; ++gk)
          o.p[gk] = *reinterpret_cast<const float4*>(sc + li * S + c * kVKeys - k0 + 16 * gk + 4 * lq);
        // ds_read_b64_tr_b8: lane i of a 16-lane row reads 8 bytes, (row i / 2, half i % 2) of an 8 x 16 byte tile, and
        // gets the tile's column i: here the wave's 16 values of keys 32 h + 4 r + lq, r = 0..7.
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int k = 32 * h + 4 * (li >> 1) + lq;
          o.v[h] = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
              (lds_v2i*)(vt + k * kD + 16 * (w ^ ((k >> 1) & 7)) + 8 * (li & 1)));
        }
      };
      auto run = [&](const Ops& o) __attribute__((always_inline)) {
        float v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) v[u] = (float)(int8_t)(o.v[u >> 3][(u >> 2) & 1] >> (8 * (u & 3)));
        __builtin_amdgcn_sched_barrier(0);  // no conversion between the MFMAs: each would wait for it
#pragma unroll
        for (int u = 0; u < 16; ++u) {
          const float4 p = o.p[u >> 2];
          const float pu = (u & 3) == 0 ? p.x : (u & 3) == 1 ? p.y : (u & 3) == 2 ? p.z : p.w;
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(pu, v[u], acc, 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      };
      // Stage c's copies have landed once at most those of the stages issued after it are outstanding.
      auto land = [&](int c) __attribute__((always_inline)) {
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): reads of the buffer refilled below are done
        wait_vm_stages<1, kVStages - 2>(min(kVStages - 2, st1 - 1 - c));
        ring_barrier();
        if (c + kVStages - 1 < st1) v_issue(c + kVStages - 1);
      };
      land(st0);
      read(A, st0);
      for (int c = st0; c < st1; c += 2) {
        if (c + 1 < st1) {
          land(c + 1);
          read(B, c + 1);
        }
        run(A);
        if (c + 1 >= st1) break;
        if (c + 2 < st1) {
          land(c + 2);
          read(A, c + 2);
        }
        run(B);
      }
      lds_barrier();  // every wave has read the coefficients and V: the next chunk, or the output, takes their place
    }
    {
      const float sum = reduce16_lanes(lane_sum);
      if (sx == 0) inv_s[sr] = 1.0f / sum;
    }
    lds_barrier();
    float* ob = reinterpret_cast<float*>(smem);  // [16][kD + 4]
#pragma unroll
    for (int i = 0; i < 4; ++i) ob[(4 * lq + i) * (kD + 4) + 16 * w + li] = acc[i] * inv_s[4 * lq + i];
    lds_barrier();
    {
      const int r = tid >> 5, x = tid & 31;
      if (r < R && ((act >> r) & 1)) {
        const float4 f = *reinterpret_cast<const float4*>(ob + r * (kD + 4) + 4 * x);
        const int64_t tr = t0 + r / G;
        const int hd = (g * G + r % G) * kD;
        float* o = out + tr * out_stride + hd + 4 * x;
        o[0] = f.x, o[1] = f.y, o[2] = f.z, o[3] = f.w;
        const float v[4] = {f.x, f.y, f.z, f.w};
        if (xq) quantize_block_lanes_n<4>(v, x & 7, xq + tr * xq_stride + (hd + 4 * x) / 32);
      }
    }
    done |= act;
    lds_barrier();  // the next pass rewrites the rows
  }
}

constexpr size_t kLds = 160 * 1024 - 1024;

}  // namespace

bool attention_mma_ok(int G, int D, const AttnAddr& a) { return D == kD && G <= kRows && a.k_perm && attn_aligned(a); }

bool attention_mma_whole(int max_keys) { return mma_lds_bytes(pad64(max_keys)) <= kLds; }

void attention_mma(hipStream_t s, const float* q, int64_t q_stride, float* out, int64_t out_stride, int n, int G, int KV,
                   float scale, const AttnAddr& a, const int32_t* seq, const int32_t* n_keys, int max_keys, BlockQ8* xq,
                   int64_t xq_stride, const int32_t* route) {
  const int TQ = kRows / G, max_pad = pad64(max_keys);
  auto go = [&]<bool LONG>(int nk_pad) {
    allow_lds<k_attention_mma<LONG>>((int)kLds);
    hipLaunchKernelGGL(k_attention_mma<LONG>, dim3(((n + TQ - 1) / TQ) * KV), dim3(kThreads), mma_lds_bytes(nk_pad), s, q, q_stride,
                       out, out_stride, G, scale, a, seq, n_keys, n, KV, max_pad, xq, xq_stride, route);
  };
  if (attention_mma_whole(max_keys))
    go.template operator()<false>(max_pad);
  else
    go.template operator()<true>(kChunk);
  check_launch("attention_mma");
}

}  // namespace mk
