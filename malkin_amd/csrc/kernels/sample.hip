// Candidate selection for stochastic sampling on the device (the first half of the reference's
// Sampler::distribution, sampler.cpp:22-40): repetition penalties applied to the logits in place, then per row the
// top k logits, highest first, ties by lower token id (where std::partial_sort leaves ties in an unspecified order).
// The host finishes the distribution over those k candidates (temperature, min-p, top-p, normalisation, draw), so a
// sampled request downloads k (value, id) pairs per row instead of the 608 KB logits row.
//
// Top-k per row: the logits become order-preserving 32-bit keys, and a workgroup selects the first of the keys that its
// threads hold in registers (select_k: a search for the k-th largest key, two bits per step, counted by wave ballots).
// A long row of few is cut into kSlices slices of every kSlices-th 64-logit chunk, one workgroup each (k_topk_part); each
// gives its slice_keep(k) first candidates through the context's workspace, and one workgroup per row selects from those
// and sorts (k_topk_final). Neighbouring ids fall into different slices, so a slice holds about k / kSlices of the
// row's first k; where all the candidates of a slice were selected, it may hold more, and that slice is then walked
// whole, in rounds of as many logits as the threads hold (the whole row: one row of 151936 whose first 1024 fall into one
// slice 282 us, that slice 55).
// What bounds it: two launches and the searches' barriers; the logits are read once (4.9 MB for 8 rows of 151936). See
// topk() for the times.
#include <algorithm>
#include <type_traits>

#include "ctx.h"
#include "ops.h"

namespace mk {
namespace {

constexpr int kSelThreads = 1024;            // k_topk_final
constexpr int kPartThreads = 256;            // k_topk_part
constexpr int kFinalPer = 8;                 // keys per thread (and round) of k_topk_final
constexpr int kMaxTopK = 1024;               // candidates per row held in LDS
constexpr int kSlices = 64, kChunk = 64;     // slice p of a row: its chunks p, p + kSlices, ...
constexpr int kOneSlice = kFinalPer * kSelThreads;  // logits of a row that one workgroup takes alone

// Candidates that a slice gives: four times the k / kSlices it holds on average, and 16.
__host__ __device__ constexpr int slice_keep(int k) { return k < 16 + k / 16 ? k : 16 + k / 16; }
static_assert(kSlices * slice_keep(kMaxTopK) <= kFinalPer * kSelThreads, "one workgroup holds a row's candidates");

// Rows that are selected from in slices at most: the workspace holds their candidates at any k (10 MB).
constexpr int kSliceRows = 256;

// Logits of a slice, some of them past the row's end.
__host__ __device__ constexpr int slice_logits(int n_vocab) {
  return (int)((n_vocab + (int64_t)kSlices * kChunk - 1) / (kSlices * kChunk)) * kChunk;
}

// Larger float -> larger key, never 0 (finite values and infinities; NaN logits are not expected).
__device__ __forceinline__ uint32_t order_key(float f) {
  const uint32_t u = __float_as_uint(f);
  return max((u & 0x80000000u) ? ~u : (u | 0x80000000u), 1u);
}

// One row per block: l[pen_id[i]] -= pen_amt[i] for this row's entries pen_off[r] .. pen_off[r + 1].
__global__ void k_penalize(float* __restrict__ logits, int64_t stride, const int32_t* __restrict__ rows,
                           const int32_t* __restrict__ pen_off, const int32_t* __restrict__ pen_id,
                           const float* __restrict__ pen_amt, int n_vocab) {
  const int r = blockIdx.x;
  float* l = logits + (int64_t)(rows ? rows[r] : r) * stride;
  for (int i = pen_off[r] + (int)threadIdx.x; i < pen_off[r + 1]; i += (int)blockDim.x) {
    const int id = pen_id[i];
    if (id >= 0 && id < n_vocab) l[id] = l[id] - pen_amt[i];
  }
}

// A T that separates the k largest of the workgroup's keys (E per thread): the largest T with at least k keys >= T, or
// any with exactly k. Two bits per step from the top, the counts of the three candidate values by wave ballots and one
// LDS add per wave; the search ends at the first prefix that k keys reach exactly (without ties about half of the 16
// steps: 8 rows of 151936 random logits at k = 40 29.5 -> 23.2 us). cnt: kSteps groups of 3 zeroed counters, fresh ones per
// step, so that one barrier per step suffices. k >= 1; where fewer keys are not 0, T = 0.
constexpr int kSteps = 16;
template <int E>
__device__ __forceinline__ uint32_t separate(const uint32_t (&key)[E], uint32_t k, uint32_t* cnt) {
  uint32_t T = 0;
  for (int st = 0; st < kSteps; ++st) {
    const int shift = 30 - 2 * st;
    uint32_t c[3] = {0, 0, 0};
#pragma unroll
    for (int e = 0; e < E; ++e)
#pragma unroll
      for (int v = 0; v < 3; ++v) c[v] += (uint32_t)__popcll(__ballot(key[e] >= (T | ((uint32_t)(v + 1) << shift))));
    if ((threadIdx.x & 63) < 3) {
      const uint32_t own = (threadIdx.x & 63) == 0 ? c[0] : (threadIdx.x & 63) == 1 ? c[1] : c[2];
      if (own) atomicAdd(&cnt[3 * st + (threadIdx.x & 63)], own);
    }
    __syncthreads();
    const uint32_t *g = cnt + 3 * st;
    const uint32_t v = g[2] >= k ? 3u : g[1] >= k ? 2u : g[0] >= k ? 1u : 0u;
    T |= v << shift;
    if (v != 0 && g[v - 1] == k) break;
  }
  return T;
}

// LDS of one selection.
struct SelLds {
  uint32_t cnt[2][3 * kSteps];  // the counters of the two searches
  uint32_t gt, eq, slot;
};

// put(slot, key, id) for the k first keys of the workgroup in the order (key desc, id asc), slots 0 .. k - 1 in any order;
// returns how many. Threads without a key hold (0, INT32_MAX), below every logit's key; where fewer than k hold one, T is 0
// and only the keys above 0 are put.
template <int E, class Put>
__device__ __forceinline__ int select_k(const uint32_t (&key)[E], const int32_t (&id)[E], int k, SelLds& L, Put put) {
  const int tid = threadIdx.x, lane = tid & 63;
  if (tid < 2 * 3 * kSteps) (&L.cnt[0][0])[tid] = 0;
  if (tid == 0) L.gt = L.eq = L.slot = 0;
  __syncthreads();
  const uint32_t T = separate(key, (uint32_t)k, L.cnt[0]);
  uint32_t ngt = 0, neq = 0;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    ngt += (uint32_t)__popcll(__ballot(key[e] > T));
    neq += (uint32_t)__popcll(__ballot(key[e] == T));
  }
  if (lane == 0) {
    if (ngt) atomicAdd(&L.gt, ngt);
    if (neq) atomicAdd(&L.eq, neq);
  }
  __syncthreads();
  // Of the keys equal to T, the need lowest ids: those with the need largest ~id among them (all of them where T
  // already separates k keys).
  const uint32_t need = (uint32_t)k - L.gt;
  uint32_t U = 0;
  if (T != 0 && L.eq > need) {
    uint32_t inv[E];
#pragma unroll
    for (int e = 0; e < E; ++e) inv[e] = key[e] == T ? ~(uint32_t)id[e] : 0u;
    U = separate(inv, need, L.cnt[1]);
  }
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const bool take = key[e] > T || (T != 0 && key[e] == T && ~(uint32_t)id[e] >= U);
    const unsigned long long bal = __ballot(take);
    if (bal == 0) continue;
    uint32_t base = 0;
    if (lane == 0) base = atomicAdd(&L.slot, (uint32_t)__popcll(bal));
    base = (uint32_t)__shfl((int)base, 0);
    if (take) put(base + (uint32_t)__popcll(bal & ((1ull << lane) - 1ull)), key[e], id[e]);
  }
  return T != 0 ? k : (int)L.gt;
}

// Slice p of a row: its slice_keep(k) first candidates (all of them, then (0, INT32_MAX), where it holds no more) to
// cand[row][p][keep]. A slice of more logits than the threads hold is walked in rounds, each over the candidates so far
// and the next logits. E: logits per thread and round.
template <int E>
__global__ __launch_bounds__(kPartThreads) void k_topk_part(const float* __restrict__ logits, int64_t stride,
                                                             const int32_t* __restrict__ rows, int n_vocab, int keep,
                                                             uint2* cand) {
  constexpr int NT = kPartThreads;
  __shared__ SelLds L;
  const int tid = threadIdx.x, r = blockIdx.y, p = blockIdx.x;
  const float* l = logits + (int64_t)(rows ? rows[r] : r) * stride;
  auto at = [&](int j) { return ((int64_t)(j / kChunk) * kSlices + p) * kChunk + j % kChunk; };  // slice logit j
  const int n = slice_logits(n_vocab);
  uint2* out = cand + ((int64_t)r * kSlices + p) * keep;
  uint32_t key[E];
  int32_t id[E];
  for (int pos = 0, held = 0;;) {  // held: entries of out that join this round (0, then keep)
    const int take = min(n - pos, E * NT - held);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int i = e * NT + tid, j = i - held;
      const int64_t v = at(pos + j);
      const bool in = j >= 0 && j < take && v < n_vocab;
      const uint2 old = i < held ? out[i] : make_uint2(0u, (uint32_t)INT32_MAX);
      id[e] = in ? (int32_t)v : (int32_t)old.y;
      key[e] = in ? order_key(l[v]) : old.x;
    }
    __syncthreads();  // out has been read
    const int got =
        select_k(key, id, keep, L, [&](uint32_t slot, uint32_t kk, int32_t ii) { out[slot] = make_uint2(kk, (uint32_t)ii); });
    for (int i = got + tid; i < keep; i += NT) out[i] = make_uint2(0u, (uint32_t)INT32_MAX);
    pos += take;
    if (pos >= n) return;
    held = keep;
    __syncthreads();  // out has been written, L has been read
  }
}

// One row's k first, sorted: from its slices' candidates (SLICED: cand[row][kSlices][keep]) and the logits of those slices
// whose candidates were all selected, or from the row's logits, in rounds of the keys the threads hold and the best so
// far. WAVES: per SIMD; 8 put two rows on a CU (512 rows of 151936 at k = 40 404 -> 294 us) but have the searches' counts
// spill to lanes of vector registers, which costs a walked row that has its CU alone 3 %.
template <int WAVES, bool SLICED>
__global__ __launch_bounds__(kSelThreads) __attribute__((amdgpu_waves_per_eu(WAVES))) void k_topk_final(
    const float* __restrict__ logits, int64_t stride, const int32_t* __restrict__ rows, int n_vocab,
    const uint2* __restrict__ cand, int k, float* __restrict__ out_v, int32_t* __restrict__ out_i) {
  constexpr int E = kFinalPer, NT = kSelThreads;
  __shared__ SelLds L;
  __shared__ uint32_t ckey[kMaxTopK];
  __shared__ int32_t cidx[kMaxTopK];
  __shared__ int taken[kSlices], full[kSlices], n_full, again;
  const int tid = threadIdx.x, r = blockIdx.x;
  const int keep = slice_keep(k);
  auto slice_of = [](int32_t i) { return (int)((uint32_t)i / kChunk % kSlices); };
  auto put = [&](uint32_t slot, uint32_t kk, int32_t ii) {
    ckey[slot] = kk;
    cidx[slot] = ii;
  };
  if constexpr (SLICED) {
    const int n = kSlices * keep;
    const uint2* c = cand + (int64_t)r * n;
    if (tid < kSlices) taken[tid] = 0;
    if (tid == 0) again = 0;
    auto from_cand = [&]<int M>() __attribute__((always_inline)) {
      uint32_t key[M];
      int32_t id[M];
#pragma unroll
      for (int e = 0; e < M; ++e) {
        const int i = e * NT + tid;
        const uint2 v = i < n ? c[i] : make_uint2(0u, (uint32_t)INT32_MAX);
        key[e] = v.x;
        id[e] = (int32_t)v.y;
      }
      select_k(key, id, k, L, put);
    };
    if (n <= 2 * NT)
      from_cand.template operator()<2>();
    else
      from_cand.template operator()<E>();
    __syncthreads();
    for (int i = tid; i < k; i += NT)
      if (atomicAdd(&taken[slice_of(cidx[i])], 1) + 1 >= keep && keep < k) again = 1;
    __syncthreads();
    if (again) {
      if (tid < kSlices) {
        const unsigned long long bal = __ballot(taken[tid] >= keep);
        if (taken[tid] >= keep) full[__popcll(bal & ((1ull << tid) - 1ull))] = tid;
        if (tid == 0) n_full = __popcll(bal);
      }
      // The walk meets these slices' candidates again. (Entry i is read there by the thread that clears it.)
      for (int i = tid; i < k; i += NT)
        if (taken[slice_of(cidx[i])] >= keep) put(i, 0u, INT32_MAX);
      __syncthreads();
    }
  }
  // The row's logits, or those of its full slices.
  using Pos = std::conditional_t<SLICED, int64_t, int>;
  const uint32_t nsl = (uint32_t)slice_logits(n_vocab);
  const Pos walk = !SLICED ? (Pos)n_vocab : again ? (Pos)n_full * nsl : 0;
  if (walk) {
    const float* l = logits + (int64_t)(rows ? rows[r] : r) * stride;
    uint32_t key[E];
    int32_t id[E];
    int held = SLICED ? k : 0;
    for (Pos pos = 0; pos < walk;) {
      const int take = (int)min(walk - pos, (Pos)(E * NT - held));
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int i = e * NT + tid, j = i - held;
        bool in = j >= 0 && j < take;
        Pos v = pos + j;
        if constexpr (SLICED)
          if (in) {
            const uint32_t q = (uint32_t)v, c = q % nsl;
            v = ((Pos)(c / kChunk) * kSlices + full[q / nsl]) * kChunk + c % kChunk;
            in = v < n_vocab;
          }
        id[e] = in ? (int32_t)v : i < held ? cidx[i] : INT32_MAX;
        key[e] = in ? order_key(l[v]) : i < held ? ckey[i] : 0u;
      }
      __syncthreads();  // the best so far have been read
      select_k(key, id, k, L, put);
      pos += take;
      held = k;
      __syncthreads();  // they have been written, L has been read
    }
  }
  // Sorted by key descending, index ascending: up to 128 by counting those before each, more by a bitonic sort
  // (padded to a power of two).
  auto before_in_order = [](uint32_t ka, int ia, uint32_t kb, int ib) { return ka > kb || (ka == kb && ia < ib); };
  auto emit = [&](int i, uint32_t u, int32_t ii) {  // order_key undone: the logit's own bits
    out_i[(int64_t)r * k + i] = ii;
    out_v[(int64_t)r * k + i] = __uint_as_float((u & 0x80000000u) ? u & 0x7FFFFFFFu : ~u);
  };
  if (k <= 128) {
    __syncthreads();
    if (tid < k) {
      const uint32_t u = ckey[tid];
      const int32_t ii = cidx[tid];
      int rank = 0;
      for (int j = 0; j < k; ++j) rank += before_in_order(ckey[j], cidx[j], u, ii) ? 1 : 0;
      emit(rank, u, ii);
    }
    return;
  }
  int n2 = 1;
  while (n2 < k) n2 <<= 1;
  for (int i = k + tid; i < n2; i += NT) {
    ckey[i] = 0u;
    cidx[i] = INT32_MAX;
  }
  __syncthreads();
  for (int size = 2; size <= n2; size <<= 1)
    for (int stride2 = size >> 1; stride2 > 0; stride2 >>= 1) {
      for (int i = tid; i < n2; i += NT) {
        const int j = i ^ stride2;
        if (j > i) {
          const bool up = (i & size) == 0;  // this run sorted in order (up) or reversed
          const bool swap = up ? before_in_order(ckey[j], cidx[j], ckey[i], cidx[i])
                               : before_in_order(ckey[i], cidx[i], ckey[j], cidx[j]);
          if (swap) {
            const uint32_t tk = ckey[i];
            const int ti = cidx[i];
            ckey[i] = ckey[j];
            cidx[i] = cidx[j];
            ckey[j] = tk;
            cidx[j] = ti;
          }
        }
      }
      __syncthreads();
    }
  for (int i = tid; i < k; i += NT) emit(i, ckey[i], cidx[i]);
}

}  // namespace

size_t topk_workspace() { return (size_t)kSliceRows * kSlices * slice_keep(kMaxTopK) * sizeof(uint2); }

void penalize(hipStream_t s, float* logits, int64_t stride, const int32_t* rows, int n_rows, int n_vocab,
              const int32_t* pen_off, const int32_t* pen_id, const float* pen_amt) {
  if (n_rows <= 0) return;
  require(pen_off != nullptr && pen_id != nullptr && pen_amt != nullptr, "penalize: missing penalty lists");
  hipLaunchKernelGGL(k_penalize, dim3(n_rows), dim3(256), 0, s, logits, stride, rows, pen_off, pen_id, pen_amt,
                     n_vocab);
  check_launch("penalize");
}

// Rows of up to kOneSlice logits take one workgroup each, and so do longer rows where there are many of them: slices pay
// while the chip would be idle, but cost a row 64 workgroups of its own. A row of n logits walked by one workgroup takes
// about as long as slices of n / 256 rows (us, walked / slices: 64 rows of 8193 at k = 40 17 / 26, 8 rows 16 / 15; 128 rows of
// 32768 51 / 42, 256 rows 51 / 70; 256 rows of 151936 209 / 228, 64 rows 209 / 68). Past kSliceRows rows the walks fill the
// chip. Against one workgroup walking each row by histograms (this file's first form): 8 rows of 151936 at k = 40
// 276 -> 21 us (1024: 287 -> 46), one row 238 -> 18, 64 rows 387 -> 68, 512 rows 461 -> 294; 8 rows of 8193 56 -> 15, 256 rows
// 59 -> 17, and of 8192, which one workgroup selects from registers in one round, 57 -> 12. A slice's threads hold 4, 8, 12
// or 16 logits each, as many as it needs: the searches' ballots are what k_topk_part spends its time on.
void topk(hipStream_t s, const float* logits, int64_t stride, const int32_t* rows, int n_rows, int n_vocab, int k,
          float* out_v, int32_t* out_i, void* workspace) {
  if (n_rows <= 0) return;
  require(k >= 1 && k <= kMaxTopK && k <= n_vocab, "topk: k must be 1..1024 and at most the vocabulary");
  const bool sliced = n_vocab > kOneSlice && n_rows <= std::min(n_vocab / 256, kSliceRows);
  uint2* cand = sliced ? static_cast<uint2*>(workspace) : nullptr;
  if (sliced) {
    auto part = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(kSlices, n_rows), dim3(kPartThreads), 0, s, logits, stride, rows, n_vocab,
                         slice_keep(k), cand);
    };
    const int per = (slice_logits(n_vocab) + kPartThreads - 1) / kPartThreads;
    per <= 4    ? part(k_topk_part<4>)
    : per <= 8  ? part(k_topk_part<8>)
    : per <= 12 ? part(k_topk_part<12>)
                : part(k_topk_part<16>);
  }
  auto final = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(n_rows), dim3(kSelThreads), 0, s, logits, stride, rows, n_vocab, cand, k, out_v, out_i);
  };
  sliced                  ? final(k_topk_final<4, true>)
  : n_rows > device_cus() ? final(k_topk_final<8, false>)
                          : final(k_topk_final<4, false>);
  check_launch("topk");
}

}  // namespace mk
