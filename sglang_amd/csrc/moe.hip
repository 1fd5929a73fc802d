// Fused-MoE side of the path for gfx950: moe_align_block_size (stable counting sort into
// block-padded expert spans), the sorted-block grouped block-FP8 GEMM (same MFMA core as
// the dense GEMM, rows gathered through the sorted token list), silu_and_mul and the
// top-k sum reduce.
#include "moe_dispatch.h"
#include "quant_core.h"
#include <algorithm>
#include <cmath>

namespace sglamd {

// ---------------------------------------------------------------------------------------
// moe_align_block_size: `parts` workgroups of 1024 lanes that never talk to each other.  The flat ids are cut
// into 16 * parts contiguous chunks; workgroup p places the ids of chunks 16 p .. 16 p + 15, one per wave.
//   1. every wave histograms its own chunk (bucket = id + 1) in LDS; the ids of the other workgroups' chunks are
//      counted by all lanes together, those in front of this workgroup's chunks and those behind them apart
//      (each workgroup reads all ids: a few hundred KB from L2, against scattered 4-byte stores that one CU
//      issues at about one per nanosecond and that the parts share),
//   2. padded totals -> exclusive prefix P (wave scans + carry), the same in every workgroup,
//   3. expert id of every block, total, cumsum buffer, padding fill (bucket b by workgroup b % parts); the per-wave
//      counts are turned into each wave's first slot per bucket (P[b] + ids in front of the workgroup's chunks +
//      counts of the waves in front),
//   4. stable scatter without workgroup barriers: a wave walks its chunk 64 ids at a time; a
//      lane's slot is the wave's running offset of the bucket plus the same-bucket lanes in
//      front of it, so every span is filled in ascending flat index.
// LDS: cnt[NB] | prefix[NB+1] | wavecnt[16][NB]   (NB = number of buckets, at most 3072; the counts of the ids in
// front share prefix[] until the scan and live in the registers of the lanes that own their buckets after it)
// ---------------------------------------------------------------------------------------
// PREP = true turns the same sort into prepare_moe_input: block size 1 (no padding), and instead of the sorted
// slot list it emits the two permutations, the expert offsets and the per-expert problem sizes.
struct MoePrepArgs {
  int32_t* expert_offsets;      // [E + 1]
  int32_t* blockscale_offsets;  // [E + 1] or null: offsets with every expert's rows rounded up to 128
  int32_t* problem_sizes1;      // [E, 3] = (rows, 2n, k)
  int32_t* problem_sizes2;      // [E, 3] = (rows, k, n)
  int32_t* input_permutation;   // [numel]: expert-major position -> token; null: no permutations are written
  int32_t* output_permutation;  // [numel]: flat (token, j) -> expert-major position
  int topk, n, k;
};

static inline size_t moe_align_lds_bytes(int nb) { return (size_t)(3 * nb + 1 + 16 * nb) * sizeof(int32_t); }
// Workgroups sharing one sort: one up to 1023 ids (the decode path: nothing to share), then one per 512 ids, 16 at most.
// Layers of 1100 to 4800 ids take 1-4 % less time than with one per 2048 from 4096 ids on.
static inline int moe_align_parts(int64_t numel) {
  if (numel < 1024) return 1;
  return (int)(numel / 512 < 16 ? numel / 512 : 16);
}

template <typename IdT, bool PREP = false>
__device__ __forceinline__ void moe_align_body(const IdT* __restrict__ topk_ids, int32_t* sorted_ids,
                                               int32_t* expert_ids, int32_t* post_pad_out, int32_t* cumsum_out, int nb,
                                               int block_size, int numel, int pad_fill, int max_padded, int part,
                                               int parts, MoePrepArgs pa = MoePrepArgs()) {
  extern __shared__ int32_t lds[];
  int32_t* cnt = lds;
  int32_t* prefix = cnt + nb;
  int32_t* wavecnt = prefix + nb + 1;
  int32_t* before = prefix;  // until the scan writes prefix[]
  __shared__ int32_t s_carry;
  __shared__ int32_t s_wsum[16];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

  for (int i = tid; i < 16 * nb; i += 1024) wavecnt[i] = 0;
  for (int i = tid; i < nb; i += 1024) cnt[i] = 0, before[i] = 0;
  if (tid == 0) s_carry = 0;
  __syncthreads();

  // Every wave owns one contiguous chunk of the flat ids (a multiple of 64 long), so ascending flat index
  // is workgroup first, wave second, position inside the wave's chunk third.
  const int chunk = ((numel + 16 * parts - 1) / (16 * parts) + 63) & ~63;
  const int wg_begin = min(numel, part * 16 * chunk), wg_end = min(numel, wg_begin + 16 * chunk);
  const int c_begin = min(numel, wg_begin + wave * chunk), c_end = min(numel, c_begin + chunk);
  int32_t* mycnt = wavecnt + wave * nb;
  // Ids are fetched ALIGN_BATCH x 64 at a time, all loads of a batch before their first use (one load per loop
  // turn would cost the wave a full memory latency per 64 ids).
  constexpr int ALIGN_BATCH = 8;
  auto bucket_at = [&](int i, int end) -> int {
    if (i >= end) return -1;
    const int b = (int)topk_ids[i] + 1;
    return (b < 0 || b >= nb) ? -1 : b;
  };
  auto bucket_of = [&](int i) -> int { return bucket_at(i, c_end); };
  for (int base = c_begin; base < c_end; base += 64 * ALIGN_BATCH) {
    int bb[ALIGN_BATCH];
#pragma unroll
    for (int u = 0; u < ALIGN_BATCH; u++) bb[u] = bucket_of(base + u * 64 + lane);
#pragma unroll
    for (int u = 0; u < ALIGN_BATCH; u++)
      if (bb[u] >= 0) atomicAdd(&mycnt[bb[u]], 1);
  }
  // the other workgroups' ids: in front of this workgroup's chunks -> before[], behind them -> cnt[]
  for (int side = 0; side < 2; side++) {
    const int lo = side ? wg_end : 0, hi = side ? numel : wg_begin;
    int32_t* dst = side ? cnt : before;
    for (int base = lo; base < hi; base += 1024 * ALIGN_BATCH) {
      int bb[ALIGN_BATCH];
#pragma unroll
      for (int u = 0; u < ALIGN_BATCH; u++) bb[u] = bucket_at(base + u * 1024 + tid, hi);
#pragma unroll
      for (int u = 0; u < ALIGN_BATCH; u++)
        if (bb[u] >= 0) atomicAdd(&dst[bb[u]], 1);
    }
  }
  __syncthreads();
  int bef[3] = {0, 0, 0};  // before[] of buckets tid, tid + 1024, tid + 2048
  for (int b = tid; b < nb; b += 1024) {
    int t = 0;
    for (int w = 0; w < 16; w++) t += wavecnt[w * nb + b];
    const int f = before[b];
    if (b < 1024) bef[0] = f;
    else if (b < 2048) bef[1] = f;
    else bef[2] = f;
    cnt[b] += t + f;
  }
  __syncthreads();

  // exclusive scan of the padded counts, 1024 buckets per round
  for (int base = 0; base < nb; base += 1024) {
    const int b = base + tid;
    const int padded = b < nb ? (cnt[b] + block_size - 1) / block_size * block_size : 0;
    int incl = padded;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int v = __shfl_up(incl, off, 64);
      if (lane >= off) incl += v;
    }
    if (lane == 63) s_wsum[wave] = incl;
    __syncthreads();
    int woff = 0;
    for (int w = 0; w < wave; w++) woff += s_wsum[w];
    const int carry = s_carry;
    if (b < nb) prefix[b] = carry + woff + incl - padded;
    __syncthreads();
    if (tid == 1023) s_carry = carry + woff + incl;
    __syncthreads();
  }
  if (tid == 0) {
    prefix[nb] = s_carry;
    if (post_pad_out && part == 0) *post_pad_out = s_carry;
  }
  __syncthreads();

  const int post_pad = prefix[nb];
  for (int b = tid; b < nb; b += 1024) {
    // per-wave counts become the slot at which each wave starts writing bucket b
    int running = prefix[b] + (b < 1024 ? bef[0] : b < 2048 ? bef[1] : bef[2]);
    for (int w = 0; w < 16; w++) {
      const int t = wavecnt[w * nb + b];
      wavecnt[w * nb + b] = running;
      running += t;
    }
    if (b % parts != part) continue;  // the outputs of bucket b come from one workgroup
    if (PREP) {
      // bucket 0 holds the ids == -1, which take no part: positions count from the end of that bucket
      if (b >= 1) {
        const int e = b - 1;
        pa.expert_offsets[e] = prefix[b] - prefix[1];
        pa.problem_sizes1[e * 3] = cnt[b];
        pa.problem_sizes1[e * 3 + 1] = 2 * pa.n;
        pa.problem_sizes1[e * 3 + 2] = pa.k;
        pa.problem_sizes2[e * 3] = cnt[b];
        pa.problem_sizes2[e * 3 + 1] = pa.k;
        pa.problem_sizes2[e * 3 + 2] = pa.n;
      }
    } else {
      for (int j = prefix[b] / block_size; j < prefix[b + 1] / block_size; j++) expert_ids[j] = b - 1;
    }
    if (cumsum_out) cumsum_out[b] = prefix[b] + cnt[b];
    if (pad_fill)
      for (int j = prefix[b] + cnt[b]; j < prefix[b + 1]; j++) sorted_ids[j] = numel;
  }
  if (cumsum_out && tid == 0 && part == 0) cumsum_out[nb] = post_pad;
  if (PREP && tid == 0 && part == 0) {
    pa.expert_offsets[nb - 1] = post_pad - prefix[1];
    if (pa.blockscale_offsets) {
      int rounded = 0;
      for (int b = 1; b < nb; b++) {
        pa.blockscale_offsets[b - 1] = rounded;
        rounded += (cnt[b] + 127) / 128 * 128;
      }
      pa.blockscale_offsets[nb - 1] = rounded;
    }
  }
  if (PREP && !pa.input_permutation) return;  // offsets and sizes only
  const int prep_base = PREP ? prefix[1] : 0;
  if (pad_fill)
    for (int j = post_pad + part * 1024 + tid; j < max_padded; j += 1024 * parts) sorted_ids[j] = numel;
  __syncthreads();

  // Stable scatter, one wave per chunk and no workgroup barrier: 64 ids at a time, a lane's slot is its wave's
  // running offset for the bucket plus the number of same-bucket lanes in front of it.
  volatile int32_t* myoff = mycnt;
  const int key_bits = 32 - __clz(max(nb - 1, 1));
  for (int base0 = c_begin; base0 < c_end; base0 += 64 * ALIGN_BATCH) {
    int bb[ALIGN_BATCH];
#pragma unroll
    for (int u = 0; u < ALIGN_BATCH; u++) bb[u] = bucket_of(base0 + u * 64 + lane);
#pragma unroll
    for (int u = 0; u < ALIGN_BATCH; u++) {
      const int i = base0 + u * 64 + lane;
      const int b = bb[u];
      // lanes of this wave with the same bucket: intersect, bit by bit of the bucket number, the lanes that agree
      unsigned long long m = __ballot(b >= 0);
      if (m == 0) continue;  // past the end of the chunk (wave-uniform)
      for (int k = 0; k < key_bits; k++) {
        const bool bit = (b >> k) & 1;
        const unsigned long long bal = __ballot(bit);
        m &= bit ? bal : ~bal;
      }
      const int rank = __popcll(m & ((1ull << lane) - 1ull));
      const int total = __popcll(m);
      const bool leader = b >= 0 && rank == 0;
      int off = 0;
      if (b >= 0) off = myoff[b];
      __builtin_amdgcn_wave_barrier();
      if (leader) myoff[b] = off + total;
      if (PREP) {
        if (b >= 1) {
          const int pos = off + rank - prep_base;
          pa.input_permutation[pos] = i / pa.topk;
          pa.output_permutation[i] = pos;
        }
      } else {
        if (b >= 0) sorted_ids[off + rank] = i;
      }
    }
  }
}

template <typename IdT>
__global__ __launch_bounds__(1024) void moe_align_kernel(const IdT* __restrict__ topk_ids, int32_t* sorted_ids,
                                                         int32_t* expert_ids, int32_t* post_pad_out,
                                                         int32_t* cumsum_out, int nb, int block_size, int numel,
                                                         int pad_fill, int max_padded) {
  moe_align_body<IdT>(topk_ids, sorted_ids, expert_ids, post_pad_out, cumsum_out, nb, block_size, numel, pad_fill,
                      max_padded, (int)blockIdx.x, (int)gridDim.x);
}

// First launch of the fused MoE layer: the first `parts` workgroups sort the tokens, the others quantise the hidden
// states (group 128, reciprocal form).  The jobs are independent, so sharing a launch only removes one launch latency
// from the decode path.  TABLES: one more workgroup behind the sorting ones writes the expert offsets and problem sizes
// that callers of the expert-major interface hand in.
template <typename IdT, typename T, bool TABLES = false>
__global__ __launch_bounds__(1024) void moe_prologue_kernel(const IdT* __restrict__ topk_ids, int32_t* sorted_ids,
                                                            int32_t* expert_ids, int32_t* post_pad_out,
                                                            int32_t* cumsum_out, int nb, int block_size, int numel,
                                                            int max_padded, int parts, GroupQuantArgs qa,
                                                            MoePrepArgs pa) {
  const int wg = (int)blockIdx.x - parts;
  if (wg < 0)
    moe_align_body<IdT>(topk_ids, sorted_ids, expert_ids, post_pad_out, cumsum_out, nb, block_size, numel, 1, max_padded,
                        (int)blockIdx.x, parts);
  else if (TABLES && wg == 0)
    moe_align_body<IdT, true>(topk_ids, nullptr, nullptr, nullptr, nullptr, nb, 1, numel, 0, 0, 0, 1, pa);
  else
    group_quant_body<T, 128, false, true>(qa, (int64_t)(wg - (TABLES ? 1 : 0)) * 1024 + threadIdx.x);
}

// The same for the row-scaled layers: one row of hidden states per workgroup behind the sorting ones.
// TEAM: 1024 / TEAM rows per workgroup (row_quant_body).
template <typename IdT, typename T, bool INT8, int NV, int TEAM = 0>
__global__ __launch_bounds__(1024) void moe_row_prologue_kernel(const IdT* __restrict__ topk_ids, int32_t* sorted_ids,
                                                                int32_t* expert_ids, int32_t* post_pad_out,
                                                                int32_t* cumsum_out, int nb, int block_size, int numel,
                                                                int max_padded, int parts, RowQuantArgs qa) {
  __shared__ float red[16];
  if ((int)blockIdx.x < parts)
    moe_align_body<IdT>(topk_ids, sorted_ids, expert_ids, post_pad_out, cumsum_out, nb, block_size, numel, 1, max_padded,
                        (int)blockIdx.x, parts);
  else
    row_quant_body<T, INT8, false, NV, TEAM>(
        qa, TEAM ? (int64_t)((int)blockIdx.x - parts) * (1024 / (TEAM ? TEAM : 1)) + threadIdx.x / (TEAM ? TEAM : 1) : (int)blockIdx.x - parts, red);
}

// prepare_moe_input: the stable sort above with block size 1, emitting permutations and problem sizes.
__global__ __launch_bounds__(1024) void moe_prepare_kernel(const int32_t* __restrict__ topk_ids, int nb, int numel,
                                                           MoePrepArgs pa) {
  moe_align_body<int32_t, true>(topk_ids, nullptr, nullptr, nullptr, nullptr, nb, 1, numel, 0, 0, (int)blockIdx.x,
                                (int)gridDim.x, pa);
}

// shuffle_rows: output row r = input row dst2src[r]; rows are moved as VEC-byte pieces.
template <typename VT>
__global__ __launch_bounds__(256) void shuffle_rows_kernel(const uint8_t* __restrict__ in, const int32_t* __restrict__ map,
                                                           uint8_t* __restrict__ out, int64_t num_dst, int64_t row_bytes) {
  const int64_t pieces = row_bytes / (int64_t)sizeof(VT);
  for (int64_t r = blockIdx.x; r < num_dst; r += gridDim.x) {
    const VT* src = (const VT*)(in + (int64_t)map[r] * row_bytes);
    VT* dst = (VT*)(out + r * row_bytes);
    for (int64_t j = threadIdx.x; j < pieces; j += 256) dst[j] = src[j];
  }
}

// apply_shuffle_mul_sum: out[i, :] = sum_j factor[i*topk + j] * in[perm[i*topk + j], :], accumulated in fp32
// in the order j = 0 .. topk-1; one workgroup per (token, 2048-column slice).
template <typename T>
__global__ __launch_bounds__(256) void shuffle_mul_sum_kernel(const u16* __restrict__ in, u16* __restrict__ out,
                                                              const int32_t* __restrict__ perm,
                                                              const u16* __restrict__ factors, int topk, int d) {
  const int i = blockIdx.x;
  const int32_t* p = perm + (int64_t)i * topk;
  const u16* f = factors ? factors + (int64_t)i * topk : nullptr;
  u16* o = out + (int64_t)i * d;
  if ((d & 7) == 0) {
    for (int j = (blockIdx.y * 256 + threadIdx.x) * 8; j < d; j += gridDim.y * 2048) {
      float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      for (int k = 0; k < topk; k++) {
        const float w = f ? T::to_f32(f[k]) : 1.f;
        const v4i v = *(const v4i*)(in + (int64_t)p[k] * d + j);
        u16 b[8];
        __builtin_memcpy(b, &v, 16);
#pragma unroll
        for (int e = 0; e < 8; e++) acc[e] = fmaf(w, T::to_f32(b[e]), acc[e]);
      }
      u16 ob[8];
#pragma unroll
      for (int e = 0; e < 8; e++) ob[e] = T::from_f32(acc[e]);
      v4i ov;
      __builtin_memcpy(&ov, ob, 16);
      *(v4i*)(o + j) = ov;
    }
  } else {
    for (int j = blockIdx.y * 256 + threadIdx.x; j < d; j += gridDim.y * 256) {
      float acc = 0.f;
      for (int k = 0; k < topk; k++)
        acc = fmaf(f ? T::to_f32(f[k]) : 1.f, T::to_f32(in[(int64_t)p[k] * d + j]), acc);
      o[j] = T::from_f32(acc);
    }
  }
}

// The same sum over rows that lie in (token, k) order already, factors as floats that are rounded to T first.
template <typename T>
__global__ __launch_bounds__(256) void weighted_sum_kernel(const u16* __restrict__ in, u16* __restrict__ out,
                                                           const float* __restrict__ factors, int topk, int d) {
  const int64_t i = blockIdx.x;
  const u16* src = in + i * topk * d;
  const float* f = factors + i * topk;
  for (int j = (blockIdx.y * 256 + threadIdx.x) * 8; j < d; j += gridDim.y * 2048) {
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < topk; k++) {
      const float w = T::to_f32(T::from_f32(f[k]));
      const v4i v = *(const v4i*)(src + (int64_t)k * d + j);
      u16 b[8];
      __builtin_memcpy(b, &v, 16);
#pragma unroll
      for (int e = 0; e < 8; e++) acc[e] = fmaf(w, T::to_f32(b[e]), acc[e]);
    }
    u16 ob[8];
#pragma unroll
    for (int e = 0; e < 8; e++) ob[e] = T::from_f32(acc[e]);
    v4i ov;
    __builtin_memcpy(&ov, ob, 16);
    *(v4i*)(out + i * d + j) = ov;
  }
}

// Sorted-block schedule of a grouped GEMM whose rows are already expert-major: expert e owns rows
// [offsets[e], offsets[e] + problem_sizes[e][0]).  Every expert gets ceil(rows / block_m) blocks; slot values
// are row numbers, slots past an expert's last row hold num_rows (the "no row" value of the GEMM kernels).  Every
// workgroup forms the prefix over the experts itself (a few KB from L2) and fills its share of the slots: one workgroup
// alone took 31 us for the 36000 slots of 4096 rows over 256 experts.
__global__ __launch_bounds__(1024) void grouped_schedule_kernel(const int32_t* __restrict__ problem_sizes,
                                                                const int32_t* __restrict__ offsets, int num_experts,
                                                                int block_m, int num_rows, int max_blocks,
                                                                int32_t* sorted_ids, int32_t* expert_ids,
                                                                int32_t* post_pad) {
  extern __shared__ int32_t lds[];  // first[E + 1]: first block of every expert
  __shared__ int32_t s_wsum[16];
  __shared__ int32_t s_carry;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (tid == 0) s_carry = 0;
  __syncthreads();
  for (int base = 0; base < num_experts; base += 1024) {
    const int e = base + tid;
    int rows = e < num_experts ? problem_sizes[e * 3] : 0;
    rows = min(max(rows, 0), num_rows);
    const int nblk = (rows + block_m - 1) / block_m;
    int incl = nblk;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int v = __shfl_up(incl, off, 64);
      if (lane >= off) incl += v;
    }
    if (lane == 63) s_wsum[wave] = incl;
    __syncthreads();
    int woff = 0;
    for (int w = 0; w < wave; w++) woff += s_wsum[w];
    const int carry = s_carry;
    if (e < num_experts) lds[e] = carry + woff + incl - nblk;
    __syncthreads();
    if (tid == 1023) s_carry = carry + woff + incl;
    __syncthreads();
  }
  const int total = min(s_carry, max_blocks);
  if (tid == 0) {
    lds[num_experts] = s_carry;
    if (blockIdx.x == 0) *post_pad = total * block_m;
  }
  __syncthreads();
  for (int idx = (int)blockIdx.x * 1024 + tid; idx < total * block_m; idx += 1024 * (int)gridDim.x) {
    const int blk = idx / block_m, r = idx - blk * block_m;
    int lo = 0, hi = num_experts - 1;  // last expert whose first block is <= blk (experts without rows share a value)
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (lds[mid] <= blk) lo = mid;
      else hi = mid - 1;
    }
    const int row_in_expert = (blk - lds[lo]) * block_m + r;
    const int rows = min(max(problem_sizes[lo * 3], 0), num_rows);
    const int row = offsets[lo] + row_in_expert;
    sorted_ids[idx] = (row_in_expert < rows && row >= 0 && row < num_rows) ? row : num_rows;
    if (r == 0) expert_ids[blk] = lo;
  }
}

// ---------------------------------------------------------------------------------------
// topk_softmax: routing of one token per wavefront.  Lane l holds experts l, l + 64, ...; the logits are
// (optionally) soft-capped and biased, soft-maxed in fp32, then k rounds
// of arg-max pick the largest remaining probability, the lower expert index winning ties; the winner's lane
// blanks its copy.  Optional renormalisation divides by the sum of the k picked probabilities.
// A chain of k dependent rounds, so latency is all there is: the rounds' maxima run on the DPP path and ballots
// (wave_pick); with butterfly shuffles of (value, index) pairs one token of 256 experts, top-8, took 7.0 us, now 4.5 (a launch of nothing: 2.5).
// ---------------------------------------------------------------------------------------
template <typename T, int EPL>
__global__ __launch_bounds__(256) void topk_softmax_kernel(const typename T::storage* __restrict__ gating,
                                                           float* __restrict__ weights, int32_t* __restrict__ ids,
                                                           int num_tokens, int num_experts, int topk, int renormalize,
                                                           float softcap, const float* __restrict__ bias) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= num_tokens) return;
  const typename T::storage* g = gating + (int64_t)row * num_experts;
  float v[EPL];
  float vmax = -INFINITY;
#pragma unroll
  for (int j = 0; j < EPL; j++) {
    const int e = lane + 64 * j;
    float x = -INFINITY;
    if (e < num_experts) {
      x = T::to_f32(g[e]);
      if (softcap != 0.f) x = tanhf(x / softcap) * softcap;
      if (bias) x += bias[e];
    }
    v[j] = x;
    vmax = fmaxf(vmax, x);
  }
  vmax = wave_max(vmax);
  float sum = 0.f;
#pragma unroll
  for (int j = 0; j < EPL; j++) {
    v[j] = (lane + 64 * j) < num_experts ? expf(v[j] - vmax) : 0.f;
    sum += v[j];
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) sum += __shfl_xor(sum, off, 64);
  const float inv = 1.f / sum;
#pragma unroll
  for (int j = 0; j < EPL; j++) v[j] = (lane + 64 * j) < num_experts ? v[j] * inv : -1.f;

  float picked = 0.f;   // lane k keeps the k-th pick
  int picked_id = 0;
  float total = 0.f;
  for (int k = 0; k < topk; k++) {
    int best_e;
    const float best = wave_pick<EPL>(v, k, -1.f, best_e);
    if (lane == (k & 63)) {
      picked = best;
      picked_id = best_e;
    }
    total += best;
    if ((k & 63) == 63 || k == topk - 1) {
      // flush up to 64 picks (renormalisation needs the total, so only the last flush can apply it when topk <= 64)
      const int base = k & ~63;
      if (base + lane <= k) {
        if (renormalize && topk <= 64) picked *= 1.f / total;  // the only flush: all picks are in
        weights[(int64_t)row * topk + base + lane] = picked;
        ids[(int64_t)row * topk + base + lane] = picked_id;
      }
    }
  }
  if (renormalize && topk > 64) {
    const float rinv = 1.f / total;
    for (int k = lane; k < topk; k += 64) weights[(int64_t)row * topk + k] *= rinv;
  }
}

// ---------------------------------------------------------------------------------------
// act_and_mul: out[t, j] = T(act_f32(x[t, j])) * x[t, d + j], product rounded to T.
// ACT 0: silu x / (1 + exp(-x)) (silu_rounded);  1: gelu x * 0.5 * (1 + erf(x / sqrt 2));  2: the tanh form of gelu.
// ---------------------------------------------------------------------------------------
template <int ACT>
__device__ __forceinline__ float act_f32(float x) {
  if constexpr (ACT == 1) {
    return x * (0.5f * (1.0f + erff(x * 0.70710678118654752440f)));
  } else {
    const float cdf = 0.5f * (1.0f + tanhf(0.7978845608028654f * (x + 0.044715f * x * x * x)));
    return x * cdf;
  }
}
template <typename T, int ACT>
__global__ __launch_bounds__(256) void act_and_mul_kernel(const u16* __restrict__ in, u16* __restrict__ out, int d) {
  const int64_t t = blockIdx.x;
  const u16* g = in + t * 2 * (int64_t)d;
  const u16* u = g + d;
  u16* o = out + t * (int64_t)d;
  for (int j = threadIdx.x * 8; j < d; j += 256 * 8) {
    v4i gv = *(const v4i*)(g + j), uv = *(const v4i*)(u + j);
    u16 gb[8], ub[8], ob[8];
    __builtin_memcpy(gb, &gv, 16);
    __builtin_memcpy(ub, &uv, 16);
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const float x = T::to_f32(gb[k]);
      float s;
      if constexpr (ACT == 0) s = silu_rounded<T>(x);
      else s = T::to_f32(T::from_f32(act_f32<ACT>(x)));
      ob[k] = T::from_f32(s * T::to_f32(ub[k]));
    }
    v4i ov;
    __builtin_memcpy(&ov, ob, 16);
    *(v4i*)(o + j) = ov;
  }
}

// moe_sum_reduce: out[t, j] = T(scale * sum_k f32(in[t, k, j]))
template <typename T>
__global__ __launch_bounds__(256) void moe_sum_reduce_kernel(const u16* __restrict__ in, u16* __restrict__ out,
                                                             int topk, int d, float scale) {
  const int64_t t = blockIdx.x;
  const u16* src = in + t * (int64_t)topk * d;
  u16* o = out + t * (int64_t)d;
  for (int j = (blockIdx.y * 256 + threadIdx.x) * 8; j < d; j += gridDim.y * 256 * 8) {
    float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int k = 0; k < topk; k++) {
      v4i v = *(const v4i*)(src + (int64_t)k * d + j);
      u16 b[8];
      __builtin_memcpy(b, &v, 16);
#pragma unroll
      for (int e = 0; e < 8; e++) acc[e] += T::to_f32(b[e]);
    }
    u16 ob[8];
#pragma unroll
    for (int e = 0; e < 8; e++) ob[e] = T::from_f32(acc[e] * scale);
    v4i ov;
    __builtin_memcpy(&ov, ob, 16);
    *(v4i*)(o + j) = ov;
  }
}

// tuning knob: SGLAMD_MOE_ACTQ=0 keeps SiLU * up and its quantisation a launch of their own behind the first GEMM
static bool moe_actq_enabled() {
  static const int v = getenv("SGLAMD_MOE_ACTQ") ? atoi(getenv("SGLAMD_MOE_ACTQ")) : 1;
  return v != 0;
}

}  // namespace sglamd

using namespace sglamd;

// More than 64 KB of dynamic LDS (above ~850 buckets) needs the kernel's limit raised, once per kernel and device.
#define SGLAMD_RAISE_LDS(kern, lds)                                                                                    \
  do {                                                                                                                 \
    if ((lds) > 64 * 1024) {                                                                                           \
      static SmemAttrOnce attr_;                                                                                       \
      const hipError_t e_ = raise_dynamic_smem(attr_, (const void*)(kern), (int)(lds));                                \
      if (e_ != hipSuccess) return fail(SGLAMD_EHIP, "hipFuncSetAttribute: %s", hipGetErrorString(e_));                \
    }                                                                                                                  \
  } while (0)

extern "C" int sglamd_moe_align_block_size(const void* topk_ids, int ids_dtype, int64_t numel, int num_experts,
                                           int block_size, int32_t* sorted_token_ids, int64_t max_num_tokens_padded,
                                           int32_t* expert_ids, int32_t* num_tokens_post_pad, int32_t* cumsum_buffer,
                                           int pad_sorted_token_ids, void* stream) {
  SGLAMD_REQUIRE(topk_ids && sorted_token_ids && expert_ids && num_tokens_post_pad, SGLAMD_EINVAL,
                 "moe_align_block_size: null pointer");
  SGLAMD_REQUIRE(ids_dtype == SGLAMD_I32 || ids_dtype == SGLAMD_I64, SGLAMD_EINVAL,
                 "moe_align_block_size: topk_ids must be int32 or int64");
  SGLAMD_REQUIRE(numel >= 0 && numel < (1ll << 30), SGLAMD_EINVAL, "moe_align_block_size: bad numel");
  SGLAMD_REQUIRE(block_size > 0, SGLAMD_EINVAL, "moe_align_block_size: block_size must be positive");
  SGLAMD_REQUIRE(num_experts > 0 && num_experts <= 2048, SGLAMD_EINVAL,
                 "moe_align_block_size: num_experts (%d) must be in [1, 2048]", num_experts);
  const size_t lds = moe_align_lds_bytes(num_experts);
  const unsigned parts = (unsigned)moe_align_parts(numel);
  hipStream_t st = (hipStream_t)stream;
  if (ids_dtype == SGLAMD_I32) {
    auto k = moe_align_kernel<int32_t>;
    SGLAMD_RAISE_LDS(k, lds);
    hipLaunchKernelGGL(k, dim3(parts), dim3(1024), lds, st, (const int32_t*)topk_ids, sorted_token_ids, expert_ids,
                       num_tokens_post_pad, cumsum_buffer, num_experts, block_size, (int)numel, pad_sorted_token_ids,
                       (int)max_num_tokens_padded);
  } else {
    auto k = moe_align_kernel<int64_t>;
    SGLAMD_RAISE_LDS(k, lds);
    hipLaunchKernelGGL(k, dim3(parts), dim3(1024), lds, st, (const int64_t*)topk_ids, sorted_token_ids, expert_ids,
                       num_tokens_post_pad, cumsum_buffer, num_experts, block_size, (int)numel, pad_sorted_token_ids,
                       (int)max_num_tokens_padded);
  }
  return check_launch("moe_align_block_size");
}

static int moe_block_gemm(int mode, const void* a, int64_t lda, const float* a_scale, int64_t as_stride_m,
                          int64_t as_stride_k, const void* w, int64_t w_stride_e, int64_t w_stride_n,
                          const float* w_scale, int64_t ws_stride_e, int64_t ws_stride_n, int64_t ws_stride_k, void* c,
                          int64_t ldc, int out_dtype, const int32_t* sorted_token_ids, const int32_t* expert_ids,
                          const int32_t* num_tokens_post_padded, const float* topk_weights, int64_t num_valid_tokens,
                          int top_k, int mul_routed_weight, int block_m, int64_t max_m_blocks, int64_t N, int64_t K,
                          void* stream, int scale_rows_padded = 0, int streams = 0) {
  const DeviceScope scope;
  SGLAMD_REQUIRE(a && a_scale && w && w_scale && c && sorted_token_ids && expert_ids && num_tokens_post_padded,
                 SGLAMD_EINVAL, "fused_moe_gemm: null pointer");
  SGLAMD_REQUIRE(!mul_routed_weight || topk_weights, SGLAMD_EINVAL, "fused_moe_gemm: topk_weights missing");
  SGLAMD_REQUIRE(N > 0 && K > 0 && K % 16 == 0 && N < (1ll << 31) && K < (1ll << 31), SGLAMD_EINVAL,
                 "fused_moe_gemm: bad N/K");
  SGLAMD_REQUIRE(top_k >= 1 && num_valid_tokens >= 0 && num_valid_tokens < (1ll << 31), SGLAMD_EINVAL,
                 "fused_moe_gemm: bad top_k / num_valid_tokens");
  SGLAMD_REQUIRE(lda % 16 == 0 && w_stride_n % 16 == 0 && w_stride_e % 16 == 0, SGLAMD_EINVAL,
                 "fused_moe_gemm: strides must be multiples of 16 bytes");
  SGLAMD_REQUIRE(((uintptr_t)a % 16) == 0 && ((uintptr_t)w % 16) == 0, SGLAMD_EINVAL,
                 "fused_moe_gemm: operands must be 16-byte aligned");
  SGLAMD_REQUIRE(max_m_blocks >= 0 && max_m_blocks < (1ll << 24), SGLAMD_EINVAL, "fused_moe_gemm: bad block count");
  if (max_m_blocks == 0 || num_valid_tokens == 0) return SGLAMD_OK;
  GemmArgs g = {};
  g.A = (const uint8_t*)a;
  g.lda = lda;
  g.B = (const uint8_t*)w;
  g.ldb = w_stride_n;
  g.b_expert_stride = w_stride_e;
  g.sa = a_scale;
  g.sa_sm = as_stride_m;
  g.sa_sk = as_stride_k;
  g.sb = w_scale;
  g.sb_se = ws_stride_e;
  g.sb_sn = ws_stride_n;
  g.sb_sk = ws_stride_k;
  g.C = c;
  g.ldc = ldc;
  g.M = (int)num_valid_tokens;
  g.N = (int)N;
  g.K = (int)K;
  g.sorted_ids = sorted_token_ids;
  g.expert_ids = expert_ids;
  g.num_post_pad = num_tokens_post_padded;
  g.topk_w = topk_weights;
  g.top_k = top_k;
  g.num_valid = (int)num_valid_tokens;
  g.mul_weight = mul_routed_weight;
  g.scale_rows_padded = scale_rows_padded;
  g.streams = streams;
  g.max_blocks_m = (int)max_m_blocks;
  hipStream_t st = (hipStream_t)stream;
  if (mode == GEMM_BLOCK_INT8) {
    if (out_dtype == SGLAMD_BF16) return dispatch_moe_gemm<GEMM_BLOCK_INT8, BF16>(g, block_m, st);
    if (out_dtype == SGLAMD_F16) return dispatch_moe_gemm<GEMM_BLOCK_INT8, F16>(g, block_m, st);
  } else {
    if (out_dtype == SGLAMD_BF16) return dispatch_moe_gemm<GEMM_BLOCK_FP8, BF16>(g, block_m, st);
    if (out_dtype == SGLAMD_F16) return dispatch_moe_gemm<GEMM_BLOCK_FP8, F16>(g, block_m, st);
  }
  return fail(SGLAMD_EINVAL, "fused_moe_gemm: out_dtype must be Half or BFloat16");
}

extern "C" int sglamd_fused_moe_block_fp8_gemm(const void* a, int64_t lda, const float* a_scale, int64_t as_stride_m,
                                               int64_t as_stride_k, const void* w, int64_t w_stride_e,
                                               int64_t w_stride_n, const float* w_scale, int64_t ws_stride_e,
                                               int64_t ws_stride_n, int64_t ws_stride_k, void* c, int64_t ldc,
                                               int out_dtype, const int32_t* sorted_token_ids,
                                               const int32_t* expert_ids, const int32_t* num_tokens_post_padded,
                                               const float* topk_weights, int64_t num_valid_tokens, int top_k,
                                               int mul_routed_weight, int block_m, int64_t max_m_blocks, int64_t N,
                                               int64_t K, void* stream) {
  return moe_block_gemm(GEMM_BLOCK_FP8, a, lda, a_scale, as_stride_m, as_stride_k, w, w_stride_e, w_stride_n, w_scale,
                        ws_stride_e, ws_stride_n, ws_stride_k, c, ldc, out_dtype, sorted_token_ids, expert_ids,
                        num_tokens_post_padded, topk_weights, num_valid_tokens, top_k, mul_routed_weight, block_m,
                        max_m_blocks, N, K, stream);
}

extern "C" int sglamd_fused_moe_block_int8_gemm(const void* a, int64_t lda, const float* a_scale, int64_t as_stride_m,
                                                int64_t as_stride_k, const void* w, int64_t w_stride_e,
                                                int64_t w_stride_n, const float* w_scale, int64_t ws_stride_e,
                                                int64_t ws_stride_n, int64_t ws_stride_k, void* c, int64_t ldc,
                                                int out_dtype, const int32_t* sorted_token_ids,
                                                const int32_t* expert_ids, const int32_t* num_tokens_post_padded,
                                                const float* topk_weights, int64_t num_valid_tokens, int top_k,
                                                int mul_routed_weight, int block_m, int64_t max_m_blocks, int64_t N,
                                                int64_t K, void* stream) {
  return moe_block_gemm(GEMM_BLOCK_INT8, a, lda, a_scale, as_stride_m, as_stride_k, w, w_stride_e, w_stride_n, w_scale,
                        ws_stride_e, ws_stride_n, ws_stride_k, c, ldc, out_dtype, sorted_token_ids, expert_ids,
                        num_tokens_post_padded, topk_weights, num_valid_tokens, top_k, mul_routed_weight, block_m,
                        max_m_blocks, N, K, stream);
}

extern "C" int sglamd_moe_list_streams(int64_t num_valid_tokens, int64_t max_m_blocks, int block_m, int64_t N, int64_t w_stride_n) {
  return block_m > 1 && moe_list_streams(num_valid_tokens, max_m_blocks, block_m, N, w_stride_n);
}

extern "C" int sglamd_topk_softmax(float* topk_weights, int32_t* topk_indices, const void* gating_output, int g_dtype,
                                  int64_t num_tokens, int64_t num_experts, int64_t topk, int renormalize,
                                  float moe_softcapping, const float* correction_bias, void* stream) {
  SGLAMD_REQUIRE(topk_weights && topk_indices && gating_output, SGLAMD_EINVAL, "topk_softmax: null pointer");
  SGLAMD_REQUIRE(num_tokens >= 0 && num_experts > 0 && topk > 0, SGLAMD_EINVAL, "topk_softmax: bad sizes");
  SGLAMD_REQUIRE(topk <= num_experts, SGLAMD_EINVAL, "topk must be less than or equal to num_experts");
  SGLAMD_REQUIRE(num_experts <= 1024, SGLAMD_ENOTSUP, "topk_softmax: more than 1024 experts");
  SGLAMD_REQUIRE(g_dtype == SGLAMD_F32 || g_dtype == SGLAMD_F16 || g_dtype == SGLAMD_BF16, SGLAMD_EINVAL,
                 "gating_output must be float32, float16, or bfloat16");
  if (num_tokens == 0) return SGLAMD_OK;
  hipStream_t st = (hipStream_t)stream;
  const unsigned blocks = (unsigned)ceil_div(num_tokens, 4);
#define SGLAMD_TOPK(TT, E)                                                                                             \
  hipLaunchKernelGGL((topk_softmax_kernel<TT, E>), dim3(blocks), dim3(256), 0, st,                                     \
                     (const typename TT::storage*)gating_output, topk_weights, topk_indices, (int)num_tokens,          \
                     (int)num_experts, (int)topk, renormalize, moe_softcapping, correction_bias)
#define SGLAMD_TOPK_E(TT)                                                                                              \
  do {                                                                                                                 \
    if (num_experts <= 64) SGLAMD_TOPK(TT, 1);                                                                         \
    else if (num_experts <= 128) SGLAMD_TOPK(TT, 2);                                                                   \
    else if (num_experts <= 256) SGLAMD_TOPK(TT, 4);                                                                   \
    else if (num_experts <= 512) SGLAMD_TOPK(TT, 8);                                                                   \
    else SGLAMD_TOPK(TT, 16);                                                                                          \
  } while (0)
  if (g_dtype == SGLAMD_F32) SGLAMD_TOPK_E(F32);
  else if (g_dtype == SGLAMD_F16) SGLAMD_TOPK_E(F16);
  else SGLAMD_TOPK_E(BF16);
#undef SGLAMD_TOPK_E
#undef SGLAMD_TOPK
  return check_launch("topk_softmax");
}

template <int ACT>
static int act_and_mul_launch(const char* name, const void* input, void* out, int dtype, int64_t rows, int64_t d,
                              void* stream) {
  SGLAMD_REQUIRE(input && out, SGLAMD_EINVAL, "%s: null pointer", name);
  SGLAMD_REQUIRE(rows >= 0 && d > 0 && d % 8 == 0 && d < (1ll << 30), SGLAMD_EINVAL,
                 "%s: d (%lld) must be a positive multiple of 8", name, (long long)d);
  SGLAMD_REQUIRE(((uintptr_t)input % 16) == 0 && ((uintptr_t)out % 16) == 0, SGLAMD_EINVAL,
                 "%s: pointers must be 16-byte aligned", name);
  SGLAMD_REQUIRE(rows < (1ll << 31), SGLAMD_EINVAL, "%s: too many rows", name);
  if (rows == 0) return SGLAMD_OK;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == SGLAMD_BF16)
    hipLaunchKernelGGL((act_and_mul_kernel<BF16, ACT>), dim3((unsigned)rows), dim3(256), 0, st, (const u16*)input,
                       (u16*)out, (int)d);
  else if (dtype == SGLAMD_F16)
    hipLaunchKernelGGL((act_and_mul_kernel<F16, ACT>), dim3((unsigned)rows), dim3(256), 0, st, (const u16*)input,
                       (u16*)out, (int)d);
  else
    return fail(SGLAMD_EINVAL, "%s: dtype must be Half or BFloat16", name);
  return check_launch(name);
}

extern "C" int sglamd_silu_and_mul(const void* input, void* out, int dtype, int64_t rows, int64_t d, void* stream) {
  return act_and_mul_launch<0>("silu_and_mul", input, out, dtype, rows, d, stream);
}
extern "C" int sglamd_gelu_and_mul(const void* input, void* out, int dtype, int64_t rows, int64_t d, void* stream) {
  return act_and_mul_launch<1>("gelu_and_mul", input, out, dtype, rows, d, stream);
}
extern "C" int sglamd_gelu_tanh_and_mul(const void* input, void* out, int dtype, int64_t rows, int64_t d,
                                        void* stream) {
  return act_and_mul_launch<2>("gelu_tanh_and_mul", input, out, dtype, rows, d, stream);
}

extern "C" int sglamd_moe_sum_reduce(const void* input, void* out, int dtype, int64_t tokens, int topk, int64_t d,
                                     float routed_scaling_factor, void* stream) {
  SGLAMD_REQUIRE(input && out, SGLAMD_EINVAL, "moe_sum_reduce: null pointer");
  SGLAMD_REQUIRE(tokens >= 0 && topk >= 1 && d > 0 && d % 8 == 0 && d < (1ll << 30), SGLAMD_EINVAL,
                 "moe_sum_reduce: hidden size (%lld) must be a positive multiple of 8", (long long)d);
  if (tokens == 0) return SGLAMD_OK;
  hipStream_t st = (hipStream_t)stream;
  int64_t gy64 = ceil_div(d, 2048);
  if (gy64 > 64) gy64 = 64;
  const unsigned gy = (unsigned)gy64;
  dim3 grid((unsigned)tokens, gy);
  if (dtype == SGLAMD_BF16)
    hipLaunchKernelGGL(moe_sum_reduce_kernel<BF16>, grid, dim3(256), 0, st, (const u16*)input, (u16*)out, topk, (int)d,
                       routed_scaling_factor);
  else if (dtype == SGLAMD_F16)
    hipLaunchKernelGGL(moe_sum_reduce_kernel<F16>, grid, dim3(256), 0, st, (const u16*)input, (u16*)out, topk, (int)d,
                       routed_scaling_factor);
  else
    return fail(SGLAMD_EINVAL, "moe_sum_reduce: dtype must be Half or BFloat16");
  return check_launch("moe_sum_reduce");
}

// ---------------------------------------------------------------------------------------
// Expert-major ("grouped") MoE interface: prepare_moe_input / shuffle_rows /
// fp8_blockwise_scaled_grouped_mm / apply_shuffle_mul_sum.
// ---------------------------------------------------------------------------------------
extern "C" int sglamd_prepare_moe_input(const int32_t* topk_ids, int64_t numel, int topk, int num_experts, int64_t n,
                                        int64_t k, int32_t* expert_offsets, int32_t* blockscale_offsets,
                                        int32_t* problem_sizes1, int32_t* problem_sizes2, int32_t* input_permutation,
                                        int32_t* output_permutation, void* stream) {
  SGLAMD_REQUIRE(topk_ids && expert_offsets && problem_sizes1 && problem_sizes2 && input_permutation &&
                     output_permutation,
                 SGLAMD_EINVAL, "prepare_moe_input: null pointer");
  SGLAMD_REQUIRE(numel >= 0 && numel < (1ll << 30) && topk >= 1, SGLAMD_EINVAL, "prepare_moe_input: bad numel/topk");
  SGLAMD_REQUIRE(num_experts > 0 && num_experts <= 2048, SGLAMD_EINVAL,
                 "prepare_moe_input: num_experts (%d) must be in [1, 2048]", num_experts);
  SGLAMD_REQUIRE(n > 0 && k > 0 && 2 * n < (1ll << 31) && k < (1ll << 31), SGLAMD_EINVAL, "prepare_moe_input: bad n/k");
  MoePrepArgs pa;
  pa.expert_offsets = expert_offsets;
  pa.blockscale_offsets = blockscale_offsets;
  pa.problem_sizes1 = problem_sizes1;
  pa.problem_sizes2 = problem_sizes2;
  pa.input_permutation = input_permutation;
  pa.output_permutation = output_permutation;
  pa.topk = topk;
  pa.n = (int)n;
  pa.k = (int)k;
  const int nb = num_experts + 1;
  const size_t lds = moe_align_lds_bytes(nb);
  auto kern = moe_prepare_kernel;
  SGLAMD_RAISE_LDS(kern, lds);
  hipLaunchKernelGGL(kern, dim3((unsigned)moe_align_parts(numel)), dim3(1024), lds, (hipStream_t)stream, topk_ids, nb, (int)numel, pa);
  return check_launch("prepare_moe_input");
}

extern "C" int sglamd_shuffle_rows(const void* input, const int32_t* dst2src_map, void* output, int64_t num_dst_rows,
                                   int64_t row_bytes, void* stream) {
  SGLAMD_REQUIRE(input && dst2src_map && output, SGLAMD_EINVAL, "shuffle_rows: null pointer");
  SGLAMD_REQUIRE(num_dst_rows >= 0 && row_bytes > 0, SGLAMD_EINVAL, "shuffle_rows: bad sizes");
  if (num_dst_rows == 0) return SGLAMD_OK;
  const unsigned blocks = (unsigned)(num_dst_rows < 65536 ? num_dst_rows : 65536);
  hipStream_t st = (hipStream_t)stream;
  const uintptr_t both = (uintptr_t)input | (uintptr_t)output | (uintptr_t)row_bytes;
  if ((both & 15) == 0)
    hipLaunchKernelGGL(shuffle_rows_kernel<v4i>, dim3(blocks), dim3(256), 0, st, (const uint8_t*)input, dst2src_map,
                       (uint8_t*)output, num_dst_rows, row_bytes);
  else if ((both & 3) == 0)
    hipLaunchKernelGGL(shuffle_rows_kernel<int32_t>, dim3(blocks), dim3(256), 0, st, (const uint8_t*)input, dst2src_map,
                       (uint8_t*)output, num_dst_rows, row_bytes);
  else
    hipLaunchKernelGGL(shuffle_rows_kernel<uint8_t>, dim3(blocks), dim3(256), 0, st, (const uint8_t*)input, dst2src_map,
                       (uint8_t*)output, num_dst_rows, row_bytes);
  return check_launch("shuffle_rows");
}

extern "C" int sglamd_apply_shuffle_mul_sum(const void* input, void* output, const int32_t* permutation,
                                            const void* factors, int dtype, int64_t m, int topk, int64_t row_stride,
                                            void* stream) {
  SGLAMD_REQUIRE(input && output && permutation, SGLAMD_EINVAL, "apply_shuffle_mul_sum: null pointer");
  SGLAMD_REQUIRE(m >= 0 && m < (1ll << 31) && topk >= 1 && row_stride > 0 && row_stride < (1ll << 30), SGLAMD_EINVAL,
                 "apply_shuffle_mul_sum: bad sizes");
  SGLAMD_REQUIRE(dtype == SGLAMD_BF16 || dtype == SGLAMD_F16, SGLAMD_EINVAL,
                 "apply_shuffle_mul_sum: dtype must be Half or BFloat16");
  SGLAMD_REQUIRE((row_stride % 8) != 0 || (((uintptr_t)input | (uintptr_t)output) % 16) == 0, SGLAMD_EINVAL,
                 "apply_shuffle_mul_sum: pointers must be 16-byte aligned");
  if (m == 0) return SGLAMD_OK;
  int64_t gy = ceil_div(row_stride, 2048);
  if (gy > 64) gy = 64;
  dim3 grid((unsigned)m, (unsigned)gy);
  hipStream_t st = (hipStream_t)stream;
  if (dtype == SGLAMD_BF16)
    hipLaunchKernelGGL(shuffle_mul_sum_kernel<BF16>, grid, dim3(256), 0, st, (const u16*)input, (u16*)output, permutation,
                       (const u16*)factors, topk, (int)row_stride);
  else
    hipLaunchKernelGGL(shuffle_mul_sum_kernel<F16>, grid, dim3(256), 0, st, (const u16*)input, (u16*)output, permutation,
                       (const u16*)factors, topk, (int)row_stride);
  return check_launch("apply_shuffle_mul_sum");
}

namespace {
struct GroupedWs {
  int64_t sorted, expert, post, total, max_padded, max_blocks;
};
GroupedWs grouped_ws_layout(int64_t rows, int E, int block_m) {
  GroupedWs w;
  const int64_t worst = rows + (int64_t)E * (block_m - 1);  // every expert may leave one block partly filled
  w.max_blocks = (worst + block_m - 1) / block_m;
  w.max_padded = w.max_blocks * block_m;
  int64_t o = 0;
  w.sorted = o; o = (o + w.max_padded * 4 + 255) & ~(int64_t)255;
  w.expert = o; o = (o + w.max_blocks * 4 + 255) & ~(int64_t)255;
  w.post = o; o += 256;
  w.total = o;
  return w;
}
int grouped_block_m(int64_t rows, int E);
}  // namespace

extern "C" int64_t sglamd_grouped_mm_workspace_bytes(int64_t total_rows, int num_experts) {
  if (total_rows <= 0 || num_experts <= 0) return 0;
  return grouped_ws_layout(total_rows, num_experts, grouped_block_m(total_rows, num_experts)).total;
}

extern "C" int sglamd_fp8_blockwise_scaled_grouped_mm(void* output, int out_dtype, const void* a, const void* b,
                                                      const float* scales_a, const float* scales_b,
                                                      const int32_t* problem_sizes, const int32_t* expert_offsets,
                                                      int num_experts, int64_t total_rows, int64_t N, int64_t K,
                                                      void* workspace, int64_t workspace_bytes, void* stream) {
  SGLAMD_REQUIRE(output && a && b && scales_a && scales_b && problem_sizes && expert_offsets, SGLAMD_EINVAL,
                 "fp8_blockwise_scaled_grouped_mm: null pointer");
  SGLAMD_REQUIRE(num_experts > 0 && num_experts <= 2048, SGLAMD_EINVAL,
                 "fp8_blockwise_scaled_grouped_mm: num_experts (%d) must be in [1, 2048]", num_experts);
  SGLAMD_REQUIRE(total_rows >= 0 && total_rows < (1ll << 30), SGLAMD_EINVAL,
                 "fp8_blockwise_scaled_grouped_mm: bad number of rows");
  SGLAMD_REQUIRE(N > 0 && K > 0 && N % 128 == 0 && K % 128 == 0 && N < (1ll << 31) && K < (1ll << 31), SGLAMD_EINVAL,
                 "fp8_blockwise_scaled_grouped_mm: N (%lld) and K (%lld) must be positive multiples of 128",
                 (long long)N, (long long)K);
  SGLAMD_REQUIRE((((uintptr_t)a | (uintptr_t)b) % 16) == 0, SGLAMD_EINVAL,
                 "fp8_blockwise_scaled_grouped_mm: operands must be 16-byte aligned");
  if (total_rows == 0) return SGLAMD_OK;
  const int block_m = grouped_block_m(total_rows, num_experts);
  const GroupedWs w = grouped_ws_layout(total_rows, num_experts, block_m);
  SGLAMD_REQUIRE(workspace && workspace_bytes >= w.total, SGLAMD_EINVAL,
                 "fp8_blockwise_scaled_grouped_mm: workspace too small (%lld < %lld bytes)", (long long)workspace_bytes,
                 (long long)w.total);
  SGLAMD_REQUIRE(((uintptr_t)workspace % 16) == 0, SGLAMD_EINVAL,
                 "fp8_blockwise_scaled_grouped_mm: workspace must be 16-byte aligned");
  uint8_t* ws = (uint8_t*)workspace;
  int32_t* sorted = (int32_t*)(ws + w.sorted);
  int32_t* expert = (int32_t*)(ws + w.expert);
  int32_t* post = (int32_t*)(ws + w.post);
  hipStream_t st = (hipStream_t)stream;
  const int64_t parts = ceil_div(w.max_padded, 2048);
  hipLaunchKernelGGL(grouped_schedule_kernel, dim3((unsigned)(parts < 64 ? parts : 64)), dim3(1024), (size_t)(num_experts + 1) * sizeof(int32_t), st,
                     problem_sizes, expert_offsets, num_experts, block_m, (int)total_rows, (int)w.max_blocks, sorted,
                     expert, post);
  int rc = check_launch("grouped_schedule");
  if (rc) return rc;
  const int64_t KB = K / 128;
  return sglamd_fused_moe_block_fp8_gemm(a, K, scales_a, KB, 1, b, N * K, K, scales_b, (N / 128) * KB, KB, 1, output, N,
                                         out_dtype, sorted, expert, post, nullptr, total_rows, 1, 0, block_m,
                                         w.max_blocks, N, K, stream);
}


// ---------------------------------------------------------------------------------------
// Whole block-FP8 MoE layer from one host call: quantise + align (one kernel) -> grouped GEMM 1 ->
// silu*mul + quantise (one kernel) -> grouped GEMM 2 (x routing weight) -> top-k sum.
// Five launches on one stream (four for up to four tokens, two for one); all intermediates live in the
// caller's workspace.
// ---------------------------------------------------------------------------------------
static_assert(GEMM_BLOCK_FP8 == (int)SGLAMD_MOE_BLOCK_FP8 && GEMM_ROW_FP8 == (int)SGLAMD_MOE_ROW_FP8 &&
                  GEMM_ROW_INT8 == (int)SGLAMD_MOE_ROW_INT8 && GEMM_BLOCK_INT8 == (int)SGLAMD_MOE_BLOCK_INT8,
              "the ABI's layer modes are the GEMM modes");

namespace {
struct MoeWs {
  int64_t sorted, expert, post, cumsum, xq, xs, c1, aq, as, c3, total;
  int64_t max_padded, max_blocks;
  int64_t few_padded, few_blocks;  // the same bounds for blocks of 4 (calls of at most four tokens), else 0
};
inline int64_t up256(int64_t v) { return (v + 255) & ~(int64_t)255; }
MoeWs moe_ws_layout(int64_t M, int64_t H, int64_t I, int E, int topk, int block_m) {
  MoeWs w;
  const int64_t T = M * topk;
  w.max_padded = T < E + 1 ? T * block_m : T + (int64_t)(E + 1) * (block_m - 1);
  w.max_blocks = (w.max_padded + block_m - 1) / block_m;
  w.few_padded = M > 4 ? 0 : (T < E + 1 ? T * 4 : ((T + (int64_t)(E + 1) * 3 + 3) / 4) * 4);
  w.few_blocks = w.few_padded / 4;
  int64_t o = 0;
  w.sorted = o; o = up256(o + (w.max_padded > w.few_padded ? w.max_padded : w.few_padded) * 4);
  w.expert = o; o = up256(o + (w.max_blocks > w.few_blocks ? w.max_blocks : w.few_blocks) * 4);
  w.post = o; o = up256(o + 4);
  w.cumsum = o; o = up256(o + (int64_t)(E + 2) * 4);
  w.xq = o; o = up256(o + M * H);
  w.xs = o; o = up256(o + M * ((H + 127) / 128) * 4);
  w.c1 = o; o = up256(o + T * 2 * I * 2);
  w.aq = o; o = up256(o + T * I);
  w.as = o; o = up256(o + T * ((I + 127) / 128) * 4);
  w.c3 = o; o = up256(o + T * H * 2);
  w.total = o;
  return w;
}
// Whether the first GEMM of a layer leaves CUs idle while every expert owns one block (0: intermediate size unknown).
bool moe_small_launch(int E, int64_t I) { return I > 0 && (int64_t)E * ceil_div(2 * I, 256) <= device_cus(); }
// A layer whose first GEMM would leave CUs idle in any height: how many tiles it has in 64-slot blocks (every expert's last
// block half full) says how short its blocks may be.  While those fit one round, a tile's time is the launch's time and
// the shortest tile wins; a little above, 128-slot blocks, up to the rows where two of them hold an expert.  0: no opinion.
// Twenty layers (4 to 256 experts of 256 to 2048, K from 1024 to 7168) at 12 to 500 rows, this rule against the bands below
// where the two differ, mean and range:
//   rows            52..72            73..104           105..169          170..215          above 215
//   block, 64   1.05 (0.93-1.21)  1.16 (1.10-1.22)  1.17 (1.00-1.39)  1.10 (1.09-1.12)  1.14 (1.00-1.23)
//   row, 64     1.09 (1.05-1.13)         -          1.11 (0.97-1.25)  1.10 (1.09-1.11)  1.11 (0.98-1.25)
// 128 slots at 105..169 rows: 1.00 (0.94-1.10) block-scaled, 0.94 (two points) row-scaled.  Where an earlier sweep was mixed
// (row-scaled at 73 to 112 rows, 128 slots above 215 rows) the bands stay.
int moe_one_round_block(double rows, int E, int64_t I, bool row_scaled) {
  if (I <= 0 || rows <= 52) return 0;
  const double tiles = E * (rows / 64 + 0.5) * (double)ceil_div(2 * I, 256) * 256.0 / device_cus();
  if (rows <= (row_scaled ? 112 : 104)) return rows <= (row_scaled ? 72 : 104) && tiles <= (row_scaled ? 80 : 96) ? 64 : 0;
  if (rows < 170) return tiles <= 200 ? 64 : tiles <= 300 ? 128 : 0;
  if (rows <= 215) return tiles <= 100 ? 64 : 0;  // (128 by the bands)
  return tiles <= 200 ? 64 : 0;
}

// Whether a layer is one for the weight-streaming tile kernel (gemm_moe_stream.h; moe_stream_takes says why).
bool moe_layer_streams(int E, int64_t H, int64_t I) { return moe_stream_enabled() && 3 * E * H * I >= MOE_STREAM_MIN_BYTES; }
// Rows per expert from which 64-slot blocks take over from the 16-slot ones of the streaming kernel on such layers.  That
// kernel reads the same bytes, but every 16 rows or 32 columns have a tile of their own and a drain at its end; rounds of tiles
// that leave part of the chip idle cost it less.  So the line follows how much of its rounds a layer fills with one block per
// expert (both GEMMs, by time).  Best lines of 98 (block FP8) and 158 (row scales) layers of 8 to 256 experts, weights from HBM:
//   filled below 0.46     11 to 18 / 13 to 20      (8 experts of 4096 x 1536, hidden x intermediate: 16 / 16)
//          0.46 to 0.59   9 to 14 / 8 to 14        (16 of 2048 x 1024: 14 / 14; 16 of 4096 x 896: level from 2 to 13 / 12)
//          0.59 to 0.75   9 to 13 / 11 to 14       (32 of 3072 x 1152: 13 / 13)
//          0.75 to 0.80   10 / 9 to 12             (32 of 5120 x 1536: 10 / 12)
//          0.80 to 0.84   2 to 7 / 2 to 11         (64 of 2048 x 768: 7 / 10)
//          0.84 to 0.94   2 to 8 / 2 to 10         (64 of 6144 x 1792: 3.5 / 6; 16 of 6144 x 2048: 8 / 10)
//          above          0.5 to 4, from 1 GB of weights on 0.5 to 3.5, either (256 of 7168 x 2048: 1 / 1; 128 of 2048 x 1024: 4 / 3)
// A second GEMM too short for the tile kernel's pipeline: block FP8 0.59 to 0.84 filled 1.3 to 5, with more than a round in the
// first 8 and more; above 0.94 0.5 to 3, with two rounds and more in the first 2.7 to 5.6; block INT8 6 to 8; row scales, whose
// 128-slot blocks have a pipeline from 512 columns on, below that 8 to 10, from three rounds in the first on 5 to 6.
// Time in 16-slot blocks over time in 64-slot ones, block FP8, at 1 / 2.5 / 5 / 10 rows: 256 of 7168 x 2048 1.01 / 1.02 / 1.06 /
// 1.19, 32 of 4096 x 1024 0.90 / 1.10 / 1.10 / 1.22, 16 of 6144 x 2048 0.85 / 0.92 / 0.93 / 1.12, 32 of 5120 x 1536 0.88 / 0.91 /
// 0.90 / 0.94, 8 of 4096 x 1536 0.71 / 0.77 / 0.92 / 0.87.
double moe_stream_from(int E, int64_t H, int64_t I, int mode) {
  const int64_t cus = device_cus(), first = E * ceil_div(2 * I, 256), second = E * ceil_div(H, 256);
  const double filled = (double)(H * first + I * second) / (cus * (H * ceil_div(first, cus) + I * ceil_div(second, cus)));
  const bool fp8 = mode == GEMM_BLOCK_FP8, block = gemm_is_block(mode);
  const bool short_second = I < (block ? 768 : 512);
  if (filled < 0.46) return 16;
  if (filled < 0.59) return 13;
  if (fp8 && short_second && filled < 0.84) return first > cus ? 8 : 4;
  if (filled < 0.80) return filled < 0.75 ? 12 : 10;
  if (filled < 0.94) return fp8 ? (filled < 0.84 ? 5 : 6) : short_second || filled < 0.84 ? 9 : 8;
  if (short_second) return fp8 ? (first >= 2 * cus ? 4.5 : 2) : block ? 7 : first >= 3 * cus ? 6 : 9;
  return 3 * E * H * I >= 1000000000ll ? 1.5 : 2.5;
}
// Rounds of tiles, one per CU, that a grouped GEMM of `cols` column tiles is expected to take in blocks of `block` slots, when
// `experts` experts hold rows of this mean and variance, drawn independently: an expert's blocks are one and one for each
// multiple of the block that its rows pass, their sum is taken as normally distributed.
double moe_rounds(int experts, double rows, double var, int block, int64_t cols, int64_t cus) {
  // P(a count of this mean and deviation > x)
  auto beyond = [](double x, double mean, double dev) { return 0.5 * std::erfc((x + 0.5 - mean) / (dev * M_SQRT2)); };
  const double dev = std::sqrt(var);
  int64_t sure = std::max<int64_t>(0, (int64_t)std::floor((rows - 5 * dev) / block));
  double blocks = experts * (1. + sure), spread = 0;
  for (int64_t j = sure + 1; j * block < rows + 5 * dev; j++) {
    const double p = beyond((double)(j * block), rows, dev);
    blocks += experts * p;
    spread += experts * p * (1 - p);
  }
  spread = std::sqrt(spread) + 1e-3;
  sure = std::max<int64_t>(0, (int64_t)std::floor((blocks - 5 * spread) * cols / cus));
  double rounds = 1. + sure;
  for (int64_t k = sure + 1; (double)(k * cus) / cols < blocks + 5 * spread + 1; k++)
    rounds += beyond((double)(k * cus / cols), blocks, spread);
  return rounds;
}
// The height of such a layer's blocks, 64 slots or more: the one whose rounds of tiles take the least time.  What a round
// takes hardly depends on how many of its slots hold a row (the weights are its time, or the products of whole tiles): it is
// linear in K, with a share of the height, relative to 192 slots.  Block scales 0.66 (64 slots, the streaming tile kernel) and 0.82
// (128, the persistent walk); row scales 0.83 and 0.90 on the streaming tile kernel, which starts and drains once a launch (460
// bytes of K), while the one-tile kernel (192 slots, and K too short for the other's pipeline) does so at every tile (630).
// What that decides: one round of short tiles against one of tall ones, a second block for an expert that overflows while
// the round has room for it, tall blocks when it has not.
// Whole layers, weights from HBM, 98 layers of every quantisation, 8 to 256 experts, 1 to 4096 rows per expert: time of the
// picked height (16 slots among them) over the fastest one, mean, and in brackets with the bands by rows that stood here:
//   block FP8 1.004 (1.012), block INT8 1.008 (1.015), per-channel FP8 1.004 (1.017), per-channel INT8 1.003 (1.019).
// 8 experts of 4096 x 1536, 150 rows 113 / 79 / 94 (two blocks of 128 are still one round); 16 of 6144 x 2048, 150 rows 269 / 217
// / 184, 190 rows 333 / 228 / 262; 64 of 4096 x 1536, 150 rows 516 / 422 / 335, 208 rows 688 / 460 / 512.
int moe_height_by_rounds(int E, int topk, int64_t H, int64_t I, double rows, bool row_scaled) {
  // every token names topk different experts of E
  const double var = std::max(1e-3, rows * (1 - (double)topk / E));
  const int64_t cus = device_cus();
  struct Round {
    int slots, pipeline;        // K from which the height's kernel is not the one-tile kernel
    double share, launch;       // what a round of it takes per K, and a launch
    double one_tile, ramp;      // what a round of the one-tile kernel takes per K, and on top
  };
  static const Round block_scaled[3] = {{64, 0, 0.66, 0, 0, 0}, {128, 0, 0.82, 0, 0, 0}, {192, 0, 1, 0, 0, 0}};
  static const Round row_scales[3] = {{64, 768, 0.83, 460, 0.47, 630}, {128, 512, 0.90, 460, 0.85, 630}, {192, 1 << 30, 0, 0, 1, 630}};
  int best = 0;
  double least = 0;
  for (const Round& r : row_scaled ? row_scales : block_scaled) {
    auto time = [&](int64_t K, int64_t N) {
      const double rounds = moe_rounds(E, rows, var, r.slots, ceil_div(N, 256), cus);
      return K >= r.pipeline ? r.share * K * rounds + r.launch : (r.one_tile * K + r.ramp) * rounds;
    };
    const double t = time(H, 2 * I) + time(I, H);
    if (!best || t < least) best = r.slots, least = t;
  }
  return best;
}

int moe_auto_block(int64_t M, int E, int topk, int64_t H, int64_t I, bool int8 = false) {
  static const int forced = getenv("SGLAMD_MOE_BLOCK_M") ? atoi(getenv("SGLAMD_MOE_BLOCK_M")) : 0;  // tuning knob
  if (forced == 16 || forced == 32 || forced == 64 || forced == 128 || forced == 192) return forced;
  const double rows = (double)M * topk / (E > 0 ? E : 1);
  // Layers whose weights come from HBM, layer time in us by block height (64: the streaming tile kernel; 128 and 192: the persistent
  // walk), 256 experts of 7168 x 2048, top-8:
  //   rows/expert    1      3      6      10     16     24     32     48     56     64     96     112    128
  //   16            1098   1670   1808   2040   2969   4115
  //   64            1079   1618   1677   1714   1755   1802   1849   1994   2129   2415   3075   3279   3779
  //   128           1243   1846   1907   1946   1987   2018   2069   2150   2189   2224   2364   2542   3017
  //   192           1271   1890   1944   1978   2016   2044   2082   2177   2217   2270   2416   2494   2564
  // (INT8 layers have no activation in the first GEMM's epilogue and no place for padded rows of scales)
  if (moe_layer_streams(E, H, I) && !(int8 && (H % 512 || I % 512))) {
    if (M <= 4 || rows < moe_stream_from(E, H, I, int8 ? GEMM_BLOCK_INT8 : GEMM_BLOCK_FP8)) return 16;
    return moe_height_by_rounds(E, topk, H, I, rows, false);
  }
  // The other layers.  Those whose tiles do not fill the chip take one round whatever the height, so the shorter block wins where it holds
  // an expert, and two full blocks of 128 beat 192 where half of the experts overflow those.  Sixteen such layers of 4 to 64
  // experts: 64 at 14..52 rows 1.05x in the mean (0.94-1.11), 128 at 170..215 rows 1.17x (0.84-1.33, two of 48 points
  // below 0.98); in the bands between, the layers disagree by as much in both directions.  Up to 8 experts the 16-slot
  // blocks stay ahead to 14 rows (8 of 7168 x 2048 1.20x, of 2048 x 1024 1.24x, of 1024 x 2048 1.24x, of 4096 x 1536 0.95x
  // at 12), from 16 experts on they are level from some 8 rows on.
  const bool small = moe_small_launch(E, I);
  if (rows < (small && E <= 8 ? 14 : 10)) return 16;
  if (const int block = moe_one_round_block(rows, E, I, false)) return block;
  if (rows < 14 || (small && rows <= 52)) return 64;
  if (rows <= 104 || (small && rows >= 170 && rows <= 215)) return 128;
  return 192;
}
// The row-scaled modes have no persistent walk and no activation in the first GEMM's epilogue; the streaming tile kernel
// takes 128 slots too (1.07-1.16x over one-tile launches of that height on layers that fill the chip).
int moe_auto_block_rows(int64_t M, int E, int topk, int64_t H, int64_t I) {
  static const int forced = getenv("SGLAMD_MOE_BLOCK_M") ? atoi(getenv("SGLAMD_MOE_BLOCK_M")) : 0;
  if (forced == 16 || forced == 32 || forced == 64 || forced == 128 || forced == 192) return forced;
  const double rows = (double)M * topk / (E > 0 ? E : 1);
  if (moe_layer_streams(E, H, I))
    return rows < moe_stream_from(E, H, I, GEMM_ROW_INT8) ? 16 : moe_height_by_rounds(E, topk, H, I, rows, true);
  // What counts without it is how few rows a tile pads: the shortest block that still holds a whole expert (its weights are
  // streamed once).  A layer that fills the chip moves on sooner, since an expert that overflows adds a tile to a full
  // round.  Sixteen layers of 4 to 64 experts that do not fill it, these bands against the ones of a layer that does: 64 at
  // 42..52 rows 1.06x in the mean (0.96-1.11), at 53..56 1.01x (0.82-1.10); 128 at 105..112 rows 1.00x (0.80-1.09), at
  // 170..215 1.10x (0.80-1.23).
  const bool small = moe_small_launch(E, I);
  if (rows < (small && E <= 8 ? 14 : 10.001)) return 16;
  if (const int block = moe_one_round_block(rows, E, I, true)) return block;
  if (rows <= (small ? 56 : 42)) return 64;
  if (rows <= (small ? 112 : 104) || (small && rows >= 170 && rows <= 215)) return 128;
  return 192;
}
int grouped_block_m(int64_t rows, int E) { return moe_auto_block(rows, E, 1, 0, 0); }
// The expert-major layer gives the bits of its separate operators, which know an expert's rows and nothing of the layer: it
// leaves the 16-slot blocks, whose kernel sums K in another order than the tile kernels, where they do.
int moe_grouped_layer_block(int64_t M, int E, int topk, int block) {  // block: the layer's own choice
  const int separate = grouped_block_m(M * topk, E);
  return separate <= 32 || block <= 32 ? separate : block;
}
}  // namespace

extern "C" int64_t sglamd_fused_moe_block_fp8_workspace(int64_t M, int64_t H, int64_t I, int E, int topk, int block_m) {
  const DeviceScope scope;
  if (M <= 0 || H <= 0 || I <= 0 || E <= 0 || topk <= 0) return 0;
  if (block_m == 0) block_m = moe_auto_block(M, E, topk, H, I);
  return moe_ws_layout(M, H, I, E, topk, block_m).total;
}

extern "C" int64_t sglamd_fused_moe_layer_workspace(int mode, int64_t M, int64_t H, int64_t I, int E, int topk,
                                                    int block_m) {
  const DeviceScope scope;
  if (M <= 0 || H <= 0 || I <= 0 || E <= 0 || topk <= 0) return 0;
  const int picked = block_m                ? block_m
                     : gemm_is_block(mode) ? moe_auto_block(M, E, topk, H, I, gemm_is_int8(mode))
                                           : moe_auto_block_rows(M, E, topk, H, I);
  int64_t total = moe_ws_layout(M, H, I, E, topk, picked).total;
  if (block_m == 0 && mode == GEMM_BLOCK_FP8) {  // (the expert-major layer is sized here too)
    const int64_t grouped = moe_ws_layout(M, H, I, E, topk, moe_grouped_layer_block(M, E, topk, picked)).total;
    if (grouped > total) total = grouped;
  }
  return total;
}

// What the expert-major form of the layer adds: the caller's tables, and routing weights that are rounded to the layer's
// type and applied in the final sum, not in the second GEMM.
struct MoeGroupedOut {
  int32_t *expert_offsets, *problem_sizes1, *problem_sizes2;
};

// `mode` is a GEMM_* mode: the two block-scaled ones with [E, 2I/128, H/128] and [E, H/128, I/128] scales, the two
// row-scaled ones with one scale per output channel ([E, 2I], [E, H]) and optional biases of that shape in `dtype`.
static int moe_layer(int mode, const void* hidden, int dtype, int64_t M, int64_t H, int64_t I, int E, int topk,
                     const void* w13, const float* w13_scale, const void* b13, const void* w2, const float* w2_scale,
                     const void* b2, const float* topk_weights, const void* topk_ids, int ids_dtype, void* out,
                     float routed_scaling_factor, int block_m, void* workspace, int64_t workspace_bytes, void* stream,
                     const MoeGroupedOut* grouped = nullptr) {
  const DeviceScope scope;
  SGLAMD_REQUIRE(hidden && w13 && w13_scale && w2 && w2_scale && topk_weights && topk_ids && out && workspace,
                 SGLAMD_EINVAL, "fused_moe: null pointer");
  SGLAMD_REQUIRE(M > 0 && E > 0 && topk > 0, SGLAMD_EINVAL, "fused_moe: bad M/E/topk");
  SGLAMD_REQUIRE(H % 128 == 0 && I % 128 == 0, SGLAMD_EINVAL,
                 "fused_moe: hidden (%lld) and intermediate (%lld) sizes must be multiples of 128", (long long)H,
                 (long long)I);
  SGLAMD_REQUIRE(dtype == SGLAMD_BF16 || dtype == SGLAMD_F16, SGLAMD_EINVAL, "fused_moe: dtype must be Half or BFloat16");
  const bool row = !gemm_is_block(mode), int8 = gemm_is_int8(mode);
  SGLAMD_REQUIRE(!row || H <= ROW_QUANT_MAX_HIDDEN, SGLAMD_ENOTSUP, "fused_moe: hidden size %lld is beyond %lld",
                 (long long)H, (long long)ROW_QUANT_MAX_HIDDEN);
  SGLAMD_REQUIRE(!row || I <= ROW_QUANT_MAX_HIDDEN, SGLAMD_ENOTSUP, "fused_moe: intermediate size %lld is beyond %lld",
                 (long long)I, (long long)ROW_QUANT_MAX_HIDDEN);
  SGLAMD_REQUIRE(row || (!b13 && !b2), SGLAMD_ENOTSUP, "fused_moe: biases go with row-scaled weights");
  if (block_m == 0) {
    block_m = row ? moe_auto_block_rows(M, E, topk, H, I) : moe_auto_block(M, E, topk, H, I, int8);
    if (grouped) block_m = moe_grouped_layer_block(M, E, topk, block_m);
  }
  SGLAMD_REQUIRE(block_m == 16 || block_m == 32 || block_m == 64 || block_m == 128 || block_m == 192, SGLAMD_EINVAL,
                 "fused_moe: block_m must be 16, 32, 64, 128 or 192");
  const MoeWs w = moe_ws_layout(M, H, I, E, topk, block_m);
  SGLAMD_REQUIRE(workspace_bytes >= w.total, SGLAMD_EINVAL, "fused_moe: workspace too small (%lld < %lld)",
                 (long long)workspace_bytes, (long long)w.total);
  SGLAMD_REQUIRE(((uintptr_t)workspace % 256) == 0, SGLAMD_EINVAL, "fused_moe: workspace must be 256-byte aligned");
  uint8_t* ws = (uint8_t*)workspace;
  int32_t* sorted = (int32_t*)(ws + w.sorted);
  int32_t* expert = (int32_t*)(ws + w.expert);
  int32_t* post = (int32_t*)(ws + w.post);
  int32_t* cumsum = (int32_t*)(ws + w.cumsum);
  const int64_t T = M * topk, KB1 = H / 128, KB2 = I / 128;
  SGLAMD_REQUIRE(ids_dtype == SGLAMD_I32 || ids_dtype == SGLAMD_I64, SGLAMD_EINVAL,
                 "fused_moe: topk_ids must be int32 or int64");
  SGLAMD_REQUIRE(E + 1 <= 2048 && T < (1ll << 30), SGLAMD_EINVAL, "fused_moe: too many experts or tokens");
  SGLAMD_REQUIRE(((uintptr_t)hidden % 16) == 0, SGLAMD_EINVAL, "fused_moe: hidden must be 16-byte aligned");
  int rc = SGLAMD_OK;
  // the last launch: the k rows of every token summed
  auto finish = [&]() -> int {
    if (!grouped) return sglamd_moe_sum_reduce(ws + w.c3, out, dtype, M, topk, H, routed_scaling_factor, stream);
    const int64_t slices = ceil_div(H, 2048);
    const dim3 grid((unsigned)M, (unsigned)(slices < 64 ? slices : 64));
    if (dtype == SGLAMD_BF16)
      hipLaunchKernelGGL(weighted_sum_kernel<BF16>, grid, dim3(256), 0, (hipStream_t)stream, (const u16*)(ws + w.c3),
                         (u16*)out, topk_weights, topk, (int)H);
    else
      hipLaunchKernelGGL(weighted_sum_kernel<F16>, grid, dim3(256), 0, (hipStream_t)stream, (const u16*)(ws + w.c3),
                         (u16*)out, topk_weights, topk, (int)H);
    return check_launch("weighted_sum");
  };
  // Decode-sized calls run with fewer launches.  Up to four tokens the activation kernel goes: the first GEMM's
  // tiles pair gate and up rows and write silu(gate) * up, the second GEMM quantises those 16-bit rows itself, at
  // most four per tile -- so these calls align the routing to blocks of 4 (a tile then holds one such block; an
  // expert named more than four times, which takes repeated ids within a token, gets several).  A single token
  // also drops the sorting / quantising launch in front, since its pairs are their own blocks and the first GEMM quantises
  // the hidden state itself (with more tokens the quantised rows of K = H bytes each would crowd the weight rings out of
  // LDS: measured 150 against 120 us at two tokens), and the sum behind: two launches.  Every variant produces the bits of
  // the five-launch sequence.
  // SGLAMD_MOE_FUSE=1 keeps the launch in front, SGLAMD_MOE_FUSE=0 the whole sequence.
  static const int fuse_level = getenv("SGLAMD_MOE_FUSE") ? atoi(getenv("SGLAMD_MOE_FUSE")) : 2;
  const bool fuse_act = mode == GEMM_BLOCK_FP8 && fuse_level >= 1 && block_m == 16 && M <= 4 && T <= 32 && I % 256 == 0 &&
                        M * H * 2 < 0x7ffffff0ll && 2 * I * H < 0x7ffffff0ll && T * I * 2 < 0x7ffffff0ll;
  // (T <= E: every pair has a block of its own; both GEMMs hold a 16-bit row in LDS beside the weight rings)
  const bool fuse_all = fuse_act && fuse_level >= 2 && M == 1 && T <= E && H <= 32768 && I <= 32768 && !grouped;
  if (row) {
    const RowQuantArgs qa = {hidden, ws + w.xq, (float*)(ws + w.xs), H, M};
    const int nb = E + 1;
    const size_t lds = moe_align_lds_bytes(nb);
    const int parts = moe_align_parts(T);
    // hidden rows in four pieces per lane, 4 or 16 to a workgroup, once that still fills the chip
    const int team = M < 1024 || H > 8192 ? 0 : H <= 2048 ? 64 : 256;
    const unsigned blocks = (unsigned)(parts + (team ? ceil_div(M, 1024 / team) : M));
    hipStream_t st = (hipStream_t)stream;
#define SGLAMD_ROW_PROLOGUE(IDT, TT, Q, NV, TEAM)                                                                            \
  do {                                                                                                                 \
    auto k = moe_row_prologue_kernel<IDT, TT, Q, NV, TEAM>;                                                                  \
    SGLAMD_RAISE_LDS(k, lds);                                                                                          \
    hipLaunchKernelGGL(k, dim3(blocks), dim3(1024), lds, st, (const IDT*)topk_ids, sorted, expert, post, cumsum, nb,   \
                       block_m, (int)T, (int)w.max_padded, parts, qa);                                                 \
  } while (0)
#define SGLAMD_ROW_PROLOGUE_NV(IDT, TT, Q)                       \
  do {                                                           \
    if (team == 64) SGLAMD_ROW_PROLOGUE(IDT, TT, Q, 4, 64);       \
    else if (team == 256) SGLAMD_ROW_PROLOGUE(IDT, TT, Q, 4, 256); \
    else if (H <= 8192) SGLAMD_ROW_PROLOGUE(IDT, TT, Q, 1, 0);     \
    else SGLAMD_ROW_PROLOGUE(IDT, TT, Q, 4, 0);                    \
  } while (0)
#define SGLAMD_ROW_PROLOGUE_T(IDT, Q)                               \
  do {                                                              \
    if (dtype == SGLAMD_BF16) SGLAMD_ROW_PROLOGUE_NV(IDT, BF16, Q); \
    else SGLAMD_ROW_PROLOGUE_NV(IDT, F16, Q);                       \
  } while (0)
    if (ids_dtype == SGLAMD_I32) {
      if (int8) SGLAMD_ROW_PROLOGUE_T(int32_t, true);
      else SGLAMD_ROW_PROLOGUE_T(int32_t, false);
    } else {
      if (int8) SGLAMD_ROW_PROLOGUE_T(int64_t, true);
      else SGLAMD_ROW_PROLOGUE_T(int64_t, false);
    }
#undef SGLAMD_ROW_PROLOGUE_T
#undef SGLAMD_ROW_PROLOGUE_NV
#undef SGLAMD_ROW_PROLOGUE
    rc = check_launch("moe_row_prologue");
    if (rc) return rc;
    GemmArgs g = {};
    g.A = ws + w.xq;
    g.lda = H;
    g.sa = (const float*)(ws + w.xs);
    g.sa_sm = 1;
    g.B = (const uint8_t*)w13;
    g.ldb = H;
    g.b_expert_stride = 2 * I * H;
    g.sb = w13_scale;
    g.sb_se = 2 * I;
    g.sb_sn = 1;
    g.bias = b13;
    g.sb_sk = 2 * I;
    g.C = ws + w.c1;
    g.ldc = 2 * I;
    g.M = (int)T;
    g.N = (int)(2 * I);
    g.K = (int)H;
    g.sorted_ids = sorted;
    g.expert_ids = expert;
    g.num_post_pad = post;
    g.top_k = topk;
    g.num_valid = (int)T;
    g.max_blocks_m = (int)w.max_blocks;
    g.streams = moe_layer_streams(E, H, I) ? 1 : -1;
    GemmArgs h = g;
    h.A = ws + w.aq;
    h.lda = I;
    h.sa = (const float*)(ws + w.as);
    h.B = (const uint8_t*)w2;
    h.ldb = I;
    h.b_expert_stride = H * I;
    h.sb = w2_scale;
    h.sb_se = H;
    h.bias = b2;
    h.sb_sk = H;
    h.C = ws + w.c3;
    h.ldc = H;
    h.N = (int)H;
    h.K = (int)I;
    h.topk_w = topk_weights;
    h.top_k = 1;
    h.mul_weight = 1;
    SGLAMD_REQUIRE(moe_rows_ok(g) && moe_rows_ok(h), SGLAMD_ENOTSUP, "fused_moe: an operand of 2 GiB or more");
    rc = moe_rows_gemm(mode, g, dtype, block_m, st);
    if (rc) return rc;
    rc = launch_row_quant(RowQuantArgs{ws + w.c1, ws + w.aq, (float*)(ws + w.as), I, T}, T, dtype, int8, true, st);
    if (rc) return rc;
    rc = moe_rows_gemm(mode, h, dtype, block_m, st);
    if (rc) return rc;
    return sglamd_moe_sum_reduce(ws + w.c3, out, dtype, M, topk, H, routed_scaling_factor, stream);
  }
  // Where the persistent walk takes the first GEMM, its epilogue applies SiLU * up and the group quantisation
  // itself and writes the second GEMM's operand directly (same bits as the two launches it replaces).
  const bool fusable = mode == GEMM_BLOCK_FP8 && moe_actq_enabled();
  const bool tall = fusable && (block_m == 192 || (block_m == 128 && moe_persist128_enabled())) && moe_persist_enabled();
  GemmArgs first = {};
  first.A = ws + w.xq;
  first.lda = H;
  first.B = (const uint8_t*)w13;
  first.ldb = H;
  first.b_expert_stride = 2 * I * H;
  first.sa = (const float*)(ws + w.xs);
  first.sa_sm = KB1;
  first.sa_sk = 1;
  first.sb = w13_scale;
  first.sb_se = (2 * I / 128) * KB1;
  first.sb_sn = KB1;
  first.sb_sk = 1;
  first.C = ws + w.aq;                 // [T, I] e4m3
  first.ldc = I;
  first.A16 = ws + w.as;               // [T, I / 128] group scales, written by the kernel
  first.lda16 = KB2;
  first.M = (int)T;
  first.N = (int)(2 * I);
  first.K = (int)H;
  first.sorted_ids = sorted;
  first.expert_ids = expert;
  first.num_post_pad = post;
  first.top_k = topk;
  first.num_valid = (int)T;
  first.max_blocks_m = (int)w.max_blocks;
  first.streams = moe_layer_streams(E, H, I) ? 1 : -1;
  // These kernels fetch activation scales in groups of four K blocks: rows of another length are padded, in the place of
  // the first GEMM's 16-bit output, which does not exist then.
  const int64_t pitch1 = (KB1 + 3) & ~(int64_t)3, pitch2 = (KB2 + 3) & ~(int64_t)3;
  const bool ragged = pitch1 != KB1 || pitch2 != KB2;
  bool padded = fusable && ragged && up256(M * pitch1 * 4) + T * pitch2 * 4 <= T * 2 * I * 2;
  GemmArgs as_padded = first;
  as_padded.sa = (const float*)(ws + w.c1);
  as_padded.sa_sm = pitch1;
  as_padded.A16 = ws + w.c1 + up256(M * pitch1 * 4);
  as_padded.lda16 = pitch2;
  as_padded.scale_rows_padded = 1;
  const bool streamed = fusable && block_m == 64 && moe_stream_takes<64>(padded ? as_padded : first, true);
  const bool act_fused = streamed || (tall && gemm8_moe_persist_ok(first) && (int64_t)(2 * I / 256) * first.max_blocks_m > device_cus());
  padded = padded && act_fused;
  if (padded) first = as_padded;
  if (!fuse_all) {
    GroupQuantArgs qa = {};
    qa.in = hidden;
    qa.q = ws + w.xq;
    qa.s = (void*)first.sa;
    qa.set_rows(M, H, 128);
    qa.layout = SGLAMD_SCALE_ROW_MAJOR;
    qa.scale_stride = first.sa_sm;
    qa.eps = 1e-10f;
    qa.min8 = int8 ? -128.f : -448.f;
    qa.max8 = int8 ? 127.f : 448.f;
    qa.form = SGLAMD_QUANT_FORM_RECIPROCAL;
    qa.q_is_fp8 = !int8;
    const int nb = E + 1;
    const size_t lds = moe_align_lds_bytes(nb);
    const int parts = moe_align_parts(T);
    const unsigned blocks = (unsigned)parts + (grouped ? 1 : 0) + (unsigned)ceil_div(qa.num_groups * 8, 1024);
    MoePrepArgs pa = {};
    if (grouped) {
      pa.expert_offsets = grouped->expert_offsets;
      pa.problem_sizes1 = grouped->problem_sizes1;
      pa.problem_sizes2 = grouped->problem_sizes2;
      pa.topk = topk;
      pa.n = (int)I;
      pa.k = (int)H;
    }
    hipStream_t st = (hipStream_t)stream;
#define SGLAMD_PROLOGUE(IDT, TT, TABLES)                                                                               \
  do {                                                                                                                 \
    auto k = moe_prologue_kernel<IDT, TT, TABLES>;                                                                     \
    SGLAMD_RAISE_LDS(k, lds);                                                                                          \
    hipLaunchKernelGGL(k, dim3(blocks), dim3(1024), lds, st, (const IDT*)topk_ids, sorted, expert, post, cumsum, nb,   \
                       fuse_act ? 4 : block_m, (int)T, (int)(fuse_act ? w.few_padded : w.max_padded), parts, qa, pa);  \
  } while (0)
    if (grouped) {
      if (dtype == SGLAMD_BF16) SGLAMD_PROLOGUE(int32_t, BF16, true);
      else SGLAMD_PROLOGUE(int32_t, F16, true);
    } else if (ids_dtype == SGLAMD_I32) {
      if (dtype == SGLAMD_BF16) SGLAMD_PROLOGUE(int32_t, BF16, false);
      else SGLAMD_PROLOGUE(int32_t, F16, false);
    } else {
      if (dtype == SGLAMD_BF16) SGLAMD_PROLOGUE(int64_t, BF16, false);
      else SGLAMD_PROLOGUE(int64_t, F16, false);
    }
#undef SGLAMD_PROLOGUE
    rc = check_launch("moe_prologue");
    if (rc) return rc;
  }
  if (fuse_act) {
    const int64_t expect = T < w.max_blocks ? T : w.max_blocks;
    GemmArgs g = {};
    if (fuse_all) {
      g.A16 = hidden;
      g.lda16 = H * 2;
      g.act_mode = 1;
      g.q_eps = 1e-10f;
      g.q_min = -448.f;
      g.q_max = 448.f;
      g.route_ids = topk_ids;
      g.route_ids_i64 = ids_dtype == SGLAMD_I64;
      g.route_experts = E;
      g.sum_count = (int*)(ws + w.xq);  // (no quantised rows in this form)
      g.sum_tiles = (int)(H / 32);
    } else {
      g.A = ws + w.xq;
      g.lda = H;
      g.sa = (const float*)(ws + w.xs);
      g.sa_sm = KB1;
      g.sa_sk = 1;
    }
    g.B = (const uint8_t*)w13;
    g.ldb = H;
    g.b_expert_stride = 2 * I * H;
    g.sb = w13_scale;
    g.sb_se = (2 * I / 128) * KB1;
    g.sb_sn = KB1;
    g.sb_sk = 1;
    g.C = ws + w.c1;  // [T, I] activations
    g.ldc = I;
    g.M = (int)T;
    g.N = (int)(2 * I);
    g.K = (int)H;
    g.sorted_ids = sorted;
    g.expert_ids = expert;
    g.num_post_pad = post;
    g.top_k = topk;
    g.num_valid = (int)T;
    g.max_blocks_m = (int)(fuse_all ? w.max_blocks : w.few_blocks);
    g.sorted_stride = fuse_all ? 0 : 4;
    g.epi_silu = 1;
    g.act_hidden = I;
    hipStream_t st = (hipStream_t)stream;
    if (!fuse_all)
      rc = dtype == SGLAMD_BF16 ? gemm8_skinny_launch_fn<1, 2, GEMM_BLOCK_FP8, BF16, true>(g, st, expect)
                                : gemm8_skinny_launch_fn<1, 2, GEMM_BLOCK_FP8, F16, true>(g, st, expect);
    else
      rc = dtype == SGLAMD_BF16 ? gemm8_skinny_launch_fn<1, 2, GEMM_BLOCK_FP8, BF16, true, 1>(g, st, expect)
                                : gemm8_skinny_launch_fn<1, 2, GEMM_BLOCK_FP8, F16, true, 1>(g, st, expect);
    if (rc) return rc;
    GemmArgs h = {};
    h.A16 = ws + w.c1;
    h.lda16 = I * 2;
    h.act_mode = 1;
    h.q_eps = 1e-10f;
    h.q_min = -448.f;
    h.q_max = 448.f;
    h.B = (const uint8_t*)w2;
    h.ldb = I;
    h.b_expert_stride = H * I;
    h.sb = w2_scale;
    h.sb_se = (H / 128) * KB2;
    h.sb_sn = KB2;
    h.sb_sk = 1;
    h.C = ws + w.c3;
    h.ldc = H;
    h.M = (int)T;
    h.N = (int)H;
    h.K = (int)I;
    h.sorted_ids = sorted;
    h.expert_ids = expert;
    h.num_post_pad = post;
    h.topk_w = topk_weights;
    h.top_k = 1;
    h.num_valid = (int)T;
    h.mul_weight = grouped ? 0 : 1;
    h.max_blocks_m = (int)(fuse_all ? w.max_blocks : w.few_blocks);
    h.sorted_stride = fuse_all ? 0 : 4;
    if (fuse_all) {
      h.route_ids = topk_ids;
      h.route_ids_i64 = ids_dtype == SGLAMD_I64;
      h.route_experts = E;
      h.sum_out = out;
      h.sum_scale = routed_scaling_factor;
      h.sum_count = (int*)(ws + w.xq);
      h.sum_tiles = (int)(H / 32);
    }
    if (!fuse_all)
      rc = dtype == SGLAMD_BF16 ? gemm8_skinny_launch_fn<1, 2, GEMM_BLOCK_FP8, BF16, true, 4>(h, st, expect)
                                : gemm8_skinny_launch_fn<1, 2, GEMM_BLOCK_FP8, F16, true, 4>(h, st, expect);
    else
      rc = dtype == SGLAMD_BF16 ? gemm8_skinny_launch_fn<1, 2, GEMM_BLOCK_FP8, BF16, true, 1>(h, st, expect)
                                : gemm8_skinny_launch_fn<1, 2, GEMM_BLOCK_FP8, F16, true, 1>(h, st, expect);
    if (rc || fuse_all) return rc;
    return finish();
  }
  if (act_fused) {
    if (streamed)
      rc = dtype == SGLAMD_BF16 ? gemm8_moe_stream_launch<GEMM_BLOCK_FP8, BF16, 64, true>(first, (hipStream_t)stream)
                                : gemm8_moe_stream_launch<GEMM_BLOCK_FP8, F16, 64, true>(first, (hipStream_t)stream);
    else if (block_m == 192)
      rc = dtype == SGLAMD_BF16 ? gemm8_moe_persist_launch<GEMM_BLOCK_FP8, BF16, 3, true>(first, (hipStream_t)stream)
                                : gemm8_moe_persist_launch<GEMM_BLOCK_FP8, F16, 3, true>(first, (hipStream_t)stream);
    else
      rc = dtype == SGLAMD_BF16 ? gemm8_moe_persist_launch<GEMM_BLOCK_FP8, BF16, 2, true>(first, (hipStream_t)stream)
                                : gemm8_moe_persist_launch<GEMM_BLOCK_FP8, F16, 2, true>(first, (hipStream_t)stream);
    if (rc) return rc;
  }
  if (!act_fused) {
    rc = moe_block_gemm(mode, ws + w.xq, H, (const float*)(ws + w.xs), KB1, 1, w13, 2 * I * H, H, w13_scale,
                        (2 * I / 128) * KB1, KB1, 1, ws + w.c1, 2 * I, dtype, sorted, expert, post, nullptr, T, topk, 0,
                        block_m, w.max_blocks, 2 * I, H, stream, 0, first.streams);
    if (rc) return rc;
    rc = sglamd_silu_mul_group_quant_8bit(ws + w.c1, dtype, ws + w.aq, int8 ? SGLAMD_I8 : SGLAMD_FP8_E4M3, ws + w.as, T,
                                          I, 128, SGLAMD_SCALE_ROW_MAJOR, 0, 1e-10f, int8 ? -128.f : -448.f,
                                          int8 ? 127.f : 448.f, SGLAMD_QUANT_FORM_RECIPROCAL, stream);
    if (rc) return rc;
  }
  rc = moe_block_gemm(mode, ws + w.aq, I, (const float*)first.A16, first.lda16, 1, w2, H * I, I, w2_scale,
                      (H / 128) * KB2, KB2, 1, ws + w.c3, H, dtype, sorted, expert, post, topk_weights, T, 1,
                      grouped ? 0 : 1, block_m, w.max_blocks, H, I, stream, first.scale_rows_padded, first.streams);
  if (rc) return rc;
  return finish();
}

extern "C" int sglamd_fused_moe_block_fp8(const void* hidden, int dtype, int64_t M, int64_t H, int64_t I, int E,
                                          int topk, const void* w13, const float* w13_scale, const void* w2,
                                          const float* w2_scale, const float* topk_weights, const void* topk_ids,
                                          int ids_dtype, void* out, float routed_scaling_factor, int block_m,
                                          void* workspace, int64_t workspace_bytes, void* stream) {
  return moe_layer(GEMM_BLOCK_FP8, hidden, dtype, M, H, I, E, topk, w13, w13_scale, nullptr, w2, w2_scale, nullptr,
                   topk_weights, topk_ids, ids_dtype, out, routed_scaling_factor, block_m, workspace, workspace_bytes,
                   stream);
}

extern "C" int sglamd_fused_moe_grouped_layer(const void* hidden, int dtype, int64_t M, int64_t H, int64_t I, int E,
                                              int topk, const void* w13, const float* w13_scale, const void* w2,
                                              const float* w2_scale, const float* topk_weights, const int32_t* topk_ids,
                                              int32_t* expert_offsets, int32_t* problem_sizes1, int32_t* problem_sizes2,
                                              void* out, void* workspace, int64_t workspace_bytes, void* stream) {
  SGLAMD_REQUIRE(expert_offsets && problem_sizes1 && problem_sizes2, SGLAMD_EINVAL, "fused_moe_grouped: null pointer");
  SGLAMD_REQUIRE(((uintptr_t)out % 16) == 0, SGLAMD_EINVAL, "fused_moe_grouped: out must be 16-byte aligned");
  const MoeGroupedOut tables = {expert_offsets, problem_sizes1, problem_sizes2};
  return moe_layer(GEMM_BLOCK_FP8, hidden, dtype, M, H, I, E, topk, w13, w13_scale, nullptr, w2, w2_scale, nullptr,
                   topk_weights, topk_ids, SGLAMD_I32, out, 1.f, 0, workspace, workspace_bytes, stream, &tables);
}

extern "C" int sglamd_fused_moe_layer(int mode, const void* hidden, int dtype, int64_t M, int64_t H, int64_t I, int E,
                                      int topk, const void* w13, const float* w13_scale, const void* b13,
                                      const void* w2, const float* w2_scale, const void* b2, const float* topk_weights,
                                      const void* topk_ids, int ids_dtype, void* out, float routed_scaling_factor,
                                      int block_m, void* workspace, int64_t workspace_bytes, void* stream) {
  SGLAMD_REQUIRE(mode >= SGLAMD_MOE_BLOCK_FP8 && mode <= SGLAMD_MOE_BLOCK_INT8, SGLAMD_EINVAL, "fused_moe: bad mode %d",
                 mode);
  return moe_layer(mode, hidden, dtype, M, H, I, E, topk, w13, w13_scale, b13, w2, w2_scale, b2, topk_weights, topk_ids,
                   ids_dtype, out, routed_scaling_factor, block_m, workspace, workspace_bytes, stream);
}

// ---------------------------------------------------------------------------------------
// The same layer for callers that cannot allocate device memory: the intermediates live in a
// file-scope device array instead of a caller workspace.
// ---------------------------------------------------------------------------------------
#define SGLAMD_MOE_STATIC_SCRATCH_BYTES (16ll << 20)
static __device__ __align__(256) uint8_t scratch[SGLAMD_MOE_STATIC_SCRATCH_BYTES];

// Device address of `scratch` on the current device.  Every GPU holds its own copy of the array at its own
// address, so the address is looked up once per device, with that device current, and kept.
static int moe_static_scratch(void** out) {
  static void* ptrs[32] = {};
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(SGLAMD_EHIP, "hipGetDevice: %s", hipGetErrorString(e));
  SGLAMD_REQUIRE(dev >= 0 && dev < 32, SGLAMD_ENOTSUP, "fused_moe_static: device index %d is beyond 31", dev);
  if (!ptrs[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) return fail(SGLAMD_EHIP, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
    ptrs[dev] = p;
  }
  *out = ptrs[dev];
  return SGLAMD_OK;
}

extern "C" int64_t sglamd_fused_moe_block_fp8_static_max_bytes(void) { return SGLAMD_MOE_STATIC_SCRATCH_BYTES; }

extern "C" int sglamd_fused_moe_block_fp8_static(const void* hidden, int dtype, int64_t M, int64_t H, int64_t I, int E,
                                                 int topk, const void* w13, const float* w13_scale, const void* w2,
                                                 const float* w2_scale, const float* topk_weights,
                                                 const void* topk_ids, int ids_dtype, void* out,
                                                 float routed_scaling_factor, int block_m, void* stream) {
  SGLAMD_REQUIRE(M > 0 && H > 0 && I > 0 && E > 0 && topk > 0, SGLAMD_EINVAL, "fused_moe_static: bad M/H/I/E/topk");
  int64_t need = sglamd_fused_moe_block_fp8_workspace(M, H, I, E, topk, block_m);
  if (block_m == 0 && need > SGLAMD_MOE_STATIC_SCRATCH_BYTES) {
    // the shortest blocks pad the sorted list least
    block_m = 16;
    need = sglamd_fused_moe_block_fp8_workspace(M, H, I, E, topk, block_m);
  }
  SGLAMD_REQUIRE(need > 0 && need <= SGLAMD_MOE_STATIC_SCRATCH_BYTES, SGLAMD_EINVAL,
                 "fused_moe_static: M=%lld tokens (H=%lld, I=%lld, E=%d, topk=%d) need %lld bytes of scratch, the "
                 "built-in array holds %lld; use sglamd_fused_moe_block_fp8 with a workspace",
                 (long long)M, (long long)H, (long long)I, E, topk, (long long)need,
                 (long long)SGLAMD_MOE_STATIC_SCRATCH_BYTES);
  void* ws = nullptr;
  const int rc = moe_static_scratch(&ws);
  if (rc) return rc;
  return sglamd_fused_moe_block_fp8(hidden, dtype, M, H, I, E, topk, w13, w13_scale, w2, w2_scale, topk_weights,
                                    topk_ids, ids_dtype, out, routed_scaling_factor, block_m, ws,
                                    SGLAMD_MOE_STATIC_SCRATCH_BYTES, stream);
}
