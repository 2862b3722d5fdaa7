// Decode partition plan: which (sequence, block range) work items a paged
// decode launch runs. Computed on the device from context_lens, so a
// hipGraph replays it with whatever lengths the step has.
//
// The reference fixes split_k per launch on the host from R * Hq
// (microinfer/layer/triton_paged_attention.py:342-349) and stripes tiles over
// the splits (:76-79). Here partitions are contiguous block ranges sized from
// the step's total context: about kTargetItems (item, KV head) workgroups of
// at least kMinPartBlocks blocks each; short sequences stay whole. A sequence's partitions occupy
// consecutive slots (first_item + part: where their partials go), but the
// launch dispatches items largest first, whatever their sequence: the
// hardware does not start a later workgroup on a CU that an early small item
// freed until well into the launch, so a small item in the first round
// leaves its CU idle, while small items at the end of the grid fill the
// tail.
#include "paged_attention.h"

namespace mi {
namespace {

// About this many (item, KV head) workgroups per launch. Fixed: the plan's
// size, and so the workspace a caller sizes, depends only on the call's
// arguments.
constexpr int32_t kTargetItems = 192;
// Merging partitions costs a launch about 2.5 us and more with their number,
// so a part covers an eighth of the longest sequence, but at least
// kMinPartPositions, and at most kMaxMinPart of up to kLongPositions and in
// proportion of longer ones; or as many as make kTargetItems. In positions,
// whatever the block size (at least one block): at 16, 64 and 256 tokens a
// block, parts of as many positions measured the same. One sequence, 8 KV
// heads, us with parts of 64 / 128 / 256 / 512 positions: of 300 tokens 7.0 /
// 7.4 / 8.4 / -, 1000 9.2 / 8.1 / 8.7 / 10.4, 2000 (96) 11.2 / 10.1 / 9.1 /
// 10.6, 4096 (176) 12.3 / - / 11.0 / 10.9, 8192 (352) 14.1 / - / - / 12.9,
// with 768 14.0; 2 KV heads, 256 / 512 / 1024: 4096 13.1 / 13.1 / 16.0, 16384
// 26.3 / 19.3 / 18.5, 32768 (352) 35.8 / 28.0 / 22.9.
// The vector kernel goes through a part's positions more slowly: half as many
// (float32, 8 KV heads, 128 / 256 / 512: 2000 tokens 12.3 / 12.0 / 16.3, 4096
// (176) 16.4 / 14.6 / 16.6; 2 KV heads, 4096 31.4 / 31.4 / 40.7, 8192 44 / 38
// / 44, 32768 (352) 69 / - / 62; head_dim 64 bf16 16.8 / 15.8 / 16.3 at 4096,
// float32 13.7 / 12.4 / 15.7, head_dim 256 bf16 32.6 / 28.3 / 33.2).
constexpr int32_t kMinPartPositions = 64;
constexpr int32_t kMaxMinPart = 512;
constexpr int32_t kMaxMinPartVector = 256;
constexpr int32_t kLongPositions = 16384;
// Sequences of up to this many positions are one item (one sequence of 130
// tokens 5.5 us whole, 6.8 in parts; float32 6.8, 9.3), and longer ones where
// the sequences alone make workgroups for a quarter of the chip (8 of 215: 6.9
// whole, 8.5 in parts; float32 8.5, 10.8). One CU streams a cold context more
// slowly than several: at 300 and at 512 the whole 300-token sequence of a
// decode step and eight float32 ones of 64-512 lost (181 against 179 us for
// four layers, 153 against 133 for eight). Up to kWholeBlocks blocks of up to
// kMaxMinPart positions too, whose parts would be few and uneven (300 tokens
// in blocks of 256: 7.3 whole, 8.8 in two; 200 in blocks of 64: 6.7, 7.4).
constexpr int32_t kWholePositions = 160;
constexpr int32_t kWholePositionsMany = 256;
constexpr int32_t kWholeBlocks = 4;
constexpr int32_t kManyItems = 64;

// Four waves: fewer waves per barrier than 1024 threads (0.06 us less per
// decode launch of a 28-layer step, whose launches share one plan).
constexpr int kPlanThreads = 256;
constexpr int kSortLimit = 1024;  // larger batches keep submission order

__device__ __forceinline__ int blocks_of(int ctx, int block_size, int lb) {
  return (ctx + block_size - 1) >> lb;
}

// Blocks per partition of a sequence of nb blocks (all but its last).
__device__ __forceinline__ int part_blocks(int nb, int split_k, int pb_global, int whole) {
  if (split_k == 0) return nb <= whole ? max(nb, 1) : pb_global;
  const int k = min(split_k, max(nb, 1));
  return max(1, (nb + k - 1) / k);
}

// The step's part size from its blocks in all and its longest sequence's.
__device__ __forceinline__ int step_part_blocks(int64_t total_blocks, int longest, int lb,
                                                int num_kv_heads, int target, int max_min_part) {
  const int64_t want = total_blocks * num_kv_heads;
  const int most = max(max_min_part >> lb, longest / (kLongPositions / max_min_part));
  const int least = min(max(longest / 8, kMinPartPositions >> lb), most);
  return max(max(least, 1), static_cast<int>((want + target - 1) / target));
}

__device__ __forceinline__ int whole_blocks(int num_seqs, int num_kv_heads, int lb) {
  const int positions =
      num_seqs * num_kv_heads >= kManyItems ? kWholePositionsMany : kWholePositions;
  return max(positions >> lb, min(kWholeBlocks, kMaxMinPart >> lb));
}

__global__ __launch_bounds__(kPlanThreads) void decode_plan_kernel(
    const int32_t* __restrict__ context_lens, int num_seqs, int num_kv_heads, int block_size,
    int lb, int width, int split_k, int target, int max_min_part, int max_items,
    PlanItem* __restrict__ plan, int32_t* __restrict__ counters, int num_counters) {
  __shared__ int s_ctx[kMaxPlanSeqs];
  __shared__ int s_order[kMaxPlanSeqs];  // rank -> sequence
  __shared__ int s_first[kMaxPlanSeqs];  // rank -> first item index
  __shared__ int s_scan[kPlanThreads];
  __shared__ int s_size[kSortLimit];  // slot -> blocks (size-ordered dispatch)
  __shared__ int s_rank[kSortLimit];  // slot -> plan position
  __shared__ int s_total_blocks;
  __shared__ int s_total_items;
  __shared__ int s_longest;
  const int whole = whole_blocks(num_seqs, num_kv_heads, lb);
  const int tid = threadIdx.x;
  const int max_ctx = width * block_size;

  // Arrival counters of the decode launch that follows (when given): zero
  // them here, so a caller whose counter memory is shared or reused needs
  // no separate clear.
  if (counters != nullptr)
    for (int i = tid; i < num_counters; i += kPlanThreads) counters[i] = 0;
  if (tid == 0) {
    s_total_blocks = 0;
    s_total_items = 0;
    s_longest = 0;
  }
  __syncthreads();
  int local = 0, longest = 0;
  for (int r = tid; r < num_seqs; r += kPlanThreads) {
    const int c = min(max(context_lens[r], 0), max_ctx);
    s_ctx[r] = c;
    local += blocks_of(c, block_size, lb);
    longest = max(longest, blocks_of(c, block_size, lb));
  }
  atomicAdd(&s_total_blocks, local);
  atomicMax(&s_longest, longest);
  __syncthreads();
  const int pb_global =
      split_k == 0 ? step_part_blocks(s_total_blocks, s_longest, lb, num_kv_heads, target,
                                    max_min_part) : 1;

  // Rank sequences by block count, longest first (ties keep batch order).
  const bool sort = num_seqs <= kSortLimit;
  for (int r = tid; r < num_seqs; r += kPlanThreads) {
    int rank = r;
    if (sort) {
      const int nb = blocks_of(s_ctx[r], block_size, lb);
      rank = 0;
      for (int s = 0; s < num_seqs; ++s) {
        const int ns = blocks_of(s_ctx[s], block_size, lb);
        rank += (ns > nb) || (ns == nb && s < r);
      }
    }
    s_order[rank] = r;
  }
  __syncthreads();

  // Exclusive scan of partition counts in rank order: each thread owns a run
  // of consecutive ranks, then the per-thread sums are scanned in LDS.
  const int per = (num_seqs + kPlanThreads - 1) / kPlanThreads;
  const int k0 = tid * per;
  const int k1 = min(num_seqs, k0 + per);
  int run = 0;
  for (int k = k0; k < k1; ++k) {
    const int nb = blocks_of(s_ctx[s_order[k]], block_size, lb);
    run += max(1, (nb + part_blocks(nb, split_k, pb_global, whole) - 1) /
                      part_blocks(nb, split_k, pb_global, whole));
  }
  s_scan[tid] = run;
  __syncthreads();
  for (int off = 1; off < kPlanThreads; off <<= 1) {
    const int v = tid >= off ? s_scan[tid - off] : 0;
    __syncthreads();
    s_scan[tid] += v;
    __syncthreads();
  }
  int first = s_scan[tid] - run;
  for (int k = k0; k < k1; ++k) {
    s_first[k] = first;
    const int nb = blocks_of(s_ctx[s_order[k]], block_size, lb);
    const int pb = part_blocks(nb, split_k, pb_global, whole);
    first += max(1, (nb + pb - 1) / pb);
  }
  if (tid == kPlanThreads - 1) s_total_items = s_scan[tid];
  __syncthreads();

  // Emit the items, then mark the rest of the launch's slots unused. Slots
  // (first_item + part) number a sequence's partitions consecutively; the
  // plan position a workgroup reads is the item's rank by size, largest
  // first (ties in slot order), so every workgroup of the first round is
  // one of the largest and the launch ends with the smallest items.
  const int total_items = min(s_total_items, max_items);
  const bool by_size = total_items <= kSortLimit;
  if (by_size) {
    for (int k = tid; k < num_seqs; k += kPlanThreads) {
      const int nb = blocks_of(s_ctx[s_order[k]], block_size, lb);
      const int pb = part_blocks(nb, split_k, pb_global, whole);
      const int np = max(1, (nb + pb - 1) / pb);
      for (int p = 0; p < np && s_first[k] + p < max_items; ++p)
        s_size[s_first[k] + p] = min(nb, (p + 1) * pb) - p * pb;
    }
    __syncthreads();
    // One thread per slot: its rank among all items (every thread reads the
    // same size at a time, an LDS broadcast).
    for (int i = tid; i < total_items; i += kPlanThreads) {
      const int sz = s_size[i];
      int r = 0;
      for (int j = 0; j < total_items; ++j) {
        const int o = s_size[j];
        r += (o > sz) || (o == sz && j < i);
      }
      s_rank[i] = r;
    }
    __syncthreads();
  }
  for (int k = tid; k < num_seqs; k += kPlanThreads) {
    const int r = s_order[k];
    const int c = s_ctx[r];
    const int nb = blocks_of(c, block_size, lb);
    const int pb = part_blocks(nb, split_k, pb_global, whole);
    const int np = max(1, (nb + pb - 1) / pb);
    const int f = s_first[k];
    for (int p = 0; p < np && f + p < max_items; ++p) {
      PlanItem it;
      it.seq = r;
      it.blk_begin = p * pb;
      it.blk_end = min(nb, (p + 1) * pb);
      it.nparts = np;
      it.first_item = f;
      it.ctx = c;
      it.part = p;
      it.unused = 0;
      plan[by_size ? s_rank[f + p] : f + p] = it;
    }
  }
  for (int i = s_total_items + tid; i < max_items; i += kPlanThreads) {
    PlanItem it{};
    it.seq = -1;
    plan[i] = it;
  }
}

// The same plan for at most a wave's width of sequences and adaptive
// partitions, the shape of every ordinary decode step: one lane per sequence
// and no LDS, so the launch is little more than one load and one store. Every
// wave derives the plan and each emits a quarter of it. All parts but a
// sequence's last (or only) one have the step's part size, so an item's rank
// by size needs only counts over sequences, not a sort over items.
// Per launch in a graph: one sequence of 16384 tokens 10.1 -> 4.3 us, 32 of
// 128-2048 8.6 -> 4.5.
__global__ __launch_bounds__(kPlanThreads) void decode_plan_wave_kernel(
    const int32_t* __restrict__ context_lens, int num_seqs, int num_kv_heads, int block_size,
    int lb, int width, int target, int max_min_part, int max_items, PlanItem* __restrict__ plan,
    int32_t* __restrict__ counters, int num_counters) {
  const int tid = threadIdx.x;
  const int lane = tid % kWave;
  const int wave = tid / kWave;
  constexpr int kWaves = kPlanThreads / kWave;
  const bool mine = lane < num_seqs;
  const int ctx = mine ? min(max(context_lens[lane], 0), width * block_size) : 0;
  if (counters != nullptr)
    for (int i = tid; i < num_counters; i += kPlanThreads) counters[i] = 0;
  const int nb = blocks_of(ctx, block_size, lb);
  int longest = nb;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) longest = max(longest, __shfl_xor(longest, o, kWave));
  const int pb = step_part_blocks(wave_sum_int(nb), longest, lb, num_kv_heads, target,
                                    max_min_part);
  const int np = nb <= whole_blocks(num_seqs, num_kv_heads, lb) ? 1 : (nb + pb - 1) / pb;
  const int last = nb - (np - 1) * pb;  // blocks of the last part, the odd one
  // Over the sequences ahead of this lane's (longer, or as long and earlier
  // in the batch): items and full parts; and the odd parts dispatched before this lane's
  // full parts (larger, or as large in an earlier slot) and before its own.
  int first = 0, full_ahead = 0, items = 0, odd_before_full = 0, odd_before_odd = 0;
  for (int s = 0; s < num_seqs; ++s) {
    const int nb_s = __builtin_amdgcn_readlane(nb, s);
    const int np_s = __builtin_amdgcn_readlane(np, s);
    const int last_s = __builtin_amdgcn_readlane(last, s);
    const bool ahead = nb_s > nb || (nb_s == nb && s < lane);
    first += ahead ? np_s : 0;
    full_ahead += ahead ? np_s - 1 : 0;
    odd_before_full += last_s > pb || (last_s == pb && ahead);
    odd_before_odd += last_s > last || (last_s == last && ahead);
    items += np_s;
  }
  const int all_full = items - num_seqs;
  // Full parts smaller than this lane's odd one come after it.
  const int full_before_odd =
      pb > last ? all_full : pb == last ? full_ahead + np - 1 : 0;
  const int full_rank = odd_before_full + full_ahead;
  const int odd_rank = odd_before_odd + full_before_odd;
  auto emit = [&](int seq, int c, int blocks, int parts, int slot, int full_at, int odd_at,
                  int p) {
    if (slot + p >= max_items) return;
    const bool odd = p == parts - 1;
    PlanItem it;
    it.seq = seq;
    it.blk_begin = p * pb;
    it.blk_end = odd ? blocks : (p + 1) * pb;
    it.nparts = parts;
    it.first_item = slot;
    it.ctx = c;
    it.part = p;
    it.unused = 0;
    plan[min(odd ? odd_at : full_at + p, max_items - 1)] = it;
  };
  if (__ballot(np > 2 * kWaves) == 0) {
    // Few parts each: every lane emits its own sequence's.
    if (mine)
      for (int p = wave; p < np; p += kWaves)
        emit(lane, ctx, nb, np, first, full_rank, odd_rank, p);
  } else {
    // Long sequences: a lane per part.
    for (int s = wave; s < num_seqs; s += kWaves) {
      const int parts = __builtin_amdgcn_readlane(np, s);
      const int c = __builtin_amdgcn_readlane(ctx, s), blocks = __builtin_amdgcn_readlane(nb, s);
      const int slot = __builtin_amdgcn_readlane(first, s);
      const int full_at = __builtin_amdgcn_readlane(full_rank, s);
      const int odd_at = __builtin_amdgcn_readlane(odd_rank, s);
      for (int p = lane; p < parts; p += kWave) emit(s, c, blocks, parts, slot, full_at, odd_at, p);
    }
  }
  for (int i = items + tid; i < max_items; i += kPlanThreads) {
    PlanItem it{};
    it.seq = -1;
    plan[i] = it;
  }
}

}  // namespace

int32_t decode_max_items(int32_t num_seqs, int32_t num_kv_heads, int32_t split_k) {
  if (split_k > 0) return num_seqs * split_k;
  return (kTargetItems + num_kv_heads - 1) / num_kv_heads + num_seqs;
}

int64_t decode_plan_bytes(int32_t num_seqs, int32_t num_kv_heads, int32_t split_k) {
  return static_cast<int64_t>(decode_max_items(num_seqs, num_kv_heads, split_k)) *
         static_cast<int64_t>(sizeof(PlanItem));
}

int32_t launch_decode_plan(const int32_t* context_lens, int32_t num_seqs, int32_t num_kv_heads,
                           int32_t block_size, int32_t block_table_width, int32_t split_k,
                           bool vector, PlanItem* plan, int32_t* counters, hipStream_t stream) {
  const int32_t max_min_part = vector ? kMaxMinPartVector : kMaxMinPart;
  if (num_seqs <= kWave && split_k == 0) {
    decode_plan_wave_kernel<<<1, kPlanThreads, 0, stream>>>(
        context_lens, num_seqs, num_kv_heads, block_size, ilog2(block_size), block_table_width,
        kTargetItems, max_min_part, decode_max_items(num_seqs, num_kv_heads, split_k), plan,
        counters, counters != nullptr ? num_seqs * num_kv_heads : 0);
    return check_launch("decode plan");
  }
  decode_plan_kernel<<<1, kPlanThreads, 0, stream>>>(
      context_lens, num_seqs, num_kv_heads, block_size, ilog2(block_size), block_table_width,
      split_k, kTargetItems, max_min_part,
      decode_max_items(num_seqs, num_kv_heads, split_k), plan, counters,
      counters != nullptr ? num_seqs * num_kv_heads : 0);
  return check_launch("decode plan");
}

}  // namespace mi

extern "C" int64_t mi_decode_plan_bytes(int32_t num_seqs, int32_t num_kv_heads,
                                        int32_t split_k) {
  if (num_seqs <= 0 || num_kv_heads <= 0 || split_k < 0) return 0;
  return mi::decode_plan_bytes(num_seqs, num_kv_heads, split_k);
}

namespace {
int32_t decode_plan(const char* who, const int32_t* context_lens, int32_t num_seqs,
                    int32_t num_kv_heads, int32_t block_size, int32_t block_table_width,
                    int32_t split_k, bool vector, void* plan, int64_t plan_bytes, void* stream) {
  using namespace mi;
  clear_error();
  const std::string fn(who);
  if (num_seqs < 0 || num_kv_heads <= 0 || split_k < 0 || block_table_width < 0)
    return fail(MI_ERR_INVALID_ARGUMENT, fn + ": invalid sizes");
  if (!is_pow2(block_size))
    return fail(MI_ERR_INVALID_ARGUMENT, fn + ": block_size must be a power of two");
  if (num_seqs > kMaxPlanSeqs)
    return fail(MI_ERR_UNSUPPORTED, fn + ": more than 4096 sequences");
  if (num_seqs == 0) return MI_OK;
  if (!context_lens || !plan) return fail(MI_ERR_INVALID_ARGUMENT, fn + ": null pointer");
  if (plan_bytes < decode_plan_bytes(num_seqs, num_kv_heads, split_k) ||
      reinterpret_cast<uintptr_t>(plan) % 32 != 0)
    return fail(MI_ERR_WORKSPACE, fn + ": plan buffer too small or misaligned");
  return launch_decode_plan(context_lens, num_seqs, num_kv_heads, block_size,
                            block_table_width, split_k, vector, static_cast<PlanItem*>(plan),
                            nullptr, static_cast<hipStream_t>(stream));
}
}  // namespace

extern "C" int32_t mi_decode_plan(const int32_t* context_lens, int32_t num_seqs,
                                  int32_t num_kv_heads, int32_t block_size,
                                  int32_t block_table_width, int32_t split_k, void* plan,
                                  int64_t plan_bytes, void* stream) {
  return decode_plan("mi_decode_plan", context_lens, num_seqs, num_kv_heads, block_size,
                     block_table_width, split_k, false, plan, plan_bytes, stream);
}

extern "C" int32_t mi_decode_plan_for(const int32_t* context_lens, int32_t num_seqs,
                                      int32_t num_q_heads, int32_t num_kv_heads,
                                      int32_t head_dim, int32_t dtype, int32_t block_size,
                                      int32_t block_table_width, int32_t split_k, void* plan,
                                      int64_t plan_bytes, void* stream) {
  if (num_kv_heads <= 0 || num_q_heads <= 0 || num_q_heads % num_kv_heads != 0 ||
      head_dim <= 0 || !mi::valid_dtype(dtype)) {
    mi::clear_error();
    return mi::fail(MI_ERR_INVALID_ARGUMENT, "mi_decode_plan_for: invalid heads or dtype");
  }
  const int32_t group = num_q_heads / num_kv_heads;
  return decode_plan("mi_decode_plan_for", context_lens, num_seqs, num_kv_heads, block_size,
                     block_table_width, split_k,
                     !mi::decode_mfma_takes(dtype, head_dim, group, block_size), plan, plan_bytes,
                     stream);
}
