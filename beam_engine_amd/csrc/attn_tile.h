// Work-list plans of the per-(item, KV head) attention kernels (gfx950): the
// plan's records, the kernels' arguments, and the epilogue pieces shared by
// attention.hip (tile and VALU kernels) and attn_block.hip (128-row blocks).
#pragma once

#include "attention.h"

namespace be {

// ------------------------------------------------------------------ plan layout
// Device plan = int32 words:
//   items      [num_items][8]   WorkItem
//   q_index    [num_queries]     query ids referenced by items
//   pages      [sum of level page lists]
//   merge_q    [num_merge]       queries the merge kernel combines
//   merge_ptr  [num_merge + 1]   CSR into merge_rows
//   merge_rows [...]             partial rows of each merged query
struct WorkItem {
  int32_t q_begin;     // first entry of q_index
  int32_t q_count;     // queries in the tile
  int32_t page_begin;  // first entry of pages[] of the item's group
  int32_t tok_begin;   // first group token covered (a multiple of 32)
  int32_t tok_count;   // tokens covered, > 0
  int32_t out_row;     // first partial row, or -1: write the final output
  int32_t vis0;        // causal: group tokens its first query sees, unclamped (query j: vis0 + j); else kNoCausal
  int32_t pad1;
};
constexpr int32_t kNoCausal = 0x3fffffff;
static_assert(sizeof(WorkItem) == 32, "WorkItem is 8 int32 words");

constexpr int kTile = 64;              // tokens per LDS tile
constexpr int kMaxPagesLds = 1024;     // page ids of one item staged in LDS
constexpr int kMaxRows = 32;       // rows (queries x GQA group) per VALU workgroup
constexpr int kMaxTileRows = 128;  // rows per MFMA workgroup (8 row tiles of 16)

struct AttnArgs {
  const void* q;
  int64_t q_sn, q_sh;
  const void* kv;
  void* out;
  int64_t o_sn, o_sh;
  float* out_lse;
  float* part_o;      // [rows, Hq, D]
  float* part_lse;    // [rows, Hq]
  const WorkItem* items;
  const int32_t* q_index;
  const int32_t* pages;
  // fused merge (null counters: the separate merge kernel runs instead)
  const int32_t* q_merge;      // per query: merge-list index or -1
  const int32_t* merge_ptr;    // CSR of partial rows per merge-list entry
  const int32_t* merge_rows;
  int32_t* counters;           // [num_merge][hkv] arrivals, zero between runs
  const int32_t* live_items;   // fixed layout: live item count (surplus workgroups exit)
  int page_size, hkv, hq, g;
  float scale_log2;   // sm_scale * log2(e)
};

// Element offset of (page, kv, slot, head, 0) in a [P, 2, page, Hkv, D] layer.
__device__ __forceinline__ int64_t kv_off(int page, int kvsel, int slot, int head, int page_size,
                                          int hkv, int d) {
  return ((((int64_t)page * 2 + kvsel) * page_size + slot) * hkv + head) * (int64_t)d;
}

// Writes the finished state of one row: o = acc / l, lse = (m + log2 l) ln 2.
template <typename T>
__device__ __forceinline__ void store_row_lse(const AttnArgs& a, const WorkItem& it, int j, int head,
                                              float m2, float l) {
  float lse = (l > 0.f) ? (m2 + log2f(l)) * 0.69314718055994531f : -INFINITY;
  if (it.out_row < 0) {
    if (a.out_lse) {
      int qi = a.q_index[it.q_begin + j];
      a.out_lse[(int64_t)qi * a.hq + head] = lse;
    }
  } else {
    a.part_lse[(int64_t)(it.out_row + j) * a.hq + head] = lse;
  }
}

// Fused split-K merge.  Called by every thread of a workgroup after it wrote
// its partial rows.  For each query of the item the workgroup counts its
// arrival on (query, kv head); the workgroup that completes the count merges
// the g heads of that query from every partial row by log-sum-exp, writes the
// output and resets the counter for the next run.  The release fence makes
// this workgroup's partial rows visible device-wide (all XCD L2s) before its
// arrival is counted; the acquire fence orders the merger's reads after it.
template <typename T, int D>
__device__ void fused_merge_epilogue(const AttnArgs& a, const WorkItem& it, int kvh, int* s_last) {
  __threadfence();
  __syncthreads();
  const int tid = threadIdx.x;
  if (tid < it.q_count) {
    const int qi = a.q_index[it.q_begin + tid];
    const int mi = a.q_merge[qi];
    const int expect = a.merge_ptr[mi + 1] - a.merge_ptr[mi];
    const int old = __hip_atomic_fetch_add(&a.counters[(int64_t)mi * a.hkv + kvh], 1, __ATOMIC_ACQ_REL,
                                           __HIP_MEMORY_SCOPE_AGENT);
    s_last[tid] = (old == expect - 1) ? mi : -1;
  }
  __syncthreads();
  bool fenced = false;
  for (int j = 0; j < it.q_count; ++j) {
    const int mi = s_last[j];
    if (mi < 0) continue;
    if (!fenced) {
      __threadfence();
      fenced = true;
    }
    const int qi = a.q_index[it.q_begin + j];
    const int rb = a.merge_ptr[mi], re = a.merge_ptr[mi + 1];
    // thread -> (head hh, column d); g * D elements over 256 threads
    for (int e = tid; e < a.g * D; e += 256) {
      const int hh = e / D, d = e - hh * D, head = kvh * a.g + hh;
      float M = -INFINITY;
      for (int r = rb; r < re; ++r) M = fmaxf(M, a.part_lse[(int64_t)a.merge_rows[r] * a.hq + head]);
      float z = 0.f, acc = 0.f;
      if (M != -INFINITY) {
        for (int r = rb; r < re; ++r) {
          const int64_t row = (int64_t)a.merge_rows[r] * a.hq + head;
          const float wgt = expf(a.part_lse[row] - M);
          z += wgt;
          acc += wgt * a.part_o[row * D + d];
        }
      }
      T* op = reinterpret_cast<T*>(a.out) + (int64_t)qi * a.o_sn + (int64_t)head * a.o_sh;
      op[d] = from_f32<T>(z > 0.f ? acc / z : 0.f);
      if (d == 0 && a.out_lse) a.out_lse[(int64_t)qi * a.hq + head] = (z > 0.f) ? M + logf(z) : -INFINITY;
    }
    if (tid == 0) a.counters[(int64_t)mi * a.hkv + kvh] = 0;
  }
}

// ---------------------------------------------------------------- 128-row blocks (attn_block.hip)
// A streaming plan's stream_loop when its causal groups run as 128-row blocks.
constexpr int kLoopBlocks = 2;
// Blocks (query tiles x KV heads) of a causal plan from which it does: below,
// the streaming kernel's split of the keys over all CUs is as fast or faster.  One
// bf16 prompt at 32 / 8 heads, head_dim 128, MI355X, streaming -> blocks: 256
// tokens (64 blocks) 13.8 -> 11.3 us, 512 23.1 -> 16.0, 1000 46.7 -> 28.1, 3000
// 243.6 -> 87 - 93; 8 x 1024 tokens 256 -> 101; 8 / 8 heads, 1000 tokens (64
// blocks) 21.5 -> 21.6.
constexpr int64_t kMinCausalBlocks = 64;

// True when the block kernel has an instantiation for this shape.
bool block_eligible(int dtype, int head_dim);

// Launches the block kernel over a work list whose items hold up to 128 rows
// (queries x GQA group): one workgroup per (item, KV head).
int block_launch(const be_attn_plan_info* info, const AttnArgs& a, hipStream_t st);

}  // namespace be
