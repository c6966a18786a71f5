// Work-list plans of the per-(item, KV head) attention kernels (gfx950): the
// plan's records, the kernels' arguments, the tile loads of attn_tile.hip (up to
// 64 rows), attn_block.hip (128-row blocks) and attn_f32.hip, and the epilogue
// pieces they share with attention.hip (the VALU kernel).
#pragma once

#include "attention.h"
#include "stream_device.h"

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
constexpr int kMaxTileRows = 128;  // rows per 16-bit MFMA item (above 64: the block kernel)

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
      const float msafe = M == -INFINITY ? 0.f : M;
      float z = 0.f, acc = 0.f;
      for (int r = rb; r < re; ++r) {
        const int64_t row = (int64_t)a.merge_rows[r] * a.hq + head;
        const float wgt = expf(a.part_lse[row] - msafe);
        z += wgt;
        // (a row of NaN scores has lse -inf and o NaN: its o counts, with weight 0)
        acc += wgt * a.part_o[row * D + d];
      }
      T* op = reinterpret_cast<T*>(a.out) + (int64_t)qi * a.o_sn + (int64_t)head * a.o_sh;
      op[d] = from_f32<T>(z > 0.f ? acc / z : acc * 0.f);
      if (d == 0 && a.out_lse) a.out_lse[(int64_t)qi * a.hq + head] = (z > 0.f) ? M + logf(z) : -INFINITY;
    }
    if (tid == 0) a.counters[(int64_t)mi * a.hkv + kvh] = 0;
  }
}

// ---------------------------------------------------------------- tile loads
static __device__ const uint4 kZeroChunk = {0, 0, 0, 0};

// K and V rows of an item, 64 tokens at a time, global -> LDS directly by the
// four waves of a workgroup: K at the stage's start, V one plane further, rows of
// RB bytes whose 16-byte chunk c sits at slot c ^ swz(row).  Load i of wave w
// moves rows (w IPW + i) RPI .. + RPI - 1 (1 KB of K and 1 KB of V); past the
// item's end K re-reads its last token (the caller masks the scores) and V reads
// zeros (a weight of 0 times an infinity would be NaN).  Pages and slots advance
// by whole tiles without a division.
//
// PAGED4: pages hold whole loads' rows (1 KB: 4 tokens of 256-byte rows), so a
// load's page is wave-uniform: its id comes from a register (64 of the item's ids)
// by v_readlane, the address is scalar, and a whole tile's loads cost no vector
// arithmetic.  Otherwise every lane looks its row's page up in pg_lds
// (the caller stages the item's page ids there and synchronises first).
template <int RB, bool PAGED4, int (*SWZ)(int)>
struct TileLoader {
  static constexpr int CPR = RB / 16;                  // 16-byte chunks per row
  static constexpr int RPI = 64 / CPR;                 // rows per wave load
  static constexpr int IPW = kTile / RPI / 4;          // loads per wave per tile (K and V each)
  static constexpr int PLANE = kTile * RB;
  static constexpr int STAGE = 2 * PLANE;

  uint64_t kvb, vplane;
  uint32_t row_bytes, off[IPW];
  int w, lane, ps, tok_count, dpage, dslot, last_page, last_slot;
  int page[IPW], slot[IPW];                            // of the next tile's loads (wave-uniform if PAGED4)
  int tok, pg_base, pg_reg;                            // next tile's first token; the register's first page
  const int32_t* pg_lds;

  __device__ __forceinline__ void init(const AttnArgs& a, const WorkItem& it, int kvh, int wave, const int32_t* lds,
                                       int first_page, int n_pages) {
    w = wave;
    lane = threadIdx.x & 63;
    ps = a.page_size;
    tok_count = it.tok_count;
    pg_lds = lds;
    row_bytes = (uint32_t)a.hkv * RB;
    vplane = (uint64_t)ps * row_bytes;
    kvb = reinterpret_cast<uint64_t>(a.kv) + (uint64_t)kvh * RB;
    dpage = kTile / ps;
    dslot = kTile % ps;
    last_page = n_pages - 1;
    last_slot = (it.tok_begin + it.tok_count - 1) % ps;
#pragma unroll
    for (int i = 0; i < IPW; ++i) {
      const int r0 = (w * IPW + i) * RPI, r = r0 + (PAGED4 ? 0 : lane / CPR);
      page[i] = (it.tok_begin + r) / ps - first_page;
      slot[i] = (it.tok_begin + r) % ps;
      off[i] = ((lane % CPR) ^ SWZ(r0 + lane / CPR)) << 4;
    }
    tok = 0;
    pg_base = 0;
    // (the first 64 ids from memory: no barrier before the first loads)
    pg_reg = PAGED4 ? a.pages[it.page_begin + first_page + min(lane, last_page)] : 0;
  }

  // A tile's loads: WHOLE, all its rows lie within the item.
  template <bool WHOLE>
  __device__ __forceinline__ void rows(uint32_t dst0) {
#pragma unroll
    for (int i = 0; i < IPW; ++i) {
      const int r0 = (w * IPW + i) * RPI;
      const uint32_t dst = dst0 + (w * IPW + i) * 1024;
      const int left = tok_count - 1 - (tok + r0);     // rows of this load up to the last token
      const bool in = WHOLE || lane / CPR <= left;
      if constexpr (PAGED4) {
        const int pg = WHOLE || left >= 0 ? page[i] : last_page, sl = WHOLE || left >= 0 ? slot[i] : last_slot;
        const int id = __builtin_amdgcn_readlane(pg_reg, pg - pg_base);
        const uint64_t base = kvb + (uint64_t)((uint32_t)id * 2u * (uint32_t)ps + (uint32_t)sl) * row_bytes;
        const uint32_t o = (uint32_t)(WHOLE ? lane / CPR : min(lane / CPR, max(left, 0))) * row_bytes + off[i];
        stream::dma16_sv(base, o, dst);
        if constexpr (WHOLE) {
          stream::dma16_sv(base + vplane, o, dst + PLANE);
        } else {
          const uint64_t src = base + vplane + o;
          stream::dma16(in ? reinterpret_cast<const void*>(src) : &kZeroChunk, dst + PLANE);
        }
      } else {
        const uint32_t rec = (uint32_t)pg_lds[in ? page[i] : last_page] * 2u * (uint32_t)ps + (uint32_t)(in ? slot[i] : last_slot);
        const uint64_t src = kvb + off[i] + (uint64_t)rec * row_bytes;
        stream::dma16(reinterpret_cast<const void*>(src), dst);
        stream::dma16(in ? reinterpret_cast<const void*>(src + vplane) : &kZeroChunk, dst + PLANE);
      }
      // (a tile that is not whole is the last; with many loads a wave the compiler
      // makes 6% slower code of leaving the step out there: fp32, head_dim 128)
      if constexpr (WHOLE || IPW > 4) {
        slot[i] += dslot;
        const bool carry = slot[i] >= ps;
        slot[i] -= carry ? ps : 0;
        page[i] += dpage + (carry ? 1 : 0);
      }
    }
  }

  // The next tile's loads, to LDS byte address dst0 (2 IPW vector memory operations).
  __device__ __forceinline__ void load(uint32_t dst0) {
    if constexpr (PAGED4) {
      // the wave's rows of a tile lie within 64 pages of its first (a page holds at least RPI tokens)
      const int p1 = min(page[IPW - 1], last_page);
      if (p1 - pg_base >= 64) {
        pg_base = min(page[0], last_page);
        pg_reg = pg_lds[min(pg_base + lane, last_page)];
      }
    }
    if (__builtin_expect(tok + kTile <= tok_count, 1)) {
      rows<true>(dst0);
    } else {
      rows<false>(dst0);
    }
    tok += kTile;
  }
};

// Whether pages of this size hold whole loads of rows of this many bytes.
inline bool paged4(int page_size, int row_bytes) { return page_size % (1024 / row_bytes) == 0; }

// Launches the 16-row-tile kernel (attn_tile.hip) over a work list whose items
// hold up to 64 rows: one workgroup per (item, KV head).
int tile_launch(const be_attn_plan_info* info, const AttnArgs& a, hipStream_t st);

// Launches the fp32 kernel (attn_f32.hip) over a work list whose items hold up to
// 64 rows: one workgroup per (item, KV head).
int f32_launch(const be_attn_plan_info* info, const AttnArgs& a, hipStream_t st);

// ---------------------------------------------------------------- 128-row blocks (attn_block.hip)
// A streaming plan's stream_loop when its causal groups run as 128-row blocks.
constexpr int kLoopBlocks = 2;
// Blocks (query tiles x KV heads) of a causal plan from which it does: below,
// the streaming kernel's split of the keys over all CUs is as fast or faster.  One
// bf16 prompt at 32 / 8 heads, head_dim 128, MI355X, streaming -> blocks: 256
// tokens (64 blocks) 13.8 -> 11.0 us, 512 23.1 -> 17.4, 1000 46.7 -> 30.4, 3000
// 243.6 -> 112; 8 x 1024 tokens 252 -> 103; 8 / 8 heads, 1000 tokens (64 blocks)
// about even.
constexpr int64_t kMinCausalBlocks = 64;
// The streaming kernel's time beyond the block kernel's fixed one: a constant, a
// 128-row x 64-token tile of a CU's share, a (query, head) row, 64 new tokens of the
// longest prompt.  Few new tokens after some cached ones leave too few blocks, each
// a long chain: 256 after 400 cached, 32 / 8 heads, 17.7 us streaming against 20.8,
// 512 after 400, 16 / 4 heads, 19.9 against 26.0; 2 x 256 after 8000, whose keys are
// split, 190 against 90.  Fitted to 426 plans (1 to 16 prompts of 16 to 4096 new
// tokens after 0 to 30000 cached ones, 4 to 128 query heads): by the block count
// alone 22 of them took up to 29% longer than on the other kernel, now 3 do, up to 7%.
constexpr double kStreamUs = 1.5, kStreamTileUs = 3.8, kStreamRowUs = 4e-4, kStreamSpanUs = 0.5;

// True when the block kernel has an instantiation for this shape.
bool block_eligible(int dtype, int head_dim);

// Launches the block kernel over a work list whose items hold up to 128 rows
// (queries x GQA group): one workgroup per (item, KV head).
int block_launch(const be_attn_plan_info* info, const AttnArgs& a, hipStream_t st);

}  // namespace be
