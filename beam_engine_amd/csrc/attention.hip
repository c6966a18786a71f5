// Paged attention over work lists on gfx950: the planner (which also decides for
// the streaming and row-block kernels), the VALU kernel, the merge kernel and the
// launches; the MFMA kernels are in attn_tile.hip, attn_block.hip, attn_f32.hip.
//
// One work-list format serves every strategy.  A work item is a tile of
// queries (a contiguous slice of q_index) attending to a contiguous token range
// of one paged group (a slice of the plan's page list).  The attention kernel
// runs one workgroup per (item, KV head) and writes either the final output
// (a query with a single item) or a partial (o, lse) row that the merge kernel
// combines by log-sum-exp.  The reference computes the same quantities with
// FlashInfer's MultiLevelCascadeAttentionWrapper (models/modeling_llama.py:
// 321-367, 732-755) and the FastTree Triton kernels
// (attention/fasttree/kernel.py:5-285).

#include <math.h>
#include <stdarg.h>

#include <algorithm>
#include <vector>

#include "attn_tile.h"

namespace be {

struct MergeArgs {
  const float* part_o;
  const float* part_lse;
  const int32_t* merge_q;
  const int32_t* merge_ptr;
  const int32_t* merge_rows;
  void* out;
  int64_t o_sn, o_sh;
  float* out_lse;
  const int32_t* live;         // fixed layout: live entry count (surplus workgroups exit)
  int hq;
};

// ================================================================== VALU kernel
// Any storage dtype and alignment, D in {64, 128, 256}, up to 32 rows per
// workgroup (blockIdx.z picks them from items of more).  K/V blocks of 32 tokens
// are converted to fp32 in LDS; scores use one thread per (token, row-group), P.V
// one thread per (head_dim column, row-group).  Runs BE_PLAN_FORCE_VALU plans, and
// any work list whose operands the other kernels' 16-byte accesses cannot take.
template <typename T, int D>
__global__ __launch_bounds__(256) void attn_valu_kernel(AttnArgs a) {
  constexpr int BT = 32;
  constexpr int NRG = 256 / D;           // row groups in the P.V phase
  constexpr int RPT = kMaxRows / NRG;    // rows per thread in the P.V phase
  constexpr int KST = D + 1;             // padded K row
  __shared__ float qs[kMaxRows][D];
  __shared__ float ks[BT * KST];
  __shared__ float vs[BT][D];
  __shared__ float psm[kMaxRows][BT];
  __shared__ float alpha_s[kMaxRows], l_s[kMaxRows], m_s[kMaxRows];
  if (a.live_items && (int)blockIdx.x >= *a.live_items) return;

  WorkItem it = a.items[blockIdx.x];
  const int kvh = blockIdx.y;
  const int tid = threadIdx.x;
  const int g = a.g;
  const int q0 = (int)blockIdx.z * (kMaxRows / g);     // this workgroup's queries of the item
  if (q0 >= it.q_count) return;
  it.q_begin += q0;
  it.q_count = min(it.q_count - q0, kMaxRows / g);
  if (it.out_row >= 0) it.out_row += q0;
  if (it.vis0 != kNoCausal) it.vis0 += q0;
  const int R = it.q_count * g;
  const T* qbase = reinterpret_cast<const T*>(a.q);
  const T* kv = reinterpret_cast<const T*>(a.kv);
  const int ps = a.page_size;

  for (int e = tid; e < kMaxRows * D; e += 256) {
    const int r = e / D, d = e % D;
    float val = 0.f;
    if (r < R) {
      const int j = r / g, hh = r - j * g;
      const int qi = a.q_index[it.q_begin + j];
      val = to_f32(qbase[(int64_t)qi * a.q_sn + (int64_t)(kvh * g + hh) * a.q_sh + d]);
    }
    qs[r][d] = val;
  }

  // score-phase ownership: token t = tid % 32, rows rg + 8k
  const int t_own = tid & 31, rg = tid >> 5;
  float m_row[4], l_row[4];
  int lim_row[4];    // item tokens row rg + 8k sees (causal: its query's limit)
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    m_row[k] = -INFINITY;
    l_row[k] = 0.f;
    const int64_t v = (int64_t)it.vis0 + (rg + 8 * k) / g - it.tok_begin;
    lim_row[k] = (int)std::min<int64_t>(it.tok_count, std::max<int64_t>(v, 0));
  }
  // P.V-phase ownership: column d = tid % D, rows rgp + NRG*k
  const int d_own = tid % D, rgp = tid / D;
  float acc[RPT];
#pragma unroll
  for (int k = 0; k < RPT; ++k) acc[k] = 0.f;

  for (int tb = 0; tb < it.tok_count; tb += BT) {
    __syncthreads();
    for (int e = tid; e < BT * D; e += 256) {
      const int t = e / D, d = e % D;
      const int tl = tb + t;
      float kx = 0.f, vx = 0.f;
      if (tl < it.tok_count) {
        const int tok = it.tok_begin + tl;
        const int page = a.pages[it.page_begin + tok / ps];
        kx = to_f32(kv[kv_off(page, 0, tok % ps, kvh, ps, a.hkv, D) + d]);
        vx = to_f32(kv[kv_off(page, 1, tok % ps, kvh, ps, a.hkv, D) + d]);
      }
      ks[t * KST + d] = kx;
      vs[t][d] = vx;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int r = rg + 8 * k;
      float sc = 0.f;
#pragma unroll 8
      for (int d = 0; d < D; ++d) sc += qs[r][d] * ks[t_own * KST + d];
      const float x = (tb + t_own) < lim_row[k] ? sc * a.scale_log2 : -INFINITY;
      float mx = x;
#pragma unroll
      for (int o = 16; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
      const float m_new = fmaxf(m_row[k], mx);
      const float msafe = (m_new == -INFINITY) ? 0.f : m_new;   // a row with nothing seen yet
      const float p = exp2f(x - msafe);
      float psum = p;
#pragma unroll
      for (int o = 16; o > 0; o >>= 1) psum += __shfl_xor(psum, o, 64);
      const float al = exp2f(m_row[k] - msafe);
      l_row[k] = l_row[k] * al + psum;
      m_row[k] = m_new;
      psm[r][t_own] = p;
      if (t_own == 0) alpha_s[r] = al;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
      const int r = rgp + NRG * k;
      float sacc = acc[k] * alpha_s[r];
#pragma unroll 8
      for (int t = 0; t < BT; ++t) sacc += psm[r][t] * vs[t][d_own];
      acc[k] = sacc;
    }
  }
  if (t_own == 0) {
#pragma unroll
    for (int k = 0; k < 4; ++k) { l_s[rg + 8 * k] = l_row[k]; m_s[rg + 8 * k] = m_row[k]; }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < RPT; ++k) {
    const int r = rgp + NRG * k;
    if (r >= R) continue;
    const int j = r / g, hh = r - j * g, head = kvh * g + hh;
    const float l = l_s[r];
    const float o = (l > 0.f) ? acc[k] / l : 0.f;
    if (it.out_row < 0) {
      const int qi = a.q_index[it.q_begin + j];
      reinterpret_cast<T*>(a.out)[(int64_t)qi * a.o_sn + (int64_t)head * a.o_sh + d_own] = from_f32<T>(o);
    } else {
      a.part_o[((int64_t)(it.out_row + j) * a.hq + head) * D + d_own] = o;
    }
    if (d_own == 0) store_row_lse<T>(a, it, j, head, m_s[r], l);
  }
  __shared__ int s_last[kMaxRows];
  if (it.out_row >= 0 && a.counters) fused_merge_epilogue<T, D>(a, it, kvh, s_last);
}

// ================================================================== merge kernel
// One thread per (merged query, head, 4 head_dim columns): eight partial rows'
// lse and o at a time (their loads issued together), combined by log-sum-exp
// with a running max.  No LDS and no barrier: the launch is a chain of dependent
// round trips (row range, row ids, lse and o) and little else, so the heads of a
// query are spread over workgroups.  One workgroup per query with the weights in
// LDS took 9.8 us for 32 queries of 17 partial rows (32 heads, head_dim 64,
// MI355X), 5.6 us now; 8 queries of 4 rows (head_dim 128) 5.3 -> 3.2 us.
constexpr int kMergeBatch = 8;

template <typename T, int D>
__global__ __launch_bounds__(256) void merge_kernel(MergeArgs a) {
  constexpr int C4 = D / 4;                       // float4 columns per head
  if (a.live && (int)blockIdx.x >= *a.live) return;
  const int i = blockIdx.y * 256 + threadIdx.x, h = i / C4, c = i - h * C4;
  const int hq = a.hq;
  if (h >= hq) return;
  const int qi = a.merge_q[blockIdx.x];
  const int b = a.merge_ptr[blockIdx.x], e = a.merge_ptr[blockIdx.x + 1];
  float M = -INFINITY, z = 0.f;
  v4f acc = {0.f, 0.f, 0.f, 0.f};
  for (int r0 = b; r0 < e; r0 += kMergeBatch) {
    float l[kMergeBatch];
    v4f o[kMergeBatch];
#pragma unroll
    for (int u = 0; u < kMergeBatch; ++u) {
      const int64_t row = (int64_t)a.merge_rows[min(r0 + u, e - 1)] * hq + h;
      l[u] = r0 + u < e ? a.part_lse[row] : -INFINITY;
      o[u] = *reinterpret_cast<const v4f*>(a.part_o + row * D + 4 * c);
    }
    float m = M;
#pragma unroll
    for (int u = 0; u < kMergeBatch; ++u) m = fmaxf(m, l[u]);
    const float msafe = m == -INFINITY ? 0.f : m;
    const float s = expf(M - msafe);              // 0 while nothing was seen
    z *= s;
    acc *= s;
#pragma unroll
    for (int u = 0; u < kMergeBatch; ++u) {
      const float wgt = expf(l[u] - msafe);
      z += wgt;
      // a row of NaN scores has lse -inf and o NaN: its o counts, with weight 0
      if (r0 + u < e) acc += o[u] * wgt;
    }
    M = m;
  }
  const float inv = (z > 0.f) ? 1.f / z : 0.f;
  T* op = reinterpret_cast<T*>(a.out) + (int64_t)qi * a.o_sn + (int64_t)h * a.o_sh + 4 * c;
#pragma unroll
  for (int k = 0; k < 4; ++k) op[k] = from_f32<T>(acc[k] * inv);
  if (a.out_lse && c == 0) a.out_lse[(int64_t)qi * hq + h] = (z > 0.f) ? M + logf(z) : -INFINITY;
}

// One wave owns one row, so outputs may alias inputs (every lane reads the
// row's lse before lane 0 overwrites it).
__global__ __launch_bounds__(256) void merge2_kernel(const float* oa, const float* la, const float* ob,
                                                    const float* lb, float* oo, float* lo, int rows,
                                                    int d) {
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (r >= rows) return;
  const float x = la[r], y = lb[r];
  const float M = fmaxf(x, y);
  float ca = 0.f, cb = 0.f;
  if (M != -INFINITY) { ca = expf(x - M); cb = expf(y - M); }
  const float z = ca + cb;
  const float inv = (z > 0.f) ? 1.f / z : 0.f;
  for (int e = lane; e < d; e += 64) {
    const int64_t i = r * d + e;
    oo[i] = (ca * oa[i] + cb * ob[i]) * inv;
  }
  if (lane == 0) lo[r] = (z > 0.f) ? M + logf(z) : -INFINITY;
}

// ================================================================== host: planner
int attn_plan(const be_level* levels, int num_levels, int num_queries, int hq, int hkv, int d,
              int page_size, int num_pages, int dtype, int flags, int num_cus, const be_plan_caps* caps,
              int32_t* out, int64_t cap, be_attn_plan_info* info) {
  BE_REQUIRE(info != nullptr && out != nullptr, "null plan buffer or info");
  memset(info, 0, sizeof(*info));
  BE_REQUIRE(num_levels >= 0 && (num_levels == 0 || levels != nullptr), "bad levels");
  BE_REQUIRE(num_queries >= 0, "num_queries must be >= 0");
  BE_REQUIRE(hq > 0 && hkv > 0 && hq % hkv == 0, "num_qo_heads (%d) must be a multiple of num_kv_heads (%d)", hq, hkv);
  BE_REQUIRE(page_size > 0 && num_pages > 0, "page_size and num_pages must be positive");
  BE_REQUIRE(dtype == BE_F32 || dtype == BE_F16 || dtype == BE_BF16, "unknown dtype %d", dtype);
  const int g = hq / hkv;
  if (d != 64 && d != 128 && d != 256) return fail(BE_ERR_UNSUPPORTED, "head_dim %d: kernels exist for 64, 128, 256", d);
  if (g > kMaxTileRows) return fail(BE_ERR_UNSUPPORTED, "GQA group %d exceeds %d", g, kMaxTileRows);
  if (num_cus <= 0) num_cus = 256;

  // ---- validate levels, collect groups
  std::vector<Group> groups;
  {
    int64_t ng = 0;
    for (int lv = 0; lv < num_levels; ++lv) ng += std::max(0, levels[lv].num_groups);
    groups.reserve((size_t)ng);
  }
  int64_t total_pages = 0;
  for (int lv = 0; lv < num_levels; ++lv) {
    const be_level& L = levels[lv];
    BE_REQUIRE(L.num_groups >= 0, "level %d: negative group count", lv);
    BE_REQUIRE(L.num_groups == 0 || (L.qo_indptr && L.kv_indptr && L.last_page_len), "level %d: null index array", lv);
    if (L.num_groups == 0) continue;
    BE_REQUIRE(L.qo_indptr[0] == 0 && L.kv_indptr[0] == 0, "level %d: indptr must start at 0", lv);
    for (int j = 0; j < L.num_groups; ++j) {
      BE_REQUIRE(L.qo_indptr[j + 1] >= L.qo_indptr[j], "level %d: qo_indptr not monotone", lv);
      BE_REQUIRE(L.kv_indptr[j + 1] >= L.kv_indptr[j], "level %d: kv_indptr not monotone", lv);
      BE_REQUIRE(L.last_page_len[j] >= 0 && L.last_page_len[j] <= page_size,
                 "level %d group %d: last_page_len %d outside [0, %d]", lv, j, L.last_page_len[j], page_size);
    }
    BE_REQUIRE(L.qo_indptr[L.num_groups] <= num_queries, "level %d: qo_indptr exceeds %d queries", lv, num_queries);
    const int np = L.kv_indptr[L.num_groups];
    BE_REQUIRE(np == 0 || L.kv_indices, "level %d: null kv_indices", lv);
    for (int i = 0; i < np; ++i)
      BE_REQUIRE(L.kv_indices[i] >= 0 && L.kv_indices[i] < num_pages, "level %d: page %d out of range [0, %d)", lv,
                 L.kv_indices[i], num_pages);
    for (int j = 0; j < L.num_groups; ++j) {
      const int npg = L.kv_indptr[j + 1] - L.kv_indptr[j];
      const int kv_len = npg == 0 ? 0 : (npg - 1) * page_size + L.last_page_len[j];
      groups.push_back(Group{lv, L.qo_indptr[j], L.qo_indptr[j + 1], (int)(total_pages + L.kv_indptr[j]), kv_len});
    }
    total_pages += np;
  }

  // ---- algorithmic bytes: distinct (page, head) valid tokens, plus Q and O
  // (a per-thread table of the pool's pages, zero between calls: only the
  // referenced entries are set, summed and cleared)
  static thread_local std::vector<int> valid;
  if ((int)valid.size() < num_pages) valid.assign((size_t)num_pages, 0);
  for (int lv = 0; lv < num_levels; ++lv) {
    const be_level& L = levels[lv];
    for (int j = 0; j < L.num_groups; ++j) {
      const int b = L.kv_indptr[j], e = L.kv_indptr[j + 1];
      for (int i = b; i < e; ++i) {
        const int v = (i + 1 < e) ? page_size : L.last_page_len[j];
        int& slot = valid[L.kv_indices[i]];
        slot = std::max(slot, v);
      }
    }
  }
  int64_t valid_tokens = 0;
  for (int lv = 0; lv < num_levels; ++lv) {
    const be_level& L = levels[lv];
    const int np = L.num_groups ? L.kv_indptr[L.num_groups] : 0;
    for (int i = 0; i < np; ++i) {
      valid_tokens += valid[L.kv_indices[i]];
      valid[L.kv_indices[i]] = 0;
    }
  }
  const int64_t es = (int64_t)dtype_size(dtype);
  double flops = 0.0;
  // causal (BE_PLAN_CAUSAL): on the last level, query q0 + i of a group of n
  // queries sees its first kv_len - n + i + 1 tokens (FlashInfer's alignment of
  // the query block to the end of the keys; one query per group masks nothing)
  const bool causal = (flags & BE_PLAN_CAUSAL) != 0;
  auto is_causal = [&](const Group& gr) { return causal && gr.level == num_levels - 1 && gr.q1 - gr.q0 > 1; };
  auto vis = [&](const Group& gr, int qi) -> int {
    if (!is_causal(gr)) return gr.kv_len;
    return std::max(0, std::min(gr.kv_len, gr.kv_len - (gr.q1 - gr.q0) + (qi - gr.q0) + 1));
  };
  bool any_causal = false;
  for (const Group& gr : groups) {
    if (gr.kv_len <= 0 || gr.q1 <= gr.q0) continue;
    any_causal = any_causal || is_causal(gr);
    if (is_causal(gr)) {
      for (int qi = gr.q0; qi < gr.q1; ++qi) flops += 4.0 * d * hq * (double)vis(gr, qi);
    } else {
      flops += 4.0 * d * hq * (double)gr.kv_len * (gr.q1 - gr.q0);
    }
  }

  bool mfma = (dtype != BE_F32) && !(flags & BE_PLAN_FORCE_VALU);
  if (!mfma && g > kMaxRows) return fail(BE_ERR_UNSUPPORTED, "GQA group %d exceeds %d (VALU kernel)", g, kMaxRows);
  if (mfma && d == 256 && g > 64) return fail(BE_ERR_UNSUPPORTED, "GQA group %d exceeds 64 at head_dim 256", g);
  // rows per workgroup: MFMA 8 row tiles (4 at head_dim 256, VGPR budget, and in
  // fp32, whose kernel is kernel 0 with tile_rows set), VALU 32
  const bool f32 = dtype == BE_F32 && !(flags & BE_PLAN_FORCE_VALU);
  // (fp32 on 64-row items: half the K / V reads, but half the items too, so more
  // key splits and fp32 partial rows; a 1000-token prompt, 32 / 8 heads, head_dim
  // 128, takes 9.8 MB of workspace where 32-row items take 12.5 KB)
  const bool less = (flags & BE_PLAN_LESS_SCRATCH) != 0;
  int rows_cap = mfma ? (d == 256 ? 64 : kMaxTileRows) : f32 && !less ? 64 : kMaxRows;
  if (caps) {
    BE_REQUIRE(!(flags & BE_PLAN_FUSED_MERGE), "the fused merge is not available with a fixed-capacity layout");
    const int tr = caps->tile_rows;
    BE_REQUIRE(tr == 16 || tr == 32 || tr == 64 || tr == 128, "caps.tile_rows must be 16, 32, 64 or 128");
    BE_REQUIRE(tr >= g, "caps.tile_rows %d smaller than the GQA group %d", tr, g);
    BE_REQUIRE(caps->max_items >= 0 && caps->max_queries >= num_queries && caps->max_pages >= 0 &&
                   caps->max_merge >= 0 && caps->max_merge_rows >= 0 && caps->max_zero >= 0,
               "bad plan capacities (max_queries %d < %d queries?)", caps->max_queries, num_queries);
    if (mfma) rows_cap = std::min(rows_cap, tr);
    // (fp32: never more items than 32-row ones, which capacities were sized for
    // whatever tile_rows said; causal ones cut their keys by their own rows)
    if (f32 && (tr <= 32 || any_causal)) rows_cap = kMaxRows;
  }
  // merge-free row blocks (decode plans, compact layout): forced by
  // BE_PLAN_ROWS, else chosen when rows_preferred says so
  bool rows_ok = false;
  if (!any_causal && !caps && stream_eligible(dtype, d, g, page_size, flags) && g <= 16 &&
      !(flags & BE_PLAN_NO_ROWS) && ((flags & BE_PLAN_ROWS) || rows_preferred(groups, num_queries, g, num_cus))) {
    memset(info, 0, sizeof(*info));
    const int rc = rows_plan(groups, levels, num_levels, total_pages, num_queries, hq, hkv, page_size, num_cus, out,
                             cap, info);
    if (rc != BE_OK && rc != BE_ERR_UNSUPPORTED) return rc;
    rows_ok = rc == BE_OK;     // unsupported: a task exceeds the kernel's LDS tables
  }
  if (rows_ok) {
    info->num_qo_heads = hq;
    info->num_kv_heads = hkv;
    info->head_dim = d;
    info->page_size = page_size;
    info->num_pages = num_pages;
    info->dtype = dtype;
    info->kv_bytes = valid_tokens * hkv * d * es * 2;
    info->qo_bytes = (int64_t)num_queries * hq * d * es * 2;
    info->flops = flops;
    return BE_OK;
  }
  const int q_tile = std::max(1, rows_cap / g);
  // Causal groups on the block kernel: a workgroup's tiles run one after the
  // other (about 1.5 us each with the CU to itself, 1.05 us per tile of the CU's
  // two workgroups together: head_dim 128, MI355X), and splitting their keys costs
  // the merge pass (about 8 us) and the fp32 partials' round trip.  The longest
  // query tile is cut into the number of chunks, a power of two, that makes the
  // slower of its own chain and the CUs' shares shortest, those costs included
  // (1000 fresh tokens, 32 / 8 heads: two chunks take 14% longer than whole).
  // Plans of at most 64 rows an item run on the tile kernel instead, in tiles of
  // half the time before a merge of few rows: where that cut leaves half the CUs
  // idle it is halved until they have a workgroup each, down to two tiles or to 16
  // chunks, whose merge is two batches (4 new tokens after 3000, 8 / 8 heads,
  // head_dim 128, page 8: 16.7 us at 4 chunks, 11.2 at 16) -- whole tiles only from
  // about 6 us, what the merge pass takes (16 after 400, head_dim 64, 7.3 us whole,
  // 9.4 in 4 chunks; after 1000 11.8 and 9.2).
  int64_t causal_chunk = 0, causal_blocks = 0, tiles = 0, queries = 0, span = 0;
  double block_us = 0;
  if (any_causal && mfma && !less && !caps && rows_cap == kMaxTileRows && block_eligible(dtype, d)) {
    int64_t longest = 0;
    int most_rows = 0;
    std::vector<int64_t> tiles_of;                     // of each query tile
    for (const Group& gr : groups) {
      if (gr.kv_len <= 0 || gr.q1 <= gr.q0) continue;
      if (is_causal(gr)) causal_blocks += ceil_div(gr.q1 - gr.q0, q_tile) * hkv;
      queries += gr.q1 - gr.q0;
      most_rows = std::max(most_rows, std::min(q_tile, gr.q1 - gr.q0) * g);
      span = std::max<int64_t>(span, gr.q1 - gr.q0);
      for (int qa = gr.q0; qa < gr.q1; qa += q_tile) {
        const int64_t t = ceil_div(vis(gr, std::min(qa + q_tile, gr.q1) - 1), kTile);
        longest = std::max(longest, t);
        tiles += t * hkv;
        tiles_of.push_back(t);
      }
    }
    const double per_d = 0.3 + 0.7 * d / 128;        // a tile's time against head_dim 128
    for (int64_t cut = 1; cut == 1 || longest / cut >= 8; cut *= 2) {
      const int64_t c = ceil_div(longest, cut);
      double t = per_d * std::max(1.5 * c, 1.05 * tiles / num_cus);
      if (cut > 1) t += 8.0 + 2.0 * cut * queries * hq * d * 4 / 5e6;
      if (cut == 1 || t < block_us) {
        block_us = t;
        causal_chunk = c * kTile;
      }
    }
    const bool cut_more = most_rows <= 64 && (causal_chunk < longest * kTile || 0.7 * per_d * longest > 6.0);
    for (int64_t c = causal_chunk / kTile; cut_more && c > 2; c = ceil_div(c, 2)) {
      int64_t wgs = 0;
      for (int64_t t : tiles_of) wgs += ceil_div(t, c) * hkv;
      if (2 * wgs > num_cus || ceil_div(longest, ceil_div(c, 2)) > 16) break;
      causal_chunk = ceil_div(c, 2) * kTile;
    }
  }
  // causal groups of enough query rows run as 128-row blocks rather than on the
  // streaming kernel, unless its even shares of the same tiles and its merge of
  // 16-bit slots take less
  const bool streams = stream_eligible(dtype, d, g, page_size, flags);
  const bool blocks = streams && !caps && !less && !(flags & BE_PLAN_NO_BLOCKS) && causal_blocks >= kMinCausalBlocks &&
                      block_us <= kStreamUs + kStreamTileUs * tiles / num_cus + kStreamRowUs * queries * hq +
                                      kStreamSpanUs * span / kTile;
  if (!(any_causal && caps) && streams && !blocks && (!caps || caps->tile_rows == 64)) {
    memset(info, 0, sizeof(*info));
    const int rc = stream_plan(groups, levels, num_levels, total_pages, num_queries, hq, hkv, d, page_size,
                               num_pages, dtype, num_cus, flags, caps, out, cap, info);
    if (rc == BE_OK) {
      info->num_qo_heads = hq;
      info->num_kv_heads = hkv;
      info->head_dim = d;
      info->page_size = page_size;
      info->num_pages = num_pages;
      info->dtype = dtype;
      info->kv_bytes = valid_tokens * hkv * d * es * 2;
      info->qo_bytes = (int64_t)num_queries * hq * d * es * 2;
      info->flops = flops;
      return BE_OK;
    }
    if (rc != BE_ERR_UNSUPPORTED) return rc;
    // a workgroup would need more segments than its table holds: tile kernel
  }

  // ---- split-K chunk: about two workgroups per CU over all (tile, chunk, head)
  // (fixed fp32 layouts: cut as 32-row items, so that partial rows stay as many)
  const int cut_tile = caps && f32 ? std::max(1, kMaxRows / g) : q_tile;
  int64_t work = 0;   // token-tiles
  for (const Group& gr : groups)
    if (gr.q1 > gr.q0 && gr.kv_len > 0) work += ceil_div(gr.q1 - gr.q0, cut_tile) * (int64_t)gr.kv_len;
  const int64_t target = 3 * (int64_t)num_cus;
  int64_t chunk = ceil_div(work * hkv, target);
  chunk = std::max<int64_t>(128, ceil_div(chunk, 64) * 64);
  // an item's page ids are staged in LDS: at most kMaxPagesLds pages per item
  const int64_t chunk_cap = std::max<int64_t>(64, ((int64_t)(kMaxPagesLds - 1) * page_size) / 64 * 64);
  if (chunk > chunk_cap) chunk = chunk_cap;

  // A chunk of a group writes rows x D x 4 bytes of partials per KV head while
  // reading 4 x D bytes per token (bf16 K + V): keep chunks >= 4 x rows tokens
  // so partial traffic stays under ~1/4 of the KV bytes it summarises.
  auto group_chunk = [&](const Group& gr) -> int64_t {
    if (causal_chunk > 0) return std::min(std::max<int64_t>(causal_chunk, kTile), chunk_cap);
    const int64_t rows = (int64_t)std::min(q_tile, gr.q1 - gr.q0) * g;
    int64_t c = std::max<int64_t>(chunk, ceil_div(4 * rows, 64) * 64);
    return std::min(c, chunk_cap);
  };

  // ---- per-query partial counts (a causal query tile stops at the chunk
  // holding its last query's last visible token)
  std::vector<int> cnt(num_queries, 0);
  for (const Group& gr : groups) {
    if (gr.kv_len <= 0 || gr.q1 <= gr.q0) continue;
    const int64_t gchunk = group_chunk(gr);
    for (int qa = gr.q0; qa < gr.q1; qa += q_tile) {
      const int qn = std::min(q_tile, gr.q1 - qa);
      const int nch = (int)ceil_div(vis(gr, qa + qn - 1), gchunk);
      for (int qi = qa; qi < qa + qn; ++qi) cnt[qi] += nch;
    }
  }

  // ---- items and partial rows
  std::vector<WorkItem> items;
  std::vector<std::vector<int>> rows_of(num_queries);
  int rows = 0, max_r = 0;
  for (const Group& gr : groups) {
    if (gr.kv_len <= 0 || gr.q1 <= gr.q0) continue;
    const int64_t gchunk = group_chunk(gr);
    for (int t0 = 0; t0 < gr.kv_len; t0 += (int)gchunk) {
      for (int qa = gr.q0; qa < gr.q1; qa += q_tile) {
        const int qn = std::min(q_tile, gr.q1 - qa);
        const int tile_vis = vis(gr, qa + qn - 1);     // the tile's last query sees the most
        if (t0 >= tile_vis) continue;
        const int tc = (int)std::min<int64_t>(gchunk, tile_vis - t0);
        bool direct = true;
        for (int qi = qa; qi < qa + qn; ++qi) direct = direct && (cnt[qi] == 1);
        // vis0: tokens the item's first query sees (group token units, before
        // clamping to [0, kv_len]: may be negative), query j of the item sees
        // vis0 + j (the kernel clamps per row); kNoCausal without the mask
        const int vis0 = gr.kv_len - (gr.q1 - gr.q0) + (qa - gr.q0) + 1;
        WorkItem w{qa, qn, gr.page_base, t0, tc, -1, is_causal(gr) ? vis0 : kNoCausal, 0};
        if (!direct) {
          w.out_row = rows;
          for (int j = 0; j < qn; ++j) rows_of[qa + j].push_back(rows + j);
          rows += qn;
        }
        max_r = std::max(max_r, qn * g);
        items.push_back(w);
      }
    }
  }

  // causal items differ in length up to the prompt's: the longest first, so that
  // the last workgroups to start are the shortest
  if (any_causal)
    std::stable_sort(items.begin(), items.end(), [](const WorkItem& x, const WorkItem& y) { return x.tok_count > y.tok_count; });

  // ---- merge list (queries with partial rows: one of a tile whose other queries
  // have more items has a row too, if only one) and zero list (no keys)
  std::vector<int> merge_q, merge_ptr{0}, merge_rows, zero_q;
  for (int qi = 0; qi < num_queries; ++qi) {
    if (cnt[qi] == 0) zero_q.push_back(qi);
    if (rows_of[qi].empty()) continue;
    merge_q.push_back(qi);
    for (int r : rows_of[qi]) merge_rows.push_back(r);
    merge_ptr.push_back((int)merge_rows.size());
  }

  // ---- serialise: header of live counts, then the regions (sized to this
  //      plan, or to the capacities of a fixed layout)
  const int64_t n_items = (int64_t)items.size();
  if (caps) {
    if (n_items > caps->max_items || total_pages > caps->max_pages || (int64_t)merge_q.size() > caps->max_merge ||
        rows > caps->max_merge_rows || (int64_t)zero_q.size() > caps->max_zero)
      return fail(BE_ERR_CAPACITY,
                  "plan exceeds its fixed capacities: items %lld/%d pages %lld/%d merge %zu/%d rows %d/%d zero %zu/%d",
                  (long long)n_items, caps->max_items, (long long)total_pages, caps->max_pages, merge_q.size(),
                  caps->max_merge, rows, caps->max_merge_rows, zero_q.size(), caps->max_zero);
  }
  const int64_t c_items = caps ? caps->max_items : n_items;
  const int64_t c_q = caps ? caps->max_queries : num_queries;
  const int64_t c_pages = caps ? caps->max_pages : total_pages;
  const int64_t c_merge = caps ? caps->max_merge : (int64_t)merge_q.size();
  const int64_t c_rows = caps ? caps->max_merge_rows : (int64_t)merge_rows.size();
  const int64_t c_zero = caps ? caps->max_zero : (int64_t)zero_q.size();
  int64_t off = kPlanHeader;
  const int64_t off_items = off;    off += c_items * 8;
  const int64_t off_qindex = off;   off += c_q;
  const int64_t off_pages = off;    off += c_pages;
  const int64_t off_mq = off;       off += c_merge;
  const int64_t off_mp = off;       off += c_merge + 1;
  const int64_t off_mr = off;       off += c_rows;
  const int64_t off_qm = off;       off += c_q;
  const int64_t off_zq = off;       off += c_zero;
  const int64_t off_zp = off;       off += c_zero + 1;
  off = ceil_div(off, 4) * 4;
  if (off > cap || off > INT32_MAX) {
    info->plan_ints = (int32_t)std::min<int64_t>(off, INT32_MAX);   // the words needed (0: a capacity of caps)
    return fail(BE_ERR_CAPACITY, "plan needs %lld int32 words, buffer holds %lld", (long long)off, (long long)cap);
  }
  for (int i = 0; i < kPlanHeader; ++i) out[i] = 0;
  out[kHdrItems] = (int32_t)n_items;
  out[kHdrMerge] = (int32_t)merge_q.size();
  out[kHdrZero] = (int32_t)zero_q.size();
  out[kHdrRows] = rows;
  memcpy(out + off_items, items.data(), n_items * sizeof(WorkItem));
  for (int i = 0; i < num_queries; ++i) out[off_qindex + i] = i;
  {
    int64_t p = off_pages;
    for (int lv = 0; lv < num_levels; ++lv) {
      const be_level& L = levels[lv];
      const int np = L.num_groups ? L.kv_indptr[L.num_groups] : 0;
      if (np) memcpy(out + p, L.kv_indices, np * sizeof(int32_t));
      p += np;
    }
  }
  if (!merge_q.empty()) memcpy(out + off_mq, merge_q.data(), merge_q.size() * 4);
  memcpy(out + off_mp, merge_ptr.data(), merge_ptr.size() * 4);
  if (!merge_rows.empty()) memcpy(out + off_mr, merge_rows.data(), merge_rows.size() * 4);
  for (int qi = 0; qi < num_queries; ++qi) out[off_qm + qi] = -1;
  for (size_t m = 0; m < merge_q.size(); ++m) out[off_qm + merge_q[m]] = (int32_t)m;
  if (!zero_q.empty()) memcpy(out + off_zq, zero_q.data(), zero_q.size() * 4);
  for (int64_t i = off_zp; i < off_zp + (int64_t)zero_q.size() + 1; ++i) out[i] = 0;   // zero_ptr: empty ranges

  memset(info, 0, sizeof(*info));
  info->num_items = (int32_t)n_items;
  info->num_part_rows = rows;
  info->num_merge = (int32_t)merge_q.size();
  info->num_queries = num_queries;
  info->num_qo_heads = hq;
  info->num_kv_heads = hkv;
  info->head_dim = d;
  info->page_size = page_size;
  info->num_pages = num_pages;
  info->dtype = dtype;
  info->kernel = blocks ? 2 : mfma ? 1 : 0;
  info->stream_loop = blocks ? kLoopBlocks : 0;
  info->tile_rows = !mfma && !f32 ? 0 : blocks ? 128 : caps ? (f32 ? rows_cap : caps->tile_rows) : (max_r <= 16 ? 16 : max_r <= 32 ? 32 : max_r <= 64 ? 64 : 128);
  info->chunk_tokens = (int32_t)std::min<int64_t>(causal_chunk > 0 ? std::min(causal_chunk, chunk_cap) : chunk, INT32_MAX);
  info->plan_ints = (int32_t)off;
  info->off_items = (int32_t)off_items;
  info->off_qindex = (int32_t)off_qindex;
  info->off_pages = (int32_t)off_pages;
  info->off_merge_q = (int32_t)off_mq;
  info->off_merge_ptr = (int32_t)off_mp;
  info->off_merge_rows = (int32_t)off_mr;
  info->off_q_merge = (int32_t)off_qm;
  info->fused_merge = (flags & BE_PLAN_FUSED_MERGE) ? 1 : 0;
  info->num_zero = (int32_t)zero_q.size();
  info->off_zero_q = (int32_t)off_zq;
  info->off_zero_ptr = (int32_t)off_zp;
  info->static_layout = caps ? 1 : 0;
  info->grid_items = (int32_t)c_items;
  info->grid_merge = (int32_t)c_merge;
  info->grid_zero = (int32_t)c_zero;
  info->part_rows_cap = (int32_t)(caps ? caps->max_merge_rows : rows);
  info->counter_offset = ceil_div((int64_t)info->part_rows_cap * hq * (d + 1) * 4, 256) * 256;
  info->counter_bytes = info->fused_merge ? (int64_t)merge_q.size() * hkv * 4 : 0;
  info->partial_bytes = info->counter_offset + info->counter_bytes;
  info->kv_bytes = valid_tokens * hkv * d * es * 2;
  info->qo_bytes = (int64_t)num_queries * hq * d * es * 2;
  info->flops = flops;
  return BE_OK;
}

// ================================================================== host: run
// Whether every row of q, out and the cache starts on 16 bytes, as the MFMA
// kernels' vector and direct-to-LDS accesses need it.
static bool rows_aligned(const be_attn_plan_info* info, const AttnArgs& a) {
  const int64_t es = (int64_t)dtype_size(info->dtype);
  const uintptr_t bits = reinterpret_cast<uintptr_t>(a.q) | reinterpret_cast<uintptr_t>(a.kv) | reinterpret_cast<uintptr_t>(a.out) |
                         (uintptr_t)(a.q_sn * es) | (uintptr_t)(a.q_sh * es) | (uintptr_t)(a.o_sn * es) | (uintptr_t)(a.o_sh * es);
  return (bits & 15) == 0;
}

template <typename T>
static int launch_attn(const be_attn_plan_info* info, AttnArgs& a, hipStream_t st) {
  // (groups beyond the VALU kernel's rows: vector accesses to q and out take any
  // alignment, only the direct loads of the cache do not)
  if (a.g > kMaxRows) BE_REQUIRE((reinterpret_cast<uintptr_t>(a.kv) & 15) == 0, "the cache must be 16-byte aligned");
  const bool aligned = a.g > kMaxRows || rows_aligned(info, a);
  const int per = std::max(1, kMaxRows / a.g);         // queries a VALU workgroup takes
  const dim3 grid(info->grid_items, info->num_kv_heads, (unsigned)ceil_div(std::max(1, info->tile_rows / a.g), per));
  if (info->kernel != 0 && aligned) {
    if (info->dtype == BE_F32) return fail(BE_ERR_UNSUPPORTED, "MFMA kernel needs fp16/bf16 storage");
    if (info->tile_rows == kMaxTileRows && block_eligible(info->dtype, info->head_dim)) return block_launch(info, a, st);
    return tile_launch(info, a, st);
  } else if (info->dtype == BE_F32 && info->tile_rows != 0 && aligned) {
    return f32_launch(info, a, st);
  } else {
    switch (info->head_dim) {
      case 64: attn_valu_kernel<T, 64><<<grid, 256, 0, st>>>(a); break;
      case 128: attn_valu_kernel<T, 128><<<grid, 256, 0, st>>>(a); break;
      case 256: attn_valu_kernel<T, 256><<<grid, 256, 0, st>>>(a); break;
      default: return fail(BE_ERR_UNSUPPORTED, "head_dim %d", info->head_dim);
    }
  }
  BE_HIP_CHECK(hipGetLastError());
  return BE_OK;
}

template <typename T>
static int launch_merge(const be_attn_plan_info* info, MergeArgs& m, int count, hipStream_t st) {
  const dim3 grid(count, (info->num_qo_heads * (info->head_dim / 4) + 255) / 256);
  switch (info->head_dim) {
    case 64: merge_kernel<T, 64><<<grid, 256, 0, st>>>(m); break;
    case 128: merge_kernel<T, 128><<<grid, 256, 0, st>>>(m); break;
    case 256: merge_kernel<T, 256><<<grid, 256, 0, st>>>(m); break;
    default: return fail(BE_ERR_UNSUPPORTED, "head_dim %d", info->head_dim);
  }
  BE_HIP_CHECK(hipGetLastError());
  return BE_OK;
}

int attn_run(const be_attn_plan_info* info, const int32_t* plan, void* partials, const void* q,
             int64_t q_sn, int64_t q_sh, const void* kv, void* out, int64_t o_sn, int64_t o_sh,
             float* lse, float sm_scale, int phases, void* stream) {
  BE_REQUIRE(phases >= 1 && phases <= 3, "phases must be a non-empty subset of attention | merge");
  BE_REQUIRE(info && plan, "null plan");
  BE_REQUIRE(q && kv && out, "null q / kv / out");
  BE_REQUIRE(info->part_rows_cap == 0 || partials, "plan needs %lld bytes of partial scratch", (long long)info->partial_bytes);
  BE_REQUIRE(info->num_qo_heads % info->num_kv_heads == 0, "corrupt plan info");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const bool worklist = info->kernel < 2 || (info->kernel == 2 && info->stream_loop == kLoopBlocks);
  BE_REQUIRE(worklist || (reinterpret_cast<uintptr_t>(kv) & 15) == 0, "the cache must be 16-byte aligned");
  if (info->kernel == 2 && info->stream_loop != kLoopBlocks)
    return stream_run(info, plan, partials, q, q_sn, q_sh, kv, out, o_sn, o_sh, lse, sm_scale, phases, st);
  if (info->kernel == 3) return rows_run(info, plan, q, q_sn, q_sh, kv, out, o_sn, o_sh, lse, sm_scale, phases, st);
  const int64_t rows = info->part_rows_cap;
  AttnArgs a;
  a.q = q; a.q_sn = q_sn; a.q_sh = q_sh;
  a.kv = kv; a.out = out; a.o_sn = o_sn; a.o_sh = o_sh; a.out_lse = lse;
  a.part_o = reinterpret_cast<float*>(partials);
  a.part_lse = a.part_o + rows * info->num_qo_heads * info->head_dim;
  a.items = reinterpret_cast<const WorkItem*>(plan + info->off_items);
  a.q_index = plan + info->off_qindex;
  a.pages = plan + info->off_pages;
  a.page_size = info->page_size;
  a.hkv = info->num_kv_heads;
  a.hq = info->num_qo_heads;
  a.g = info->num_qo_heads / info->num_kv_heads;
  a.scale_log2 = sm_scale * 1.4426950408889634f;
  a.q_merge = plan + info->off_q_merge;
  a.merge_ptr = plan + info->off_merge_ptr;
  a.merge_rows = plan + info->off_merge_rows;
  a.live_items = info->static_layout ? plan + kHdrItems : nullptr;
  a.counters = (info->fused_merge && info->num_merge > 0)
                   ? reinterpret_cast<int32_t*>(reinterpret_cast<char*>(partials) + info->counter_offset)
                   : nullptr;
  int rc = BE_OK;
  if ((phases & BE_RUN_ATTENTION) && info->grid_items > 0) {
    switch (info->dtype) {
      case BE_F32: rc = launch_attn<float>(info, a, st); break;
      case BE_F16: rc = launch_attn<f16_t>(info, a, st); break;
      case BE_BF16: rc = launch_attn<bf16_t>(info, a, st); break;
      default: return fail(BE_ERR_INVALID, "dtype %d", info->dtype);
    }
    if (rc) return rc;
  }
  if (!(phases & BE_RUN_MERGE)) return rc;
  MergeArgs m;
  m.part_o = a.part_o; m.part_lse = a.part_lse;
  m.merge_rows = plan + info->off_merge_rows;
  m.out = out; m.o_sn = o_sn; m.o_sh = o_sh; m.out_lse = lse; m.hq = info->num_qo_heads;
  for (int pass = 0; pass < 2; ++pass) {
    // pass 0: split-K merge (separate-merge plans); pass 1: queries without keys
    const int count = pass == 0 ? (info->fused_merge ? 0 : info->grid_merge) : info->grid_zero;
    if (count == 0) continue;
    m.live = info->static_layout ? plan + (pass == 0 ? kHdrMerge : kHdrZero) : nullptr;
    m.merge_q = plan + (pass == 0 ? info->off_merge_q : info->off_zero_q);
    m.merge_ptr = plan + (pass == 0 ? info->off_merge_ptr : info->off_zero_ptr);
    switch (info->dtype) {
      case BE_F32: rc = launch_merge<float>(info, m, count, st); break;
      case BE_F16: rc = launch_merge<f16_t>(info, m, count, st); break;
      case BE_BF16: rc = launch_merge<bf16_t>(info, m, count, st); break;
    }
    if (rc) return rc;
  }
  return rc;
}

}  // namespace be

extern "C" {

int be_attn_plan(const be_level* levels, int num_levels, int num_queries, int num_qo_heads,
                 int num_kv_heads, int head_dim, int page_size, int num_pages, int dtype, int flags,
                 int num_cus, const be_plan_caps* caps, int32_t* host_plan, int64_t host_plan_capacity,
                 be_attn_plan_info* info) {
  return be::attn_plan(levels, num_levels, num_queries, num_qo_heads, num_kv_heads, head_dim, page_size,
                       num_pages, dtype, flags, num_cus, caps, host_plan, host_plan_capacity, info);
}

int be_attn_run(const be_attn_plan_info* info, const int32_t* dev_plan, void* partials, const void* q,
                int64_t q_stride_n, int64_t q_stride_h, const void* kv_layer, void* out, int64_t o_stride_n,
                int64_t o_stride_h, float* lse, float sm_scale, int phases, void* stream) {
  return be::attn_run(info, dev_plan, partials, q, q_stride_n, q_stride_h, kv_layer, out, o_stride_n,
                      o_stride_h, lse, sm_scale, phases, stream);
}

int be_merge_states(const float* o_a, const float* lse_a, const float* o_b, const float* lse_b, float* o_out,
                    float* lse_out, int n, int heads, int head_dim, void* stream) {
  BE_REQUIRE(o_a && lse_a && o_b && lse_b && o_out && lse_out, "null pointer");
  BE_REQUIRE(n >= 0 && heads > 0 && head_dim > 0, "bad shape");
  const int64_t rows = (int64_t)n * heads;
  const int64_t total = rows * head_dim;
  if (total == 0) return BE_OK;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  be::merge2_kernel<<<(unsigned)((rows + 3) / 4), 256, 0, st>>>(o_a, lse_a, o_b, lse_b, o_out, lse_out,
                                                              (int)rows, head_dim);
  BE_HIP_CHECK(hipGetLastError());
  return BE_OK;
}

}  // extern "C"
