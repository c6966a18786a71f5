// Paged attention for up to 64 query rows per KV head (gfx950): decode groups and
// short query blocks of plans the streaming kernel does not take.  16-bit storage,
// head_dim 64, 128 or 256, any page size.
//
// One workgroup of four waves per (work item, KV head): RT 16-row tiles of the
// item's rows (queries x GQA group) over its tokens in 64-token tiles.  With
// RT <= 2 row tiles the four waves also split a tile's tokens (4 / RT ways) and
// are combined through LDS at the end; with RT = 4 every wave sees all tokens of
// its row tile, so K and V are read once per workgroup.
//
// Scores: Sᵀ = K Qᵀ with v_mfma_f32_16x16x32 (A = 8 consecutive head_dim elements
// of a token row, B = Q from registers).  The C layout of a 16-token Sᵀ tile
// (lane (lg, lc): tokens 4 lg .. + 3 of row lc) is the B operand of Oᵀ += Vᵀ Pᵀ:
// two token sub-tiles to a v_mfma_f32_16x16x32, or one to a 16x16x16; Vᵀ is read
// from row-major V with ds_read_b64_tr_b16.
//
// What bounds it: latency.  An item of a decode plan is two tiles or so, and the
// launch is a chain of round trips: item, page ids, K / V, result.  K and V go
// global -> LDS directly with two tiles in flight from the start (no registers
// held, no LDS stores), the first page ids come straight from memory, and a
// tile's operand reads are issued ahead of its MFMAs.  Measured on MI355X (rocprof,
// per launch) against K / V staged through registers with V transposed by 2-byte
// LDS stores: 8 beams x 344 + 24 tokens, 32 / 8 heads, fp16, page 8, 9.2 -> 7.0 us;
// 4 x 8 beams x 2048 + 128 tokens, head_dim 64, 11.9 -> 10.0 us (2.1 TB/s).

#include <math.h>

#include "attn_tile.h"

namespace be {
namespace tile {

using stream::lds_addr;
using stream::lds_v4s_t;
using stream::pack4;
using stream::rfl;

// The value XORed into the 16-byte chunk index of K / V row r in LDS: eight
// consecutive rows (a half wave's transposed V read: 8 rows x 2 chunks) take
// eight chunk pairs, and 16 consecutive rows' chunk (a K read's quarter wave)
// 16 slots.
template <int D>
__device__ __forceinline__ int swz(int r) {
  return D >= 128 ? ((r & 7) << 1 | ((r >> 3) & 1)) : (((r >> 1) & 3) << 1 | ((r >> 3) & 1));
}

template <typename T, int D, int RT, bool PAGED4>
__global__ __launch_bounds__(256, D == 64 ? 4 : D == 128 ? 2 : 1) void attn_tile_kernel(AttnArgs a) {
  constexpr int RB = D * 2;                          // bytes of a K or V row
  using Loader = TileLoader<RB, PAGED4, swz<D>>;
  constexpr int PLANE = Loader::PLANE, STAGE = Loader::STAGE;
  constexpr int KS = D / 32;                         // QK contraction steps
  constexpr int MT = D / 16;                         // Oᵀ head_dim tiles
  constexpr int TSPLIT = 4 / RT;                     // waves sharing a row tile (token split)
  constexpr int NSUB = RT;                           // 16-token sub-tiles per wave per tile
  constexpr int COMB_SLOT = (MT * 64 * 4 + 2 * 64) * 4;   // bytes: Oᵀ frags + m + l of one wave
  static_assert(TSPLIT == 1 || (TSPLIT - 1) * RT * COMB_SLOT <= 2 * STAGE, "combine scratch must fit");

  __shared__ __attribute__((aligned(1024))) unsigned char stage[2 * STAGE];
  __shared__ int32_t pg_lds[kMaxPagesLds];
  if (a.live_items && (int)blockIdx.x >= *a.live_items) return;

  const WorkItem it = a.items[blockIdx.x];
  const int kvh = blockIdx.y;
  const int tid = threadIdx.x;
  const int w = rfl(tid >> 6), lane = tid & 63, lg = lane >> 4, lc = lane & 15;
  const int g = a.g, R = it.q_count * g, ps = a.page_size;

  // ---- the item's pages; the first two tiles' loads
  const int first_page = it.tok_begin / ps;
  const int n_pages = (it.tok_begin + it.tok_count - 1) / ps - first_page + 1;
  const int n_tiles = (it.tok_count + kTile - 1) / kTile;
  const uint32_t lds0 = lds_addr(stage);
  Loader ld;
  if constexpr (PAGED4) {
    // (a window of 64 ids covers the first two tiles; later ones come from LDS)
    ld.init(a, it, kvh, w, pg_lds, first_page, n_pages);
    for (int i = 64 + tid; i < n_pages; i += 256) pg_lds[i] = a.pages[it.page_begin + first_page + i];
    if (tid < min(n_pages, 64)) pg_lds[tid] = ld.pg_reg;   // wave 0 holds them
  } else {
    for (int i = tid; i < n_pages; i += 256) pg_lds[i] = a.pages[it.page_begin + first_page + i];
    __syncthreads();
    ld.init(a, it, kvh, w, pg_lds, first_page, n_pages);
  }

  // ---- wave role
  const int rt = w % RT, ts = w / RT;
  const bool active = rt * 16 < R;
  const int row = rt * 16 + lc;
  // row / g for row < 256 (the quotient's distance from an integer is at least 1 / (2 g))
  const int j = (int)(((float)row + 0.5f) * (1.f / (float)g)), hh = row - j * g;

  // ---- Q as the B operand: lane holds Q[row][32 ks + 8 lg .. + 7]
  v8s qf[KS];
  if (row < R) {
    const T* qp = reinterpret_cast<const T*>(a.q) + (int64_t)(it.q_begin + j) * a.q_sn + (int64_t)(kvh * g + hh) * a.q_sh;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = *reinterpret_cast<const v8s*>(qp + ks * 32 + lg * 8);
  } else {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = v8s{0, 0, 0, 0, 0, 0, 0, 0};
  }
  // Q, which left with the page ids, has landed before the tile loads go out: a
  // later first use would make the compiler wait for them too
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(qf[ks]));
  ld.load(lds0);
  if (n_tiles > 1) ld.load(lds0 + STAGE);
  // item tokens this lane's row sees (causal: its query's limit)
  int lim;
  {
    const int64_t v = (int64_t)it.vis0 + j - it.tok_begin;
    lim = (int)std::min<int64_t>(it.tok_count, std::max<int64_t>(v, 0));
  }
  // ---- operand offsets (rows 16 sub + .. add 16 sub RB: swz repeats every 16 rows)
  uint32_t koff[KS], voff[MT];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) koff[ks] = lc * RB + (((4 * ks + lg) ^ swz<D>(lc)) << 4);
  const int vr = 4 * lg + (lc >> 2);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) voff[mt] = vr * RB + (((2 * mt + ((lc & 3) >> 1)) ^ swz<D>(vr)) << 4) + (lc & 1) * 8;

  float m_run = -INFINITY, l_run = 0.f;
  v4f o_acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) o_acc[mt] = v4f{0.f, 0.f, 0.f, 0.f};

  for (int tile = 0; tile < n_tiles; ++tile) {
    const int st = tile & 1;
    // this wave's loads of the tile have landed (the next tile's may be in
    // flight); after the barrier everyone's have
    if (tile + 1 < n_tiles) {
      if constexpr (Loader::IPW == 2) asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      else if constexpr (Loader::IPW == 4) asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(16) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
    const int s0 = tile * kTile + ts * NSUB * 16;      // first token of the wave's sub-tiles
    if (active && s0 < it.tok_count) {
      const unsigned char* kt = stage + st * STAGE + ts * NSUB * 16 * RB;
      const unsigned char* vt = kt + PLANE;
      float x[NSUB][4];
#pragma unroll
      for (int k = 0; k < NSUB; ++k) {
        v8s kf[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) kf[ks] = *reinterpret_cast<const v8s*>(kt + k * 16 * RB + koff[ks]);
        v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) acc = mfma_qk<T>(kf[ks], qf[ks], acc);
#pragma unroll
        for (int r = 0; r < 4; ++r) x[k][r] = acc[r] * a.scale_log2;
      }
      if (__builtin_amdgcn_ballot_w64(lim < s0 + NSUB * 16) != 0) {
        const int left = lim - s0 - 4 * lg;
#pragma unroll
        for (int k = 0; k < NSUB; ++k)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (k * 16 + r >= left) x[k][r] = -INFINITY;
      }
      float mx = -INFINITY;
#pragma unroll
      for (int k = 0; k < NSUB; ++k)
#pragma unroll
        for (int r = 0; r < 4; ++r) mx = fmaxf(mx, x[k][r]);
      mx = rows4_max(mx);
      const float m_new = fmaxf(m_run, mx);
      const float msafe = (m_new == -INFINITY) ? 0.f : m_new;
      if (__builtin_amdgcn_ballot_w64(m_new > m_run) != 0) {
        const float alpha = __builtin_amdgcn_exp2f(m_run - msafe);    // 0 while nothing was seen
        l_run *= alpha;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) o_acc[mt] *= alpha;
      }
      m_run = m_new;
      v4s pf[NSUB];
#pragma unroll
      for (int k = 0; k < NSUB; ++k) {
        float p[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          p[r] = __builtin_amdgcn_exp2f(x[k][r] - msafe);
          l_run += p[r];
        }
        pf[k] = pack4<T>(p[0], p[1], p[2], p[3]);
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        if constexpr (NSUB == 1) {
          o_acc[mt] = mfma_pv<T>(__builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t)(vt + voff[mt])), pf[0], o_acc[mt]);
        } else {
#pragma unroll
          for (int k = 0; k < NSUB; k += 2) {
            const v4s v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t)(vt + k * 16 * RB + voff[mt]));
            const v4s v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t)(vt + (k + 1) * 16 * RB + voff[mt]));
            o_acc[mt] = mfma_qk<T>(__builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7),
                                   __builtin_shufflevector(pf[k], pf[k + 1], 0, 1, 2, 3, 4, 5, 6, 7), o_acc[mt]);
          }
        }
      }
    }
    if (tile + 2 < n_tiles) {
      // everyone is done with this stage
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      ld.load(lds0 + st * STAGE);
    }
  }
  l_run = rows4_sum(l_run);

  // ---- token-split waves (ts > 0) hand their state to the ts == 0 wave of the row tile
  if constexpr (TSPLIT > 1) {
    float* comb = reinterpret_cast<float*>(stage);
    __syncthreads();                                   // tiles no longer needed
    if (ts > 0 && active) {
      float* slot = comb + ((ts - 1) * RT + rt) * (COMB_SLOT / 4);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) *reinterpret_cast<v4f*>(slot + (mt * 64 + lane) * 4) = o_acc[mt];
      slot[MT * 256 + lane] = m_run;
      slot[MT * 256 + 64 + lane] = l_run;
    }
    __syncthreads();
    if (ts == 0 && active) {
#pragma unroll
      for (int s2 = 1; s2 < TSPLIT; ++s2) {
        const float* slot = comb + ((s2 - 1) * RT + rt) * (COMB_SLOT / 4);
        const float mb = slot[MT * 256 + lane], lb = slot[MT * 256 + 64 + lane];
        const float M = fmaxf(m_run, mb);
        const float ca = (M == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(m_run - M);
        const float cb = (M == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(mb - M);
        l_run = l_run * ca + lb * cb;
        m_run = M;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          o_acc[mt] = o_acc[mt] * ca + *reinterpret_cast<const v4f*>(slot + (mt * 64 + lane) * 4) * cb;
      }
    }
  }

  // ---- writes: lane holds Oᵀ[16 mt + 4 lg + i][row]
  if (ts == 0 && active && row < R) {
    const int head = kvh * g + hh;
    const float inv = (l_run > 0.f) ? 1.f / l_run : 0.f;
    if (it.out_row < 0) {
      T* op = reinterpret_cast<T*>(a.out) + (int64_t)(it.q_begin + j) * a.o_sn + (int64_t)head * a.o_sh;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        *reinterpret_cast<v4s*>(op + mt * 16 + 4 * lg) =
            pack4<T>(o_acc[mt][0] * inv, o_acc[mt][1] * inv, o_acc[mt][2] * inv, o_acc[mt][3] * inv);
    } else {
      float* op = a.part_o + ((int64_t)(it.out_row + j) * a.hq + head) * D;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) *reinterpret_cast<v4f*>(op + mt * 16 + 4 * lg) = o_acc[mt] * inv;
    }
    if (lg == 0) store_row_lse<T>(a, it, j, head, m_run, l_run);
  }
  __shared__ int s_last[64];
  if (it.out_row >= 0 && a.counters) fused_merge_epilogue<T, D>(a, it, kvh, s_last);
}

template <typename T, int D>
static int launch(const be_attn_plan_info* info, const AttnArgs& a, hipStream_t st) {
  const dim3 grid(info->grid_items, info->num_kv_heads);
  const bool p4 = paged4(info->page_size, D * 2);
#define BE_TILE_LAUNCH(RT)                                                     \
  if (p4) attn_tile_kernel<T, D, RT, true><<<grid, 256, 0, st>>>(a);            \
  else attn_tile_kernel<T, D, RT, false><<<grid, 256, 0, st>>>(a);
  switch (info->tile_rows) {
    case 16: BE_TILE_LAUNCH(1) break;
    case 32: BE_TILE_LAUNCH(2) break;
    case 64: BE_TILE_LAUNCH(4) break;
    case 128: return fail(BE_ERR_UNSUPPORTED, "128-row tiles at head_dim %d", D);
    default: return fail(BE_ERR_INVALID, "corrupt plan: tile_rows %d at head_dim %d", info->tile_rows, D);
  }
#undef BE_TILE_LAUNCH
  BE_HIP_CHECK(hipGetLastError());
  return BE_OK;
}

template <typename T>
static int launch_d(const be_attn_plan_info* info, const AttnArgs& a, hipStream_t st) {
  switch (info->head_dim) {
    case 64: return launch<T, 64>(info, a, st);
    case 128: return launch<T, 128>(info, a, st);
    case 256: return launch<T, 256>(info, a, st);
    default: return fail(BE_ERR_UNSUPPORTED, "head_dim %d", info->head_dim);
  }
}

}  // namespace tile

int tile_launch(const be_attn_plan_info* info, const AttnArgs& a, hipStream_t st) {
  return info->dtype == BE_BF16 ? tile::launch_d<bf16_t>(info, a, st) : tile::launch_d<f16_t>(info, a, st);
}

}  // namespace be
