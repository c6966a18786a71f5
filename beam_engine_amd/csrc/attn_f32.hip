// Paged attention on fp32 storage (gfx950): any decode or prefill plan, head_dim
// 64, 128 or 256, any page size, up to 64 query rows per KV head and item.
//
// One workgroup of four waves per (work item, KV head), the 16-bit tile kernel's
// structure (attn_tile.hip) with the contractions on v_mfma_f32_16x16x4 (fp32
// products, fp32 accumulation): Sᵀ = K Qᵀ takes its four head_dim elements of a
// step from 16-byte reads (lane (lg, lc): elements 16 s + 4 lg .. + 3 of row lc, K
// and Q alike, one MFMA per element), and Oᵀ += Vᵀ Pᵀ the token 4 lg + r of the
// scores' register r, its Vᵀ from 16-byte reads of V's rows (lane lc: columns
// 4 lc .. + 3, one MFMA per column), so neither K nor V is transposed in LDS and
// the probabilities never leave registers.
//
// What bounds it: decode, the chain of round trips of a small launch; prefill, the
// fp32 MFMA rate (a 16 x 16 x 4 product takes 32 cycles: 157 TFLOP/s).  Measured on
// MI355X against the VALU kernel, us per layer: 1 x 4 beams x 512 + 32 tokens, 8 / 8
// heads, head_dim 64, 42.2 -> 13.6; 5 x 27 beams x 2204 tokens 122.8 -> 32.6 (1.6
// TB/s); 2 x 16 x 8000, head_dim 128, 339 -> 57 (2.5 TB/s); prompts of 1000 tokens
// 146 -> 32, 2000 510 -> 67 (61 TFLOP/s).

#include <math.h>

#include "attn_tile.h"

namespace be {
namespace f32 {

using stream::lds_addr;
using stream::rfl;

// Chunks of K row r sit at c ^ swz(r): 16 consecutive rows' chunk take 16 slots.
__device__ __forceinline__ int swz(int r) { return r & 15; }

__device__ __forceinline__ v4f mfma4(float a, float b, v4f c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

template <int D, int RT, bool PAGED4>
__global__ __launch_bounds__(256, D == 64 ? 2 : 1) void attn_f32_kernel(AttnArgs a) {
  constexpr int RB = D * 4;
  using Loader = TileLoader<RB, PAGED4, swz>;
  constexpr int PLANE = Loader::PLANE, STAGE = Loader::STAGE;
  constexpr int NST = D == 256 ? 1 : 2;              // stages (128 KB each at head_dim 256)
  constexpr int KC = D / 16;                         // 16-element groups of the QK contraction
  constexpr int MB = D / 64;                         // 64-column blocks of V
  constexpr int TSPLIT = 4 / RT;                     // waves sharing a row tile (token split)
  constexpr int NSUB = RT;                           // 16-token sub-tiles per wave per tile
  constexpr int COMB_SLOT = (MB * 4 * 64 * 4 + 2 * 64) * 4;
  static_assert(TSPLIT == 1 || (TSPLIT - 1) * RT * COMB_SLOT <= NST * STAGE, "combine scratch must fit");

  __shared__ __attribute__((aligned(1024))) unsigned char stage[NST * STAGE];
  __shared__ int32_t pg_lds[kMaxPagesLds];
  if (a.live_items && (int)blockIdx.x >= *a.live_items) return;

  const WorkItem it = a.items[blockIdx.x];
  const int kvh = blockIdx.y;
  const int tid = threadIdx.x;
  const int w = rfl(tid >> 6), lane = tid & 63, lg = lane >> 4, lc = lane & 15;
  const int g = a.g, R = it.q_count * g, ps = a.page_size;

  // ---- the item's pages
  const int first_page = it.tok_begin / ps;
  const int n_pages = (it.tok_begin + it.tok_count - 1) / ps - first_page + 1;
  const int n_tiles = (it.tok_count + kTile - 1) / kTile;
  const uint32_t lds0 = lds_addr(stage);
  Loader ld;
  if constexpr (PAGED4) {
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

  // ---- Q as the B operand: lane holds Q[row][16 s + 4 lg + e]
  v4f qf[KC];
  if (row < R) {
    const float* qp = reinterpret_cast<const float*>(a.q) + (int64_t)(it.q_begin + j) * a.q_sn + (int64_t)(kvh * g + hh) * a.q_sh;
#pragma unroll
    for (int s = 0; s < KC; ++s) qf[s] = *reinterpret_cast<const v4f*>(qp + s * 16 + lg * 4);
  } else {
#pragma unroll
    for (int s = 0; s < KC; ++s) qf[s] = v4f{0.f, 0.f, 0.f, 0.f};
  }
  // Q, which left with the page ids, has landed before the tile loads go out: a
  // later first use would make the compiler wait for them too
#pragma unroll
  for (int s = 0; s < KC; ++s) asm volatile("" : "+v"(qf[s]));
  ld.load(lds0);
  if (NST > 1 && n_tiles > 1) ld.load(lds0 + STAGE);
  // item tokens this lane's row sees (causal: its query's limit)
  int lim;
  {
    const int64_t v = (int64_t)it.vis0 + j - it.tok_begin;
    lim = (int)std::min<int64_t>(it.tok_count, std::max<int64_t>(v, 0));
  }
  // rows are in query order: the row tile's last row sees the most
  const int lim_most = __builtin_amdgcn_readlane(lim, min(15, max(R - 1 - rt * 16, 0)));

  // ---- operand offsets (a 16-token sub-tile further: 16 RB)
  uint32_t koff[KC], voff[4];
#pragma unroll
  for (int s = 0; s < KC; ++s) koff[s] = lc * RB + (((4 * s + lg) ^ swz(lc)) << 4);
#pragma unroll
  for (int r = 0; r < 4; ++r) voff[r] = (4 * lg + r) * RB + ((lc ^ swz(4 * lg + r)) << 4);

  float m_run = -INFINITY, l_run = 0.f;
  v4f o_acc[MB][4];                                  // [block][e]: lane holds column 64 b + 4 (4 lg + i) + e of row lc
#pragma unroll
  for (int b = 0; b < MB; ++b)
#pragma unroll
    for (int e = 0; e < 4; ++e) o_acc[b][e] = v4f{0.f, 0.f, 0.f, 0.f};

  for (int tile = 0; tile < n_tiles; ++tile) {
    const int st = tile % NST;
    // this wave's loads of the tile have landed (the next tile's may be in
    // flight); after the barrier everyone's have
    if (NST > 1 && tile + 1 < n_tiles) {
      if constexpr (Loader::IPW == 4) asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(16) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
    const int s0 = tile * kTile + ts * NSUB * 16;      // first token of the wave's sub-tiles
    if (active && s0 < lim_most) {
      const unsigned char* kt = stage + st * STAGE + ts * NSUB * 16 * RB;
      const unsigned char* vt = kt + PLANE;
      float x[NSUB][4];
#pragma unroll
      for (int k = 0; k < NSUB; ++k) {
        v4f acc[2] = {v4f{0.f, 0.f, 0.f, 0.f}, v4f{0.f, 0.f, 0.f, 0.f}};   // two chains
#pragma unroll
        for (int s = 0; s < KC; ++s) {
          const v4f kf = *reinterpret_cast<const v4f*>(kt + k * 16 * RB + koff[s]);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[e & 1] = mfma4(kf[e], qf[s][e], acc[e & 1]);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) x[k][r] = (acc[0][r] + acc[1][r]) * a.scale_log2;
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
        const float alpha = exp2f(m_run - msafe);      // 0 while nothing was seen
        l_run *= alpha;
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
          for (int e = 0; e < 4; ++e) o_acc[b][e] *= alpha;
      }
      m_run = m_new;
#pragma unroll
      for (int k = 0; k < NSUB; ++k) {
        float p[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          p[r] = exp2f(x[k][r] - msafe);
          l_run += p[r];
        }
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const v4f vf = *reinterpret_cast<const v4f*>(vt + k * 16 * RB + b * 256 + voff[r]);
#pragma unroll
            for (int e = 0; e < 4; ++e) o_acc[b][e] = mfma4(vf[e], p[r], o_acc[b][e]);
          }
      }
    }
    if (tile + NST < n_tiles) {
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
      for (int b = 0; b < MB; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) *reinterpret_cast<v4f*>(slot + ((b * 4 + e) * 64 + lane) * 4) = o_acc[b][e];
      slot[MB * 1024 + lane] = m_run;
      slot[MB * 1024 + 64 + lane] = l_run;
    }
    __syncthreads();
    if (ts == 0 && active) {
#pragma unroll
      for (int s2 = 1; s2 < TSPLIT; ++s2) {
        const float* slot = comb + ((s2 - 1) * RT + rt) * (COMB_SLOT / 4);
        const float mb = slot[MB * 1024 + lane], lb = slot[MB * 1024 + 64 + lane];
        const float M = fmaxf(m_run, mb);
        const float ca = (M == -INFINITY) ? 0.f : exp2f(m_run - M);
        const float cb = (M == -INFINITY) ? 0.f : exp2f(mb - M);
        l_run = l_run * ca + lb * cb;
        m_run = M;
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            o_acc[b][e] = o_acc[b][e] * ca + *reinterpret_cast<const v4f*>(slot + ((b * 4 + e) * 64 + lane) * 4) * cb;
      }
    }
  }

  // ---- writes: o_acc[b][e][i] is column 64 b + 16 lg + 4 i + e
  if (ts == 0 && active && row < R) {
    const int head = kvh * g + hh;
    const float inv = (l_run > 0.f) ? 1.f / l_run : 0.f;
    float* op = it.out_row < 0 ? reinterpret_cast<float*>(a.out) + (int64_t)(it.q_begin + j) * a.o_sn + (int64_t)head * a.o_sh
                               : a.part_o + ((int64_t)(it.out_row + j) * a.hq + head) * D;
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<v4f*>(op + b * 64 + lg * 16 + i * 4) =
            v4f{o_acc[b][0][i] * inv, o_acc[b][1][i] * inv, o_acc[b][2][i] * inv, o_acc[b][3][i] * inv};
    if (lg == 0) store_row_lse<float>(a, it, j, head, m_run, l_run);
  }
  __shared__ int s_last[64];
  if (it.out_row >= 0 && a.counters) fused_merge_epilogue<float, D>(a, it, kvh, s_last);
}

template <int D>
static int launch(const be_attn_plan_info* info, const AttnArgs& a, hipStream_t st) {
  const dim3 grid(info->grid_items, info->num_kv_heads);
  const bool p4 = paged4(info->page_size, D * 4);
#define BE_F32_LAUNCH(RT)                                                \
  if (p4) attn_f32_kernel<D, RT, true><<<grid, 256, 0, st>>>(a);          \
  else attn_f32_kernel<D, RT, false><<<grid, 256, 0, st>>>(a);
  switch (info->tile_rows) {
    case 16: BE_F32_LAUNCH(1) break;
    case 32: BE_F32_LAUNCH(2) break;
    case 64: BE_F32_LAUNCH(4) break;
    default: return fail(BE_ERR_INVALID, "corrupt plan: tile_rows %d on fp32", info->tile_rows);
  }
#undef BE_F32_LAUNCH
  BE_HIP_CHECK(hipGetLastError());
  return BE_OK;
}

}  // namespace f32

int f32_launch(const be_attn_plan_info* info, const AttnArgs& a, hipStream_t st) {
  switch (info->head_dim) {
    case 64: return f32::launch<64>(info, a, st);
    case 128: return f32::launch<128>(info, a, st);
    case 256: return f32::launch<256>(info, a, st);
    default: return fail(BE_ERR_UNSUPPORTED, "head_dim %d", info->head_dim);
  }
}

}  // namespace be
