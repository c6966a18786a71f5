// Paged attention for many query rows per KV head (gfx950): prefill and large
// shared groups.  16-bit storage, head_dim 64 or 128, any page size.
//
// One workgroup of four waves per (work item, KV head): up to 128 query rows
// (queries x GQA group), 32 per wave, over the item's tokens in 64-token tiles.
// Each wave's tile step is Sᵀ = K Qᵀ and Oᵀ += Vᵀ Pᵀ with
// v_mfma_f32_32x32x16: Q stays in registers as the B operand, and the C layout
// of Sᵀ (lane l: row l % 32, tokens 8 (i / 4) + 4 (l / 32) + i % 4) is, eight
// registers at a time, the B operand of the second product over a permuted token
// order that the Vᵀ reads follow, so P never leaves registers.
//
// K and V rows go global -> LDS directly (global_load_lds_dwordx4), two stages
// deep: the next tile's loads are in flight during a whole tile step and one
// barrier per tile both publishes a stage and frees the other.  Rows keep their
// 16-byte chunks XOR-swizzled by row (chosen by each lane's global address); V
// stays row-major and is read transposed with ds_read_b64_tr_b16.  Every operand
// read of a tile is issued ahead of its use: K before the first MFMA, V before
// the softmax.
//
// What bounds it: per wave and tile (head_dim 128) 32 MFMAs of 32 cycles, about
// 180 VALU instructions (32 of them quarter-rate exponentials) and 32 KB of LDS
// operand reads, in waves of which only two fit a SIMD (about 242 VGPRs), so
// they overlap in part: 2.1 us per tile for a CU's two workgroups, 38% MFMA and
// 50% VALU busy; a workgroup's prologue and epilogue (about 6 us beside another
// workgroup's tiles) weigh on short prompts.  Measured on MI355X, us per layer,
// 32 / 8 heads, head_dim 128: 8 x 1024 tokens 250 (275 TFLOP/s, the streaming
// kernel's 64-row tiles) -> 92 to 99 (695 to 748), 4 x 2048 436 -> 157 to 167 (823
// to 876); page 8 fp16, three ragged prompts of up to 1500 tokens after up to 400
// cached 292 (the 16-row-tile kernel, V transposed by 2-byte LDS stores) -> 64.

#include <math.h>

#include <type_traits>

#include "attn_tile.h"

namespace be {
namespace block {

using stream::lds_addr;
using stream::lds_v4s_t;
using stream::pack2;
using stream::rfl;

constexpr int kRows = 128;            // query rows per workgroup
constexpr int kWaveRows = 32;
typedef float v16f __attribute__((ext_vector_type(16)));

template <typename T> __device__ __forceinline__ v16f mfma32(v8s a, v8s b, v16f c);
template <> __device__ __forceinline__ v16f mfma32<bf16_t>(v8s a, v8s b, v16f c) {
  typedef __bf16 v8b __attribute__((ext_vector_type(8)));
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8b, a), __builtin_bit_cast(v8b, b), c, 0, 0, 0);
}
template <> __device__ __forceinline__ v16f mfma32<f16_t>(v8s a, v8s b, v16f c) {
  typedef _Float16 v8h __attribute__((ext_vector_type(8)));
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0, 0);
}

// The value XORed into the 16-byte chunk index of K / V row r in LDS: the row's
// low two bits select the chunk quad, so that the four rows x four chunks a
// half wave reads with ds_read_b64_tr_b16, and any 16 consecutive rows' chunk
// read with ds_read_b128, fall on all 64 banks.  (Plain r & 15 put two of the
// transposed read's four rows on the same banks: 14 M conflict cycles per launch
// against 0.8 M, 8 x 1024-token prompts, 109 -> 103 us.)
template <int D>
__device__ __forceinline__ int swz(int r) {
  return D == 128 ? ((r & 3) << 2 | ((r >> 2) & 3)) : (((r >> 1) & 1) << 2 | ((r >> 2) & 3));
}

// The other 32-lane half's value of the same row.
__device__ __forceinline__ float other_half_max(float x) {
  typedef unsigned int u2 __attribute__((ext_vector_type(2)));
  const unsigned xb = __float_as_uint(x);
  const u2 r = __builtin_amdgcn_permlane32_swap(xb, xb, false, false);
  const unsigned a = r.x, b = r.y;
  return fmaxf(__uint_as_float(a), __uint_as_float(b));
}
__device__ __forceinline__ float other_half_sum(float x) {
  typedef unsigned int u2 __attribute__((ext_vector_type(2)));
  const unsigned xb = __float_as_uint(x);
  const u2 r = __builtin_amdgcn_permlane32_swap(xb, xb, false, false);
  const unsigned a = r.x, b = r.y;
  return __uint_as_float(a) + __uint_as_float(b);
}

template <typename T, int D, bool PAGED4>
__global__ __launch_bounds__(256, 2) void attn_block_kernel(AttnArgs a, int n_items) {
  constexpr int KS = D / 16;                         // QK contraction steps
  constexpr int MB = D / 32;                         // Oᵀ head_dim blocks
  constexpr int RB = D * 2;                          // bytes of a K or V row
  using Loader = TileLoader<RB, PAGED4, swz<D>>;
  constexpr int CPR = Loader::CPR, RPI = Loader::RPI, PLANE = Loader::PLANE, STAGE = Loader::STAGE;

  __shared__ __attribute__((aligned(1024))) unsigned char stage[2 * STAGE];
  __shared__ int32_t pg_lds[kMaxPagesLds];
  // consecutive workgroups are the KV heads of one item: with 8 (or a divisor)
  // heads an XCD keeps the same heads' K and V in its L2
  const int item = (int)blockIdx.x / a.hkv, kvh = (int)blockIdx.x - item * a.hkv;
  if (a.live_items && item >= *a.live_items) return;
  if (item >= n_items) return;

  const WorkItem it = a.items[item];
  const int tid = threadIdx.x;
  const int w = rfl(tid >> 6), lane = tid & 63, h = lane >> 5, lr = lane & 31;
  const int g = a.g, R = it.q_count * g, ps = a.page_size;

  // ---- the item's pages
  const int first_page = it.tok_begin / ps;
  const int n_pages = (it.tok_begin + it.tok_count - 1) / ps - first_page + 1;
  for (int i = tid; i < n_pages; i += 256) pg_lds[i] = a.pages[it.page_begin + first_page + i];

  // ---- this wave's rows: lane's row, the tokens it sees, the wave's most
  const int row = w * kWaveRows + lr;
  const bool wave_on = w * kWaveRows < R;
  // row / g for row < 256 (the quotient's distance from an integer is at least 1 / (2 g))
  const float inv_g = 1.f / (float)g;
  auto query_of = [&](int r) { return (int)(((float)r + 0.5f) * inv_g); };
  int lim;
  {
    const int64_t v = (int64_t)it.vis0 + query_of(min(row, R - 1)) - it.tok_begin;
    lim = (int)std::min<int64_t>(it.tok_count, std::max<int64_t>(v, 0));
  }
  // rows are in query order, so the wave's last row sees the most
  const int lim_most = __builtin_amdgcn_readlane(lim, 31);

  // ---- Q as the B operand: lane holds Q[row][16 ks + 8 h .. +7].  The softmax
  // takes the max of unscaled scores, so the scale must be positive: a negative
  // one moves its sign into Q, a zero one zeroes Q.
  const float scale = a.scale_log2 == 0.f ? 1.f : fabsf(a.scale_log2);
  v8s qf[KS];
  if (row < R) {
    const int j = query_of(row), hh = row - j * g;
    const T* qp = reinterpret_cast<const T*>(a.q) + (int64_t)(it.q_begin + j) * a.q_sn + (int64_t)(kvh * g + hh) * a.q_sh;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = *reinterpret_cast<const v8s*>(qp + ks * 16 + h * 8);
    if (a.scale_log2 <= 0.f) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) qf[ks] = a.scale_log2 == 0.f ? (v8s)(short)0 : qf[ks] ^ (v8s)(short)0x8000;
    }
  } else {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = v8s{0, 0, 0, 0, 0, 0, 0, 0};
  }
  if constexpr (!PAGED4) __syncthreads();            // page ids staged (else by the first tile's barrier)
  Loader ld;
  ld.init(a, it, kvh, w, pg_lds, first_page, n_pages);
  const uint32_t lds0 = lds_addr(stage);
  ld.load(lds0);
  // Q has landed before the loop: the compiler would otherwise wait for it, and
  // with it for the tile loads issued since, in every iteration
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(qf[ks]));

  // ---- operand offsets
  const int r16 = lane & 15, q4 = r16 >> 2, e4 = ((lane >> 4) & 1) * 2 + ((r16 & 3) >> 1);
  uint32_t koff[KS], voff[MB][2];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) koff[ks] = lr * RB + (((2 * ks + h) ^ swz<D>(lr)) << 4);
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int vr = 8 * u + 4 * h + q4;             // the row's low four bits
      voff[mb][u] = vr * RB + (((mb * 4 + e4) ^ swz<D>(vr)) << 4) + (r16 & 1) * 8;
    }

  float m_run = -INFINITY, m_top = -INFINITY, l_run = 0.f;   // reference of the sums, the largest score, the weights' sum
  v16f o_acc[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int i = 0; i < 16; ++i) o_acc[mb][i] = 0.f;

  const int n_tiles = (it.tok_count + kTile - 1) / kTile;
  auto step = [&](auto one, int tile) {
    constexpr bool ONE = decltype(one)::value;       // the item's only tile
    const int st = tile & 1;
    // this wave's loads of the tile have landed; after the barrier everyone's
    // have, and everyone is done with the other stage
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (!ONE && tile + 1 < n_tiles) ld.load(lds0 + (st ^ 1) * STAGE);
    const int t0 = tile * kTile;
    if (!wave_on || t0 >= lim_most) return;
    const unsigned char* kt = stage + st * STAGE;
    const unsigned char* vt = kt + PLANE;

    // Sᵀ of both 32-token blocks, every K fragment read ahead of the MFMAs
    v8s kf[2][KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int tb = 0; tb < 2; ++tb) kf[tb][ks] = *reinterpret_cast<const v8s*>(kt + tb * 32 * RB + koff[ks]);
    __builtin_amdgcn_sched_barrier(0);
    v16f x[2];
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
#pragma unroll
      for (int i = 0; i < 16; ++i) x[tb][i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int tb = 0; tb < 2; ++tb) x[tb] = mfma32<T>(kf[tb][ks], qf[ks], x[tb]);
    // the Vᵀ fragments: their reads run under the softmax
    v4s vf[4][MB][2];
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int u = 0; u < 2; ++u)
          vf[s][mb][u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t)(vt + s * 16 * RB + voff[mb][u]));
    __builtin_amdgcn_sched_barrier(0);
    if (__builtin_amdgcn_ballot_w64(lim < t0 + kTile) != 0) {
      const int left = lim - t0 - 4 * h;
#pragma unroll
      for (int tb = 0; tb < 2; ++tb)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (tb * 32 + 8 * (i >> 2) + (i & 3) >= left) x[tb][i] = -INFINITY;
    }
    // (maximum rather than fmax: no canonicalising of the MFMA results; a NaN
    // score makes the row NaN either way)
    float mx[2] = {-INFINITY, -INFINITY};
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
#pragma unroll
      for (int i = 0; i < 16; i += 2)
        mx[tb] = __builtin_elementwise_maximum(__builtin_elementwise_maximum(x[tb][i], x[tb][i + 1]), mx[tb]);
    // When a row's largest score (m_top) grows, every row of the wave takes the
    // tile's largest as its reference -- in an item's only tile each 32-token
    // block's -- so that this weight is exactly 1 in the 16-bit P, unless it lies
    // 2^8 below m_top: weights, l and Oᵀ stay within 2^8 of their scale at m_top.
    // With m_top itself as the reference only the row's largest weight is exact,
    // where the streaming kernel, which splits the tokens over two waves, has two:
    // bf16 prompts were 2.00e-3 from the 64-bit result against 1.98e-3 (8 x 1024
    // tokens; 1.96e-3 now) and 1.84e-3 against 1.83e-3 (8 x 64; 1.83e-3 now).  It
    // costs 0 to 2% of the launch (8 x 1024 tokens 91.4 -> 91.7 us, 512 35.9 -> 36.6).
    auto refer = [&](float top) {
      top = other_half_max(top) * scale;
      if (__builtin_amdgcn_ballot_w64(top > m_top) != 0) {
        m_top = fmaxf(m_top, top);
        const float m_new = top >= m_top - 8.f ? top : m_run;
        const float alpha = __builtin_amdgcn_exp2f(m_run - (m_new == -INFINITY ? 0.f : m_new));
        l_run *= alpha;
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) o_acc[mb] *= alpha;
        m_run = m_new;
      }
    };
    constexpr int NB = ONE ? 1 : 2;                  // 32-token blocks per reference
#pragma unroll
    for (int b = 0; b < 2; b += NB) {
      refer(ONE ? mx[b] : __builtin_elementwise_maximum(mx[0], mx[1]));
      const float msafe = m_run == -INFINITY ? 0.f : m_run;
      v8s pf[2 * NB];
#pragma unroll
      for (int s = 0; s < 2 * NB; ++s) {
        const int tb = b + (s >> 1);
        uint32_t pw[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float p0 = __builtin_amdgcn_exp2f(fmaf(x[tb][8 * (s & 1) + 2 * j], scale, -msafe));
          const float p1 = __builtin_amdgcn_exp2f(fmaf(x[tb][8 * (s & 1) + 2 * j + 1], scale, -msafe));
          l_run += p0 + p1;
          pw[j] = pack2<T>(p0, p1);
        }
        typedef uint32_t u4 __attribute__((ext_vector_type(4)));
        pf[s] = __builtin_bit_cast(v8s, (u4){pw[0], pw[1], pw[2], pw[3]});
      }
#pragma unroll
      for (int s = 0; s < 2 * NB; ++s)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
          const v4s *v = vf[2 * b + s][mb];
          o_acc[mb] = mfma32<T>(__builtin_shufflevector(v[0], v[1], 0, 1, 2, 3, 4, 5, 6, 7), pf[s], o_acc[mb]);
        }
    }
  };
  if (n_tiles == 1) {
    step(std::true_type(), 0);
  } else {
    for (int tile = 0; tile < n_tiles; ++tile) step(std::false_type(), tile);
  }

  // ---- writes: lane holds Oᵀ[32 mb + 8 (i / 4) + 4 h + i % 4][row]
  l_run = other_half_sum(l_run);
  const float inv = l_run > 0.f ? 1.f / l_run : 0.f;
  const int j = query_of(row), hh = row - j * g, head = kvh * g + hh;
  if (it.out_row < 0) {
    // through LDS (the wave's own 32 rows, chunks swizzled by row), so that the
    // stores are whole rows, 16 bytes a lane
    __syncthreads();                                 // every wave is done with the stages
    unsigned char* ol = stage + w * kWaveRows * RB;
    typedef uint32_t u2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const u2 pk = {pack2<T>(o_acc[mb][4 * b] * inv, o_acc[mb][4 * b + 1] * inv),
                       pack2<T>(o_acc[mb][4 * b + 2] * inv, o_acc[mb][4 * b + 3] * inv)};
        *reinterpret_cast<u2*>(ol + lr * RB + (((mb * 4 + b) ^ swz<D>(lr)) << 4) + 8 * h) = pk;
      }
    // (a wave reads only what it wrote: the compiler's lgkmcnt waits order it)
#pragma unroll
    for (int i = 0; i < kWaveRows / RPI; ++i) {
      const int lrow = i * RPI + lane / CPR, orow = w * kWaveRows + lrow;
      const uint4 v = *reinterpret_cast<const uint4*>(ol + lrow * RB + (((lane % CPR) ^ swz<D>(lrow)) << 4));
      if (orow < R) {
        const int oj = query_of(orow), oh = kvh * g + (orow - oj * g);
        T* op = reinterpret_cast<T*>(a.out) + (int64_t)(it.q_begin + oj) * a.o_sn + (int64_t)oh * a.o_sh;
        *reinterpret_cast<uint4*>(op + (lane % CPR) * 8) = v;
      }
    }
  } else if (row < R) {
    float* op = a.part_o + ((int64_t)(it.out_row + j) * a.hq + head) * D;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const v4f v = {o_acc[mb][4 * b] * inv, o_acc[mb][4 * b + 1] * inv, o_acc[mb][4 * b + 2] * inv,
                       o_acc[mb][4 * b + 3] * inv};
        *reinterpret_cast<v4f*>(op + mb * 32 + 8 * b + 4 * h) = v;
      }
  }
  if (row < R && h == 0) store_row_lse<T>(a, it, j, head, m_run, l_run);
  __shared__ int s_last[kRows];
  if (it.out_row >= 0 && a.counters) fused_merge_epilogue<T, D>(a, it, kvh, s_last);
}

}  // namespace block

bool block_eligible(int dtype, int head_dim) {
  return (dtype == BE_BF16 || dtype == BE_F16) && (head_dim == 64 || head_dim == 128);
}

int block_launch(const be_attn_plan_info* info, const AttnArgs& a, hipStream_t st) {
  const int n = info->grid_items;
  const unsigned blocks = (unsigned)n * (unsigned)info->num_kv_heads;
  const bool p4 = paged4(info->page_size, info->head_dim * 2);
#define BE_BLOCK_LAUNCH(TY, DD)                                                        \
  if (p4) block::attn_block_kernel<TY, DD, true><<<blocks, 256, 0, st>>>(a, n);         \
  else block::attn_block_kernel<TY, DD, false><<<blocks, 256, 0, st>>>(a, n);
  if (info->dtype == BE_BF16) {
    if (info->head_dim == 64) { BE_BLOCK_LAUNCH(bf16_t, 64) }
    else { BE_BLOCK_LAUNCH(bf16_t, 128) }
  } else {
    if (info->head_dim == 64) { BE_BLOCK_LAUNCH(f16_t, 64) }
    else { BE_BLOCK_LAUNCH(f16_t, 128) }
  }
#undef BE_BLOCK_LAUNCH
  BE_HIP_CHECK(hipGetLastError());
  return BE_OK;
}

}  // namespace be
