"""128-row block attention (prefill and large groups) on the GPU against the
float64 oracle, at the edges of its query blocks, token tiles, load groups and
page windows.  Tolerances are the attention tests' own (16-bit storage: 2e-2
relative, 1e-2 absolute, against the oracle on the same rounded inputs)."""

import math

import numpy as np
import pytest
import torch

from oracle import attention as oa
from tests.test_gpu_prefill import TOL, _check, _levels

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ws():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return torch.empty(256 << 20, dtype=torch.uint8, device="cuda")


def _run(ws, dtype, q_lens, kv_lens, hq, hkv, d, page, causal=True, sm_scale=None, shuffle=3, cus=None, kernel=None):
    from beam_engine_amd import BatchPrefillWithPagedKVCacheWrapper
    (qo, kvp, kvi, lpl), pages = _levels(q_lens, kv_lens, page)
    g = torch.Generator().manual_seed(shuffle)
    kvi = torch.randperm(pages, generator=g).tolist()
    kv = torch.randn((pages, 2, page, hkv, d), generator=g).to(dtype)
    q = torch.randn((qo[-1], hq, d), generator=g).to(dtype)
    w = BatchPrefillWithPagedKVCacheWrapper(ws)
    w._num_cus = cus
    w.plan(qo, kvp, kvi, lpl, hq, hkv, d, page, causal=causal, sm_scale=sm_scale, q_data_type=dtype)
    assert kernel is None or w.stats.launches[0] == kernel
    out, lse = w.run(q.cuda(), kv.cuda(), return_lse=True)
    torch.cuda.synchronize()
    ref_o, ref_lse = oa.cascade_attention(q, kv, [qo], [kvp], [kvi], [lpl], page, sm_scale, causal=causal)
    _check(out, lse, ref_o, ref_lse, dtype)
    return w


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("page", [1, 3, 4, 8, 12, 16, 64, 100])
@pytest.mark.parametrize("d", [64, 128])
def test_pages_and_head_dims(ws, dtype, page, d):
    """Page sizes that hold whole load groups (4 rows at head_dim 128, 8 at 64)
    and ones that do not, prompts around the 32-query block and 64-token tile,
    with cached tokens before them (longer ones where the streaming kernel, which
    takes head_dim 128 on pages of 16, would run few blocks)."""
    print(f"[case] block page {page} d {d} {dtype}", flush=True)
    if d == 128 and page % 16 == 0:
        q_lens, kv_lens = [65, 290, 128], [65, 361, 129]
    else:
        q_lens, kv_lens = [33, 129, 64], [33, 200, 65]
    _run(ws, dtype, q_lens, kv_lens, 16, 4, d, page, kernel="attn_block_kernel")


@pytest.mark.parametrize("hq,hkv", [(8, 8), (12, 4), (40, 8), (64, 2), (48, 1), (128, 1)])
def test_group_sizes(ws, hq, hkv):
    """GQA groups that divide the 128-row block and ones that leave rows unused."""
    print(f"[case] block group {hq}/{hkv}", flush=True)
    n = 140 if hq // hkv < 32 else 12
    _run(ws, torch.bfloat16, [n], [n + 77], hq, hkv, 64, 16, kernel="attn_block_kernel")


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("scale", [0.3, -0.2, 0.0])
def test_scales_and_unmasked(ws, causal, scale):
    """Any sign of the scale (the block softmax takes the max of unscaled
    scores), masked and unmasked."""
    print(f"[case] block scale {scale} causal {causal}", flush=True)
    _run(ws, torch.bfloat16, [70, 5], [70, 130], 32, 8, 64, 8, causal=causal, sm_scale=scale, kernel="attn_block_kernel")


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("page", [1, 2, 3, 8, 16])
@pytest.mark.parametrize("rows", [(4, 1), (3, 4), (5, 8), (1, 40)])
def test_few_rows(ws, d, page, rows):
    """Items of one to four 16-row tiles (the waves split the tokens of few rows
    and are combined), token counts around one and two tiles and beyond 64 page
    ids, causal, at every head_dim."""
    n, g = rows
    print(f"[case] tile rows {n} x {g} d {d} page {page}", flush=True)
    # (head_dim 128 on pages of 16 streams)
    _run(ws, torch.bfloat16, [n, n, n], [63, 130, 400], 2 * g, 2, d, page,
         kernel=None if d == 128 and page == 16 else "attn_tile_kernel")


@pytest.mark.parametrize("page", [1, 4, 16])
def test_keys_split_over_blocks(ws, page):
    """Few queries over many cached tokens: the keys are cut into chunks and
    merged; page 1 also meets the page-id limit of one item."""
    print(f"[case] block split page {page}", flush=True)
    w = _run(ws, torch.float16, [40], [3000], 32, 8, 64, page, kernel="attn_block_kernel")
    assert w.stats.num_merge == 40


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("q_lens,kv_lens,page", [([256], [8256], 16), ([100, 40], [4000, 3000], 8), ([70], [2000], 5)])
def test_keys_split_over_blocks_d128(ws, dtype, q_lens, kv_lens, page):
    """The same at head_dim 128: partial rows of several chunks per query, on
    plans of both kinds that run blocks, and the merge."""
    print(f"[case] block split d128 page {page} {dtype}", flush=True)
    w = _run(ws, dtype, q_lens, kv_lens, 32, 8, 128, page, kernel="attn_block_kernel")
    assert w.stats.num_merge == sum(q_lens) and w.stats.launches == ("attn_block_kernel", "merge_kernel")
    assert (w._info.kernel, w._info.stream_loop) == ((2, 2) if page == 16 else (1, 0))


@pytest.mark.parametrize("d,page,n,kv_len", [(128, 4, 70, 1400), (128, 8, 70, 2500), (64, 8, 70, 2500), (128, 8, 600, 4000),
                                             (128, 1, 70, 900), (128, 12, 70, 2000)])
def test_long_items(ws, d, page, n, kv_len):
    """Items of hundreds of pages (one CU: the keys stay whole): where pages hold
    whole load groups the page ids pass through windows of 64, elsewhere every
    lane looks its row's up."""
    print(f"[case] block windows d {d} page {page}", flush=True)
    w = _run(ws, torch.bfloat16, [n], [kv_len], 32, 8, d, page, cus=1, kernel="attn_block_kernel")
    assert w.stats.num_merge == 0 and kv_len // page > 128


@pytest.mark.parametrize("dtype,hq,hkv,page,n,kv_len,small", [
    (torch.bfloat16, 32, 8, 16, 256, 8256, "stream"), (torch.float32, 32, 8, 16, 1000, 1000, "f32")])
def test_plan_for_a_small_workspace(dtype, hq, hkv, page, n, kv_len, small):
    """A causal plan whose fp32 partial rows do not fit the workspace is planned
    again with less scratch: 16-bit storage for the streaming kernel, fp32 in
    32-row items.  Both plans run."""
    from beam_engine_amd import BatchPrefillWithPagedKVCacheWrapper
    print(f"[case] small workspace {dtype}", flush=True)
    d = 128
    (qo, kvp, kvi, lpl), pages = _levels([n], [kv_len], page)
    g = torch.Generator().manual_seed(4)
    kv = torch.randn((pages, 2, page, hkv, d), generator=g).to(dtype)
    q = torch.randn((n, hq, d), generator=g).to(dtype)
    ref_o, ref_lse = oa.cascade_attention(q, kv, [qo], [kvp], [kvi], [lpl], page, None, causal=True)

    def run(nbytes):
        w = BatchPrefillWithPagedKVCacheWrapper(torch.empty(nbytes, dtype=torch.uint8, device="cuda"))
        w.plan(qo, kvp, kvi, lpl, hq, hkv, d, page, causal=True, q_data_type=dtype)
        out, lse = w.run(q.cuda(), kv.cuda(), return_lse=True)
        torch.cuda.synchronize()
        _check(out, lse, ref_o, ref_lse, dtype)
        return w
    full = run(256 << 20)
    assert full._info.partial_bytes > 8 << 20
    less = run(full._need(full._info) - 4096)
    assert less._need(less._info) < full._need(full._info)
    if small == "stream":
        assert full._info.stream_loop == 2 and less._info.kernel == 2 and less._info.stream_loop != 2
    else:
        assert full._info.tile_rows == 64 and less._info.tile_rows == 32


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("reqs,n,cached", [(8, 64, 0), (8, 256, 0), (2, 1024, 0), (2, 300, 400)])
def test_no_further_from_64_bits_than_streaming(ws, dtype, reqs, n, cached):
    """The block kernel's distance (2-norm) from the float64 result is no larger
    than the streaming kernel's on the same inputs: both round P and the output
    to the storage type, so only how many weights are exact differs.  0.1% is
    left for the draw: where both have the same exact weights (8 x 64 tokens),
    0.5 M outputs of independent roundings agree to 0.006%; one exact weight
    fewer is 0.7%."""
    from beam_engine_amd import BatchPrefillWithPagedKVCacheWrapper
    print(f"[case] block error {reqs} x {n} + {cached} {dtype}", flush=True)
    hq, hkv, d, page = 32, 8, 128, 16
    (qo, kvp, kvi, lpl), pages = _levels([n] * reqs, [n + cached] * reqs, page)
    g = torch.Generator().manual_seed(n)
    kv = torch.randn((pages, 2, page, hkv, d), generator=g).to(dtype)
    q = torch.randn((qo[-1], hq, d), generator=g).to(dtype)
    ref, _ = oa.cascade_attention(q, kv, [qo], [kvp], [kvi], [lpl], page, None, causal=True)
    err = []
    for no_blocks in (False, True):
        w = BatchPrefillWithPagedKVCacheWrapper(ws)
        w._no_blocks = no_blocks
        w.plan(qo, kvp, kvi, lpl, hq, hkv, d, page, causal=True, q_data_type=dtype)
        assert w._info.kernel == 2 and (w._info.stream_loop == 2) != no_blocks
        out = w.run(q.cuda(), kv.cuda()).double().cpu().numpy()
        err.append(np.linalg.norm(out - ref) / np.linalg.norm(ref))
    assert err[0] <= 1.001 * err[1], err


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("page", [1, 2, 3, 8, 16])
@pytest.mark.parametrize("rows", [(4, 1), (20, 2), (3, 32)])
def test_fp32(ws, d, page, rows):
    """fp32 storage on the fp32 MFMA kernel: one to four row tiles, all page
    shapes, within 1e-5 of the float64 oracle."""
    n, g = rows
    print(f"[case] f32 rows {n} x {g} d {d} page {page}", flush=True)
    w = _run(ws, torch.float32, [n, n, 1], [64, 131, 390], 2 * g, 2, d, page)
    assert w.stats.kernel == "valu" and w._info.tile_rows in (16, 32, 64)
    assert w.stats.launches[0] == "attn_f32_kernel"


@pytest.mark.parametrize("dtype,n,hq,page,d,fused", [
    (torch.float32, 40, 8, 16, 128, False), (torch.float32, 5, 8, 3, 64, True), (torch.bfloat16, 70, 16, 8, 128, False),
    (torch.float16, 300, 16, 16, 128, False), (torch.bfloat16, 9, 8, 8, 256, False), (torch.bfloat16, 30, 8, 16, 64, True)])
def test_unaligned_cache(ws, dtype, n, hq, page, d, fused):
    """A cache that starts one element off an allocation: the kernels that load
    16 bytes a lane, or straight to LDS, leave the work list to the VALU kernel
    (items of more rows than it holds are shared by its workgroups)."""
    from beam_engine_amd import BatchPrefillWithPagedKVCacheWrapper
    print(f"[case] unaligned cache {dtype} n {n} page {page} d {d}", flush=True)
    (qo, kvp, kvi, lpl), pages = _levels([n, 3], [n + 900, 40], page)
    g = torch.Generator().manual_seed(8)
    kv = torch.randn((pages, 2, page, 2, d), generator=g).to(dtype)
    q = torch.randn((n + 3, hq, d), generator=g).to(dtype)
    off = torch.empty(kv.numel() + 1, dtype=dtype, device="cuda")[1:].view(kv.shape)
    off.copy_(kv)
    assert off.data_ptr() % 16 != 0 and off.is_contiguous()
    w = BatchPrefillWithPagedKVCacheWrapper(ws)
    w._fused_merge, w._tile_kernel, w._num_cus = fused, page % 16 != 0, 8
    w.plan(qo, kvp, kvi, lpl, hq, 2, d, page, causal=True, q_data_type=dtype)
    if w._info.kernel == 2 and w._info.stream_loop != 2:
        with pytest.raises(ValueError, match="aligned"):
            w.run(q.cuda(), off)
        return
    out, lse = w.run(q.cuda(), off, return_lse=True)
    torch.cuda.synchronize()
    ref_o, ref_lse = oa.cascade_attention(q, kv, [qo], [kvp], [kvi], [lpl], page, None, causal=True)
    _check(out, lse, ref_o, ref_lse, dtype)


@pytest.mark.parametrize("tile_rows", [16, 32, 64])
def test_fp32_fixed_layout(ws, tile_rows):
    """fp32 in a fixed-capacity layout sized for 32-row items."""
    from beam_engine_amd import BatchPrefillWithPagedKVCacheWrapper
    print(f"[case] f32 fixed layout {tile_rows}", flush=True)
    (qo, kvp, kvi, lpl), pages = _levels([64], [500], 16)
    g = torch.Generator().manual_seed(6)
    kv = torch.randn((pages, 2, 16, 2, 128), generator=g)
    q = torch.randn((64, 8, 128), generator=g)
    w = BatchPrefillWithPagedKVCacheWrapper(ws)
    w.use_fixed_layout(32, 64, 32, 64, 256, 0, tile_rows)
    w.plan(qo, kvp, kvi, lpl, 8, 2, 128, 16, causal=False, q_data_type=torch.float32)
    out, lse = w.run(q.cuda(), kv.cuda(), return_lse=True)
    ref_o, ref_lse = oa.cascade_attention(q, kv, [qo], [kvp], [kvi], [lpl], 16, None)
    _check(out, lse, ref_o, ref_lse, torch.float32)


@pytest.mark.parametrize("dtype,d,page", [(torch.bfloat16, 128, 8), (torch.float32, 128, 16), (torch.float16, 64, 16),
                                          (torch.bfloat16, 256, 16)])
@pytest.mark.parametrize("fused", [False, True])
def test_queries_with_one_item_beside_others(ws, dtype, d, page, fused):
    """Two levels on the work-list kernels, some queries without keys on the
    second or the first: a query's only item may share its tile with queries of
    more items, and its partial row is the whole result."""
    from beam_engine_amd import MultiLevelCascadeAttentionWrapper
    print(f"[case] one item beside others {dtype} d {d} page {page} fused {fused}", flush=True)
    hq, hkv, nq = 8, 2, 24
    (qo0, kvp0, kvi0, lpl0), p0 = _levels([16, 8], [700, 0], page)
    (qo1, kvp1, kvi1, lpl1), p1 = _levels([1] * nq, [0 if i % 3 == 0 else 5 + 11 * i for i in range(nq)], page)
    levels = ([qo0, qo1], [kvp0, kvp1], [kvi0, [p0 + x for x in kvi1]], [lpl0, lpl1])
    g = torch.Generator().manual_seed(12)
    kv = torch.randn((p0 + p1, 2, page, hkv, d), generator=g).to(dtype)
    q = torch.randn((nq, hq, d), generator=g).to(dtype)
    w = MultiLevelCascadeAttentionWrapper(2, ws)
    w._fused_merge = fused
    w.plan(*levels, hq, hkv, d, page, q_data_type=dtype)
    out, lse = w.run(q.cuda(), kv.cuda(), return_lse=True)
    torch.cuda.synchronize()
    ref_o, ref_lse = oa.cascade_attention(q, kv, *levels, page)
    _check(out, lse, ref_o, ref_lse, dtype)


@pytest.mark.parametrize("dtype,d,page,n,hq", [
    (torch.float32, 64, 16, 2, 8), (torch.float32, 128, 3, 8, 8), (torch.float32, 256, 8, 30, 8), (torch.bfloat16, 64, 8, 2, 8),
    (torch.bfloat16, 256, 3, 20, 8), (torch.float16, 128, 8, 8, 8), (torch.float16, 64, 16, 40, 8), (torch.bfloat16, 128, 5, 90, 8)])
@pytest.mark.parametrize("kv_len", [1, 63, 70, 127, 200])
def test_infinite_value_of_the_last_token(ws, dtype, d, page, n, hq, kv_len):
    """An infinite value element of a group's last token makes its column
    infinite: what fills the token tile beyond the group's end does not meet it
    (0 x infinity)."""
    from beam_engine_amd import BatchPrefillWithPagedKVCacheWrapper
    print(f"[case] inf d {d} page {page} {dtype} n {n} kv {kv_len}", flush=True)
    (qo, kvp, kvi, lpl), pages = _levels([n], [kv_len], page)
    g = torch.Generator().manual_seed(5)
    kv = torch.randn((pages, 2, page, 2, d), generator=g).to(dtype)
    kv[kvi[(kv_len - 1) // page], 1, (kv_len - 1) % page, 1, 7] = math.inf
    q = torch.randn((n, hq, d), generator=g).to(dtype)
    w = BatchPrefillWithPagedKVCacheWrapper(ws)
    w._tile_kernel = True
    w.plan(qo, kvp, kvi, lpl, hq, 2, d, page, causal=False, q_data_type=dtype)
    out = w.run(q.cuda(), kv.cuda()).float().cpu()
    assert not out.isnan().any()
    want = torch.zeros_like(out, dtype=torch.bool)
    want[:, hq // 2:, 7] = True
    assert torch.equal(out == math.inf, want)


@pytest.mark.parametrize("dtype,d,page,n", [(torch.bfloat16, 64, 8, 4), (torch.float32, 64, 16, 4), (torch.float32, 128, 16, 4),
                                            (torch.bfloat16, 64, 16, 64)])
@pytest.mark.parametrize("where", ["k", "v", "q"])
@pytest.mark.parametrize("fused", [False, True])
def test_nan_survives_the_merge(ws, dtype, d, page, n, where, fused):
    """A NaN key makes every row of its KV head NaN, a NaN value its column and a
    NaN query its row, also where the keys are split: the NaN piece is merged with
    finite ones, or (a query's) every piece is NaN."""
    from beam_engine_amd import BatchPrefillWithPagedKVCacheWrapper
    print(f"[case] nan {where} d {d} page {page} {dtype}", flush=True)
    (qo, kvp, kvi, lpl), pages = _levels([n], [3000], page)
    g = torch.Generator().manual_seed(5)
    kv = torch.randn((pages, 2, page, 2, d), generator=g).to(dtype)
    q = torch.randn((n, 8, d), generator=g).to(dtype)
    if where == "q":
        q[2, 5, 7] = math.nan
    else:
        kv[kvi[1700 // page], 0 if where == "k" else 1, 1700 % page, 1, 7] = math.nan
    w = BatchPrefillWithPagedKVCacheWrapper(ws)
    w._fused_merge = fused
    w.plan(qo, kvp, kvi, lpl, 8, 2, d, page, causal=False, q_data_type=dtype)
    out = w.run(q.cuda(), kv.cuda()).float().cpu()
    assert w.stats.num_merge == n and w.stats.kernel != "stream"
    want = torch.zeros_like(out, dtype=torch.bool)
    if where == "q":
        want[2, 5] = True
    elif where == "k":
        want[:, 4:] = True
    else:
        want[:, 4:, 7] = True
    assert torch.equal(out.isnan(), want)
