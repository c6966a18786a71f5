"""The decoder's fused passes on the GPU against float64: residual add + RMSNorm
and SiLU(gate) * up, at row lengths around the vector, workgroup and largest row.

Bounds are the storage roundings: the sum and the norm round once each (half an
ulp: 2^-8 of a bf16 value with its 8 significant bits, 2^-11 of an fp16 one with
its 11), SiLU * up twice; one percent
and a subnormal's half ulp are left for the fp32 arithmetic."""

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

HALF_ULP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _decoder(n, inter, dtype):
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from beam_engine_amd.llama import LlamaConfig, LlamaDecoder
    cfg = LlamaConfig(vocab_size=64, hidden_size=n, intermediate_size=inter, num_hidden_layers=1, num_attention_heads=1,
                      num_key_value_heads=1, head_dim=64, max_position_embeddings=16)
    return LlamaDecoder(cfg, dtype=dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,n", [(1, 8), (3, 2040), (2, 2048), (5, 2056), (300, 4096), (2, 8192), (2, 8200), (2, 100)])
def test_add_rms_norm(dtype, rows, n):
    m = _decoder(n, 8, dtype)
    g = torch.Generator(device="cuda").manual_seed(n)
    x, d = (torch.randn((rows, n), generator=g, device="cuda").mul(2).to(dtype) for _ in range(2))
    w = torch.rand(n, generator=g, device="cuda").add(0.5).to(dtype)
    keep = x.clone(), d.clone()
    s, h = m._add_rms(x, d, w)
    assert torch.equal(x, keep[0]) and torch.equal(d, keep[1]) and torch.equal(s, x + d)
    v = s.double()
    ref = v * torch.rsqrt(v.square().mean(-1, keepdim=True) + m.cfg.rms_norm_eps) * w.double()
    assert ((h.double() - ref).abs() <= 1.01 * HALF_ULP[dtype] * ref.abs() + 2.0 ** -25).all()
    s, h = m._add_rms(x, None, w)
    assert s is x and torch.equal(h, m._rms(x, w))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,inter", [(1, 8), (3, 2040), (5, 2056), (130, 14336), (2, 100)])
def test_silu_mul(dtype, rows, inter):
    """Through the MLP with an identity down projection."""
    m = _decoder(inter, inter, dtype)
    g = torch.Generator(device="cuda").manual_seed(inter)
    gu = torch.randn((rows, 2 * inter), generator=g, device="cuda").mul(4).to(dtype)
    gu[0, :4] = torch.tensor([30000.0, -30000.0, 0.0, -20.0], device="cuda").to(dtype)
    calls = []

    def linear(a, wgt):
        calls.append(a)
        return gu if len(calls) == 1 else a
    old, F.linear = F.linear, linear
    try:
        y = m._mlp(m.layers[0], gu)
    finally:
        F.linear = old
    a, b = gu.double().chunk(2, dim=-1)
    ref = a / (1 + torch.exp(-a)) * b
    # twice half an ulp, SiLU's subnormals scaled by |up|
    err = (y.double() - ref).abs()
    fin = ref.abs() < 6e4
    assert (err[fin] <= (2.02 * HALF_ULP[dtype] * ref.abs() + 2.0 ** -25 * (1 + b.abs()))[fin]).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16])
def test_silu_mul_special_values(dtype):
    """NaN and infinities as the tensor code gives them."""
    m = _decoder(8, 8, dtype)
    inf, nan = float("inf"), float("nan")
    gu = torch.tensor([[inf, -inf, nan, 1.0, 2.0, -inf, 0.0, 1.0, 1.0, 1.0, 1.0, nan, inf, 2.0, inf, -inf]], device="cuda").to(dtype)
    calls = []

    def linear(a, wgt):
        calls.append(a)
        return gu if len(calls) == 1 else a
    old, F.linear = F.linear, linear
    try:
        y = m._mlp(m.layers[0], gu)
    finally:
        F.linear = old
    a, b = gu.chunk(2, dim=-1)
    assert torch.equal((F.silu(a) * b).nan_to_num(7.0, 8.0, 9.0), y.nan_to_num(7.0, 8.0, 9.0))
