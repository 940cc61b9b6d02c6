"""Prefill attention at head_dim 16 and 32 (dg_attn_small.hip) against float64,
at the edges of its 16-query tiles and 16-key tiles, and with values that are
not finite behind the mask."""

import pytest
import torch

pytestmark = pytest.mark.gpu

TDT = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
# half an ulp of p significant bits is at most 2^-p of the value
HALF = {"f32": 2.0**-24, "bf16": 2.0**-8, "f16": 2.0**-11}


def _case(dev, B, H, Tq, Tk, D, dt, seed=0, scale=1.0):
    g = torch.Generator(device=dev).manual_seed(seed)
    wide = (torch.randn(B, Tq, 2, H, D, generator=g, device=dev) * scale).to(dt)
    pages = torch.randn(2, B, H, Tk + 3, D, generator=g, device=dev).to(dt)  # cache pages, (B,H,T,D)
    return wide[:, :, 1], pages[0, :, :, :Tk].transpose(1, 2), pages[1, :, :, :Tk].transpose(1, 2)


def _attend64(q, k, v):
    Tq, Tk = q.size(1), k.size(1)
    q, k, v = (t.double().transpose(1, 2) for t in (q, k, v))
    s = q @ k.transpose(-1, -2).contiguous() * q.size(-1) ** -0.5
    hidden = torch.ones(Tq, Tk, dtype=torch.bool, device=q.device).triu(Tk - Tq + 1)
    return (s.masked_fill(hidden, float("-inf")).softmax(-1) @ v).transpose(1, 2)


@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("D", [16, 32])
@pytest.mark.parametrize("B,H,Tq,Tk", [(1, 1, 16, 16), (3, 4, 17, 17), (2, 4, 138, 138), (1, 3, 31, 95), (2, 2, 64, 65),
                                       (1, 2, 16, 1000), (5, 1, 129, 129), (1, 2, 400, 401)])
def test_small_prefill_matches_float64(dev, dtype, D, B, H, Tq, Tk):
    """Within the rounding of the result plus fp32 arithmetic: scores up to about 6
    and sums of up to 1001 probabilities, 2e-6 of the largest output."""
    from diff_gpt import _native

    q, k, v = _case(dev, B, H, Tq, Tk, D, TDT[dtype], seed=Tq + D)
    y = torch.empty(B, Tq, H, D, dtype=TDT[dtype], device=dev)
    _native.attention_(q, k, v, y, D**-0.5)
    assert _native.last_kernel() == "prefill_small_kernel"
    ref = _attend64(q, k, v)
    assert bool(((y.double() - ref).abs() <= HALF[dtype] * ref.abs() + 2e-6 * ref.abs().max()).all())


@pytest.mark.parametrize("D", [16, 32])
def test_small_prefill_large_scores_rescale(dev, D):
    """Scores of several hundred that grow along the keys: the running maximum is
    raised chunk after chunk.  A score's fp32 rounding, some 16 ulps of its
    largest partial sum (2^-24 * 16 * 600 = 6e-4), moves a probability by as much."""
    from diff_gpt import _native

    q, k, v = _case(dev, 1, 2, 200, 200, D, torch.float32, seed=3, scale=30.0)
    k = k * torch.linspace(0.2, 3.0, 200, device=dev).view(1, 200, 1, 1)
    y = torch.empty(1, 200, 2, D, device=dev)
    _native.attention_(q, k, v, y, D**-0.5)
    assert _native.last_kernel() == "prefill_small_kernel"
    ref = _attend64(q, k, v)
    assert bool(((y.double() - ref).abs() <= 2 * 6e-4 * ref.abs().max()).all())


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("D", [16, 32])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
def test_small_prefill_keeps_hidden_rows_out(dev, dtype, D, bad):
    """A key and value row that is not finite (an id outside the vocabulary gives
    NaN rows) stays out of every query before it, and makes the queries from it on
    what arithmetic makes them.  The tile holding it sums its 16 products in
    another order: 2e-6 of the largest output, and for 16-bit types two roundings
    to either side of the same value."""
    from diff_gpt import _native

    B, H, T, j = 2, 2, 75, 37
    q, k, v = _case(dev, B, H, T, T, D, TDT[dtype], seed=8)
    y0, y1, y2 = (torch.empty(B, T, H, D, dtype=TDT[dtype], device=dev) for _ in range(3))
    _native.attention_(q, k, v, y0, D**-0.5)
    v2 = v.clone()
    v2[:, j, :, 3] = bad
    _native.attention_(q, k, v2, y1, D**-0.5)
    assert _native.last_kernel() == "prefill_small_kernel"

    def close(a, b):
        a, b = a.double(), b.double()
        return bool(((a - b).abs() <= 2 * HALF[dtype] * b.abs() + 2e-6 * b.abs().max()).all())

    assert close(y1[:, :j], y0[:, :j])
    col = y1[:, j:, :, 3]
    assert bool(col.isnan().all()) if bad != bad else torch.equal(col, torch.full_like(col, bad))
    others = [d for d in range(D) if d != 3]
    assert close(y1[:, j:][..., others], y0[:, j:][..., others])
    k2 = k.clone()
    k2[:, j] = float("nan")
    _native.attention_(q, k2, v2, y2, D**-0.5)
    assert close(y2[:, :j], y0[:, :j]) and bool(y2[:, j:].isnan().all())
