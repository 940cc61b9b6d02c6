"""The vector forms of the row kernels around attention (dg_block.hip) against
their general forms on the same values, at the sizes where a vector form can go
wrong: rows whose vector count does not divide the workgroup, one row, launches
with one and with four vectors per thread, and a last workgroup that is partly
empty.  The general form runs on rows one element off their alignment."""

import pytest
import torch

pytestmark = pytest.mark.gpu

TDT = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}


def _rows(M, C, dtype, dev, seed, offset, scale=3.0):
    """(M, C) values that depend on the seed alone, rows ``offset`` elements off
    their alignment (32 elements more a row keep a wide row's lanes aligned too)."""
    g = torch.Generator(device=dev).manual_seed(seed)
    x = (torch.randn(M, C, generator=g, device=dev) * scale).to(dtype)
    wide = torch.zeros(M, C + 32, dtype=dtype, device=dev)
    wide[:, offset : offset + C] = x
    return wide[:, offset : offset + C]


SHAPES = [(1, 8), (3, 24), (1, 512), (37, 200), (4100, 64), (131075, 64), (2051, 4104)]


@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("M,C", SHAPES, ids=lambda v: str(v))
def test_gate_and_swiglu_vector_rows_equal_the_general_form(dev, dtype, M, C):
    from diff_gpt import _native

    dt = TDT[dtype]
    got, ref = (_rows(M, C, dt, dev, 1, off) for off in (0, 1))
    ga, gb = (_rows(M, C, dt, dev, 2, off) for off in (0, 1))
    _native.gate_(got, ga)
    assert _native.last_kernel() == "gate_vec_kernel"
    _native.gate_(ref, gb)
    assert _native.last_kernel() == "gate_kernel"
    assert torch.equal(got, ref)
    xa, xb = (_rows(M, C, dt, dev, 3, off) for off in (0, 1))
    oa, ob = (torch.empty(M, C // 2, dtype=dt, device=dev) for _ in range(2))
    _native.swiglu_(xa, oa, 1.702, 7.0)
    assert _native.last_kernel() == "swiglu_vec_kernel"
    _native.swiglu_(xb, ob, 1.702, 7.0)
    assert _native.last_kernel() == "swiglu_kernel"
    assert torch.equal(oa, ob)


@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
def test_gate_limits(dev, dtype):
    """sigmoid at infinities, NaN and arguments beyond exp's range: the values of
    torch's own sequence within one rounding of the type (2^-7, 2^-10 or, for
    fp32, 4 ulps of 2^-23, relative)."""
    from diff_gpt import _native

    g = torch.tensor([float("inf"), float("-inf"), float("nan"), 0.0, -0.0, 88.0, -86.0, 200.0, -200.0, 3e4, -3e4,
                      1e-6, -1e-6, 1.5, -1.5, 9.0] * 4, dtype=TDT[dtype])
    y = torch.full_like(g, 1.25)
    got = y.to(dev).view(1, -1).clone()
    _native.gate_(got, g.to(dev).view(1, -1))
    ref = (y * torch.sigmoid(g)).view(1, -1)
    tol = {"f32": 2.0**-21, "bf16": 2.0**-7, "f16": 2.0**-10}[dtype]
    assert torch.equal(got.isnan().cpu(), ref.isnan())
    d = (got.cpu().double() - ref.double()).abs().nan_to_num(0.0)
    assert bool((d <= tol * ref.double().abs().nan_to_num(0.0) + torch.finfo(TDT[dtype]).tiny).all())


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_sigmoid_of_every_argument(dev, dtype):
    """The gate and the SwiGLU of all 65536 arguments of a 16-bit type, in their
    vector and general forms, are torch's own sequence on the device bit for bit:
    subnormal results (arguments from -87.5 to -88.5 in bf16) included.  NaN
    arguments go to the gate alone (swi_glu.py's clamp passes them on, the
    kernel's minimum does not)."""
    from diff_gpt import _native

    dt = TDT[dtype]
    bits = lambda t: t.contiguous().view(torch.int16)  # noqa: E731
    x = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(dt).to(dev).view(256, 256)
    nan = x.isnan()
    for y in (1.0, 1.25):
        ref = torch.full_like(x, y) * torch.sigmoid(x)
        for off in (0, 1):
            g, got = (torch.zeros(256, 264, dtype=dt, device=dev)[:, off : off + 256] for _ in range(2))
            g.copy_(x)
            got.fill_(y)
            _native.gate_(got, g)
            assert torch.equal(got.isnan(), nan) and torch.equal(bits(got)[~nan], bits(ref)[~nan])
    gate = x.clamp(max=7.0)
    ref = gate * torch.sigmoid(1.702 * gate) * (torch.zeros_like(x) + 1)
    for off in (0, 1):
        pairs = torch.zeros(256, 520, dtype=dt, device=dev)[:, off : off + 512]
        pairs[:, ::2] = x
        out = torch.empty(256, 256, dtype=dt, device=dev)
        _native.swiglu_(pairs, out, 1.702, 7.0)
        assert torch.equal(bits(out)[~nan & ~ref.isnan()], bits(ref)[~nan & ~ref.isnan()])
        assert bool(out[~nan & ref.isnan()].isnan().all())


@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("C", [64, 256, 512, 1024, 2048])
@pytest.mark.parametrize("n", [1, 2, 4, 5, 7, 8, 12, 13])
def test_mixture_forms_agree(dev, dtype, C, n):
    """Aligned full-width rows (every source held in registers where they fit),
    rows off their alignment (the general form) and few rows (a workgroup per
    row) give the same bits, with source 1 being source 0 itself or a copy of
    it."""
    from diff_gpt import _native

    dt, M = TDT[dtype], 4099
    aligned, shifted = ([_rows(M, C, dt, dev, 50 + i, off, 0.5 + 0.2 * i) for i in range(n)] for off in (0, 1))
    if n > 1:
        aligned[1], shifted[1] = aligned[0], shifted[0]
    copied = [s.clone() for s in aligned]  # no two are the same rows
    w = torch.randn(1, C, generator=torch.Generator(device=dev).manual_seed(9), device=dev).to(dt)
    # rows that fill a wave (64 lanes of 16 bytes or more), at most 96 registers of sources
    full = C * dt.itemsize >= 1024
    wave = full and any(n <= s and C // 64 * dt.itemsize // 4 * s <= 96 for s in (4, 6, 8, 12))
    outs = []
    for srcs, held in ((aligned, wave), (shifted, False), (copied, wave)):
        out = torch.empty(M, C, dtype=dt, device=dev)
        _native.attn_res_norm_(srcs, w, out)
        assert _native.last_kernel() == ("attn_res_norm_wave_kernel" if held else "attn_res_norm_kernel")
        outs.append(out)
    few = torch.empty(33, C, dtype=dt, device=dev)
    _native.attn_res_norm_([s[:33] for s in aligned], w, few)
    assert _native.last_kernel() == ("attn_res_norm_split_kernel" if full else "attn_res_norm_kernel")
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    assert torch.equal(outs[0][:33], few)


def test_mixture_f32_error(dev):
    """fp32 rows of 1024 against float64: the rounding of the result alone leaves
    about 3e-8 of its norm and the sums the rest.  Measured 9.4e-8 (one chain of
    products per lane: 9.9e-8); the bound lies between."""
    from diff_gpt import _native

    M, C, eps, errs = 8192, 1024, torch.finfo(torch.float32).eps, []
    for n in (2, 3, 5, 6, 9):
        g = torch.Generator().manual_seed(n)
        srcs = [(torch.randn(M, C, generator=g) * (0.5 + 0.3 * i)).to(dev) for i in range(n)]
        w = (torch.randn(1, C, generator=g) * C**-0.5).to(dev)
        out = torch.empty(M, C, device=dev)
        _native.attn_res_norm_(srcs, w, out)
        V = torch.stack(srcs).double()
        rms = lambda x: x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)  # noqa: E731
        ref = rms(((rms(V) @ w.view(-1).double()).softmax(0).unsqueeze(-1) * V).sum(0))
        errs.append(float((out.double() - ref).norm() / ref.norm()))
    assert sum(errs) / len(errs) < 9.7e-8


@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,Tq,past", [(2, 16, 0), (1, 129, 0), (3, 33, 47), (2, 300, 1)])
def test_prefill_gate_equals_prefill_then_gate(dev, dtype, D, B, Tq, past):
    """dg_prefill_rope_gate against dg_prefill_rope and dg_gate, bit for bit:
    ragged query counts, chunks, both softmax forms, the gate a column slice of
    the projections; a gate off its alignment is declined."""
    from diff_gpt import _native

    dt, H = TDT[dtype], 3
    g = torch.Generator(device=dev).manual_seed(5)
    wide = torch.randn(B, Tq, 2, H, D, generator=g, device=dev).to(dt)
    q, gate = wide[:, :, 0], wide[:, :, 1]
    k = torch.nn.functional.normalize(torch.randn(B, past + Tq, H, D, generator=g, device=dev), dim=-1)
    k = (k * D**0.5).to(dt)
    v = torch.randn(B, past + Tq, H, D, generator=g, device=dev).to(dt)
    ang = torch.rand(Tq, D // 2, generator=g, device=dev) * 6.0
    freqs = torch.stack((ang.cos(), ang.sin()), dim=-1).to(dt).view(1, Tq, 1, D // 2, 2)
    for normed in (False, True):
        ya, yb = torch.empty_like(v[:, :Tq]), torch.empty_like(v[:, :Tq])
        assert _native.prefill_rope_(q, freqs, k, v, ya, D**-0.5, True, normed)
        _native.gate_(ya.view(B, Tq, H * D), gate.reshape(B, Tq, H * D))
        assert _native.prefill_rope_(q, freqs, k, v, yb, D**-0.5, True, normed, gate=gate)
        assert torch.equal(ya, yb)
    off = torch.zeros(B, Tq, H, D + 8, dtype=dt, device=dev)[..., 1 : D + 1]
    assert not _native.prefill_rope_(q, freqs, k, v, yb, D**-0.5, True, True, gate=off)


@pytest.mark.parametrize("n_embd,n_head", [(512, 8), (1024, 8)])
def test_layers_gating_in_the_prefill_equal_the_gate_launch(dev, n_embd, n_head, monkeypatch):
    """A Block and a MultiHeadAttention whose output passes the fused gate's size
    give the bits of the same call with the gate launched apart."""
    from diff_gpt.model import mha as mha_mod
    from diff_gpt.model.block import Block
    from diff_gpt.model.kv_cache import KVCache
    from diff_gpt.model.rope import precompute_freqs_cis

    torch.manual_seed(0)
    block = Block(n_embd, n_head, 1.702, 7.0, layer_idx=0).eval().to(dev).to(torch.bfloat16)
    B, T, D = 2, 700, n_embd // n_head  # more rows than dg_linear_rows takes, whose sums are ordered differently
    x = torch.randn(B, T, n_embd, device=dev).to(torch.bfloat16)
    other = torch.randn(B, T, n_embd, device=dev).to(torch.bfloat16)
    freqs = precompute_freqs_cis(D, T, 10000.0).to(dev).to(torch.bfloat16).view(1, T, 1, D // 2, 2)
    calls = []
    real = mha_mod._native.prefill_rope_

    def spy(*a, **k):
        calls.append("gate" in k)
        return real(*a, **k)

    monkeypatch.setattr(mha_mod._native, "prefill_rope_", spy)
    results = []
    for limit in (0, 1 << 40):
        monkeypatch.setattr(mha_mod, "_FUSED_GATE_BYTES", limit)
        cache = KVCache(batch_size=B, num_heads=n_head, seq_len=T, head_dim=D, num_layers=1)
        with torch.no_grad():
            results.append((block.sa(x, freqs, None), block((x,), other, freqs_cis=freqs, kv_cache=cache)[1]))
    assert calls == [True, True, False, False]
    for fused, apart in zip(*results):
        assert torch.equal(fused, apart)
