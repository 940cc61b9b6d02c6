"""dg_linear_rows (dg_linear.hip) against float64 at the edges of its row tiles,
feature tiles and contraction chunks, and a Block with and without it."""

import pytest
import torch

pytestmark = pytest.mark.gpu

TDT = {"bf16": torch.bfloat16, "f16": torch.float16}
HALF = {"bf16": 2.0**-8, "f16": 2.0**-11}  # half an ulp, relative to the value




@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("M,N,K", [(1, 32, 512), (31, 64, 1024), (32, 512, 512), (33, 320, 1536), (100, 512, 1024),
                                   (257, 1024, 512), (300, 512, 2048)])
def test_linear_rows(dev, dtype, M, N, K):
    from diff_gpt import _native

    dt = TDT[dtype]
    g = torch.Generator(device=dev).manual_seed(M + N)
    r = lambda *s: torch.randn(*s, generator=g, device=dev).to(dt)  # noqa: E731
    wide = r(M, 2 * K + 8)  # rows with a stride of their own
    x, gate, res = wide[:, :K], wide[:, K : 2 * K], r(M, N)
    w = (r(N, K).float() * K**-0.5).to(dt)
    out = torch.full((M, N), 7.0, dtype=dt, device=dev)
    assert _native.linear_rows_(x, w, out)
    ref = x.double() @ w.double().T
    size = x.double().abs() @ w.double().abs().T * 2.0**-2 + ref.abs()  # fp32 sums of up to 2048 products
    plain = out.clone()
    assert bool(((out.double() - ref).abs() <= HALF[dtype] * ref.abs() + 2.0**-18 * size + 2.0**-24).all())
    # the residual: the rounded product plus the row, rounded
    assert _native.linear_rows_(x, w, out, residual=res)
    assert torch.equal(out, plain + res)
    # the gate: the rows as dg_gate stores them
    gated = x.clone(memory_format=torch.contiguous_format)
    _native.gate_(gated, gate)
    assert _native.linear_rows_(gated, w, plain)
    assert _native.linear_rows_(x, w, out, gate=gate)
    assert torch.equal(out, plain)
    assert _native.linear_rows_(x, w, out, gate=gate, residual=res)
    assert torch.equal(out, plain + res)
    # SwiGLU of the rounded product, as dg_swiglu (these sizes take as many waves in both)
    if N % 64 == 0:
        assert _native.linear_rows_(x, w, plain)
        hid = torch.empty(M, N // 2, dtype=dt, device=dev)
        assert _native.linear_rows_(x, w, hid, swiglu=(1.702, 7.0))
        assert torch.equal(hid, _native.ops().swiglu(plain, 1.702, 7.0))


def test_linear_rows_declines(dev):
    from diff_gpt import _native

    for M, N, K, dt in ((4, 64, 512, torch.float32), (4, 48, 512, torch.bfloat16), (4, 64, 256, torch.bfloat16)):
        out = torch.full((M, N), 3.0, dtype=dt, device=dev)
        assert not _native.linear_rows_(torch.ones(M, K, dtype=dt, device=dev), torch.ones(N, K, dtype=dt, device=dev), out)
        assert bool((out == 3.0).all())
    x = torch.ones(4 * 512 + 1, dtype=torch.bfloat16, device=dev)[1:].view(4, 512)  # misaligned rows
    out = torch.full((4, 64), 3.0, dtype=torch.bfloat16, device=dev)
    assert not _native.linear_rows_(x, torch.ones(64, 512, dtype=torch.bfloat16, device=dev), out)


@pytest.mark.parametrize("layer_idx", [0, 1])  # with two layers per block: one adds to its input, one commits it
def test_block_with_and_without(dev, layer_idx, monkeypatch):
    """The layer's output within bf16's bar of the separate launches; infinities
    and NaN reach the same rows."""
    from diff_gpt.model import block

    torch.manual_seed(3)
    blk = block.Block(512, 8, 1.702, 7.0, layer_idx, layers_per_block=2).eval().to(dev).to(torch.bfloat16)
    x = torch.randn(33, 1, 512, device=dev).to(torch.bfloat16)
    x[5, 0, 7], x[6, 0, 8] = float("inf"), float("nan")
    from diff_gpt.model.rope import precompute_freqs_cis

    freqs = precompute_freqs_cis(64, 4, 10000.0).to(dev)[:1].view(1, 1, 1, 32, 2)
    with torch.inference_mode():
        one = blk((x,), x * 2, freqs, None)[1]
        monkeypatch.setattr(block, "_few_rows", lambda *a: False)
        apart = blk((x,), x * 2, freqs, None)[1]
    assert torch.equal(one.isfinite(), apart.isfinite())
    ok = apart.isfinite()
    assert (one[ok].double() - apart[ok].double()).abs().max() <= 2e-2 * apart[ok].double().abs().max()


def test_a_replaced_output_projection_is_heard(dev, monkeypatch):
    """c_proj with a forward of its own, in the instance or the class, or watched
    by a hook on all modules, is called as it is with a hook of its own."""
    from torch import nn
    from torch.nn.modules.module import register_module_forward_hook

    from diff_gpt.model.block import Block
    from diff_gpt.model.rope import precompute_freqs_cis

    torch.manual_seed(3)
    blk = Block(512, 8, 1.702, 7.0, 0).eval().to(dev).to(torch.bfloat16)
    x = torch.randn(33, 1, 512, device=dev).to(torch.bfloat16)
    freqs = precompute_freqs_cis(64, 4, 10000.0).to(dev)[:1].view(1, 1, 1, 32, 2)
    proj, inner = blk.sa.c_proj, nn.Linear.forward

    @torch.inference_mode()
    def out():
        return blk((x,), x * 2, freqs, None)[1]

    plain = out()
    hook = proj.register_forward_hook(lambda m, i, o: o * 2)
    ref = out()
    hook.remove()
    assert not torch.equal(ref, plain)
    proj.forward = lambda y: inner(proj, y) * 2
    assert torch.equal(out(), ref)
    del proj.forward
    with monkeypatch.context() as m:
        m.setattr(nn.Linear, "forward", lambda self, y: inner(self, y) * (2 if self is proj else 1))
        assert torch.equal(out(), ref)
    hook = register_module_forward_hook(lambda m, i, o: o * 2 if m is proj else None)
    try:
        assert torch.equal(out(), ref)
    finally:
        hook.remove()
    assert torch.equal(out(), plain)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("n_embd,n_head", [(64, 4), (128, 4), (512, 8), (1024, 8)])
@pytest.mark.parametrize("layer_idx", [0, 1])
def test_block_takes_permuted_inputs(dev, dtype, n_embd, n_head, layer_idx):
    """Committed blocks and a partial sum whose dimensions lie in another order
    than (B, T, C), at few rows and at many: the contiguous copies' result."""
    from diff_gpt.model.block import Block
    from diff_gpt.model.rope import precompute_freqs_cis

    torch.manual_seed(3)
    dt = {"f32": torch.float32, **TDT}[dtype]
    blk = Block(n_embd, n_head, 1.702, 7.0, layer_idx, layers_per_block=2).eval().to(dev).to(dt)
    for B, T in ((3, 5), (16, 100)):
        freqs = precompute_freqs_cis(n_embd // n_head, T, 10000.0).to(dev).view(1, T, 1, -1, 2)
        first, partial = (torch.randn(T, B, n_embd, device=dev).to(dt).transpose(0, 1) for _ in range(2))
        with torch.inference_mode():
            got = blk((first,), partial, freqs, None)[1]
            ref = blk((first.contiguous(),), partial.contiguous(), freqs, None)[1]
        assert torch.equal(got, ref)
