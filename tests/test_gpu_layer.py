"""dg_block_in and dg_block_out (dg_layer.hip) at the edges of their 16-row
groups, of the rows that fill the chip once (a workgroup then walks several
groups) and of the sources held in registers."""

import pytest
import torch

pytestmark = pytest.mark.gpu

TDT = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
BAR = {"f32": 1e-5, "bf16": 2e-2, "f16": 2e-2}


def _sources(M, C, n, dt, dev, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    s = [(torch.randn(M, C, generator=g, device=dev) * (0.5 + 0.1 * i)).to(dt) for i in range(n)]
    if n > 1:
        s[1] = s[0]
    return s


def _weight(rows, C, dt, dev, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    return (torch.randn(rows, C, generator=g, device=dev) * C**-0.5).to(dt)


def _rel(a, b):
    return ((a.double() - b.double()).abs().max() / b.double().abs().max()).item()


@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("C", [64, 128])
@pytest.mark.parametrize("M,n", [(1, 1), (1, 3), (16, 2), (17, 4), (100, 5), (333, 8), (40, 9), (70, 32), (8193, 3),
                                 (20000, 4)])
def test_block_in_is_the_mixture_then_the_projection(dev, dtype, C, M, n):
    """Against the mixture kernel and float64 products of its rows: within the
    bars, the mixture's roundings being the same."""
    from diff_gpt import _native

    dt = TDT[dtype]
    srcs = _sources(M, C, n, dt, dev, 3 + n)
    w_mix, w = _weight(1, C, dt, dev, 5) * 4, _weight(4 * C, C, dt, dev, 6)
    out = torch.empty(M, 4 * C, dtype=dt, device=dev)
    assert _native.block_in_(srcs, w_mix, w, out)
    xn = torch.empty(M, C, dtype=dt, device=dev)
    _native.attn_res_norm_(srcs, w_mix, xn)
    ref = xn.double() @ w.double().T
    assert _rel(out, ref) <= BAR[dtype]
    plain = torch.empty_like(out)
    assert _native.block_in_([xn], None, w, plain)
    half = {"f32": 0.0, "bf16": 2.0**-8, "f16": 2.0**-11}[dtype]
    # one rounding of an fp32 sum of C products
    assert bool(((plain.double() - ref).abs() <= half * ref.abs() + C * 2.0**-23 * (xn.double().abs() @ w.double().abs().T)).all())


@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("C", [64, 128])
@pytest.mark.parametrize("n", [3, 8, 9])
def test_layer_rows_do_not_depend_on_the_launch(dev, dtype, C, n):
    """A row's bits are the same alone, among a few rows and in a launch whose
    workgroups walk several groups; dg_block_out_norm's norm is dg_rms_norm's."""
    from diff_gpt import _native

    dt, M = TDT[dtype], 16 * 512 * 2 + 5
    srcs = _sources(M, C, n, dt, dev, 11)
    y, qkvg = _sources(M, C, 1, dt, dev, 12)[0], _sources(M, 4 * C, 1, dt, dev, 13)[0]
    wm, wq, wp = _weight(1, C, dt, dev, 1) * 4, _weight(4 * C, C, dt, dev, 2), _weight(C, C, dt, dev, 3)
    wu, wd = _weight(4 * C, C, dt, dev, 4) * 2, _weight(C, 2 * C, dt, dev, 5)

    def run(sl):
        s = [t[sl] for t in srcs]
        rows = s[0].size(0)
        qo = torch.empty(rows, 4 * C, dtype=dt, device=dev)
        assert _native.block_in_(s, wm, wq, qo)
        outs = [qo]
        for pin in (None, s[-1]):
            o, xn = (torch.empty(rows, C, dtype=dt, device=dev) for _ in range(2))
            assert _native.block_out_(y[sl], qkvg[sl][:, 3 * C :], wp, pin, s, wm, wu, wd, 1.702, 7.0, o, xn)
            assert torch.equal(xn, _native.ops().rms_norm(o))
            outs.append(o)
        return outs

    full = run(slice(0, M))
    for sl in (slice(0, 1), slice(100, 137), slice(M - 20, M), slice(16 * 512 - 3, 16 * 512 + 30)):
        for part, whole in zip(run(sl), full):
            assert torch.equal(part, whole[sl])


@pytest.mark.parametrize("C", [32, 96, 256])
def test_block_in_declines_other_widths(dev, C):
    from diff_gpt import _native

    out = torch.full((4, 4 * C), 3.0, device=dev)
    assert not _native.block_in_(_sources(4, C, 2, torch.float32, dev, 1), _weight(1, C, torch.float32, dev, 1),
                                 _weight(4 * C, C, torch.float32, dev, 2), out)
    assert bool((out == 3.0).all())
