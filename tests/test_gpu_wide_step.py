"""The fused decode step over shared prefixes at head_dim 64 and 128
(dg_attn_wide.hip): against float64, the appended rows against the RoPE kernel's
bits, and its forms against each other, at the edges of its row tiles, key
chunks, groups and own-key trips."""

import pytest
import torch

pytestmark = pytest.mark.gpu

TDT = {"bf16": torch.bfloat16, "f16": torch.float16}
HALF = {"bf16": 2.0**-8, "f16": 2.0**-11}  # half an ulp, relative to the value

CASES = [  # (rows, group, H, prefix, cached own keys, spare capacity)
    (1616, 16, 8, 16, 0, 1),    # whole tiles, no own key: the new one alone
    (442, 17, 8, 63, 1, 3),     # every second tile of one row
    (600, 100, 8, 64, 15, 10),
    (560, 32, 8, 65, 16, 10),   # ragged last group, whole tiles
    (105, 20, 8, 500, 33, 20),  # ragged last group inside a tile
    (160, 16, 8, 513, 100, 30),
    (66, 33, 5, 1031, 7, 5),
    (20, 32, 16, 1100, 40, 2),  # fewer rows than a group
    (20, 32, 16, 1068, 40, 2),  # the first prefix below the line: the vector kernel
    (17, 17, 1, 63, 1, 3),
]
VECTOR_CASES = CASES[-2:]


def _case(dev, dtype, D, case, seed=0):
    from diff_gpt.model.rope import precompute_freqs_cis

    B, G, H, P, own, spare = case
    dt, groups, cap = TDT[dtype], (B + G - 1) // G, P + own + 1 + spare
    g = torch.Generator(device=dev).manual_seed(seed + P + own)
    r = lambda *s: torch.randn(*s, generator=g, device=dev)  # noqa: E731
    unit = lambda x: torch.nn.functional.normalize(x, dim=-1) * D**0.5  # noqa: E731
    pages = torch.stack((unit(r(groups, H, P, D)), r(groups, H, P, D))).to(dt)
    rows = torch.full((2, B, H, cap - P, D), float("nan"), dtype=dt, device=dev)  # unwritten positions
    rows[0, :, :, :own], rows[1, :, :, :own] = unit(r(B, H, own, D)).to(dt), r(B, H, own, D).to(dt)
    qkv = (r(B, 1, 3, H, D) * 2).to(dt)
    table = precompute_freqs_cis(D, 2 * cap, 10000.0).to(dev)
    return pages, rows, [qkv[:, :, i] for i in range(3)], table, P + own


def _step(pages, rows, qkv, table, pos, case, device_pos=False):
    from diff_gpt import _native

    q, k, v = qkv
    P = case[3]
    y = torch.empty_like(q.contiguous())
    pre = _native.Prefix(P, case[1], pages[0].transpose(1, 2), pages[1].transpose(1, 2), P)
    p, f = (torch.tensor([pos], dtype=torch.int32, device=q.device), table) if device_pos else (pos, table[pos])
    _native.decode_step_(q, k, v, f, rows[0].transpose(1, 2), rows[1].transpose(1, 2), y, q.size(-1) ** -0.5, p,
                         prefix=pre)
    return y


@pytest.mark.parametrize("f32_table", [False, True])
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_wide_step(dev, dtype, D, case, f32_table):
    """y within half an ulp of the type plus 2e-5 (fp32 probabilities and sums) of
    the largest value, of float64 attention over the rotated query; cache rows the
    RoPE kernel's bits, nothing else written; host and device positions, prefix
    pages and broadcast rows alike."""
    from diff_gpt import _native

    B, G, H, P, own, spare = case
    pages, rows, qkv, table, pos = _case(dev, dtype, D, case)
    if not f32_table:
        table = table.to(TDT[dtype])
    before = rows.clone()
    y = _step(pages, rows, qkv, table, pos, case)
    assert (_native.last_kernel() == "attn_wide_kernel") == (case not in VECTOR_CASES)
    q_rot, k_rot = (torch.empty(B, 1, H, D, dtype=TDT[dtype], device=dev) for _ in range(2))
    _native.rope_qknorm_append_(qkv[0], qkv[1], None, table[pos].view(1, 1, 1, D // 2, 2), q_rot, k_rot, None, True)
    assert torch.equal(rows[0, :, :, own], k_rot[:, 0]) and torch.equal(rows[1, :, :, own], qkv[2][:, 0])
    others = [i for i in range(rows.size(3)) if i != own]
    assert torch.equal(rows[:, :, :, others].nan_to_num(5.0), before[:, :, :, others].nan_to_num(5.0))
    group = torch.arange(B, device=dev) // G
    keys, vals = (torch.cat((pages[i][group], rows[i][:, :, : own + 1]), dim=2).double() for i in (0, 1))
    s = (keys @ q_rot[:, 0].double().unsqueeze(-1)).squeeze(-1) * D**-0.5
    ref = (s.softmax(-1).unsqueeze(-2) @ vals).squeeze(-2)
    err = (y[:, 0].double() - ref).abs()
    assert bool((err <= HALF[dtype] * ref.abs() + 2e-5 * vals.abs().max()).all())

    rows2 = before.clone()
    assert torch.equal(_step(pages, rows2, qkv, table, pos, case, device_pos=True), y)
    assert (_native.last_kernel() == "attn_wide_kernel") == (case not in VECTOR_CASES)
    assert torch.equal(rows2.nan_to_num(5.0), rows.nan_to_num(5.0))
    # the prefix in every row instead of pages of its own
    dense = torch.cat((pages[:, group], before), dim=3)
    y3 = torch.empty_like(y)
    _native.decode_step_(*qkv, table[pos], dense[0].transpose(1, 2), dense[1].transpose(1, 2), y3, D**-0.5, pos, P, G)
    assert torch.equal(y3, y)
    # a device position outside the pages writes nothing
    rows4 = before.clone()
    for bad in (P - 1, rows.size(3) + P):
        _step(pages, rows4, qkv, table, bad, case, device_pos=True)
    torch.cuda.synchronize()
    assert torch.equal(rows4.nan_to_num(5.0), before.nan_to_num(5.0))


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("D", [64, 128])
def test_wide_step_values_not_finite(dev, dtype, D):
    """An infinity or a NaN among the prefix's values gives float64 attention's
    infinity or NaN in its column, whatever the rounding error of its probability
    (every row of the group weighs it by another), and the other columns what they
    have without it; opposite infinities in one column give NaN."""
    from diff_gpt import _native

    case = (400, 100, 8, 1024, 40, 56)
    B, G, H, P, own, spare = case
    pages, rows, qkv, table, pos = _case(dev, dtype, D, case)
    inf = float("inf")
    clean = _step(pages, rows.clone(), qkv, table, pos, case)
    for grp, h, t, d, x in [(0, 0, 5, 3, inf), (1, 2, 77, 9, -inf), (2, 1, 3, 1, float("nan")),
                            (3, 7, 1023, D - 1, inf), (3, 4, 600, 20, inf), (3, 4, 601, 20, -inf),
                            (0, 5, 0, 0, inf), (0, 5, 64, 0, inf)]:
        pages[1, grp, h, t, d] = x
    y = _step(pages, rows, qkv, table, pos, case)
    assert _native.last_kernel() == "attn_wide_kernel"
    q_rot, k_rot = (torch.empty(B, 1, H, D, dtype=TDT[dtype], device=dev) for _ in range(2))
    _native.rope_qknorm_append_(qkv[0], qkv[1], None, table[pos].view(1, 1, 1, D // 2, 2), q_rot, k_rot, None, True)
    group = torch.arange(B, device=dev) // G
    keys, vals = (torch.cat((pages[i][group], rows[i][:, :, : own + 1]), dim=2).double() for i in (0, 1))
    p = ((keys @ q_rot[:, 0].double().unsqueeze(-1)).squeeze(-1) * D**-0.5).softmax(-1)
    bad = (p.unsqueeze(-1) * (vals - vals.nan_to_num(0.0, 0.0, 0.0))).sum(-2)  # inf, -inf, NaN or 0
    finite = bad == 0
    assert int((~finite).sum()) == 6 * G
    kinds = lambda x: x.float().nan_to_num(7.0, 8.0, 9.0)  # noqa: E731
    assert torch.equal(kinds(y[:, 0][~finite]), kinds(bad[~finite]))
    assert torch.equal(y[:, 0][finite], clean[:, 0][finite])


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("own", [1, 41, 43, 44])  # the last slot holds one key, some or all it can
def test_wide_step_own_values_not_finite(dev, dtype, D, own):
    """The same for the values of a row's own keys, the newest cached one and the
    new one among them: the infinity or NaN reaches its row and column alone."""
    from diff_gpt import _native

    case = (400, 100, 8, 1024, own, 50)
    B, G, H, P, _, _ = case
    pages, rows, qkv, table, pos = _case(dev, dtype, D, case)
    clean = _step(pages, rows.clone(), qkv, table, pos, case)
    assert _native.last_kernel() == "attn_wide_kernel"
    inf = float("inf")
    hit = torch.full((B, H, D), 0.0, device=dev)
    for b, h, t, d, x in [(0, 0, own - 1, 3, inf), (17, 3, own - 1, 5, -inf), (33, 7, 0, 9, inf), (399, 1, own - 1, D - 1, inf),
                          (200, 2, own // 2, 4, float("nan")), (55, 6, own, 7, -inf)]:
        if t < own:
            rows[1, b, h, t, d] = x
        else:
            qkv[2][b, 0, h, d] = x
        hit[b, h, d] = x
    y = _step(pages, rows, qkv, table, pos, case)[:, 0].float()
    kinds = lambda t: t.nan_to_num(7.0, 8.0, 9.0)  # noqa: E731
    bad = ~hit.isfinite()
    assert torch.equal(kinds(y[bad]), kinds(hit[bad]))
    assert torch.equal(y[~bad], clean[:, 0].float()[~bad])


def test_wide_step_large_scores(dev):
    """Queries and keys that are not normalised: scores of several hundred, the
    maximum raised chunk after chunk.  Their fp32 sums are off by up to some
    2^-24 * 64 * 600, and a probability by as much."""
    from diff_gpt import _native

    D, case = 64, (40, 40, 16, 700, 20, 2)
    pages, rows, qkv, table, pos = _case(dev, "bf16", D, case)
    pages[0] *= torch.linspace(0.1, 20, case[3], device=dev).view(-1, 1).to(pages.dtype)
    qkv[0].mul_(10)
    y = torch.empty(40, 1, 16, D, dtype=torch.bfloat16, device=dev)
    pre = _native.Prefix(700, 40, pages[0].transpose(1, 2), pages[1].transpose(1, 2), 700)
    _native.decode_step_(*qkv, table[pos], rows[0].transpose(1, 2), rows[1].transpose(1, 2), y, D**-0.5, pos,
                         qknorm=False, prefix=pre)
    assert _native.last_kernel() == "attn_wide_kernel"
    q_rot = torch.empty_like(y)
    _native.rope_qknorm_append_(qkv[0], None, None, table[pos].view(1, 1, 1, D // 2, 2), q_rot, None, None, False)
    keys, vals = (torch.cat((pages[i].expand(40, -1, -1, -1), rows[i][:, :, :21]), dim=2).double() for i in (0, 1))
    s = (keys @ q_rot[:, 0].double().unsqueeze(-1)).squeeze(-1) * D**-0.5
    ref = (s.softmax(-1).unsqueeze(-2) @ vals).squeeze(-2)
    assert s.max() > 300
    assert bool(((y[:, 0].double() - ref).abs() <= HALF["bf16"] * ref.abs() + 5e-3 * vals.abs().max()).all())
