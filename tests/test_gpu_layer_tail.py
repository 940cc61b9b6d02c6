"""Launches joined at few rows (dg_layer.hip): dg_embed_in, dg_block_out_in and
dg_block_out_head against the separate launches, bit for bit, and GPT.forward
with and without them."""

import pytest
import torch

from diff_gpt.model.block import Block
from diff_gpt.model.rms_norm import rms_norm

pytestmark = pytest.mark.gpu

TDT = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}


def _rand(seed, dev, dt, *shape, scale=1.0):
    g = torch.Generator(device=dev).manual_seed(seed)
    return (torch.randn(*shape, generator=g, device=dev) * scale).to(dt)


def _layer(M, C, nblk, dt, dev):
    r = lambda seed, *s, scale=1.0: _rand(seed, dev, dt, *s, scale=scale)  # noqa: E731
    blocks = [r(20 + i, M, C, scale=0.5 + 0.1 * i) for i in range(nblk)]
    if nblk > 1:
        blocks[1] = blocks[0]
    w = dict(proj=r(1, C, C, scale=C**-0.5), mix=r(2, 1, C, scale=4 * C**-0.5), up=r(3, 4 * C, C, scale=2 * C**-0.5),
             down=r(4, C, 2 * C, scale=C**-0.5))
    return r(5, M, C), r(6, M, 4 * C)[:, 3 * C :], r(7, M, C), blocks, w


@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("C", [64, 128])
@pytest.mark.parametrize("M,nblk,pin", [(1, 1, False), (16, 3, True), (17, 2, False), (100, 8, True), (333, 9, False),
                                        (40, 31, False), (5000, 3, False)])
def test_block_out_with_what_follows(dev, dtype, C, M, nblk, pin):
    from diff_gpt import _native

    if dtype == "f32" and C == 128:
        pytest.skip("declined: test_block_out_leaves_other_tails_undone")
    dt = TDT[dtype]
    y, g, p, blocks, w = _layer(M, C, nblk, dt, dev)
    args = (y, g, w["proj"], p if pin else None, blocks, w["mix"], w["up"], w["down"], 1.702, 7.0)
    out, xn = torch.empty(M, C, dtype=dt, device=dev), torch.empty(M, C, dtype=dt, device=dev)
    assert _native.block_out_(*args, out, xn)
    # the next layer's projections
    mix, wq = _rand(8, dev, dt, 1, C, scale=4 * C**-0.5), _rand(9, dev, dt, 4 * C, C, scale=C**-0.5)
    qkvg = torch.empty(M, 4 * C, dtype=dt, device=dev)
    assert _native.block_in_([*blocks, out], mix, wq, qkvg)
    tail = _native.Tail(mix, wq, torch.full_like(qkvg, 3.0))
    out2 = torch.empty_like(out)
    assert _native.block_out_(*args, out2, tail=tail) and tail.done
    assert torch.equal(out2, out) and torch.equal(tail.out, qkvg)
    # the head, with and without a cap, the norm and the ids
    for V, cap in ((64, 15.0), (256, 15.0), (256, 0.0), (1024, 3.0)):
        table = _rand(V, dev, dt, V, C)
        table[V // 2] = table[3]  # equal logits: the first wins
        logits, ids = torch.empty(M, V, dtype=dt, device=dev), torch.empty(M, dtype=torch.int64, device=dev)
        assert _native.lm_head_(xn, table, cap, logits, ids)
        tail = _native.Tail(None, table, torch.empty_like(logits), cap, torch.empty_like(ids))
        out3, xn3 = torch.empty_like(out), torch.empty_like(xn)
        assert _native.block_out_(*args, out3, xn3, tail=tail) and tail.done
        assert torch.equal(out3, out) and torch.equal(xn3, xn)
        assert torch.equal(tail.out, logits) and torch.equal(tail.ids, ids)
        plain = _native.Tail(None, table, torch.empty_like(logits), cap)
        assert _native.block_out_(*args, out3, tail=plain) and plain.done
        assert torch.equal(plain.out, logits)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_pseudo_queries_with_a_stride(dev, dtype):
    """Pseudo-queries that are columns of another tensor are copied for the launch,
    each into memory of its own."""
    from diff_gpt import _native

    C, dt = 64, TDT[dtype]
    y, g, _, blocks, w = _layer(20, C, 3, dt, dev)
    mixes = [_rand(i, dev, dt, 1, C, scale=4 * C**-0.5) for i in (11, 12)]
    wq = _rand(9, dev, dt, 4 * C, C, scale=C**-0.5)
    results = []
    for strided in (False, True):
        mix, t_mix = (_rand(1, dev, dt, C, 3).copy_(m.view(C, 1).expand(C, 3))[:, 1:2].T if strided else m for m in mixes)
        assert mix.is_contiguous() != strided
        out, tail = torch.empty(20, C, dtype=dt, device=dev), _native.Tail(t_mix, wq)
        assert _native.block_out_(y, g, w["proj"], None, blocks, mix, w["up"], w["down"], 1.702, 7.0, out, tail=tail)
        results.append((out, tail.out))
    assert all(torch.equal(a, b) for a, b in zip(*results))


def test_block_out_leaves_other_tails_undone(dev):
    """A vocabulary that the head does not take, a table without unit stride,
    fp32 at n_embd 128: the layer alone."""
    from diff_gpt import _native

    for table in (_rand(1, dev, torch.float32, 96, 64), _rand(1, dev, torch.float32, 64, 256).T,
                  _rand(1, dev, torch.float32, 256, 128)):
        C = table.size(1)
        y, g, _, blocks, w = _layer(20, C, 2, torch.float32, dev)
        args = (y, g, w["proj"], None, blocks, w["mix"], w["up"], w["down"], 1.702, 7.0)
        out, out2 = torch.empty(20, C, device=dev), torch.empty(20, C, device=dev)
        assert _native.block_out_(*args, out)
        tail = _native.Tail(None, table, torch.full((20, table.size(0)), 3.0, device=dev))
        assert _native.block_out_(*args, out2, tail=tail)
        assert not tail.done and bool((tail.out == 3.0).all()) and torch.equal(out2, out)


@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("C", [64, 128])
@pytest.mark.parametrize("M", [1, 16, 17, 100, 5000])
def test_embed_in_is_the_two_launches(dev, dtype, C, M):
    from diff_gpt import _native

    dt, V = TDT[dtype], 96
    table, w = _rand(1, dev, dt, V, C), _rand(2, dev, dt, 4 * C, C, scale=C**-0.5)
    ids = torch.randint(0, V, (M,), generator=torch.Generator().manual_seed(3)).to(dev)
    ids[M // 2] = V if M > 1 else 5  # outside: a NaN row
    ids[M // 3] = -1 if M > 16 else 7
    x, xn, x2 = (torch.empty(M, C, dtype=dt, device=dev) for _ in range(3))
    q, q2 = (torch.empty(M, 4 * C, dtype=dt, device=dev) for _ in range(2))
    assert _native.embed_norm_(ids, table, x, xn) and _native.block_in_([xn], None, w, q)
    assert _native.embed_norm_(ids, table, x2, None, w, q2)
    bits = {4: torch.int32, 2: torch.int16}[x.element_size()]
    assert torch.equal(x.isnan(), x2.isnan()) and torch.equal(q.isnan(), q2.isnan())
    assert torch.equal(x.nan_to_num(9.0).view(bits), x2.nan_to_num(9.0).view(bits))
    assert torch.equal(q.nan_to_num(9.0).view(bits), q2.nan_to_num(9.0).view(bits))


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("embd,layers_per_block", [(64, 1), (64, 2), (128, 1)])
def test_gpt_with_joined_launches(dev, dtype, embd, layers_per_block, monkeypatch):
    """Logits, argmax, the last position's logits and a decode step: the bits of
    the launches one by one.  A hook on a block keeps its place."""
    from diff_gpt.model import gpt
    from diff_gpt.model.kv_cache import KVCache

    torch.manual_seed(0)
    model = gpt.GPT(vocab_size=128, n_embd=embd, block_size=32, n_head=4, n_layer=3, use_checkpoint=False,
                    attn_res_layers_per_block=layers_per_block).eval().to(dev).to(TDT[dtype])
    idx = torch.randint(0, 128, (3, 17), generator=torch.Generator().manual_seed(4)).to(dev)

    def run():
        kv = KVCache(batch_size=3, num_heads=4, seq_len=18, head_dim=embd // 4, num_layers=3)
        am, am1 = (torch.empty(3, t, dtype=torch.int64, device=dev) for t in (17, 1))
        with torch.inference_mode():
            first = model(idx, kv_cache=kv, _argmax_out=am)[0]
            step = model(am[:, -1:], kv_cache=kv)[0]
            last = model(idx, _last_only=True, _argmax_out=am1)[0]
        return first, am, step, last, am1

    joined = run()
    hook = model.blocks[1].register_forward_hook(lambda m, i, o: (o[0], o[1] * 2))
    hooked = run()
    monkeypatch.setattr(gpt.GPT, "_joins", lambda self, rows: False)
    hooked_apart = run()
    hook.remove()
    apart = run()
    assert all(torch.equal(a, b) for a, b in zip(joined, apart))
    assert all(torch.equal(a, b) for a, b in zip(hooked, hooked_apart))
    assert not torch.equal(hooked[0], joined[0])


class _Doubled(Block):
    """A layer with a forward of its own, of the arguments a Block took before
    launches were joined."""

    def forward(self, blocks, partial_block, freqs_cis, kv_cache, *, _last_only=False, _xn=None, _xn_out=None):
        blocks, out = super().forward(blocks, partial_block, freqs_cis, kv_cache, _last_only=_last_only, _xn=_xn)
        out = out * 2
        if _xn_out is not None:
            _xn_out.copy_(rms_norm(out))
        return blocks, out


@pytest.mark.parametrize("embd", [64, 128])
@pytest.mark.parametrize("layer", [0, 1, 2])
def test_an_overridden_layer_is_heard(dev, embd, layer, monkeypatch):
    """A layer's output replaced by a subclass, by a forward put into the instance
    or the class, or by a hook on all modules is what the next layer and the head
    read, as it is with a hook on the layer (whose head reads the last layer's
    norm by way of _xn_out, so only the next layer's input shows there)."""
    from torch.nn.modules.module import register_module_forward_hook

    from diff_gpt.model import gpt

    def build():
        torch.manual_seed(0)
        return gpt.GPT(vocab_size=128, n_embd=embd, block_size=32, n_head=4, n_layer=3,
                       use_checkpoint=False).eval().to(dev).to(torch.bfloat16)

    idx = torch.randint(0, 128, (3, 17), generator=torch.Generator().manual_seed(4)).to(dev)

    @torch.inference_mode()
    def logits(model):
        return model(idx)[0]

    plain = logits(build())
    model = build()
    model.blocks[layer].__class__ = _Doubled
    doubled = logits(model)
    assert not torch.equal(doubled, plain) or layer == 2  # 2 x keeps the head's norm but for its epsilon
    model = build()
    with monkeypatch.context() as m:
        m.setattr(gpt.GPT, "_joins", lambda self, rows: False)
        model.blocks[layer].__class__ = _Doubled
        assert torch.equal(logits(model), doubled)
    # the same by an instance's forward
    model = build()
    block = model.blocks[layer]
    inner = Block.forward

    def doubling(blocks, partial_block, freqs_cis, kv_cache, *, _last_only=False, _xn=None, _xn_out=None):
        blocks, out = inner(block, blocks, partial_block, freqs_cis, kv_cache, _last_only=_last_only, _xn=_xn)
        out = out * 2
        if _xn_out is not None:
            _xn_out.copy_(rms_norm(out))
        return blocks, out

    block.forward = doubling
    assert torch.equal(logits(model), doubled)
    del block.forward
    assert torch.equal(logits(model), plain)
    # by the class's, and by a hook on all modules
    if layer < 2:
        hook = block.register_forward_hook(lambda mod, i, o: (o[0], o[1] * 2))
        hooked = logits(model)
        hook.remove()
        assert torch.equal(hooked, doubled)
        with monkeypatch.context() as m:
            m.setattr(Block, "forward",
                      lambda self, *a, **k: (lambda o: (o[0], o[1] * 2) if self is block else o)(inner(self, *a, **k)))
            assert torch.equal(logits(model), doubled)
        hook = register_module_forward_hook(lambda mod, i, o: (o[0], o[1] * 2) if mod is block else None)
        try:
            assert torch.equal(logits(model), doubled)
        finally:
            hook.remove()
    assert torch.equal(logits(model), plain)


def test_a_joined_head_stores_no_norm(dev, monkeypatch):
    """With the head in the last layer's launch the norm of its rows goes nowhere;
    a head of its own launch reads it from memory."""
    from diff_gpt import _native
    from diff_gpt.model import gpt

    torch.manual_seed(0)
    idx = torch.randint(0, 128, (3, 17), generator=torch.Generator().manual_seed(4)).to(dev)
    lib, stored = _native.lib(), []
    for name in ("dg_block_out_head", "dg_block_out_norm"):
        real = getattr(lib, name)
        xn = 23  # the argument after out and its row stride
        monkeypatch.setattr(lib, name, lambda *a, real=real: (stored.append(a[xn].value is not None), real(*a))[1])
    for vocab, norm in ((128, False), (192, True)):
        model = gpt.GPT(vocab_size=vocab, n_embd=64, block_size=32, n_head=4, n_layer=2).eval().to(dev)
        for last_only in (False, True):
            stored.clear()
            with torch.inference_mode():
                model(idx, _last_only=last_only)
            assert stored == [norm]


@pytest.mark.parametrize("vocab", [1536, 1024])
def test_logits_are_allocated_once(dev, vocab, monkeypatch):
    """Peak memory of a forward with joined launches: no second (B, T, V) beside
    the logits, whether the layer's launch takes the head or not."""
    from diff_gpt.model import gpt

    torch.manual_seed(0)
    model = gpt.GPT(vocab_size=vocab, n_embd=64, block_size=64, n_head=4, n_layer=2).eval().to(dev)
    idx = torch.randint(0, vocab, (256, 64), generator=torch.Generator().manual_seed(4)).to(dev)
    logits_bytes = idx.numel() * vocab * 4

    @torch.inference_mode()
    def peak():
        model(idx)
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        model(idx)
        torch.cuda.synchronize()
        return torch.cuda.max_memory_allocated() - before

    joined = peak()
    monkeypatch.setattr(gpt.GPT, "_joins", lambda self, rows: False)
    assert joined < peak() + logits_bytes // 2


def test_an_overridden_head_is_heard(dev):
    from diff_gpt.model import gpt

    class Halved(gpt.GPT):
        def _head(self, partial, argmax_out, xn=None):
            return super()._head(partial, argmax_out, xn) * 0.5

    torch.manual_seed(0)
    model = gpt.GPT(vocab_size=128, n_embd=64, block_size=32, n_head=4, n_layer=2).eval().to(dev)
    idx = torch.randint(0, 128, (3, 17), generator=torch.Generator().manual_seed(4)).to(dev)
    with torch.inference_mode():
        full = model(idx)[0]
        model.__class__ = Halved
        assert torch.equal(model(idx)[0], full * 0.5)


def test_a_captured_step_of_an_overridden_model(dev):
    """A forward put into the model's instance, of the arguments GPT.forward took
    before the head's launch could advance the position, is captured as it is."""
    from diff_gpt.model import gpt
    from diff_gpt.model.engine import Engine
    from diff_gpt.sampler.temperature import TemperatureSampler

    torch.manual_seed(0)
    model = gpt.GPT(vocab_size=128, n_embd=64, block_size=32, n_head=4, n_layer=2).eval().to(dev)
    inner = model.forward

    def forward(idx, targets=None, kv_cache=None, *, _argmax_out=None, _last_only=False):
        logits, loss = inner(idx, targets, kv_cache, _argmax_out=_argmax_out, _last_only=_last_only)
        return -logits, loss

    def tokens(use_graph):
        return Engine(model, use_graph=use_graph).generate_batch([1, 2, 3], num_samples=4, max_tokens=6,
                                                                 sampler=TemperatureSampler(0.0))

    plain = tokens(True)
    model.forward = forward
    assert tokens(True) == tokens(False) != plain


def test_head_advances_the_position(dev):
    """A device position moves on by one with the head's launch, at one
    workgroup and at many; the layer without a joined head adds it itself."""
    from diff_gpt import _native

    for M in (1, 100, 5000):
        y, g, _, blocks, w = _layer(M, 64, 2, torch.float32, dev)
        out, pos = torch.empty(M, 64, device=dev), torch.tensor([41, 7], dtype=torch.int32, device=dev)
        table = _rand(1, dev, torch.float32, 256, 64)
        tail = _native.Tail(None, table, torch.empty(M, 256, device=dev), 15.0, advance=pos)
        assert _native.block_out_(y, g, w["proj"], None, blocks, w["mix"], w["up"], w["down"], 1.702, 7.0, out, tail=tail)
        assert pos.tolist() == [42, 7]


@pytest.mark.parametrize("vocab", [128, 192])  # 192: no joined head
def test_step_advances_the_cache(dev, vocab):
    from diff_gpt.model import gpt
    from diff_gpt.model.kv_cache import KVCache

    torch.manual_seed(0)
    model = gpt.GPT(vocab_size=vocab, n_embd=64, block_size=32, n_head=4, n_layer=2, use_checkpoint=False).eval().to(dev)
    kv = KVCache(batch_size=3, num_heads=4, seq_len=20, head_dim=16, num_layers=2)
    ids = torch.randint(0, vocab, (3, 9), generator=torch.Generator().manual_seed(4)).to(dev)
    with torch.inference_mode():
        model(ids, kv_cache=kv)
        kv.pos_dev = torch.tensor([9], dtype=torch.int32, device=dev)
        model(ids[:, :1], kv_cache=kv, _advance=True)
        assert kv.pos_dev.item() == 10
        kv.pos = 10
        model(ids[:, :1], kv_cache=kv)
        assert kv.pos_dev.item() == 10
