"""Timing cases of the framework: the work its users have it do, over the real range of sizes.

Each case is a dict of plain values.  ``kind`` says which path it takes:

  gpt_step     GPT.forward over one new token per row, captured once and replayed, as a
               decode loop replays it (rows of unrelated prompts)
  engine       one Engine.generate_batch call: prefill of one prompt, then num_samples
               trajectories, the logits of every step recorded by the sampler
  gpt_score    GPT.forward over whole windows, logits of every position (scoring, and the
               sliding-window sampler's forward)
  block_step   one Block over one new token per row, captured and replayed; the rows either
               have caches of their own (samples = 1) or share their prompt's (samples > 1)
  block_prefill  one Block over whole prompts into a KV cache, from position ``past`` on
  mha_prefill  one MultiHeadAttention over whole prompts, without a cache
"""

import math
import sys
from pathlib import Path

import torch

_PKG = str(Path(__file__).resolve().parent.parent / "diff-gpt_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from diff_gpt.model.block import Block  # noqa: E402
from diff_gpt.model.engine import Engine  # noqa: E402
from diff_gpt.model.gpt import GPT  # noqa: E402
from diff_gpt.model.kv_cache import KVCache  # noqa: E402
from diff_gpt.model.mha import MultiHeadAttention  # noqa: E402
from diff_gpt.model.rope import precompute_freqs_cis  # noqa: E402
from diff_gpt.sampler.sampler import Sampler  # noqa: E402

_DEV = "cuda"
_THETA, _ALPHA, _LIMIT, _CAP = 10000.0, 1.702, 7.0, 15.0
_DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}
_BYTES = {"f32": 4, "bf16": 2}


def listed():
    return [
        # 32 sequences of the small model, one greedy decode step: the smallest call of a
        # decode loop, bound by latency
        dict(name="gpt_step_f32", kind="gpt_step", rows=32, prompt=119, embd=64, heads=4, layers=2, vocab=256,
             dtype="f32"),
        # one series forecast by 100 trajectories of 48 tokens after a 96-token prompt
        dict(name="engine_series_f32", kind="engine", samples=100, prompt=96, steps=48, embd=64, heads=4, layers=2,
             vocab=256, dtype="f32"),
        # 256 windows of 138 tokens (half the small model's RoPE table) scored in one forward
        dict(name="gpt_score_f32", kind="gpt_score", batch=256, tokens=138, embd=64, heads=4, layers=2, vocab=256,
             dtype="f32"),
        # a decode step's layer over 64 series x 100 trajectories, halfway through 48 new tokens
        dict(name="step_series_f32", kind="block_step", prompts=64, samples=100, prefix=96, own=24, room=48, embd=64,
             heads=4, layer=1, dtype="f32"),
        # the same in bf16 with counts that divide nothing
        dict(name="step_series_bf16", kind="block_step", prompts=37, samples=50, prefix=131, own=17, room=48, embd=64,
             heads=4, layer=1, dtype="bf16"),
        # 512 unrelated rows, head_dim 64, in the middle of 512 new tokens after 1024
        dict(name="step_rows_bf16", kind="block_step", prompts=512, samples=1, prefix=1024, own=271, room=512,
             embd=512, heads=8, layer=4, dtype="bf16"),
        # 64 unrelated rows, head_dim 128, long prompts
        dict(name="step_long_bf16", kind="block_step", prompts=64, samples=1, prefix=3584, own=48, room=96, embd=1024,
             heads=8, layer=2, dtype="bf16"),
        # the wider model forecasting 4 series by 100 trajectories each
        dict(name="step_samples_bf16", kind="block_step", prompts=4, samples=100, prefix=1024, own=40, room=96,
             embd=512, heads=8, layer=4, dtype="bf16"),
        # a middle layer of the wider model over 64 prompts of 1024 tokens
        dict(name="prefill_bf16", kind="block_prefill", batch=64, tokens=1024, past=0, embd=512, heads=8, layer=4,
             dtype="bf16"),
        # a layer of the widest model over 8 prompts of 3584 tokens
        dict(name="prefill_long_bf16", kind="block_prefill", batch=8, tokens=3584, past=0, embd=1024, heads=8,
             layer=2, dtype="bf16"),
        # the reference's default type at the wider model's geometry, ragged length
        dict(name="prefill_f32", kind="block_prefill", batch=16, tokens=1000, past=0, embd=512, heads=8, layer=4,
             dtype="f32"),
        # the attention sub-layer alone over 256 prompts of 1024 tokens
        dict(name="mha_prefill_bf16", kind="mha_prefill", batch=256, tokens=1024, embd=512, heads=8, dtype="bf16"),
    ]


def _spread(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm; odd more often than not."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(lo, min(hi, n | 1 if rng.random() < 0.6 else n))


def draw(rng):
    kind = rng.choice(["gpt_step", "engine", "gpt_score", "series", "series", "rows", "long", "samples", "samples",
                       "prefill_small", "prefill", "prefill", "prefill_long", "prefill_f32", "mha_prefill"])
    small = dict(embd=64, heads=4) if rng.random() < 0.7 else dict(embd=128, heads=4)
    either = rng.choice(["f32", "bf16"])
    wide = rng.random() < 0.5
    if kind == "gpt_step":
        return dict(kind=kind, rows=_spread(rng, 1, 64), prompt=_spread(rng, 16, 250), layers=2, vocab=256,
                    dtype="f32", **small)
    if kind == "engine":
        return dict(kind=kind, samples=_spread(rng, 16, 100), prompt=_spread(rng, 32, 160),
                    steps=rng.randint(16, 48), embd=64, heads=4, layers=2, vocab=256, dtype="f32")
    if kind == "gpt_score":
        return dict(kind=kind, batch=_spread(rng, 16, 256), tokens=_spread(rng, 24, 138), layers=2, vocab=256,
                    dtype="f32", embd=64, heads=4)
    if kind == "series":
        room = rng.randint(16, 64)
        return dict(kind="block_step", prompts=_spread(rng, 2, 64), samples=_spread(rng, 16, 100),
                    prefix=_spread(rng, 32, 200), own=rng.randint(0, room - 1), room=room, layer=1, dtype=either,
                    **small)
    if kind == "rows":
        return dict(kind="block_step", prompts=_spread(rng, 32, 512), samples=1, prefix=_spread(rng, 128, 1024),
                    own=rng.randint(0, 255), room=256, embd=512, heads=8, layer=4, dtype="bf16")
    if kind == "long":
        return dict(kind="block_step", prompts=_spread(rng, 4, 64), samples=1, prefix=_spread(rng, 512, 3584),
                    own=rng.randint(0, 95), room=96, embd=1024, heads=8, layer=2, dtype="bf16")
    if kind == "samples":
        return dict(kind="block_step", prompts=_spread(rng, 1, 6), samples=_spread(rng, 20, 128),
                    prefix=_spread(rng, 200, 2000), own=rng.randint(0, 95), room=96, embd=1024 if wide else 512,
                    heads=8, layer=2, dtype="bf16")
    if kind == "prefill_small":
        return dict(kind="block_prefill", batch=_spread(rng, 32, 256), tokens=_spread(rng, 24, 200), past=0, layer=1,
                    dtype=either, **small)
    if kind == "prefill":
        tokens = _spread(rng, 64, 1024)
        past = rng.choice([0, 0, 0, _spread(rng, 16, 512)])
        return dict(kind="block_prefill", batch=_spread(rng, 2, 48), tokens=tokens, past=past, embd=512, heads=8,
                    layer=rng.randint(0, 5), dtype="bf16")
    if kind == "prefill_long":
        return dict(kind="block_prefill", batch=_spread(rng, 1, 6), tokens=_spread(rng, 512, 3584), past=0,
                    embd=1024, heads=8, layer=rng.randint(0, 3), dtype="bf16")
    if kind == "prefill_f32":
        return dict(kind="block_prefill", batch=_spread(rng, 1, 12), tokens=_spread(rng, 64, 1000), past=0, embd=512,
                    heads=8, layer=rng.randint(0, 5), dtype="f32")
    return dict(kind="mha_prefill", batch=_spread(rng, 4, 200), tokens=_spread(rng, 64, 1024),
                embd=1024 if wide and rng.random() < 0.3 else 512, heads=8, dtype="bf16")


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------


def _gen(seed):
    g = torch.Generator(device=_DEV)
    g.manual_seed(seed)
    return g


def _randn(g, *shape, dtype=torch.float32, scale=1.0):
    x = torch.empty(shape, dtype=dtype, device=_DEV).normal_(0.0, scale, generator=g)
    return x


def _unit_rows(x):
    """Rows of root mean square 1 in place: what the QK-norm leaves in a cache."""
    for part in x:  # one batch entry at a time bounds the temporary
        part.copy_(torch.nn.functional.normalize(part.float(), dim=-1) * math.sqrt(x.size(-1)))
    return x


def _seeded(seed, make):
    with torch.random.fork_rng(devices=[]):
        torch.manual_seed(seed)
        return make()


def _gpt(case, seed):
    model = _seeded(seed, lambda: GPT(vocab_size=case["vocab"], n_embd=case["embd"], block_size=138,
                                      n_head=case["heads"], n_layer=case["layers"], use_checkpoint=False))
    return model.eval().to(_DEV).to(_DTYPES[case["dtype"]])


def _block(case, seed):
    block = _seeded(seed, lambda: Block(n_embd=case["embd"], n_head=case["heads"], swiglu_alpha=_ALPHA,
                                        swiglu_limit=_LIMIT, layer_idx=case["layer"]))
    return block.eval().to(_DEV).to(_DTYPES[case["dtype"]])


def _states(case, g, *lead):
    """The committed blocks and the partial sum that enter layer ``layer`` of a model that
    commits after every layer: the normalised embedding (block 0, and committed once more by
    layer 0), then one partial sum per layer."""
    dtype, C = _DTYPES[case["dtype"]], case["embd"]
    x = _unit_rows(_randn(g, *lead, C)).to(dtype)
    if case["layer"] == 0:
        return (x,), x
    later = [_randn(g, *lead, C, scale=0.7).to(dtype) for _ in range(case["layer"])]
    return (x, x, *later[:-1]), later[-1]


def _table(case, end):
    return precompute_freqs_cis(case["embd"] // case["heads"], end, _THETA).to(_DEV).to(_DTYPES[case["dtype"]])


def _capture(step):
    """step() captured as a graph, as a decode loop captures it (warmed up on a side stream)."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    return graph, out


class _Teacher(Sampler):
    """Records the logits it is handed and answers with the tokens of a prepared table."""

    def __init__(self, table):
        self.table = table  # (steps, rows, 1)
        self.logits = []

    def __call__(self, logits, rng=None):
        self.logits.append(logits.clone())
        return self.table[len(self.logits) - 1]


@torch.no_grad()
def prepare(case, seed):
    g = _gen(seed)
    kind, H, C = case["kind"], case["heads"], case["embd"]
    D, dtype = C // H, _DTYPES[case["dtype"]]
    st = {"case": case}

    if kind == "gpt_step":
        B, P = case["rows"], case["prompt"]
        model = _gpt(case, seed)
        ids = torch.randint(0, case["vocab"], (B, P + 1), generator=g, device=_DEV)
        cache = KVCache(batch_size=B, num_heads=H, seq_len=P + 16, head_dim=D, num_layers=case["layers"])
        model.forward(ids[:, :P], kv_cache=cache)
        cache.pos_dev = torch.full((1,), P, dtype=torch.int32, device=_DEV)
        last = ids[:, P:].contiguous()

        def step():
            cache.pos = P
            logits, _ = model.forward(last, kv_cache=cache)
            rows = [r[:, P] for i in range(case["layers"]) for r in cache.decode_views(i)[:2]]
            return {"logits": logits, "cache_rows": rows}

        graph, out = _capture(step)
        st.update(model=model, ids=ids, cache=cache, last=last, graph=graph, out=out)
        return st

    if kind == "engine":
        model = _gpt(case, seed)
        tokens = torch.randint(0, case["vocab"], (case["prompt"],), generator=g, device=_DEV)
        table = torch.randint(0, case["vocab"], (case["steps"], case["samples"], 1), generator=g, device=_DEV)
        st.update(model=model, engine=Engine(model), tokens=tokens.tolist(), table=table)
        return st

    if kind == "gpt_score":
        ids = torch.randint(0, case["vocab"], (case["batch"], case["tokens"]), generator=g, device=_DEV)
        st.update(model=_gpt(case, seed), ids=ids)
        return st

    if kind == "mha_prefill":
        mha = _seeded(seed, lambda: MultiHeadAttention(n_embd=C, n_head=H, layer_idx=0)).eval().to(_DEV).to(dtype)
        B, T = case["batch"], case["tokens"]
        x = _unit_rows(_randn(g, B, T, C)).to(dtype)
        st.update(mha=mha, x=x, freqs=_table(case, T).view(1, T, 1, D // 2, 2))
        return st

    block = _block(case, seed)
    L = case["layer"] + 1
    if kind == "block_prefill":
        B, T, past = case["batch"], case["tokens"], case["past"]
        cache = KVCache(batch_size=B, num_heads=H, seq_len=past + T, head_dim=D, num_layers=L)
        table = _table(case, past + T)
        if past:  # what an earlier chunk of the prompt left in the cache
            blocks, partial = _states(case, g, B, past)
            block(blocks, partial, freqs_cis=table[:past].view(1, past, 1, D // 2, 2), kv_cache=cache)
        blocks, partial = _states(case, g, B, T)
        st.update(block=block, blocks=blocks, partial=partial, cache=cache,
                  freqs=table[past:].view(1, T, 1, D // 2, 2))
        return st

    # block_step
    G, S, P, own = case["prompts"], case["samples"], case["prefix"], case["own"]
    B, cap = G * S, P + case["room"]
    k = _unit_rows(_randn(g, G, H, P, D, dtype=dtype))
    v = _randn(g, G, H, P, D, dtype=dtype)
    kw = dict(num_heads=H, head_dim=D, num_layers=L)
    prompts = KVCache(batch_size=G, seq_len=P if S > 1 else cap, **kw)
    prompts.insert_kv(L - 1, k, v)
    cache = prompts
    if S > 1:  # every prompt's cache shared by its trajectories, as Engine lays it out
        cache = KVCache(batch_size=B, seq_len=cap, **kw)
        cache._prefill_groups(prompts, S)
    del prompts, k, v
    k_pages, v_pages, _ = cache.decode_views(L - 1)  # (B, positions, H, D) from own_start on
    first = P - cache.own_start
    if own:
        k_pages[:, first : first + own].copy_(_unit_rows(_randn(g, B, own, H, D, dtype=dtype)))
        v_pages[:, first : first + own].copy_(_randn(g, B, own, H, D, dtype=dtype))
    pos = P + own
    cache.pos = pos
    cache.pos_dev = torch.full((1,), pos, dtype=torch.int32, device=_DEV)
    table = _table(case, cap)
    blocks, partial = _states(case, g, B, 1)

    def step():
        cache.pos = pos
        _, out = block(blocks, partial, freqs_cis=table, kv_cache=cache)
        return {"out": out, "key": k_pages[:, first + own], "value": v_pages[:, first + own]}

    graph, out = _capture(step)
    st.update(block=block, blocks=blocks, partial=partial, cache=cache, freqs=table, graph=graph, out=out)
    return st


@torch.no_grad()
def run(state):
    kind = state["case"]["kind"]
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    if kind == "engine":
        teacher = _Teacher(state["table"])
        case = state["case"]
        rows, _ = state["engine"].generate_batch(state["tokens"], num_samples=case["samples"],
                                                 max_tokens=case["steps"], sampler=teacher)
        return {"logits": torch.stack(teacher.logits), "tokens": torch.tensor(rows)}
    if kind == "gpt_score":
        return state["model"].forward(state["ids"])[0]
    if kind == "mha_prefill":
        return state["mha"](state["x"], state["freqs"], None)
    cache, past = state["cache"], state["case"]["past"]
    cache.pos = past
    _, out = state["block"](state["blocks"], state["partial"], freqs_cis=state["freqs"], kv_cache=cache)
    keys, values = cache.layer_views(state["case"]["layer"], past + state["case"]["tokens"])
    return {"out": out, "keys": keys[:, :, past:], "values": values[:, :, past:]}


# ---------------------------------------------------------------------------
# work and tolerance
# ---------------------------------------------------------------------------


def _layer_work(rows, C, H, keys_per_row, key_bytes, es, sources):
    """One Block: its weights and sources read once, its output and new K/V written once; the
    projections, the attention over keys_per_row keys, the FFN."""
    weights = 5 * C * C + 6 * C * C + 2 * C
    nbytes = es * (weights + rows * C * (sources + 1 + 2)) + key_bytes
    flops = 2 * rows * C * (5 * C + 6 * C) + 4 * rows * C * keys_per_row
    return nbytes, flops


def work(case):
    C, H, es, kind = case["embd"], case["heads"], _BYTES[case["dtype"]], case["kind"]
    if kind == "mha_prefill":
        B, T = case["batch"], case["tokens"]
        return {"bytes": es * (2 * B * T * C + 5 * C * C + T * (C // H)),
                "flops": 2 * B * T * 5 * C * C + 2 * B * C * T * (T + 1)}
    if kind == "block_prefill":
        B, T, past = case["batch"], case["tokens"], case["past"]
        b, f = _layer_work(B * T, C, H, past + (T + 1) / 2, es * 2 * B * past * C, es, max(1, case["layer"] + 1))
        return {"bytes": int(b), "flops": int(f)}
    if kind == "block_step":
        G, S, P, own = case["prompts"], case["samples"], case["prefix"], case["own"]
        held = 2 * C * es * (G * P + G * S * own)
        b, f = _layer_work(G * S, C, H, P + own + 1, held, es, case["layer"] + 1)
        return {"bytes": int(b), "flops": int(f)}
    L, V = case["layers"], case["vocab"]
    weights = es * (L * (11 * C * C + 2 * C) + V * C)
    per_token = 2 * (L * 11 * C * C)
    if kind == "gpt_step":
        B, P = case["rows"], case["prompt"]
        return {"bytes": weights + es * (B * (2 * L * C * (P + 1) + V)),
                "flops": B * (per_token + 2 * V * C + 4 * L * C * (P + 1))}
    if kind == "gpt_score":
        B, T = case["batch"], case["tokens"]
        return {"bytes": weights + B * T * (8 + es * V),
                "flops": B * T * (per_token + 2 * V * C + 2 * L * C * (T + 1))}
    P, N, S = case["prompt"], case["steps"], case["samples"]
    forwards = N - 1  # the last column's logits are not computed
    keys = sum(P + s + 1 for s in range(forwards))
    own = sum(s + 1 for s in range(forwards))
    return {"bytes": N * weights + es * 2 * L * C * (forwards * P + S * own) + N * S * (V * es + 8),
            "flops": P * (per_token + 2 * L * C * (P + 1)) + forwards * S * (per_token + 2 * V * C) + 4 * L * C * S * keys}


def tolerance(case):
    # Against 64 bits the paths measure, relative / largest: fp32 8e-7 / 6e-6 (a layer of n_embd
    # 512) and 3.4e-7 / 3e-6 (the small model), bf16 5.9e-3 / 3.6e-2 (a layer) and 5.1e-3 / 0.13
    # (the attention sub-layer, whose sums of many values are small).  Two correct forms differ by
    # the roundings of both.
    if case["dtype"] == "f32":
        return {"rel": 4e-6, "max": 4e-5}
    return {"rel": 1.2e-2, "max": 0.4 if case["kind"] == "mha_prefill" else 0.15}


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------


def _rms64(x):
    return x * torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + torch.finfo(torch.float32).eps)


def _rope64(x, table):
    """x (B, T, H, D), table (T, D/2, 2)."""
    re, im = x[..., 0::2], x[..., 1::2]
    c, s = table[None, :, None, :, 0], table[None, :, None, :, 1]
    return torch.stack((re * c - im * s, re * s + im * c), dim=-1).flatten(-2)


def _mixture64(sources, w):
    V = torch.stack(sources)
    p = (_rms64(V) @ w.view(-1)).softmax(dim=0)
    return (p.unsqueeze(-1) * V).sum(dim=0)


def _attend64(q, k, v, past):
    """q (B, T, H, D) after RoPE and QK-norm, k and v (B, Tk, H, D): causal from position past."""
    q, k, v = (t.transpose(1, 2) for t in (q, k, v))
    s = (q @ k.transpose(-1, -2).contiguous()) / math.sqrt(q.size(-1))
    T, Tk = s.shape[-2:]
    if T > 1:
        hidden = torch.ones((T, Tk), dtype=torch.bool, device=s.device).triu(past + 1)
        s = s.masked_fill_(hidden, float("-inf"))
    return (s.softmax(dim=-1) @ v).transpose(1, 2)


def _sa64(w, x, table, H, keys, past):
    """The attention sub-layer on x (B, T, C); keys(b0, b1) gives the cached K and V of those
    rows (None without any).  Returns the output and the new K and V rows (B, T, H, D)."""
    B, T, C = x.shape
    D = C // H
    out, ks, vs = [], [], []
    chunk = max(1, (1 << 29) // (H * T * (past + T) * 8 + (past + T) * C * 16))
    for b in range(0, B, chunk):
        xb = x[b : b + chunk]
        q, k, v = ((xb @ w[n].T).view(-1, T, H, D) for n in ("c_q", "c_k", "c_v"))
        q, k = _rms64(_rope64(q, table)), _rms64(_rope64(k, table))
        ks.append(k)
        vs.append(v)
        if keys is not None:
            k0, v0 = keys(b, min(B, b + chunk))
            k, v = torch.cat((k0, k), dim=1), torch.cat((v0, v), dim=1)
        y = _attend64(q, k, v, past).reshape(-1, T, C)
        out.append((y * torch.sigmoid(xb @ w["c_g"].T)) @ w["c_proj"].T)
    return torch.cat(out), torch.cat(ks), torch.cat(vs)


def _sa_weights(mha):
    return {n: getattr(mha, n).weight.double() for n in ("c_q", "c_k", "c_v", "c_g", "c_proj")}


def _block64(block, blocks, partial, table, H, keys, past):
    up, down = block.ffwd.net[0].weight.double(), block.ffwd.net[2].weight.double()
    first = len(blocks) == 1 and partial is blocks[0]
    h = partial if first else _mixture64([*blocks, partial], block.attn_res_proj.weight.double())
    blocks = (*blocks, partial)
    a, k, v = _sa64(_sa_weights(block.sa), _rms64(h), table, H, keys, past)
    h = _rms64(_mixture64([*blocks, a], block.mlp_res_proj.weight.double()))
    out = torch.empty_like(a)
    for b in range(0, h.size(0), 16):  # one slice of the batch at a time bounds the 4C-wide temporaries
        z = h[b : b + 16] @ up.T
        gate, lin = z[..., 0::2].clamp(max=_LIMIT), z[..., 1::2].clamp(-_LIMIT, _LIMIT)
        out[b : b + 16] = a[b : b + 16] + (gate * torch.sigmoid(_ALPHA * gate) * (lin + 1)) @ down.T
    return blocks, out, k, v


def _gpt64(model, ids):
    """Logits of every position of ids (B, T), and each layer's K and V rows."""
    emb = model.token_embedding_table.weight.double()
    table = model.freqs_cis.double()[: ids.size(1)]
    x = _rms64(emb[ids])
    blocks, partial, rows = (x,), x, []
    for block in model.blocks:
        blocks, partial, k, v = _block64(block, blocks, partial, table, model.n_head, None, 0)
        rows += [k, v]
    return _CAP * torch.tanh((_rms64(partial) @ emb.T) / _CAP), rows


@torch.no_grad()
def exact(case, seed):
    st = prepare(case, seed)
    kind, H = case["kind"], case["heads"]
    if kind == "gpt_step":
        logits, rows = _gpt64(st["model"], st["ids"])
        return {"logits": logits[:, -1:], "cache_rows": [r[:, -1] for r in rows]}
    if kind == "engine":
        prompt = torch.tensor(st["tokens"], device=_DEV).expand(case["samples"], -1)
        ids = torch.cat((prompt, st["table"][..., 0].T), dim=1)
        logits, _ = _gpt64(st["model"], ids)
        P = case["prompt"]
        return {"logits": logits[:, P - 1 : -1].transpose(0, 1).contiguous(), "tokens": None}
    if kind == "gpt_score":
        return torch.cat([_gpt64(st["model"], part)[0] for part in st["ids"].split(32)])
    if kind == "mha_prefill":
        table = st["freqs"].double().view(case["tokens"], -1, 2)
        w = _sa_weights(st["mha"])
        parts = [_sa64(w, part.double(), table, H, None, 0)[0] for part in st["x"].split(16)]
        return torch.cat(parts)
    double = {}
    for t in (*st["blocks"], st["partial"]):
        double.setdefault(id(t), t.double())
    blocks = tuple(double[id(t)] for t in st["blocks"])
    partial = double[id(st["partial"])]
    if kind == "block_prefill":
        T, past, layer = case["tokens"], case["past"], case["layer"]
        keys = None
        if past:
            k0, v0 = st["cache"].layer_views(layer, past)
            keys = lambda a, b: (k0[a:b].transpose(1, 2).double(), v0[a:b].transpose(1, 2).double())  # noqa: E731
        table = st["freqs"].double().view(T, -1, 2)
        _, out, k, v = _block64(st["block"], blocks, partial, table, H, keys, past)
        return {"out": out, "keys": k.transpose(1, 2), "values": v.transpose(1, 2)}
    P, own, S = case["prefix"], case["own"], case["samples"]
    pos = P + own
    k_pages, v_pages, prefix = st["cache"].decode_views(case["layer"])

    def keys(a, b):
        if prefix is None:
            return k_pages[a:b, :pos].double(), v_pages[a:b, :pos].double()
        group = torch.arange(a, b, device=_DEV) // S
        return (torch.cat((prefix.k[group], k_pages[a:b, :own]), dim=1).double(),
                torch.cat((prefix.v[group], v_pages[a:b, :own]), dim=1).double())

    table = st["freqs"].double()[pos : pos + 1]
    _, out, k, v = _block64(st["block"], blocks, partial, table, H, keys, pos)
    return {"out": out, "key": k[:, 0], "value": v[:, 0]}
