"""Transformer block with Block Attention Residuals (src/diff_gpt/model/block.py:10-107).

Each sub-layer (attention, MLP) reads a per-token softmax mixture over the
committed block states plus the running partial sum, weighted by a learned
pseudo-query; a block boundary every ``layers_per_block`` layers commits the
partial sum.  In Block.forward the mixture and the RMSNorm after it are one
dg_attn_res_norm launch, the clamped SwiGLU of the MLP one dg_swiglu launch,
and the attention sub-layer is the HIP path of MultiHeadAttention.  At
n_embd 64 or 128 everything before the attention -- the mixture, its norm and
the four projections -- is one dg_block_in launch, and everything after it --
gate, c_proj, the partial sum, the MLP's mixture and norm, the FFN and the
residual -- one dg_block_out launch instead of six.
``block_attn_res`` keeps the reference's torch formulation for direct callers.
"""

import torch
import torch.nn.functional as F
from torch import nn
from torch.nn.modules import module as _modules

from diff_gpt import _native
from diff_gpt.model.feed_forward import FeedForward
from diff_gpt.model.kv_cache import KVCache
from diff_gpt.model.mha import MultiHeadAttention
from diff_gpt.model.rms_norm import rms_norm

# dg_attn_res_norm takes at most this many sources of at most this width
ATTN_RES_MAX_SOURCES = 32
ATTN_RES_MAX_WIDTH = 2048
# the widths dg_block_in and dg_block_out take
LAYER_WIDTHS = (64, 128)
_LINEAR_FORWARD = nn.Linear.forward
_PLAIN_TENSORS = (torch.Tensor, nn.Parameter)


def _empty_rows(x: torch.Tensor) -> torch.Tensor:
    """An output shaped as x whose rows follow each other; empty_like would keep
    the order of a permuted x's dimensions."""
    return torch.empty(x.shape, dtype=x.dtype, device=x.device)


def _few_rows(x: torch.Tensor, w: torch.Tensor, tile: int, *others: torch.Tensor | None) -> bool:
    """Whether F.linear(x, w) and the elementwise work around it, with the tensors
    ``others``, go to dg_linear_rows: where F.linear would be the plain product
    (autograd records nothing, autocast changes no type, the weight has no class
    of its own that would answer for it), in 16-bit types, with workgroups, of 32
    rows and ``tile`` features, that times K stay within 256 x 1024, K at most 1024
    (512 for the FFN's first product).  Beyond, its tiles read the operands too
    often.  us, the separate launches -> one, bf16:
      gate, c_proj, sum    n_embd  512: 64 rows 9.5 -> 6.3, 512 9.0 -> 6.5, 1024 9.9 -> 9.2, 1056 10.1 -> 12.3
                           n_embd 1024: 64 rows 10.8 -> 8.9, 256 10.7 -> 9.3, 400 11.6 -> 15.9
      FFN up, SwiGLU       n_embd  512: 64 rows 7.9 -> 5.5, 512 9.2 -> 8.2, 768 11.0 -> 11.4
                           n_embd 1024: 16 rows 6.6 -> 7.5, 200 10.8 -> 13.7
      FFN down, residual   n_embd  512: 64 rows 8.7 -> 6.1, 512 7.8 -> 6.3, 768 8.7 -> 9.7
                           n_embd 1024: 16 rows 7.2 -> 8.3, 256 9.1 -> 9.9"""
    if x.dtype not in (torch.bfloat16, torch.float16):
        return False
    N, K = w.shape
    if K > 1024 or K % 512:
        return False
    if type(w) not in _PLAIN_TENSORS or torch.is_autocast_enabled("cuda"):
        return False
    if torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in (x, w, *others)):
        return False
    return (x.numel() // K + 31) // 32 * (N // tile) * K <= 256 * 1024


def as_written(m: nn.Module, cls: type, forward) -> bool:
    """Whether calling m runs cls's own ``forward`` and nothing else: not a
    subclass's, not one put into the instance or the class since, no hooks on the
    module or on all modules, not compiled."""
    return (type(m) is cls and cls.forward is forward and "forward" not in m.__dict__
            and not m._forward_hooks and not m._forward_pre_hooks
            and not _modules._global_forward_hooks and not _modules._global_forward_pre_hooks
            and m._compiled_call_impl is None)


def _plain_linear(m: nn.Module) -> bool:
    """A Linear that nothing watches or replaces, whose product may be taken
    from its weight."""
    return as_written(m, nn.Linear, _LINEAR_FORWARD) and m.bias is None


def block_attn_res(
    blocks: tuple[torch.Tensor, ...],
    partial_block: torch.Tensor,
    proj: nn.Linear,
) -> torch.Tensor:
    """softmax_n(rms_norm(V_n) . w) weighted sum of V_n over V = (*blocks, partial),
    per token (block.py:10-44).  With a single committed block that *is* the
    partial sum (layer 0) the mixture is that tensor itself."""
    if len(blocks) == 1 and partial_block is blocks[0]:
        return partial_block
    V = torch.stack((*blocks, partial_block), dim=0)  # (N+1, B, T, C)
    scores = rms_norm(V).matmul(proj.weight.view(-1))  # (N+1, B, T)
    weights = scores.softmax(dim=0).unsqueeze(-1)
    return (weights * V).sum(dim=0)


def attn_res_norm(
    blocks: tuple[torch.Tensor, ...],
    partial_block: torch.Tensor,
    proj: nn.Linear,
) -> torch.Tensor:
    """rms_norm(block_attn_res(blocks, partial_block, proj)) in one launch
    (dg_attn_res_norm), with block_attn_res's single-block short cut."""
    if len(blocks) == 1 and partial_block is blocks[0]:
        return rms_norm(partial_block)
    if len(blocks) + 1 > ATTN_RES_MAX_SOURCES or partial_block.size(-1) > ATTN_RES_MAX_WIDTH:
        # beyond the fused kernel's limits: the mixture as device torch ops,
        # then the RMSNorm kernel
        return rms_norm(block_attn_res(blocks, partial_block, proj))
    return _native.ops().attn_res_norm([*blocks, partial_block], proj.weight)


class Block(nn.Module):
    def __init__(
        self,
        n_embd: int,
        n_head: int,
        swiglu_alpha: float,
        swiglu_limit: float,
        layer_idx: int,
        layers_per_block: int = 1,
    ) -> None:
        super().__init__()
        assert layers_per_block >= 1
        self.layer_idx = layer_idx
        self.layers_per_block = layers_per_block
        self.sa = MultiHeadAttention(n_embd=n_embd, n_head=n_head, layer_idx=layer_idx)
        self.ffwd = FeedForward(
            n_embd=n_embd, swiglu_alpha=swiglu_alpha, swiglu_limit=swiglu_limit
        )
        # one (1, C) pseudo-query per sub-layer
        self.attn_res_proj = nn.Linear(n_embd, 1, bias=False)
        self.mlp_res_proj = nn.Linear(n_embd, 1, bias=False)

    def _at_boundary(self) -> bool:
        return (self.layer_idx + 1) % self.layers_per_block == 0

    def forward(
        self,
        blocks: tuple[torch.Tensor, ...],
        partial_block: torch.Tensor,
        freqs_cis: torch.Tensor,
        kv_cache: KVCache | None,
        *,
        _last_only: bool = False,
        _xn: torch.Tensor | None = None,
        _xn_out: torch.Tensor | None = None,
        _qkvg: torch.Tensor | None = None,
        _tail: _native.Tail | None = None,
    ) -> tuple[tuple[torch.Tensor, ...], torch.Tensor]:
        """block.py:87-107.  With _last_only the attention still runs over
        every position (its keys and values go to the cache), and the rest of
        the layer only for the last one: the outputs are that position's
        (B, 1, C) rows, for a last layer whose other rows only the logits of
        their own positions would read.  _xn, when given, is the attention
        sub-layer's input attn_res_norm(blocks, partial_block) computed by the
        caller (layer 0's, from the embedding launch).  _xn_out, when given
        (shaped as the returned partial sum), receives rms_norm of it: the
        head's input after the last layer, from the same launch when
        dg_block_out takes the layer.  _qkvg, when given, is this layer's
        q/k/v/g projections, computed by an earlier launch; _tail what follows
        this layer (its ``done`` says whether the launch took it)."""
        _native.require_device("Block", partial_block)
        sa = self.sa
        qkvg = self._project(blocks, partial_block, _xn) if _qkvg is None else _qkvg
        committed = self._at_boundary()
        partial_in = partial_block
        if committed:
            blocks = (*blocks, partial_block)
        # a large prefill's gate goes with the attention's stores, unless
        # dg_block_out takes the ungated output below or only one row goes on
        gated = not _last_only and sa.n_embd not in LAYER_WIDTHS and sa._gates_in_prefill(qkvg)
        y = sa._attend(qkvg, freqs_cis, kv_cache, gated=True) if gated else sa._attend(qkvg, freqs_cis, kv_cache)
        g = sa._gate_logits(qkvg)
        if _last_only:
            y, g, partial_in = y[:, -1:], g[:, -1:], partial_in[:, -1:]
            blocks = tuple(b[:, -1:] for b in blocks)
        up, swiglu, down = self.ffwd.net
        if not gated and sa.n_embd in LAYER_WIDTHS and len(blocks) + 1 <= ATTN_RES_MAX_SOURCES:
            # gate, c_proj, the partial sum, the MLP's mixture and norm, the FFN
            # and the residual in one launch (n_embd 64 or 128)
            out = _empty_rows(partial_in)
            if _native.block_out_(y, g, sa.c_proj.weight, None if committed else partial_in, list(blocks),
                                  self.mlp_res_proj.weight, up.weight, down.weight, swiglu.alpha, swiglu.limit,
                                  out, _xn_out, tail=_tail):
                return blocks, out
        joined = None
        if not gated and _few_rows(y, sa.c_proj.weight, 32, g, partial_in) and _plain_linear(sa.c_proj):
            # the gate, c_proj and the partial sum in one launch
            joined = _empty_rows(partial_in)
            if not _native.linear_rows_(y, sa.c_proj.weight, joined, gate=g,
                                        residual=None if committed else partial_in):
                joined = None
        if joined is not None:
            partial_block = joined
        else:
            if not gated:
                _native.ops().gate_(y, g)  # y * sigmoid(g), mha.py:84
            attn_out = sa.c_proj(y)
            partial_block = attn_out if committed else partial_in + attn_out
        out = self._mlp(blocks, partial_block)
        if _xn_out is not None:
            _native.rms_norm_(out, _xn_out)
        return blocks, out

    def _project(self, blocks: tuple[torch.Tensor, ...], partial_block: torch.Tensor,
                 xn: torch.Tensor | None) -> torch.Tensor:
        """The q/k/v/g projections (..., 3*inner + C) of the attention's input
        attn_res_norm(blocks, partial_block), or of xn when the caller computed
        it: one dg_block_in launch at n_embd 64 or 128, else the mixture's
        launch and a GEMM."""
        w = self.sa._projection_weight()
        if w.size(1) in LAYER_WIDTHS and w.size(0) == 4 * w.size(1):
            if xn is None and len(blocks) == 1 and partial_block is blocks[0]:
                xn = rms_norm(partial_block)
            out = torch.empty((*partial_block.shape[:-1], w.size(0)), dtype=w.dtype, device=partial_block.device)
            if xn is not None:
                if _native.block_in_([xn], None, w, out):
                    return out
            elif len(blocks) + 1 <= ATTN_RES_MAX_SOURCES:
                if _native.block_in_([*blocks, partial_block], self.attn_res_proj.weight, w, out):
                    return out
        if xn is None:
            xn = attn_res_norm(blocks, partial_block, self.attn_res_proj)
        return F.linear(xn, w)

    def _mlp(self, blocks: tuple[torch.Tensor, ...], partial_block: torch.Tensor) -> torch.Tensor:
        xn = attn_res_norm(blocks, partial_block, self.mlp_res_proj)
        up, swiglu, down = self.ffwd.net
        hidden = None
        if _few_rows(xn, up.weight, 64) and xn.size(-1) <= 512:
            hidden = torch.empty((*xn.shape[:-1], up.weight.size(0) // 2), dtype=xn.dtype, device=xn.device)
            if not _native.linear_rows_(xn, up.weight, hidden, swiglu=(swiglu.alpha, swiglu.limit)):
                hidden = None
        if hidden is None:
            hidden = _native.ops().swiglu(F.linear(xn, up.weight), swiglu.alpha, swiglu.limit)
        if _few_rows(hidden, down.weight, 32, partial_block):
            out = _empty_rows(partial_block)
            if _native.linear_rows_(hidden, down.weight, out, residual=partial_block):
                return out
        return partial_block + F.linear(hidden, down.weight)


_BLOCK_FORWARD = Block.forward


def plain_block(m: nn.Module) -> bool:
    """Whether m's output is what Block.forward returned, so that the launch inside
    may go on with what reads it."""
    return as_written(m, Block, _BLOCK_FORWARD)
