"""GPT over the MI355X attention path (src/diff_gpt/model/gpt.py:15-242).

Same constructor, parameter names (state_dicts load both ways), parameter
creation order (so a seeded construction gives the same weights), forward
signature and generation API as the reference.  Inference only: the HIP
kernels have no backward, so a forward that would need autograd raises.
"""

from abc import ABC, abstractmethod

import torch
import torch.nn as nn
from torch.nn import functional as F

from diff_gpt import _native
from diff_gpt.model.block import Block, plain_block
from diff_gpt.model.kv_cache import KVCache
from diff_gpt.model.rms_norm import rms_norm
from diff_gpt.model.rope import precompute_freqs_cis
from diff_gpt.sampler.sampler import Sampler
from diff_gpt.sampler.temperature import TemperatureSampler, draw_one

# (n_embd, bytes of an element) -> the most rows whose launches are joined
# (GPT._joins).  Whole forwards over a vocabulary of 256, us one by one -> joined:
#   n_embd  64 fp32  2 layers:   100 rows 43.4 -> 35.8, 35328 245 -> 236, 41400 274 -> 271, 70656 408 -> 417
#                    6 layers:   100 rows  118 ->  109, 35328 666 -> 669, 41400 749 -> 785, 70656 1155 -> 1269
#   n_embd  64 bf16  2 layers:   100 rows 37.7 -> 30.8, 8192 86.8 -> 77.3, 16384 142 -> 140
#                    6 layers:   100 rows  102 -> 90.1, 8192 243 -> 226, 16384 390 -> 395 (70656 728 -> 752)
#   n_embd 128 bf16  2 layers:   100 rows 49.7 -> 45.1, 4096 78.0 -> 70.0, 8192 119 -> 123
#                    6 layers:   100 rows  138 ->  141, 4096 231 -> 206, 8192 332 -> 362
#   n_embd 128 fp32 (the embedding's launch alone joins)  2 layers: 100 rows 70.9 -> 69.1, 8192 181 -> 176
# Beyond the lines the launches of their own take 32-row groups, which joined
# ones have no registers for.  A vocabulary of 1024 gains more (fp32, 2 layers,
# 70656 rows: 566 -> 542), many layers less.
JOINED_ROWS = {(64, 4): 36864, (64, 2): 8192, (128, 4): 4096, (128, 2): 4096}


def _ordinal_target_table(V: int, sigma: float, dtype: torch.dtype, device) -> torch.Tensor:
    """(V, V) table whose row t is the soft target for token t: a discretised
    Gaussian over the bin indices centred on t with standard deviation sigma
    (in bins), normalised to sum to 1."""
    bins = torch.arange(V, device=device, dtype=torch.float64)
    z = (bins[None, :] - bins[:, None]) / sigma
    return torch.softmax(-0.5 * z * z, dim=-1).to(dtype)


def _ordinal_soft_ce(
    logits: torch.Tensor,
    targets: torch.Tensor,
    sigma: float,
    ignore_index: int = -100,
) -> torch.Tensor:
    """Mean over the rows whose target is not ignore_index of the cross-entropy
    between the row's log-softmax and its Gaussian soft target (the training
    loss of gpt.py:15-35 for label_smoothing_sigma > 0); 0 when every row is
    ignored."""
    valid = targets != ignore_index
    soft = _ordinal_target_table(logits.size(-1), sigma, logits.dtype, logits.device)
    rows = soft[torch.where(valid, targets, 0)]
    per_row = -(rows * F.log_softmax(logits, dim=-1)).sum(dim=-1)
    return torch.where(valid, per_row, 0.0).sum() / valid.sum().clamp(min=1)


class BaseGPT(nn.Module, ABC):
    def __init__(
        self,
        block_size: int,
        vocab_size: int,
        n_embd: int,
        n_head: int,
        n_layer: int,
    ) -> None:
        super().__init__()
        self.block_size = block_size
        self.vocab_size = vocab_size
        self.n_embd = n_embd
        self.n_head = n_head
        self.n_layer = n_layer

    @abstractmethod
    def forward(
        self,
        idx: torch.Tensor,
        targets: torch.Tensor | None = None,
        kv_cache: KVCache | None = None,
    ) -> tuple[torch.Tensor, torch.Tensor | None]:
        pass

    @abstractmethod
    def generate(
        self,
        idx: torch.Tensor,
        max_new_tokens: int,
        sampler: Sampler | None,
        seed: int | None = None,
    ) -> torch.Tensor:
        pass

    @property
    @abstractmethod
    def device_type(self) -> str:
        pass


class GPT(BaseGPT):
    def __init__(
        self,
        vocab_size: int,
        n_embd: int = 64,
        block_size: int = 32,
        n_head: int = 4,
        n_layer: int = 4,
        rope_theta: float = 10000,
        swiglu_alpha: float = 1.702,
        swiglu_limit: float = 7.0,
        use_checkpoint: bool = True,
        logit_softcap: float = 15.0,
        pad_vocab_size_to: int = 64,
        attn_res_layers_per_block: int = 1,
        label_smoothing_sigma: float = 0.0,
    ) -> None:
        super().__init__(
            block_size=block_size,
            vocab_size=vocab_size,
            n_embd=n_embd,
            n_head=n_head,
            n_layer=n_layer,
        )
        assert logit_softcap >= 0, "logit_softcap must be non-negative (0 disables it)"
        assert label_smoothing_sigma >= 0, (
            "label_smoothing_sigma must be non-negative (0 disables it)"
        )
        assert pad_vocab_size_to >= 1, "pad_vocab_size_to must be >= 1"
        assert attn_res_layers_per_block >= 1, "attn_res_layers_per_block must be >= 1"
        assert vocab_size % pad_vocab_size_to == 0, (
            f"vocab_size ({vocab_size}) must be a multiple of "
            f"pad_vocab_size_to ({pad_vocab_size_to}); pad it in the encoder"
        )
        self.token_embedding_table = nn.Embedding(vocab_size, n_embd)
        self.blocks = nn.ModuleList(
            Block(
                n_embd=n_embd,
                n_head=n_head,
                swiglu_alpha=swiglu_alpha,
                swiglu_limit=swiglu_limit,
                layer_idx=i,
                layers_per_block=attn_res_layers_per_block,
            )
            for i in range(n_layer)
        )
        # lm_head is created (consuming the seeded RNG) and then tied
        self.lm_head = nn.Linear(n_embd, vocab_size, bias=False)
        self.lm_head.weight = self.token_embedding_table.weight
        # RoPE table for 2*block_size positions; not saved in the state_dict
        self.register_buffer(
            "freqs_cis",
            precompute_freqs_cis(n_embd // n_head, block_size * 2, theta=rope_theta),
            persistent=False,
        )
        self.use_checkpoint = use_checkpoint
        self.logit_softcap = logit_softcap
        self.label_smoothing_sigma = label_smoothing_sigma

    def _head(self, partial: torch.Tensor, argmax_out: torch.Tensor | None,
              xn: torch.Tensor | None = None) -> torch.Tensor:
        """rms_norm -> tied lm_head -> softcap (gpt.py:180-186): one dg_lm_head
        launch after the norm (xn, when the last layer's launch wrote it),
        which also writes each row's argmax into argmax_out (B, T) when given;
        F.linear + dg_softcap (+ torch.argmax) for shapes it does not take."""
        if xn is None:
            xn = rms_norm(partial)
        B, T, C = xn.shape
        V = self.lm_head.weight.size(0)
        cap = float(self.logit_softcap)
        logits = torch.empty((B, T, V), dtype=xn.dtype, device=xn.device)
        ids = None if argmax_out is None else argmax_out.view(B * T)
        if _native.lm_head_(xn.view(B * T, C), self.lm_head.weight, cap, logits.view(B * T, V), ids):
            return logits
        logits = self.lm_head(xn)
        if cap > 0:
            _native.ops().softcap_(logits, cap)  # cap * tanh(logits / cap)
        if argmax_out is not None:
            argmax_out.copy_(torch.argmax(logits, dim=-1))
        return logits

    def _embed(self, idx: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor | None, torch.Tensor | None]:
        """x = rms_norm(token_embedding_table(idx)) (gpt.py:154-155) and, when
        there is a layer 0, what it begins with: its q/k/v/g projections of
        rms_norm(x) at few rows (one dg_embed_in launch), else rms_norm(x) (one
        dg_embed_norm launch).  An id outside the vocabulary gives a NaN row
        (nn.Embedding raises).  fp64 tables take nn.Embedding and the RMSNorm
        kernel."""
        table = self.token_embedding_table.weight
        _native.require_device("GPT", idx, table)
        _native.require_inference("GPT", table)
        C = table.size(1)
        x = torch.empty((*idx.shape, C), dtype=table.dtype, device=table.device)
        if self.blocks and self._joins(idx.numel()):
            w = self.blocks[0].sa._projection_weight()
            qkvg = torch.empty((*idx.shape, w.size(0)), dtype=table.dtype, device=table.device)
            if _native.embed_norm_(idx, table, x, None, w, qkvg):
                return x, None, qkvg
        xn0 = torch.empty_like(x) if self.blocks else None
        if _native.embed_norm_(idx, table, x, xn0):
            return x, xn0, None
        return rms_norm(self.token_embedding_table(idx)), None, None

    def _joins(self, rows: int) -> bool:
        """Whether, over ``rows`` rows, the embedding, the layers' projections and
        the head go with the launch before them: only where every layer is a Block
        as written, since an overridden forward or a hook may read or replace what
        lies between."""
        w = self.token_embedding_table.weight
        if rows > JOINED_ROWS.get((w.size(1), w.element_size()), -1):
            return False
        return all(plain_block(b) for b in self.blocks)

    def _tail(self, i: int, ids: torch.Tensor | None, advance: torch.Tensor | None) -> _native.Tail | None:
        """What follows layer i: layer i + 1's projections or the head (not an
        overridden one).  None where no launch would take it."""
        w = self.lm_head.weight
        if not _native.takes_tail(w.dtype, w.size(1)):
            return None
        if i + 1 < len(self.blocks):
            block = self.blocks[i + 1]
            return _native.Tail(block.attn_res_proj.weight, block.sa._projection_weight())
        if w.size(0) not in _native.TAIL_VOCABS or type(self)._head is not _GPT_HEAD or "_head" in self.__dict__:
            return None
        return _native.Tail(None, w, None, float(self.logit_softcap), ids, advance, keep_norm=False)

    def forward(
        self,
        idx: torch.Tensor,
        targets: torch.Tensor | None = None,
        kv_cache: KVCache | None = None,
        *,
        _argmax_out: torch.Tensor | None = None,
        _last_only: bool = False,
        _advance: bool = False,
    ) -> tuple[torch.Tensor, torch.Tensor | None]:
        """gpt.py:140-200.  _argmax_out (B, T) int64, when given, receives the
        first maximum of every logits row (greedy sampling without a separate
        argmax launch).  _last_only returns the (B, 1, V) logits of the last
        position only (a prefill whose caller reads no others; _argmax_out is
        then (B, 1)): every layer still attends and caches every position, but
        the last layer's work after its attention and the head run for that
        position alone."""
        B, T = idx.shape
        assert not (_last_only and targets is not None), "_last_only returns the last position's logits alone"
        start = 0 if kv_cache is None else kv_cache.get_pos()
        end = start + T
        assert end <= self.freqs_cis.shape[0]
        if kv_cache is not None and kv_cache.pos_dev is not None:
            # captured decode step: the kernels index the whole table with the
            # position they read on the device
            freqs_cis = self.freqs_cis
        else:
            freqs_cis = self.freqs_cis[start:end].view(1, T, 1, -1, 2)

        # the normalised embedding and, when layer 0 reads it, layer 0's
        # attention input rms_norm(x) (its one-block mixture) in one launch
        x, xn0, qkvg = self._embed(idx)
        # Block-AttnRes state: the normalised embedding is block 0 and also the
        # first partial sum
        blocks: tuple[torch.Tensor, ...] = (x,)
        partial = x
        last = len(self.blocks) - 1
        # the head's input rms_norm(partial), written by the last layer
        xn_head = None
        if self.blocks:
            xn_head = torch.empty((B, 1 if _last_only else T, x.size(-1)), dtype=x.dtype, device=x.device)
        advance = kv_cache.pos_dev if _advance else None
        joins = self._joins(B * T)
        joins_last = self._joins(B) if _last_only else joins
        tail = None
        for i, block in enumerate(self.blocks):
            one = _last_only and i == last
            tail = self._tail(i, _argmax_out, advance) if (joins_last if one else joins) else None
            # a Block with a forward of its own is not handed what joined launches pass on
            joined = {} if qkvg is None and tail is None else {"_qkvg": qkvg, "_tail": tail}
            blocks, partial = block(blocks, partial, freqs_cis=freqs_cis, kv_cache=kv_cache,
                                    _last_only=_last_only and i == last, _xn=xn0 if i == 0 else None,
                                    _xn_out=xn_head if i == last else None, **joined)
            qkvg = tail.out if tail is not None and tail.done else None
        if _last_only and not self.blocks:
            partial = partial[:, -1:]

        if tail is not None and tail.done:
            logits = tail.out
        else:
            logits = self._head(partial, _argmax_out, xn_head)
            if advance is not None:
                advance.add_(1)

        loss = None
        if targets is not None:
            flat_logits = logits.view(B * T, -1)
            flat_targets = targets.view(B * T)
            if self.label_smoothing_sigma > 0:
                loss = _ordinal_soft_ce(
                    flat_logits, flat_targets, sigma=self.label_smoothing_sigma
                )
            else:
                loss = F.cross_entropy(flat_logits, flat_targets)
        return logits, loss

    @torch.inference_mode()
    def generate(
        self,
        idx: torch.Tensor,
        max_new_tokens: int,
        sampler: Sampler | None,
        seed: int | None = None,
    ) -> torch.Tensor:
        """Cache-free sliding-window sampling (gpt.py:202-237): every step
        re-runs the last block_size tokens through the causal prefill path."""
        device = idx.device
        rng = None
        if seed is not None:
            rng = torch.Generator(device=device)
            rng.manual_seed(seed)
        B, T = idx.shape
        out = torch.zeros((B, T + max_new_tokens), dtype=torch.int64, device=device)
        out[:, :T] = idx
        # greedy: the argmax comes out of the lm_head launch (temperature.py:22-23)
        greedy = type(sampler) is TemperatureSampler and sampler.temperature == 0
        for cur in range(T, T + max_new_tokens):
            window = out[:, max(0, cur - self.block_size) : cur]
            # only the last position's logits are read
            if greedy:
                am = torch.empty((B, 1), dtype=torch.int64, device=device)
                self(window, _argmax_out=am, _last_only=True)
                out[:, cur] = am[:, -1]
                continue
            logits, _ = self(window, _last_only=True)
            last = logits[:, -1]
            if sampler is not None:
                nxt = sampler(last, rng=rng)
            else:
                nxt = draw_one(F.softmax(last, dim=-1), rng)
            out[:, cur] = nxt.squeeze()
        return out

    @property
    def device_type(self) -> str:
        return str(self.freqs_cis.device.type)


_GPT_HEAD = GPT._head
_GPT_FORWARD = GPT.forward


def plain_gpt(model: nn.Module) -> bool:
    """Whether model.forward is GPT.forward as written, which takes the private
    arguments of a captured step."""
    return type(model) is GPT and GPT.forward is _GPT_FORWARD and "forward" not in model.__dict__
