"""Token embedding with an optional input projection, and the output head.

x0[t] = Etok[id[t]] (+ position rows), reference src/csrc/kernel/embedding.cu:25-35.
When the embedding width differs from the hidden width, the token vector is
projected first (no bias) and the position rows are added to the projected
vector; the reference has no such model (README.md:42 tells users to avoid it).
The head computes logits = y * Wlm^T in float (src/csrc/model/gpt/gpt.cc:192-201),
after an optional output projection, and falls back to the embedding table when
the file has no separate head tensor (tied weights, scripts/lib/converter_lib.py:272).
``HashedPairEmbedding`` adds a row of a second table chosen by a hash of the token and the token before it
in its sequence, and multiplies the token's own row by a factor; the head may multiply its logits by a factor
and limit them smoothly, cap * tanh(logit / cap).  The reference has neither."""
from __future__ import annotations

from typing import Dict, List, Optional

import torch

from ..ops import kernels as K
from ..weights.loader import TensorSpec
from .base import Part


class TokenEmbedding(Part):
    """params: vocab_size, embed_dim (width of the table; projected to hidden if different), norm
    (optional: the ``PartSpec`` of a norm applied to the embedded rows before the first layer)."""

    def __init__(self, spec, hidden_size, dtype):
        super().__init__(spec, hidden_size, dtype)
        self.vocab_size = int(self.param("vocab_size"))
        self.embed_dim = int(self.param("embed_dim", hidden_size))
        self.projected = self.embed_dim != hidden_size
        self.table = None
        self.w_in = None
        self.norm = None
        if spec.params.get("norm") is not None:
            from .base import build_part
            self.norm = build_part("norm", spec.params["norm"], hidden_size, dtype)

    def tensor_specs(self) -> List[TensorSpec]:
        specs = [TensorSpec(self.name("weight"), (self.vocab_size, self.embed_dim), "table")]
        if self.projected:
            specs.append(TensorSpec(self.name("project_in"), (self.hidden_size, self.embed_dim), "matrix"))
        if self.norm is not None:
            specs += self.norm.tensor_specs()
        return specs

    def bind(self, tensors: Dict[str, torch.Tensor]) -> None:
        self.table = tensors[self.name("weight")]
        if self.projected:
            self.w_in = tensors[self.name("project_in")]
        if self.norm is not None:
            self.norm.bind(tensors)

    def forward(self, ctx, position) -> torch.Tensor:
        x32 = self._embed(ctx, position)
        if self.norm is not None:
            _, x32 = self.norm.forward(x32, out_t=False, out_f32=True)
        return x32

    def _embed(self, ctx, position) -> torch.Tensor:
        T = ctx.num_tokens
        dev = self.table.device
        addend = position.embedding_addend(ctx) if position is not None else None
        x32 = K.empty((T, self.hidden_size), torch.float32, dev)
        if not self.projected:
            if addend is None:
                K.lookup(ctx.token_ids, self.table, out_f32=x32)
            else:
                ptab, pidx, poff = addend
                K.lookup(ctx.token_ids, self.table, add_ids=pidx, add_offset=poff, add_table=ptab,
                         out_f32=x32)
            return x32
        tok = K.empty((T, self.embed_dim), self.dtype, dev)
        K.lookup(ctx.token_ids, self.table, out_t=tok)
        K.gemm(tok, self.w_in, out=x32, out_f32=True)
        if addend is not None:
            ptab, pidx, poff = addend
            K.lookup(None, None, add_ids=pidx, add_offset=poff, add_table=ptab, out_f32=x32,
                     accumulate=True)
        return x32


class HashedPairEmbedding(Part):
    """params: vocab_size, scale (float, default 1: the factor on the token's row), buckets, mul_prev, mul_cur
    (ints: the row of ``pairs`` is (previous token * mul_prev + token * mul_cur) mod buckets; a sequence's first
    token takes row ``buckets``, the last one; buckets 0: no second table).  names: weight [vocab, hidden], pairs [buckets + 1, hidden].

    The previous token of a step's first row is the request's last token of an earlier step: one int a
    request in its state slot (``cache_need``), which the model hands to ``forward`` as ``cache``."""

    def __init__(self, spec, hidden_size, dtype):
        super().__init__(spec, hidden_size, dtype)
        self.vocab_size = int(self.param("vocab_size"))
        self.scale = float(spec.params.get("scale", 1.0))
        self.buckets = int(self.param("buckets"))
        self.mul_prev = int(spec.params.get("mul_prev", 1))
        self.mul_cur = int(spec.params.get("mul_cur", 1))
        if self.buckets < 0:
            raise ValueError(f"the number of buckets is not negative ({self.buckets}); 0: no table of pairs")
        self.table = self.pairs = None

    def tensor_specs(self) -> List[TensorSpec]:
        specs = [TensorSpec(self.name("weight"), (self.vocab_size, self.hidden_size), "table")]
        if self.buckets:
            specs.append(TensorSpec(self.name("pairs"), (self.buckets + 1, self.hidden_size), "table"))
        return specs

    def bind(self, tensors: Dict[str, torch.Tensor]) -> None:
        self.table = tensors[self.name("weight")]
        self.pairs = tensors[self.name("pairs")] if self.buckets else None

    def cache_need(self):
        from .base import CacheNeed
        return CacheNeed("state", state_shape=(1,), state_dtype=torch.int32) if self.buckets else None

    def forward(self, ctx, position, cache=None) -> torch.Tensor:
        if self.buckets and (cache is None or cache.state is None):
            raise ValueError("the pair embedding keeps each request's last token in its state slot")
        return K.hashed_embed(ctx.token_ids, ctx.positions, (ctx.token_item, ctx.item_len, ctx.item_tok_off, ctx.item_slot),
                              cache.state if self.buckets else None, self.table, self.pairs, self.mul_prev,
                              self.mul_cur, self.scale)


class LMHead(Part):
    """params: vocab_size, embed_dim (input width of the head matrix), tied_to (file name of
    the tensor used when the head's own tensor is absent, or None), logit_scale (float, default 1) and
    softcap (float, default 0 = none): logits leave as softcap * tanh(logit_scale * logit / softcap)."""

    def __init__(self, spec, hidden_size, dtype):
        super().__init__(spec, hidden_size, dtype)
        self.vocab_size = int(self.param("vocab_size"))
        self.embed_dim = int(self.param("embed_dim", hidden_size))
        self.projected = self.embed_dim != hidden_size
        self.tied_to: Optional[str] = spec.params.get("tied_to")
        self.logit_scale = float(spec.params.get("logit_scale", 1.0))
        self.softcap = float(spec.params.get("softcap", 0.0) or 0.0)
        self.weight = None
        self.w_out = None

    def tensor_specs(self) -> List[TensorSpec]:
        specs = [TensorSpec(self.name("weight"), (self.vocab_size, self.embed_dim), "matrix",
                            optional=self.tied_to is not None)]
        if self.projected:
            specs.append(TensorSpec(self.name("project_out"), (self.embed_dim, self.hidden_size), "matrix"))
        return specs

    def bind(self, tensors: Dict[str, torch.Tensor]) -> None:
        own = tensors.get(self.name("weight"))
        if own is None:
            if self.tied_to is None or self.tied_to not in tensors:
                raise KeyError("the head has neither its own tensor nor a table to be tied to")
            own = tensors[self.tied_to]
        self.weight = own
        if self.projected:
            self.w_out = tensors[self.name("project_out")]

    def takes_norm(self, rows: int, norm) -> bool:
        """Whether ``forward`` can take ``norm`` (a norm part) of picked rows as its input instead of
        normalised rows, and report the rows' best outputs: the product with the head matrix then
        runs in the kernel that walks a very wide matrix with few rows."""
        # (the rows' best outputs are found before the factor and the limit: both must keep their order)
        return (self.logit_scale > 0 and not self.projected and hasattr(norm, "as_input") and getattr(norm, "width", None) == self.embed_dim
                and K.wide_offered(rows, self.vocab_size, self.embed_dim, self.dtype))

    def offers_best(self, rows: int) -> bool:
        """Whether ``forward`` of that many normalised rows reports the rows' best outputs.  (Not through a factor or a limit: they may
        make two different outputs equal, and the best is then the lower index.)"""
        return (self.logit_scale == 1.0 and self.softcap == 0 and not self.projected
                and K.wide_offered(rows, self.vocab_size, self.embed_dim, self.dtype))

    def forward(self, y_t, best: Optional[torch.Tensor] = None) -> torch.Tensor:
        """float32 logits [rows, vocab] of ``y_t``: normalised rows, or (where ``takes_norm``) what a
        norm's ``as_input`` returned.  ``best`` (int32 [rows], where ``takes_norm`` or ``offers_best``): receives every
        row's best output, the lowest index on ties."""
        if self.projected:
            y_t = K.gemm(y_t, self.w_out)
        logits = K.gemm(y_t, self.weight, out_f32=True, best=best)
        if self.logit_scale != 1.0 or self.softcap > 0:
            K.scale_softcap(logits, self.logit_scale, self.softcap)
        return logits
