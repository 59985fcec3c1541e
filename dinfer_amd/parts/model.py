"""A decoder model assembled from a ModelSpec: embedding (-> an operation on it, if the spec names one) -> run list
of blocks -> final norm on the wanted rows -> LM head (-> an operation on the logits, if the spec names one).
Knows no architecture by name.
"""
from __future__ import annotations

import math

import torch

from ..kernels import gemm, ops
from .base import BuildContext, Carried
from .linear import Linear
from .registry import BLOCKS, NORMS, STREAM_OPS
from .spec import ModelSpec, RunEntry, TensorSpec


def _build_blocks(spec: ModelSpec):
    return [BLOCKS.get(l.block.kind)(hidden=spec.hidden_size, layer=l, **l.block.params) for l in spec.layers]


def _stream_ops(spec: ModelSpec) -> list:
    """[(weight-name prefix, part)] of the operations on the embeddings and on the logits, None where there is none."""
    made = []
    for part, width, prefix in ((spec.embed_post, spec.hidden_size, spec.embed_name), (spec.logits_post, spec.vocab_size, spec.head_name)):
        made.append(None if part is None else (prefix + ".post.", STREAM_OPS.get(part.kind)(width, **part.params)))
    return made


def _before_ops(spec: ModelSpec) -> list:
    """Per run entry: the part applied to the stream right before it, or None."""
    return [None if e.before is None else STREAM_OPS.get(e.before.kind)(spec.hidden_size, **e.before.params)
            for e in spec.run]


def expected_tensors(spec: ModelSpec, blocks=None) -> tuple[dict[str, TensorSpec], set[str]]:
    """(name -> TensorSpec for every tensor the model reads, names that may be present or absent)."""
    blocks = blocks or _build_blocks(spec)
    exp = {spec.embed_name: TensorSpec((spec.vocab_size, spec.hidden_size))}
    for l, b in zip(spec.layers, blocks):
        for n, s in b.tensors().items():
            exp[l.prefix + n] = s
    fn = NORMS.get(spec.final_norm.kind)(spec.hidden_size, **spec.final_norm.params)
    for n, s in fn.tensors().items():
        exp[spec.final_norm_name + n] = s
    for op in _stream_ops(spec):
        if op is not None:
            for n, ts in op[1].tensors().items():
                exp[op[0] + n] = ts
    for op in _before_ops(spec):
        if op is not None:
            exp.update(op.tensors())      # under the names they give themselves; several entries may read one table
    optional = set()
    if spec.tie_embeddings:
        # A tied checkpoint may still ship the head; it is used when present (model.rs:487-496).
        optional.add(spec.head_name)
    else:
        exp[spec.head_name] = TensorSpec((spec.vocab_size, spec.hidden_size))
    return exp, optional


class DecoderModel:
    def __init__(self, spec: ModelSpec):
        self.spec = spec
        self.blocks = _build_blocks(spec)
        self.final_norm = NORMS.get(spec.final_norm.kind)(spec.hidden_size, **spec.final_norm.params)
        self.head = Linear(spec.hidden_size, spec.vocab_size)
        self.embed_post, self.logits_post = _stream_ops(spec)
        self.embed: torch.Tensor | None = None
        self.run = [RunEntry(e.layer, i if e.cache is None else e.cache, e.before) for i, e in enumerate(spec.run)]
        self.before = _before_ops(spec)
        # the embeddings as they entered the stream, kept for an entry's `before` part that adds them again
        self.keeps_embedding = any(getattr(op, "needs_embedding", False) for op in self.before if op is not None)
        for i, e in enumerate(self.run):
            if not (0 <= e.layer < len(self.blocks)):
                raise ValueError(f"run entry {i} names layer {e.layer}, but the model has {len(self.blocks)} layers")
            if not (0 <= e.cache <= i):
                raise ValueError(f"run entry {i} reads the cache of entry {e.cache}, which does not run before it")
            if self.run[e.cache].cache != e.cache:
                raise ValueError(f"run entry {i} reads the cache of entry {e.cache}, which has no cache of its own")

    # ---- weights -------------------------------------------------------------------------------
    def expected_tensors(self):
        return expected_tensors(self.spec, self.blocks)

    def layer_weights(self) -> int:
        """Weights of a layer, all of its experts' among them, on the average over the layers."""
        return sum(math.prod(t.shape) for b in self.blocks for t in b.tensors().values()) // max(len(self.blocks), 1)

    def load(self, loader) -> None:
        exp, optional = self.expected_tensors()
        loader.check(exp, optional)
        self._load_from(lambda name, compute=False: loader.fetch(name, compute=compute), loader.has)

    def load_random(self, seed: int, device, dtype: torch.dtype) -> None:
        """Draws every tensor on the device by the rule of the random-weights mode (weights/random_init.py: each
        tensor from (seed, its name)); for measurements at sizes where writing a file first would only cost time."""
        from ..weights.random_init import draw_on_device
        exp, _ = self.expected_tensors()
        self._load_from(lambda name, compute=False: draw_on_device(seed, name, exp[name], dtype, device),
                        lambda name: name in exp)

    def _load_from(self, get, has) -> None:
        s = self.spec
        self.embed = get(s.embed_name, compute=True)
        for l, b in zip(s.layers, self.blocks):
            b.load(lambda n, _p=l.prefix, **kw: get(_p + n, **kw))
        self.final_norm.load(lambda n, **kw: get(s.final_norm_name + n, **kw))
        if has(s.head_name):
            self.head.set_weight(get(s.head_name, compute=True))
        elif s.tie_embeddings:
            self.head.set_weight(self.embed)  # one buffer for both
        else:
            raise ValueError(f"no {s.head_name} in the weights and tie_word_embeddings is false")
        for op in (self.embed_post, self.logits_post):
            if op is not None:
                op[1].load(lambda n, _p=op[0], **kw: get(_p + n, **kw))
        for op in self.before:
            if op is not None:
                op.load(get)

    # ---- cache needs ---------------------------------------------------------------------------
    def cache_needs(self) -> list:
        """Per run entry: the CacheSpec of the cache it owns; None if it has none or borrows one."""
        out = []
        for i, e in enumerate(self.run):
            block = self.blocks[e.layer]
            # a block that keeps something of its own between steps answers for its mixer too
            need = block.cache_spec() if hasattr(block, "cache_spec") else block.mixer.cache_spec()
            out.append(need if e.cache == i else None)
        return out

    def capturable(self) -> bool:
        """Whether a step of single rows may be captured once and replayed for other requests."""
        ops_ = [op[1] for op in (self.embed_post, self.logits_post) if op is not None]
        ops_ += [op for op in self.before if op is not None]
        return (all(self.blocks[e.layer].capturable for e in self.run) and self.final_norm.capturable
                and all(o.capturable for o in ops_))

    def capturable_portions(self) -> bool:
        """The same for steps with prompt portions (Mixer.capturable_portions)."""
        return (self.capturable() and all(self.blocks[e.layer].capturable_portions for e in self.run)
                and self.final_norm.capturable_portions)

    def wants_lengths(self, batch) -> bool:
        """Whether the step in `batch` is better launched one by one than padded and replayed, because parts then know its requests'
        lengths: where one finds a better way by them, and the device has as much to do in the usual way as the host to launch.

        That is some 110 us a layer; what of it the usual way (Part.choices) and the weights (read at 4.7 TB/s, or multiplied at 1
        PFLOP/s) leave to its other kernels is 65. Replayed the usual way, and launched one by one the other, us a step (us of these 45):
          6 layers of 3 million weights, 4 heads: one request of 128 (12) 504 and 761, three of 200 behind 300 (45) 729 and 762, one of
            128 behind 1,000 (89) 893 and 757
          8 of 10, 8 heads: 128 (15) 718 and 983, 384 (40) 957 and 996, 512 (54) 1,042 and 1,005, 8 of 130 (39) 1,006 and 1,007, three of
            200 behind 300 (55) 1,102 and 987
          8 of 30, 16 heads: 128 (24) 915 and 982, 256 (39) 1,057 and 1,002, 4 of 128 (48) 1,153 and 1,071
          4 of 316 with 64 experts: 128 (146) 1,006 and 978"""
        usual, better = 0.0, False
        for choice, times in self._choices:
            us = choice.usual_way(batch)
            if us is not None:
                usual, better = usual + us * times, True
        return better and usual / len(self.run) + self._weights * max(2 / 4.7e6, 2e-9 * batch.num_tokens) >= 45.0

    # ---- execution -----------------------------------------------------------------------------
    def bind(self, ctx: BuildContext) -> None:
        self.ctx = ctx
        for b in self.blocks:
            b.bind(ctx)
        # (asked once: steps are launched against the clock)
        met = [c for e in self.run for c in self.blocks[e.layer].choices()]
        self._choices = [(c, sum(x is c for x in met)) for i, c in enumerate(met) if not any(x is c for x in met[:i])]
        self._weights = self.layer_weights()
        for op in (self.embed_post, self.logits_post):
            if op is not None:
                op[1].bind(ctx)
        for op in self.before:
            if op is not None:
                op.bind(ctx)
        ws = ctx.workspace
        stream = torch.float32 if self.spec.stream_dtype == "float32" else None
        self.streams = int(self.spec.streams or 1)
        if self.streams > 1:
            # several residual streams a token: the embedding is gathered into a row of its own and copied into
            # every stream; the sum of the streams of the wanted rows is what the final norm reads
            if self.spec.stream_dtype != "float32":
                raise ValueError("several residual streams are kept in float32 (stream_dtype)")
            self.embedded_once = ws.buffer("embedded_once", self.spec.hidden_size, dtype=stream)
            self.hidden = ws.buffer("hidden_streams", self.streams * self.spec.hidden_size, dtype=stream)
            self.summed = ws.buffer("streams_summed", self.spec.hidden_size, dtype=stream, rows=ctx.max_rows)
            self.ones = torch.ones(self.streams, dtype=torch.float32, device=ctx.device)
            if self.keeps_embedding or self.embed_post is not None:
                raise ValueError("several residual streams with operations on the embeddings are not built")
        else:
            self.hidden = ws.buffer("hidden", self.spec.hidden_size, dtype=stream)
        self.embedded = ws.buffer("embedded", self.spec.hidden_size, dtype=stream) if self.keeps_embedding else None
        self.final_normed = ws.buffer("final_normed", self.spec.hidden_size, rows=ctx.max_rows)
        self.logits = torch.empty((ctx.max_rows, self.spec.vocab_size), dtype=torch.float32, device=ctx.device)

    def forward(self, batch, caches: list) -> torch.Tensor:
        """Runs the batch's tokens through all run entries; returns float32 logits [num_rows, vocab]
        at batch.logits_rows (a view of a fixed buffer)."""
        T, R = batch.num_tokens, batch.num_rows
        first = self.hidden if self.streams == 1 else self.embedded_once
        ops.embedding(batch.input_ids[:T], self.embed, first, getattr(batch, "feedback_src", None),
                      getattr(batch, "last_tokens", None), scale=self.spec.embed_scale)
        if self.streams > 1:
            ops.streams_expand(first, self.hidden, T, self.streams)
        if self.embed_post is not None:
            self.embed_post[1].forward(self.hidden, T)
        if self.embedded is not None:
            if self.embed_post is None:     # gathered a second time: a kernel of the engine's own in a captured step
                ops.embedding(batch.input_ids[:T], self.embed, self.embedded, getattr(batch, "feedback_src", None),
                              getattr(batch, "last_tokens", None), scale=self.spec.embed_scale)
            else:
                self.embedded[:T].copy_(self.hidden[:T])
        pending = None
        for i, e in enumerate(self.run):
            block = self.blocks[e.layer]
            if self.before[i] is not None:
                # the stream must be whole before something is added to it from outside the blocks
                if isinstance(pending, Carried):
                    pending = None
                elif hasattr(pending, "settle"):
                    pending.settle(T)
                    pending = None
                elif pending is not None:
                    ops.add_rows(self.hidden, T, a=pending)
                    pending = None
                if getattr(self.before[i], "needs_embedding", False):
                    self.before[i].forward(self.hidden, T, embedding=self.embedded)
                else:
                    self.before[i].forward(self.hidden, T)
            # the input norm of the block that runs next, if that block lets the one before carry it (and nothing
            # touches the stream between the two)
            if block.carries_norms and i + 1 < len(self.run) and self.before[i + 1] is None:
                nxt = self.blocks[self.run[i + 1].layer].input_norm()
                pending = block.forward(self.hidden, pending, batch, caches[i], next_norm=nxt)
            else:
                pending = block.forward(self.hidden, pending, batch, caches[i])
        if R == 0:
            return self.logits[:0]
        if self.streams > 1:
            # the last write into the streams happens on the wanted rows only, inside the pass that sums them
            kw = {}
            if hasattr(pending, "settle"):
                kw = dict(branch=pending.branch, mix=pending.mix, out_weights=pending.out)
            ops.streams_step(self.hidden, R, self.streams, dtype=self.final_normed.dtype, read=self.ones,
                             u_out=self.summed, rows=batch.logits_rows, **kw)
            self.final_norm.forward(self.summed, self.final_normed, R)
        elif hasattr(pending, "settle"):
            pending.settle(T)
            self.final_norm.forward(self.hidden, self.final_normed, R, rows=batch.logits_rows)
        elif pending is None or isinstance(pending, Carried):
            self.final_norm.forward(self.hidden, self.final_normed, R, rows=batch.logits_rows)
        else:
            # the last add happens on the wanted rows only, inside the norm kernel
            self.final_norm.forward(pending, self.final_normed, R, residual=self.hidden, rows=batch.logits_rows)
        gemm.matmul_nt(self.final_normed, self.head.weight, self.logits, R, may_pad=True)  # both are buffers of max_rows rows
        if self.logits_post is not None:
            self.logits_post[1].forward(self.logits, R)
        return self.logits[:R]
