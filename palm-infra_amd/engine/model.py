"""A decoder built from a description: embedding, layers in their run order, final norm, head.

This replaces the reference's graph builder and executor for the one path a request takes
(models/qwen3.py:171-251, graph/execute.cpp:244-833): the description is walked directly, every part
launches its kernels, and nothing is serialised.  The model knows no architecture by name.
"""
from __future__ import annotations

import torch

from ..config.spec import ModelSpec
from ..kernels import ops
from ..parts import Builder, ResidualSink, cache_needs, cache_needs_beside_shared


class DecoderModel:
    def __init__(self, spec: ModelSpec, weights, dtype: torch.dtype, device):
        self.spec, self.dtype, self.device = spec, dtype, torch.device(device)
        builder = Builder(weights, dtype, device)
        self.embedding = builder.build(spec.embedding)
        self.layers = [builder.build(layer) for layer in spec.layers]
        self.final_norm = builder.build(spec.final_norm)
        self.head = builder.build(spec.head)
        builder.finish()
        self.order = spec.order
        self.weights = weights
        self._choosing = list(builder.choosing.values())

    @property
    def capturable(self) -> bool:
        """Whether a decode step of this model may be recorded into a HIP graph: every part says of itself
        that it launches the same kernels whatever the step holds (a part that plans on the host does not)."""
        parts = [self.embedding, *self.layers, self.final_norm, self.head]
        return all(getattr(p, "capturable", False) for p in parts)

    def decode_forms(self, starts: list[int], max_total: int) -> tuple:
        """What the lengths of a decode step's sequences choose among the parts' kernels: a recorded step serves only steps that choose the same."""
        return tuple(part.decode_form(starts, max_total) for part in self._choosing)

    def cache_plan(self):
        """For each entry of the run order: what it keeps per sequence, and whose cache it reads."""
        needs, shares = [], []
        for call in self.order:
            if call.cache_of is None:
                needs.append(cache_needs(self.spec.layers[call.layer]))
                shares.append(None)
            else:
                # what the entry keeps of its own beside the storage that it reads (a state of its own projections)
                needs.append(cache_needs_beside_shared(self.spec.layers[call.layer]))
                shares.append(call.cache_of)
        return needs, shares

    def forward(self, ctx, cache, want_rows: torch.Tensor | None) -> torch.Tensor:
        """Run the step's tokens through all layers; logits (float32) at the rows ``want_rows`` of the
        packed tokens (all rows if None)."""
        if self.spec.keeps_results and self.order:
            # layers read earlier layers' results: plane 0 holds the embedding rows, plane i + 1 the i-th run's result
            ctx.results = torch.empty((len(self.order) + 1, ctx.n_tokens, self.spec.hidden_size), dtype=torch.float32,
                                      device=self.device)
            x = self.embedding.forward(ctx.token_ids, out=ctx.results[0]).clone()
        else:
            x = self.embedding.forward(ctx.token_ids)
        if self.spec.streams is not None and self.spec.streams > 1:
            x = ops.streams_spread(x, self.spec.streams)        # every copy starts as the embedding's rows
        if not self.order:
            return self.head.forward(self.final_norm(x, rows=want_rows))
        # a layer gets its first norm's output and returns the output of the norm after it: the next layer's
        # first norm, at the end the final norm over the wanted rows
        # entries that add the embedding's rows again need them as they left the embedding
        x0 = x.clone() if any(call.adds_embedding for call in self.order) else None
        h = self.layers[self.order[0].layer].entry_norm(x)
        for i, call in enumerate(self.order):
            ctx.layer_cache = cache.layer_caches[i]
            if call.adds_embedding:
                # the sum is made in 32-bit in the pass that norms it for this entry
                h = self.layers[call.layer].entry_norm(x, delta=x0, update=True)
            if i + 1 < len(self.order):
                after = self.layers[self.order[i + 1].layer]
                sink = ResidualSink(x, after.entry_norm, reader=getattr(after, "entry_reader", None))
            else:
                sink = ResidualSink(x, self.final_norm, rows=want_rows, reader=self.head)
            h = self.layers[call.layer].forward(x, h, ctx, sink)
        ctx.layer_cache = None
        ctx.results = None
        return self.head.forward(h)
