"""A decoder assembled from a `ModelSpec`: embedding, the blocks in schedule order, final norm
and logits at the wanted rows (`inferrs-models/src/models/qwen3.rs:398-440`,
`attention_utils.rs:382-395`).  Nothing here names an architecture."""
from __future__ import annotations

from typing import Dict, Optional

import torch

from .. import ops
from ..config.spec import ModelSpec, SpecError
from ..parts.base import block_class, part_class
from ..parts.layer_run import LayerRun
from ..parts.linear import Linear
from ..parts.norm import build_norm
from .batch import StepContext

DTYPES = {"float32": torch.float32, "f32": torch.float32, "fp32": torch.float32,
          "bfloat16": torch.bfloat16, "bf16": torch.bfloat16}


def parse_dtype(name) -> torch.dtype:
    if isinstance(name, torch.dtype):
        if name not in (torch.float32, torch.bfloat16):
            raise ValueError(f"the engine computes in float32 or bfloat16, not {name}")
        return name
    try:
        return DTYPES[str(name).lower()]
    except KeyError:
        raise ValueError(f"unknown dtype {name!r}; choose bfloat16 or float32") from None


class DecoderModel:
    def __init__(self, spec: ModelSpec, tensors: Dict[str, torch.Tensor], dtype: torch.dtype, device):
        """`tensors`: every tensor of `model_tensors(spec)` by name, in its stored precision,
        on any device.  Entries are dropped from the dict as they are taken over."""
        spec.validate()
        self.spec, self.dtype, self.device = spec, dtype, torch.device(device)

        def take(names) -> Dict[str, torch.Tensor]:
            return {n: tensors.pop(n) for n in list(names) if n in tensors}

        embedding_cls = part_class("embedding", spec.embedding)
        self.embedding = embedding_cls(spec.embedding, take(embedding_cls.tensors(spec.embedding)), dtype, device)
        head_cls = part_class("head", spec.head)
        self.head = head_cls(spec.head, take(head_cls.tensors(spec.head)), dtype, device, embedding=self.embedding)
        self.blocks = []
        for layer in spec.layers:
            cls = block_class(layer)
            self.blocks.append(cls(layer, take(cls.tensors(layer)), dtype, device))
        self.pass_input = None
        if spec.pass_input is not None:
            pass_cls = part_class("pass_input", spec.pass_input)
            self.pass_input = pass_cls(spec.pass_input, take(pass_cls.tensors(spec.pass_input)), dtype, device)
        self.final_norm = None
        if spec.final_norm is not None:
            self.final_norm = build_norm(spec.final_norm_name, spec.final_norm, tensors, dtype, device, pop=True)
        self.layer_run = LayerRun.of_model(spec, self.blocks)

    @property
    def graph_safe(self) -> bool:
        """Whether every part allows a decode step to be captured and replayed."""
        return all(getattr(p, "graph_safe", False) for p in self.all_parts())

    def all_parts(self):
        parts = [self.embedding, self.head, self.final_norm, self.pass_input]
        for b in self.blocks:
            parts += list(b.parts())
        return [p for p in parts if p is not None]

    def load_notes(self, page_size: int):
        """What the parts have to say once about how they will run (a part may offer `load_notes(page_size)`):
        every different note once, in the order of the parts."""
        notes = []
        for p in self.all_parts():
            for note in (p.load_notes(page_size) if hasattr(p, "load_notes") else []):
                if note not in notes:
                    notes.append(note)
        return notes

    def cache_needs(self) -> Dict[int, object]:
        """Schedule stop that owns a cache -> what its mixer keeps per request."""
        needs: Dict[int, object] = {}
        for stop, e in enumerate(self.spec.schedule):
            if e.cache_of is None:
                mixer = self.spec.layers[e.layer].mixer
                needs[stop] = part_class("mixer", mixer).cache_need(mixer)
        return needs

    def forward(self, ctx: StepContext, storage) -> torch.Tensor:
        """Runs the step's tokens through every stop of the schedule (which appends to the
        caches) and returns float32 logits `[n_want, vocab]`."""
        x = first_rows = self.embedding.forward(ctx)
        first = self.blocks[self.spec.schedule[0].layer]
        if hasattr(first, "enter"):                  # an arrangement whose stream is not the embedding's rows
            x = first.enter(ctx, x)
        pending = None                               # a block's output that is not added to x yet
        of_run, in_run = self.layer_run.takes(ctx, x, storage) if self.layer_run is not None else None, 0
        if of_run is not None:                       # the first layers in one kernel, which leaves nothing to be added
            x, in_run = self.layer_run.forward(ctx, x, of_run, storage), self.layer_run.length
        for stop, e in enumerate(self.spec.schedule):
            if stop < in_run:
                continue
            cache = storage.layers.get(self.spec.cache_stop(stop))
            if cache is not None and e.cache_of is not None:
                cache = cache.reader()
            after = self.spec.schedule[stop + 1].layer if stop + 1 < len(self.spec.schedule) else None
            next_norm = self.blocks[after].first_norm if after is not None else None
            if e.pass_index is not None and self.pass_input is not None:
                ctx.pass_input = self.pass_input.inputs(first_rows, e.pass_index)
            x, pending = self.blocks[e.layer].forward(ctx, x, pending, cache, next_norm)
            if ctx.pass_input is not None:
                raise SpecError(f"the arrangement {self.spec.layers[e.layer].arrangement!r} does not take what enters the "
                                "stream before a pass of a looped range")
        n_want = ctx.want_rows.numel()
        if n_want == 0:
            return torch.empty((0, self.spec.vocab_size), dtype=torch.float32, device=x.device)
        last = self.blocks[self.spec.schedule[-1].layer]
        if hasattr(last, "leave"):                   # such an arrangement hands over the final norm's output itself
            return self.head.forward(last.leave(ctx, x, pending, ctx.want_rows, self.final_norm))
        if isinstance(pending, ops.Partials):        # the last product is still split along k
            pending = pending.materialize()
        xs = ops.gather_rows(x, ctx.want_rows)
        added = pending is None or isinstance(pending, ops.Added)   # the last block has left nothing to add
        if self.final_norm is None:
            h = xs if added else ops.add_inplace(xs, ops.gather_rows(pending, ctx.want_rows))
        elif added:
            h = self.final_norm.forward(xs)
        else:
            h = self.final_norm.add_forward(xs, ops.gather_rows(pending, ctx.want_rows))
        return self.head.forward(h)

    def weight_bytes(self) -> int:
        seen, total = set(), 0
        def add(t):
            nonlocal total
            if t is not None and t.data_ptr() not in seen:
                seen.add(t.data_ptr()); total += t.numel() * t.element_size()
        for part in self.all_parts():
            for v in vars(part).values():
                if isinstance(v, torch.Tensor):
                    add(v)
                elif isinstance(v, Linear):
                    add(v.weight)
                    add(v.bias)
        return total
