"""Runs of like layers that decode steps of few rows take in one kernel (`ops.layer_run`): pre-norm blocks of plain grouped-query
attention over caches of their own and a SiLU feed-forward, without biases, windows or sinks, heads of 128 that are normed and
turned whole.  The model asks for the run that begins with its first layer; steps that the kernel does not take, and layers behind the run, go
through the blocks."""
from __future__ import annotations

from typing import List, Optional, Tuple

import torch

from .. import ops
from .attention import Attention
from .block import Block
from .mlp import GatedMlp
from .norm import RMSNorm


def _kind(block) -> Optional[Tuple]:
    """What two layers of one run have in common; None for a layer that the kernel does not take."""
    if type(block) is not Block or type(block.mixer) is not Attention or type(block.ffn) is not GatedMlp:
        return None
    a, f, norms = block.mixer, block.ffn, (block.norm_mixer, block.norm_ffn)
    if not a.plain or any(type(n) is not RMSNorm for n in norms):
        return None
    s = a.spec
    if (a.qkv.weight.dtype != torch.bfloat16 or s.head_dim != 128 or s.window or s.sink or a.q_norm_w is None or a.position.rot_dim != 128
            or a.position.interleaved or a.qkv.bias is not None or a.o.bias is not None):
        return None
    if f.spec.activation != "silu" or f.gate_up.bias is not None or f.down.bias is not None:
        return None
    return (s.hidden, f.spec.intermediate, s.n_heads, s.n_kv_heads, s.softmax_scale, a.position.spec, a.norm_eps, a.norm_add_one,
            norms[0].eps, norms[0].add_one, norms[1].eps, norms[1].add_one)


class LayerRun:
    """The first `length` stops of a model's schedule as one run.  One layer or two gain as well (us a step at 700 keys, five kernels a layer / a run,
    1 row: models of one layer, 0.6B shape 45 / 36, 8B 114 / 103, of two 73 / 51 and 199 / 165; the first of five layers 155 / 149 and 460 / 458, the
    first two 155 / 136 and 462 / 433)."""

    def __init__(self, blocks: List[Block], stops: List[int]):
        self.blocks, self.length = blocks, len(blocks)
        self.stops = stops                               # whose caches the layers write, in the order of the run

    @classmethod
    def of_model(cls, spec, blocks) -> Optional["LayerRun"]:
        run, stops, first = [], [], None
        for stop, e in enumerate(spec.schedule):
            kind = _kind(blocks[e.layer]) if e.cache_of is None and e.pass_index is None else None
            if kind is None or (run and kind != first):
                break
            first = kind
            run.append(blocks[e.layer])
            stops.append(stop)
        return cls(run, stops) if run else None

    def takes(self, ctx, x: torch.Tensor, storage) -> Optional[List[Tuple[torch.Tensor, ...]]]:
        """The layers' arrays where this step goes through the kernel, else None: one token a request, few of them, all layers' pages in one table."""
        if ctx.max_q_len != 1 or ctx.run_words is None or not (0 < x.shape[0] <= ops.RUN_MAX_ROWS):
            return None
        b, caches = self.blocks[0], [storage.layers.get(s) for s in self.stops]
        s = b.mixer.spec
        sizes = (x.shape[0], s.hidden, b.ffn.spec.intermediate, s.n_heads, s.n_kv_heads)
        if (ops.MID_PRODUCTS != "own" or ops.MID_FROM_ROWS is not None) and x.shape[0] >= ops.mid_from_rows(s.hidden):
            return None                                  # (a switch says which kernels the products of so many rows take)
        if (not all(c is not None and c.writable and c.group == caches[0].group for c in caches)
                or not ops.layer_run_fits(*sizes, ctx.groups[caches[0].group].page_size) or not ops.layer_run_pays(*sizes, ctx.max_kv_len, self.length)):
            return None
        layers = [(m.mixer.qkv.weight, m.mixer.o.weight, m.ffn.gate_up.weight, m.ffn.down.weight, m.norm_mixer.weight, m.norm_ffn.weight,
                   m.mixer.q_norm_w, m.mixer.k_norm_w, c.k, c.v) for m, c in zip(self.blocks, caches)]
        return layers if ops.layer_run_aligned(layers) else None

    def forward(self, ctx, x: torch.Tensor, layers: List[Tuple[torch.Tensor, ...]], storage) -> torch.Tensor:
        """The stream after the run, in place; `layers` as `takes` has given them."""
        b = self.blocks[0]
        a, s, group = b.mixer, b.mixer.spec, ctx.groups[storage.layers[self.stops[0]].group]
        cos, sin = ctx.position_table(a.position)
        return ops.layer_run(x, layers, ctx.run_words, ctx.positions, group.slots, group.block_table, cos, sin, nq=s.n_heads, nkv=s.n_kv_heads,
                             ff=b.ffn.spec.intermediate, max_kv_len=ctx.max_kv_len, eps=(b.norm_mixer.eps, b.norm_ffn.eps, a.norm_eps),
                             add_one=(b.norm_mixer.add_one, b.norm_ffn.add_one, a.norm_add_one), scale=s.softmax_scale)
