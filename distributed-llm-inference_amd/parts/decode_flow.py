"""All layers of a decode step of one row in one launch (``csrc/decode_flow.hip``).

A small model's decode step of a single request is mostly the launches of its five kernels a layer. Where every
block of the model is the pre-norm arrangement of RMSNorm, rotary grouped-query attention over pages and a gated
feed-forward, in bfloat16, all of one size, the blocks describe themselves once (:meth:`Part.native_fields`, as for the loop
in C) and one kernel runs them all. Anything else, and sizes that the kernel does not take, run block by block.

The words by which the kernel's workgroups hand their results on belong to one bound list of caches, whose steps follow one
another: they are made with the description and live as long as it does."""

from __future__ import annotations

from typing import Any, Optional, Sequence

import torch

from ..kernels import ops
from .base import DecodeStream

# Of the longest context that the step's tables can hold. Up to here a wave has one pair of tiles of keys (4,096 keys) or two, all of them
# on their way at once; longer contexts the attention's own kernel cuts over more workgroups than the sixteen a kv head of this one. Kernel by
# kernel -> in one launch, a step and seven more, ms, at 8,000, 12,000, 16,000, 33,000 and 66,000 keys: 135M sizes 5.74 4.22, 6.17 4.98,
# 6.30 5.26, 7.43 7.84, 8.33 11.7; 12 layers of 1,024 with 8 heads of 128 on 2 2.99 2.30, 3.12 2.76, 3.15 2.86, 4.09 4.80, 4.76 7.43; 16 heads
# of 64 on 16 4.04 2.99, 4.42 3.47, 4.69 3.73, 6.32 5.59, 9.01 8.94. (Tables grow in powers of two: the next one holds 16,384, its tests end
# here.)
MOST_KEYS = 8192


class DecodeFlow:
    def __init__(self, fields: Sequence[dict], caches: Sequence[Any], position: Any, device: torch.device) -> None:
        f = fields[0]
        self.sizes = (len(fields), f["hidden"], f["q_heads"], f["kv_heads"], f["head_dim"], f["intermediate"])
        self.eps, self.scale, self.group, self.position = f["eps1"], f["scale"], caches[0].group, position
        rows = []
        self.keep = []   # tensors whose addresses the table holds
        for f, cache in zip(fields, caches):
            tensors = [f[n] for n in ("norm1_w", "norm2_w", "w_qkv", "w_o", "w_gate_up", "w_down")] + [cache.k_pages, cache.v_pages]
            self.keep += tensors
            rows.append([t.data_ptr() for t in tensors])
        self.table = torch.tensor(rows, dtype=torch.int64).to(device)
        self.words = torch.zeros(ops.decode_flow_bytes(*self.sizes) // 4, dtype=torch.int32, device=device)
        self.tickets = torch.zeros(1, dtype=torch.int64, device=device)

    @staticmethod
    def build(model: Any, caches: Sequence[Any]) -> Optional["DecodeFlow"]:
        """``None`` unless the kernel runs exactly these blocks on these caches."""
        if not model.rt.is_bf16 or not model.spec.schedule:
            return None
        fields = []
        for entry, cache in zip(model.spec.schedule, caches):
            layer = model.layers[entry.layer]
            f = layer.block.native_fields(layer.parts)
            if f is None or cache is None or cache.kind != "paged" or not cache.writable or cache.group != caches[0].group:
                return None
            if any(f[n] is not None for n in ("b_qkv", "b_o", "b_gate_up", "b_down")) or f["window"] or f["rotary_dim"] != f["head_dim"]:
                return None
            if (cache.window or cache.k_pages.dtype != torch.bfloat16 or cache.k_pages.shape[2] % 16
                    or tuple(cache.k_pages.shape[1:]) != (f["kv_heads"], cache.k_pages.shape[2], f["head_dim"])
                    or tuple(cache.v_pages.shape) != (cache.k_pages.shape[0], f["kv_heads"], f["head_dim"], cache.k_pages.shape[2])):
                return None
            if any(t.data_ptr() % 16 or not t.is_contiguous() for t in (f["norm1_w"], f["norm2_w"], f["w_qkv"], f["w_o"], f["w_gate_up"], f["w_down"])):
                return None
            fields.append(f)
        same = ("hidden", "q_heads", "kv_heads", "head_dim", "intermediate", "eps1", "eps2", "scale")
        first = fields[0]
        if (any(f[n] != first[n] for f in fields for n in same) or first["eps1"] != first["eps2"]
                or any(f["inv_freq"].data_ptr() != first["inv_freq"].data_ptr() for f in fields)):
            return None
        if not ops.decode_flow_bytes(len(fields), *(first[n] for n in ("hidden", "q_heads", "kv_heads", "head_dim", "intermediate"))):
            return None
        return DecodeFlow(fields, caches, model.layers[model.spec.schedule[0].layer].parts["mixer"].position, model.rt.device)

    def run(self, stream: DecodeStream, ctx: Any) -> bool:
        """All blocks on a stream of one row; False (and nothing has run) where the step is not the kernel's."""
        grp = ctx.groups[self.group]
        tables = grp.block_tables
        if stream.x.shape[0] != 1 or not stream.x.is_contiguous() or tables.shape[1] * ctx.page_size > MOST_KEYS:
            return False
        ssq = torch.empty(ops.decode_flow_parts(*self.sizes), 1, device=stream.x.device, dtype=torch.float32)
        ops.decode_flow(self.table, self.words, self.tickets, stream.x, ssq, self.position.step_angles(ctx, stream.x.dtype), grp.slots,
                        ctx.kv_len, tables, self.sizes, ctx.page_size, self.eps, self.scale)
        stream.wrote(ssq)
        return True
