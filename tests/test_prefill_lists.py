"""What a step's layers share of the prompt attention's tile lists, where they differ in their heads; which masked portions it takes."""

import numpy as np
import pytest
import torch


def _context(monkeypatch, new):
    from dli_amd.engine import batch
    from dli_amd.kernels import ops

    monkeypatch.setattr(ops, "compute_units", lambda device: 256)
    monkeypatch.setattr(batch, "upload", lambda arrays, device: [torch.from_numpy(np.ascontiguousarray(a)) for a in arrays])
    empty, width = torch.zeros(0, dtype=torch.int32), -(-max(new) // 16)
    q_start = np.concatenate([[0], np.cumsum(new)]).astype(np.int32)
    return batch.StepContext(device=torch.device("cpu"), page_size=16, num_tokens=int(q_start[-1]), num_entries=len(new), num_decode=0,
                             token_ids=empty, positions=empty, q_start=empty, kv_len=empty, state_slots=empty, logit_rows=empty,
                             groups=[batch.GroupView(empty, torch.zeros(len(new), width, dtype=torch.int32), width)],
                             q_start_host=q_start, kv_len_host=np.asarray(new, np.int32))


# the smaller heads first and the larger; more heads and fewer on the same tiles; prompts that are cut and one that is not
@pytest.mark.parametrize("tokens", [300, 1600, 2048])
@pytest.mark.parametrize("shapes", [[(64, 32, 8), (128, 32, 8), (32, 32, 8)], [(128, 32, 8), (64, 32, 8)], [(64, 16, 4), (64, 32, 8), (112, 16, 4)]])
def test_every_shape_has_buffers_of_its_own_size(monkeypatch, tokens, shapes):
    from dli_amd.kernels import ops
    from dli_amd.parts.attention_kernels import prefill_tiles

    ctx = _context(monkeypatch, [tokens])
    made = [prefill_tiles(ctx, *shape, 0, ctx.device) for shape in shapes]
    for (dim, heads, kv), t in zip(shapes, made):
        assert (t.cut is None) == (tokens == 300)
        if t.cut is not None:
            assert t.cut_buf.numel() == t.cut_tiles * t.cut_room * ops.attention_prefill_cut_floats(dim, heads, kv)
            assert t.cut_count.numel() == t.cut_tiles * heads
    assert [prefill_tiles(ctx, *shape, 0, ctx.device) for shape in shapes] == made   # one a shape and step
    alike = [t for (_, heads, kv), t in zip(shapes, made) if (heads, kv) == (32, 8)]
    assert all(t.entry is alike[0].entry and t.q0 is alike[0].q0 and t.cut is alike[0].cut for t in alike)   # the list is one


def test_which_portions_share_key_tiles():
    from dli_amd.parts.attention_kernels import PLAIN_FROM_PAIRS, plain_pays

    many, more = 40 << 20, 64 << 20
    assert PLAIN_FROM_PAIRS <= many
    assert all(plain_pays(*s) for s in [(64, 32, 8, many, 0), (64, 32, 8, many, 32), (128, 16, 8, many, 48), (64, 32, 32, many, 80), (64, 16, 8, more, 48),
                                        (48, 24, 8, more, 80), (128, 32, 8, many, 2048), (64, 16, 4, more, 1024)])
    assert not any(plain_pays(*s) for s in [(64, 32, 8, PLAIN_FROM_PAIRS - 1, 0), (64, 32, 8, many, 16), (128, 16, 8, many, 32), (64, 32, 32, many, 64),
                                            (48, 24, 8, more, 48), (16, 32, 8, more, 0), (16, 32, 8, more, 2048), (64, 32, 32, 16 * many, 64),
                                            (64, 16, 4, many, 1024), (64, 16, 4, many, 0)])


def test_a_no_is_asked_for_once_a_step(monkeypatch):
    """Layers of a step whose portions stay with the kernel for changed scores ask for its plan, which is made once all the same."""
    from types import SimpleNamespace

    from dli_amd.parts import attention_kernels as A

    ctx, asked = _context(monkeypatch, [100]), []
    monkeypatch.setattr(A, "plain_pays", lambda *a: asked.append(a))
    q, k, v = torch.zeros(100, 256).bfloat16(), torch.zeros(7, 2, 16, 64).bfloat16(), torch.zeros(7, 2, 64, 16).bfloat16()
    for _ in range(3):
        assert not A.plain_portions(q, k, v, torch.zeros_like(q), ctx, SimpleNamespace(group=0), 4, 0.125, chunk=48)
    assert len(asked) == 1
