"""Portions whose mask is all that changes their attention: the kernel that shares key tiles against the one for changed scores."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


class _Cache:
    def __init__(self, k, v):
        self.group, self.k_pages, self.v_pages = 0, k, v


def _context(page, old, new, decode):
    """A step of `decode` single tokens and then portions, over pages in no order."""
    from dli_amd.engine.batch import GroupView, StepContext

    kv = np.asarray(old, np.int32) + np.asarray(new, np.int32)
    q_start = np.concatenate([[0], np.cumsum(new)]).astype(np.int32)
    width = int(-(-kv.max() // page)) + 1
    tables = np.random.default_rng(1).permutation(len(new) * width).reshape(len(new), width).astype(np.int32)
    on = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    empty = torch.zeros(0, dtype=torch.int32, device="cuda")
    positions = np.concatenate([np.arange(o, o + n) for o, n in zip(old, new)]).astype(np.int32)
    ctx = StepContext(device=torch.device("cuda"), page_size=page, num_tokens=int(q_start[-1]), num_entries=len(new), num_decode=decode,
                      token_ids=empty, positions=on(positions), q_start=on(q_start), kv_len=on(kv), state_slots=empty, logit_rows=empty,
                      groups=[GroupView(empty, on(tables), width)], q_start_host=q_start, kv_len_host=kv)
    return ctx, len(new) * width


# chunks that are met and not, whose edges rows and cached keys lie on and beside, one key a piece; windows met, not met, and not met beside kept
# positions; heads of all kinds that share tiles; pages of one tile and of several; single tokens in front
@pytest.mark.parametrize("masks,page", [({"chunk": 64}, 16), ({"chunk": 192}, 32), ({"chunk": 4096}, 16), ({"window": 100}, 16), ({}, 64),
                                        ({"window": 4096, "keep_first": 4}, 16), ({"chunk": 64, "window": 4096}, 16)])
@pytest.mark.parametrize("heads,kv,dim", [(4, 1, 64), (8, 8, 64), (6, 2, 128), (3, 3, 48)])
def test_same_results(monkeypatch, masks, page, heads, kv, dim):
    from dli_amd.kernels import ops
    from dli_amd.parts import attention_kernels as A

    monkeypatch.setattr(A, "PLAIN_FROM_PAIRS", 0)
    old, new = [70, 0, 63, 64, 65, 0, 130], [1, 200, 1, 64, 63, 3, 700]
    ctx, pages = _context(page, old, new, 1)
    gen = torch.Generator(device="cuda").manual_seed(heads + page)
    draw = lambda *s: torch.randn(*s, device="cuda", generator=gen).bfloat16()
    n = ctx.num_tokens
    q, k, v = draw(n, heads * dim), draw(pages, kv, page, dim), draw(pages, kv, dim, page)
    got, want = torch.zeros(n, heads * dim, device="cuda").bfloat16(), torch.zeros(n, heads * dim, device="cuda").bfloat16()
    assert A.plain_portions(q, k, v, got, ctx, _Cache(k, v), heads, dim ** -0.5, **masks)
    tiles = ctx.q_tiles(ops.attention_grouped_tile_tokens(heads, kv), first_entry=1)
    ops.attention_grouped(q, k, v, want, ctx.q_start, ctx.kv_len, ctx.groups[0].block_tables, tiles[0], tiles[1], heads, dim ** -0.5, **masks)
    # weights are rounded to bfloat16 (2^-9 each at most) against one reference point or another, and the results once more
    assert (got[1:].float() - want[1:].float()).abs().max() <= 3 * 2.0 ** -9 * want.float().abs().max()
    assert not got[0].any()   # the single token's row is another kernel's


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("spread", [1, 2, 4])
@pytest.mark.parametrize("masks", [{}, {"chunk": 512}, {"window": 300}])
def test_no_further_from_64_bits(monkeypatch, masks, spread, dim):
    """Scores of this standard deviation, up to one key for all there is: as far from 64-bit arithmetic as the kernel for changed scores
    (2-norm over 12,000 rows of a head, whose chance is well below 1%), with 2% for that chance."""
    from dli_amd.kernels import ops
    from dli_amd.parts import attention_kernels as A

    monkeypatch.setattr(A, "PLAIN_FROM_PAIRS", 0)
    heads, kv, n = 8, 2, 1500
    ctx, pages = _context(16, [0], [n], 0)
    gen = torch.Generator(device="cuda").manual_seed(spread)
    draw = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    q, k, v = (draw(n, heads * dim) * spread).bfloat16(), draw(pages, kv, 16, dim).bfloat16(), draw(pages, kv, dim, 16).bfloat16()
    got, other = torch.zeros_like(q), torch.zeros_like(q)
    assert A.plain_portions(q, k, v, got, ctx, _Cache(k, v), heads, dim ** -0.5, **masks)
    tiles = ctx.q_tiles(ops.attention_grouped_tile_tokens(heads, kv))
    ops.attention_grouped(q, k, v, other, ctx.q_start, ctx.kv_len, ctx.groups[0].block_tables, tiles[0], tiles[1], heads, dim ** -0.5, **masks)
    table = ctx.groups[0].block_tables[0].long()
    keys, values = k[table].transpose(1, 2).reshape(-1, kv, dim)[:n], v[table].permute(0, 3, 1, 2).reshape(-1, kv, dim)[:n]
    keys, values = (t.double().repeat_interleave(heads // kv, 1).transpose(0, 1) for t in (keys, values))
    scores = torch.matmul(q.view(n, heads, dim).transpose(0, 1).double(), keys.transpose(1, 2).contiguous()) * dim ** -0.5
    at = torch.arange(n, device="cuda")
    seen = at[None] <= at[:, None]
    if "chunk" in masks:
        seen &= at[None] // 512 == at[:, None] // 512
    if "window" in masks:
        seen &= at[None] > at[:, None] - 300
    want = torch.matmul(scores.masked_fill(~seen, -torch.inf).softmax(-1), values).transpose(0, 1).reshape(n, -1)
    far, far_other = ((o.double() - want).norm().item() for o in (got, other))
    assert far <= 1.02 * far_other, far / far_other


def test_layers_with_heads_of_two_sizes_in_one_step():
    """A prompt whose longest tiles have their keys cut, in a step whose layers differ in their head size."""
    from dli_amd.kernels import ops
    from dli_amd.parts import attention_kernels as A

    heads, kv, n = 32, 8, 1600
    ctx, pages = _context(16, [0], [n], 0)
    gen = torch.Generator(device="cuda").manual_seed(2)
    draw = lambda *s: torch.randn(*s, device="cuda", generator=gen).bfloat16()
    for dim in (64, 128, 64):
        q, k, v = draw(n, heads * dim), draw(pages, kv, 16, dim), draw(pages, kv, dim, 16)
        got, want = torch.zeros_like(q), torch.zeros_like(q)
        assert A.plain_portions(q, k, v, got, ctx, _Cache(k, v), heads, dim ** -0.5, chunk=4096)
        tiles = ctx.q_tiles(ops.attention_grouped_tile_tokens(heads, kv))
        ops.attention_grouped(q, k, v, want, ctx.q_start, ctx.kv_len, ctx.groups[0].block_tables, tiles[0], tiles[1], heads, dim ** -0.5, chunk=4096)
        assert (got.float() - want.float()).abs().max() <= 3 * 2.0 ** -9 * want.float().abs().max()   # as above
    assert A.prefill_tiles(ctx, 64, heads, kv, 0, q.device).cut is not None


def test_what_stays_with_the_kernel_for_changed_scores(monkeypatch):
    from dli_amd.parts import attention_kernels as A

    monkeypatch.setattr(A, "PLAIN_FROM_PAIRS", 0)

    def takes(page=16, v_dim=64, out=torch.bfloat16, scale=0.125, **masks):
        ctx, pages = _context(page, [0], [300], 0)
        k, v = torch.zeros(pages, 2, page, 64, device="cuda").bfloat16(), torch.zeros(pages, 2, v_dim, page, device="cuda").bfloat16()
        q = torch.zeros(300, 256, device="cuda").bfloat16()
        return A.plain_portions(q, k, v, torch.zeros(300, 4 * v_dim, device="cuda", dtype=out), ctx, _Cache(k, v), 4, scale, **masks)

    assert takes() and takes(chunk=64)
    assert not any([takes(chunk=40), takes(page=8), takes(v_dim=32), takes(out=torch.float32), takes(scale=-0.125), takes(window=64, keep_first=4),
                    takes(chunk=64, window=100)])
    monkeypatch.setattr(A, "PLAIN_FROM_PAIRS", 4 * 300 * 151)
    assert not takes()
