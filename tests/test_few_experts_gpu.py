"""Experts with few rows: against 64-bit arithmetic, and bit for bit against the kernels for many rows."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from dli_amd.kernels import ops as module

    return module


@pytest.mark.parametrize("width,ff", [(32, 32), (256, 64), (288, 544), (1056, 96), (1024, 800), (64, 1312)])
@pytest.mark.parametrize("weighted", [False, True])
def test_few_rows_have_the_many_rows_bits(ops, width, ff, weighted):
    gen = torch.Generator().manual_seed(width + ff)
    experts, rows = 2, 40
    w_gate, w_up = (torch.randn(experts, ff, width, generator=gen).mul_(width ** -0.5).bfloat16() for _ in range(2))
    w_down = torch.randn(experts, width, ff, generator=gen).mul_(ff ** -0.5).bfloat16()
    h = torch.randn(rows, width + 8, generator=gen).bfloat16()[:, :width]
    ids = torch.tensor([[r % 5 // 3] for r in range(rows)], dtype=torch.int32)       # 24 rows and 16
    weights = torch.rand(rows, 1, generator=gen) if weighted else None
    held = torch.zeros(rows, width + 8, dtype=torch.bfloat16, device="cuda")
    held[:, :width] = h.cuda()
    moved = [t.cuda() for t in (w_gate, w_up, w_down)]

    def run(chosen):
        x = held if len(chosen) == rows else held[chosen[0]:chosen[-1] + 1]
        return ops.expert_products(ids[chosen].cuda(), x[:, :width], *moved, 7.0, 1.702, 1.0,
                                   in_weights=None if weights is None else weights[chosen].cuda()).cpu()

    many = run(list(range(rows)))                                                     # more than 16 slots an expert
    for first, n in ((0, 1), (3, 2), (0, 17), (7, 32)):
        assert torch.equal(run(list(range(first, first + n))), many[first:first + n]), (first, n)
    x, pick = h.double(), ids[:, 0].long()
    scale = 1.0 if weights is None else weights.double()
    gate = scale * torch.einsum("rk,rfk->rf", x, w_gate.double()[pick])
    up = scale * torch.einsum("rk,rfk->rf", x, w_up.double()[pick])
    gate, up = gate.clamp(max=7.0), up.clamp(-7.0, 7.0)
    y = (gate * torch.sigmoid(1.702 * gate) * (up + 1)).bfloat16().double()
    want = torch.einsum("rf,rwf->rw", y, w_down.double()[pick])
    # a few of the intermediate's values round to bfloat16 the other way, by 2^-8 of up to about eight, times weights of ff^-0.5
    assert (many.double() - want).abs().max() < 2 ** -8 * 8 * 4 * ff ** -0.5 + 1e-5


@pytest.mark.parametrize("rows,k,ff", [(1, 32, 8), (4, 96, 24), (5, 1024, 304), (16, 2048, 40), (8, 4096, 2048), (16, 4096, 2048), (17, 64, 24)])
def test_shared_expert(rows, k, ff):
    """A mixture whose shared expert is all there is: the streaming product with the activation inside, and the library's product with
    the activation behind it (more than 16 rows, or many of wide weights), against 64-bit arithmetic."""
    from dli_amd.parts import Runtime
    from dli_amd.parts.experts import RoutedExperts

    gen, rt = torch.Generator().manual_seed(rows + k), Runtime(torch.device("cuda"), torch.bfloat16)
    part = RoutedExperts(rt, hidden_size=k, experts=0, top=1, expert_size=0, limit=7.0, identity=1, shared_size=ff, shared_limit=1.5,
                         shared_gate=False, up_shift=0.5, correction=False)
    draw = lambda *s: torch.randn(*s, generator=gen).mul_(s[-1] ** -0.5).bfloat16()
    t = {"shared.gate": draw(ff, k), "shared.up": draw(ff, k), "shared.down": draw(k, ff), "router": draw(1, k)}
    missing = set(part.weight_specs()) - set(t)
    assert not missing, missing
    part.load_weights({n: w.cuda() for n, w in t.items() if n in part.weight_specs()})
    x = draw(rows, k).mul_(k ** 0.5 * 2)
    got = part.forward(x.cuda(), None).float().cpu().double()
    xd, d = x.double(), {n: w.double() for n, w in t.items()}
    gate, up = xd @ d["shared.gate"].T, xd @ d["shared.up"].T
    gate, up = gate.bfloat16().double().clamp(max=1.5), up.bfloat16().double().clamp(-1.5, 1.5)
    want = (gate * torch.sigmoid(part.alpha * gate) * (up + 0.5)).bfloat16().double() @ d["shared.down"].T + xd
    # gate, up and their product round to 2^-9 of up to three, some the other way (2^-8), summed with weights of ff^-0.5; the
    # identity expert's row is the input, the sums stay 32-bit
    assert (got - want).abs().max() < 2 ** -8 * 3 * 4


# choices a wave sorts for itself: one, a token's, as many as there are lanes; an expert with more than a tile's rows, experts without rows,
# choices that have none (identity experts), nothing but those
@pytest.mark.parametrize("rows", [1, 3, 16])
@pytest.mark.parametrize("kind", ["spread", "one", "identity", "none"])
@pytest.mark.parametrize("table", [False, True])
def test_choices_sorted_on_the_way(ops, rows, kind, table):
    experts, top, width, ff, vocab = 8, 4, 96, 64, 40
    gen = torch.Generator().manual_seed(rows)
    most = {"spread": experts, "one": 1, "identity": experts + 4, "none": experts}[kind]
    choices = torch.randint(0, most, (vocab, top), generator=gen, dtype=torch.int32) + (experts if kind == "none" else 0)
    tokens = torch.randint(0, vocab, (rows + 20,), generator=gen, dtype=torch.int32)
    w_gate, w_up, w_down = ((torch.randn(experts, *s, generator=gen) * s[1] ** -0.5).bfloat16().cuda() for s in ((ff, width), (ff, width), (width, ff)))
    h = torch.randn(rows + 20, width, generator=gen).bfloat16().cuda()

    def run(n):
        ids = choices[tokens[:n].long()].cuda()
        given = torch.full_like(ids, -7) if table else ids.clone()
        weights = torch.zeros(n, top, device="cuda")
        z = ops.expert_products(given, h[:n], w_gate, w_up, w_down, 7.0, 1.702, 1.0,
                                choose=(choices.cuda(), tokens[:n].cuda(), weights) if table else None)
        assert torch.equal(given, ids) and (not table or (weights == 1 / top).all())
        real = (ids < experts).reshape(-1)
        return z[:rows * top][real[:rows * top]]

    assert torch.equal(run(rows), run(rows + 20))   # (80 choices and more: sorted by a kernel of its own)


# weights on the inputs of experts that a table names: the table's own, which the products' launch writes, and others
@pytest.mark.parametrize("rows", [1, 3, 4, 16])   # the most choices that the products sort themselves, and more
@pytest.mark.parametrize("own", [True, False])
def test_table_with_weights_on_the_inputs(ops, rows, own):
    experts, top, width, ff, vocab, many = 8, 4, 96, 64, 40, 36
    gen = torch.Generator().manual_seed(rows)
    choices = torch.rand(vocab, experts, generator=gen).argsort(1)[:, :top].int().contiguous()
    tokens = torch.randint(0, vocab, (many,), generator=gen, dtype=torch.int32)
    w_gate, w_up, w_down = ((torch.randn(experts, *s, generator=gen) * s[1] ** -0.5).bfloat16().cuda() for s in ((ff, width), (ff, width), (width, ff)))
    h, other = torch.randn(many, width, generator=gen).bfloat16().cuda(), torch.rand(many, top, generator=gen).cuda()

    def run(n):
        weights = torch.full((n, top), float("nan"), device="cuda")
        z = ops.expert_products(torch.full((n, top), -7, dtype=torch.int32, device="cuda"), h[:n], w_gate, w_up, w_down, 7.0, 1.702, 1.0,
                                in_weights=weights if own else other[:n], choose=(choices.cuda(), tokens[:n].cuda(), weights))
        assert (weights == 1 / top).all()
        return z[:rows * top]

    got = run(rows)
    assert got.isfinite().all() and torch.equal(got, run(many))   # (144 choices: the weights are there a launch earlier)
