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
