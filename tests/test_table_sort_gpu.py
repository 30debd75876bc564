"""Choices that a table names, looked up by the kernel that sorts them: the same choices, weights and results as looked up before."""

import pytest
import torch

pytestmark = pytest.mark.gpu


# slots: one, a few, one a thread, several a thread
@pytest.mark.parametrize("n,top", [(1, 1), (2, 4), (256, 4), (700, 3)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_choices_looked_up_by_the_sort(n, top, dtype):
    from dli_amd.kernels import ops

    g = torch.Generator(device="cuda").manual_seed(n)
    experts, width, ff, vocab = 7, 64, 32, 50
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").to(dtype)
    table = torch.rand(vocab, experts, generator=g, device="cuda").argsort(1)[:, :top].int().contiguous()
    tokens = torch.randint(-2, vocab + 2, (n,), generator=g, device="cuda").int()   # (ids outside the table take its first and last row)
    h, w = r(n, width), (r(experts, ff, width), r(experts, ff, width), r(experts, width, ff))
    ids, weights = torch.empty(n, top, device="cuda", dtype=torch.int32), torch.empty(n, top, device="cuda")
    ops.table_choose(table, tokens, ids, weights)
    want = ops.expert_products(ids, h, *w, 7.0, 1.0)
    ids2, weights2 = torch.full_like(ids, -1), torch.zeros_like(weights)
    got = ops.expert_products(ids2, h, *w, 7.0, 1.0, choose=(table, tokens, weights2))
    assert torch.equal(ids2, ids) and torch.equal(weights2, weights) and torch.equal(got, want)
