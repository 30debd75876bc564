"""Rotation and cache write of many rows (sixteen neighbours to an XCD) against the same rows a hundred at a time: the same bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from dli_amd.kernels import ops as o
    return o


def _pages(n, kv, d):
    return [torch.full(s, 3.0, device="cuda", dtype=torch.bfloat16) for s in ((n // 16 + 2, kv, 16, d), (n // 16 + 2, kv, d, 16))]


# rows: the first that are taken so, a block's end and past it; `shift`: bias and norm weights that begin at no whole vector
@pytest.mark.parametrize("n", [127, 128, 129, 1100])
@pytest.mark.parametrize("heads,kv,d,rot,shift", [(4, 2, 64, 32, 0), (4, 2, 64, 64, 1), (3, 1, 20, 8, 0), (2, 1, 10, 6, 0)])
def test_rotary_cache_of_many_rows(ops, n, heads, kv, d, rot, shift):
    g = torch.Generator(device="cuda").manual_seed(n + d)
    width = (heads + 2 * kv) * d
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    proj, bias, norm = r(n, width + 4), r(width + 5)[shift:shift + width + 4], (r(heads * d + 1)[shift:shift + heads * d], r(kv * d + 1)[shift:shift + kv * d], 1e-6)
    positions, slots = torch.arange(5, 5 + n, device="cuda").int(), torch.arange(n, device="cuda").int()
    slots[n // 2] = -1
    freq = torch.rand(rot // 2, device="cuda", generator=g)
    results = []
    for cut in (n, 100):
        (k, v), q = _pages(n, kv, d), torch.empty(n, heads * d, device="cuda", dtype=torch.bfloat16)
        for a in range(0, n, cut):
            s = slice(a, min(n, a + cut))
            ops.rotary_cache(proj[s], 0, heads * d, (heads + kv) * d, positions[s], freq, rot, False, q[s], slots[s].contiguous(), k, v, heads,
                             bias=bias, row_norm=norm)
        results.append((q, k, v))
    assert all(torch.equal(one, other) for one, other in zip(*results))


@pytest.mark.parametrize("n", [127, 128, 129, 1100])
def test_unit_keys_of_many_rows(ops, n):
    g = torch.Generator(device="cuda").manual_seed(n)
    heads, kv, d = 6, 2, 48
    proj, slots = torch.randn(n, (heads + 2 * kv) * d, generator=g, device="cuda"), torch.arange(n, device="cuda").int()
    slots[n // 2] = -1
    results = []
    for cut in (n, 100):
        (k, v), q = _pages(n, kv, d), torch.empty(n, heads * d, device="cuda", dtype=torch.bfloat16)
        for a in range(0, n, cut):
            s = slice(a, min(n, a + cut))
            ops.qk_unit_cache(proj[s], 0, heads * d, (heads + kv) * d, q[s], slots[s].contiguous(), k, v, heads, 1e-6)
        results.append((q, k, v))
    assert all(torch.equal(one, other) for one, other in zip(*results))
