"""Experts combined into the residual stream with the norms behind it: the stream bit for bit as combination and sum give it one
after the other, the norms within rounding of the pair's own kernel."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from dli_amd.kernels import ops as o
    return o


# widths: one piece of four, less than and more than a piece a thread (256 and 512 threads), beyond the two that are kept
@pytest.mark.parametrize("n,top,width", [(1, 1, 4), (2, 4, 1024), (3, 5, 1028), (2, 4, 2048), (300, 6, 2052), (5, 2, 4100), (2, 9, 8192)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("form", ["plain", "shared", "gated", "ones"])
def test_combined_into_the_stream(ops, n, top, width, dtype, form):
    g = torch.Generator(device="cuda").manual_seed(n * width + top)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    experts = 6
    ids = torch.randint(0, experts + 2, (n, top), generator=g, device="cuda").int()   # two identity experts among them
    z, h, x, a, weights = r(n * top, width), r(n, width).to(dtype), r(n, width), r(n, width), torch.rand(n, top, generator=g, device="cuda")
    z[(ids >= experts).reshape(-1)] = float("nan")                                    # rows that nobody has written
    w1, w2 = 1 + 0.1 * r(width), 1 + 0.1 * r(width)
    kw = dict(shared=r(n, width + 4)[:, :width]) if form in ("shared", "gated") else {}
    if form == "gated":
        kw["shared_gate"] = r(n, 3)[:, 1:2]
    weights = None if form == "ones" else weights
    out, want, h1, h2 = torch.empty_like(x), x.clone(), torch.empty_like(h), torch.empty_like(h)
    ops.expert_combine(ids, weights, z, h, experts, out, **kw)
    ops.add_pair_into_stream(want, a, out)
    ops.rms_norm_pair(want, w1, w2, 1e-6, h1, h2)
    alone, both, g1, g2 = x.clone(), x.clone(), torch.empty_like(h), torch.empty_like(h)
    assert ops.expert_combine_stream_supports(alone, a, z, kw.get("shared"))
    ops.expert_combine_stream(ids, weights, z, h, experts, alone, a, **kw)
    ops.expert_combine_stream(ids, weights, z, h, experts, both, a, w1=w1, w2=w2, eps=1e-6, out1=g1, out2=g2, **kw)
    assert torch.equal(alone, want) and torch.equal(both, want)
    # sums of squares in another order: a few of the last bits of 24, of a value or of its rounding to eight
    for one, other in ((g1, h1), (g2, h2)):
        assert ((one.double() - other.double()).abs() <= other.double().abs() * (2 ** -7 if dtype == torch.bfloat16 else 2 ** -20)).all()
