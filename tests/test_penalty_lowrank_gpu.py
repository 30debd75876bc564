"""The grouped attention's penalty on the distance, and the low-rank projection's second half with many rows."""

from __future__ import annotations

import pytest
import torch

import plain_makodra as P
from test_makodra_gpu import i32, paged

pytestmark = pytest.mark.gpu
F = torch.float64


@pytest.fixture(scope="module")
def ops():
    from dli_amd.kernels import ops as module

    return module


@pytest.mark.parametrize("H,G,D,V,ps", [(4, 2, 32, 16, 16), (8, 2, 64, 64, 16), (6, 2, 40, 128, 8), (66, 1, 16, 48, 16), (3, 3, 104, 100, 8)])
@pytest.mark.parametrize("scale", [0.7, -0.4])
def test_grouped_attention_with_a_penalty(ops, H, G, D, V, ps, scale):
    gen = torch.Generator().manual_seed(H * 100 + D)
    n = 150
    q = P.rms(torch.randn(n, H, D, dtype=F, generator=gen), 1e-6).bfloat16().double()
    k = P.rms(torch.randn(n, G, D, dtype=F, generator=gen), 1e-6).bfloat16().double()
    v = torch.randn(n, G, V, dtype=F, generator=gen).bfloat16().double()
    r1, r2 = 0.2 + torch.rand(H, generator=gen), 0.1 + 2 * torch.rand(H, generator=gen)
    gate = torch.randn(n, H * V, generator=gen)
    kp, vp, table = paged(k, v, ps, torch.bfloat16)
    tokens = ops.attention_grouped_tile_tokens(H, G)
    for case in (dict(), dict(sink=True), dict(chunk=64, sink=True), dict(chunk=37), dict(window=50), dict(window=1, chunk=64)):
        ref = P.scored_attention_core(q, k, v, scale, chunk=case.get("chunk", 0), window=case.get("window", 0),
                                      sink=case.get("sink", False), r1=r1.double(), r2=r2.double()).reshape(n, H * V)
        for first in (0, 63, 64, n - 3):
            rows = n - first
            starts = range(0, rows, tokens)
            for out32 in (False, True):
                out = torch.empty(rows, H * V, dtype=torch.float32 if out32 else torch.bfloat16, device="cuda")
                ops.attention_grouped(q[first:].reshape(rows, H * D).bfloat16().cuda(), kp.cuda(), vp.cuda(), out, i32([0, rows]),
                                      i32([n]), i32(table).view(1, -1), i32([0] * len(starts)), i32(list(starts)), H, scale,
                                      r1=r1.cuda(), r2=r2.cuda(), gate=gate[first:].cuda(), **case)
                want = ref[first:] * torch.sigmoid(gate[first:].double())
                # weights are rounded to bfloat16 for the second product: 2^-9 of values of up to about four
                assert (out.cpu().double() - want).abs().max() < 3e-2, (case, first, out32)


@pytest.mark.parametrize("rows,features,rank", [(rows, *sizes) for rows in (767, 768, 769, 1000)
                                                for sizes in ((4, 4), (260, 8), (1024, 64), (96, 512))]
                         + [(1009, 4100, 4), (2050, 1604, 8), (770, 2308, 64), (257, 4612, 128), (1023, 772, 512), (300, 100, 128),
                            (300, 1028, 100), (7, 33, 21)])
def test_lowrank_rows_have_the_single_rows_bits(ops, rows, features, rank):
    """Rows made sixteen a workgroup, rows of few and of many workgroups of their own: the bits of a row alone."""
    assert bool(ops.library().dli_lowrank_takes_rows(rows, features, rank)) == (
        (rows, features, rank) in ((1009, 4100, 4), (2050, 1604, 8), (770, 2308, 64), (257, 4612, 128), (1023, 772, 512)))
    gen = torch.Generator(device="cuda").manual_seed(rows + features)
    t = torch.randn(rows, rank + 3, device="cuda", generator=gen)[:, :rank]
    w2t, bias = torch.randn(rank, features, device="cuda", generator=gen), torch.randn(features, device="cuda", generator=gen)
    rate, rate_bias = torch.randn(rows, features + 4, device="cuda", generator=gen)[:, :features], bias * 0.5
    for act, out_act in (("tanh", "delta_decay"), ("tanh", "double_exp_decay"), ("none", "softplus")):
        many, rates = torch.empty(rows, features, device="cuda"), rate.clone()
        wide = torch.empty(rows, features + 4, device="cuda")[:, :features]
        wide.copy_(rate)
        ops.lowrank_out(t, w2t, bias, many, act=act, out_act=out_act, rate=wide, rate_bias=rate_bias)
        for r in (0, rows // 2, rows - 1):
            one, one_rate = torch.empty(1, features, device="cuda"), rates[r:r + 1].contiguous()
            ops.lowrank_out(t[r:r + 1], w2t, bias, one, act=act, out_act=out_act, rate=one_rate, rate_bias=rate_bias)
            assert torch.equal(one[0], many[r]) and torch.equal(one_rate[0], wide[r])
