"""A row's sum of squares behind a norm, alone in its step and among others."""

from __future__ import annotations

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from dli_amd.kernels import ops as o

    o.library()
    return o


@pytest.mark.parametrize("k,parts", [(256, 16), (576, 36), (1024, 64), (1920, 600)])
def test_a_row_alone_is_summed_as_among_others(ops, k, parts):
    """The q/k/v product behind a norm gives a row of fewer than 2,048 values the same bits in a step of one request and of
    several: its sum of squares is added in the same order (parts whose sums depend on it)."""
    gen = torch.Generator().manual_seed(k)
    qh, kvh, d = 4, 2, 64
    wq = ops.tile_weights_qkv_rope((torch.randn((qh + 2 * kvh) * d, k, generator=gen) / math.sqrt(k)).bfloat16().cuda(), qh, kvh, d)
    norm_w = (1 + 0.1 * torch.randn(k, generator=gen)).cuda()
    kp, vp = torch.zeros(4, kvh, 16, d, device="cuda").bfloat16(), torch.zeros(4, kvh, d, 16, device="cuda").bfloat16()
    angles = torch.rand(3, 2, d // 2, generator=gen).cuda()
    slots = torch.arange(3, dtype=torch.int32, device="cuda")
    for _ in range(40):
        x = torch.randn(3, k, generator=gen).bfloat16().cuda()
        ssq = (torch.rand(parts, 3, generator=gen) * k / parts * 2).cuda()
        got = {}
        for rows in (1, 3):
            q = torch.empty(rows, qh * d, dtype=torch.bfloat16, device="cuda")
            ops.skinny_gemm_qkv_rope(x[:rows], wq, q, angles[:rows], slots[:rows], kp, vp, qh, norm_w=norm_w, eps=1e-5,
                                     ssq_in=ssq[:, :rows].contiguous())
            got[rows] = q[0], kp[0, :, 0].clone(), vp[0, :, :, 0].clone()
        assert all(torch.equal(a, b) for a, b in zip(got[1], got[3]))


# parts: one trip, and more than a workgroup asks for at once (64 a wave of four or eight)
@pytest.mark.parametrize("k,parts", [(256, 16), (640, 40), (1024, 64), (1024, 520), (1920, 600)])
@pytest.mark.parametrize("n", [16, 512, 1536])
def test_a_gated_row_alone_is_summed_as_among_others(ops, n, k, parts):
    """The same for the gated product."""
    gen = torch.Generator().manual_seed(n + k)
    w = (torch.randn(2 * n, k, generator=gen) / math.sqrt(k)).bfloat16().cuda()
    tiled, norm_w = ops.tile_weights(w), (1 + 0.1 * torch.randn(k, generator=gen)).cuda()
    assert all(ops.skinny_gemm_plan(rows, n, k, ops.SKINNY_SWIGLU, w.device, tiled=True)[0] == "tiles16" for rows in (1, 3))
    for _ in range(40):
        x = torch.randn(3, k, generator=gen).bfloat16().cuda()
        ssq = (torch.rand(parts, 3, generator=gen) * k / parts * 2).cuda()
        got = {}
        for rows in (1, 3):
            out = torch.empty(rows, n, dtype=torch.bfloat16, device="cuda")
            ops.skinny_gemm(x[:rows], w, w_tiled=tiled, epilogue=ops.SKINNY_SWIGLU, out=out, norm_w=norm_w, eps=1e-5,
                            ssq_in=ssq[:, :rows].contiguous())
            got[rows] = out[0]
        assert torch.equal(got[1], got[3])
