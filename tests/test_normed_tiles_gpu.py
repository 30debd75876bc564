"""The gated decode product behind a norm, rows normalised once a workgroup: at the edges of its pieces of 256 values, its blocks
of 128 k, its loads of the parts of the sums of squares, and of the sizes that it leaves to the general kernel."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [0, 1, 4])
@pytest.mark.parametrize("k,parts", [(128, 1), (256, 64), (384, 600), (1152, 129), (3072, 257), (4096, 1030)])
def test_gated_product_behind_a_norm(k, parts, shape):
    from dli_amd.kernels import ops

    n, eps = 48, 1e-5   # three tiles of 16: one too many for whole pairs
    gen = torch.Generator().manual_seed(k + shape)
    w = torch.randn(2 * n, k, generator=gen).mul_(k ** -0.5).bfloat16()
    bias = (0.3 * torch.randn(2 * n, generator=gen)).bfloat16()
    norm_w = 1 + 0.1 * torch.randn(k, generator=gen)
    wt = ops.tile_weights(w.cuda())
    for rows in (1, 2, 3, 4, 6, 8, 9, 15, 16):
        x = (2 * torch.randn(rows, k, generator=gen)).bfloat16()
        x[0] *= 30.0   # rows that a mixed-up sum of squares would show
        cut = torch.linspace(0, k, parts + 1).long().tolist()
        ssq = torch.stack([x[:, a:b].float().pow(2).sum(1) for a, b in zip(cut[:-1], cut[1:])]).contiguous()
        wide = torch.full((rows, k + 24), float("nan")).bfloat16()   # rows that lie further apart than they are long
        wide[:, :k] = x
        out = torch.full((rows, n + 8), 7.0, dtype=torch.bfloat16, device="cuda")
        ops.skinny_gemm(wide.cuda()[:, :k], w.cuda(), w_tiled=wt, epilogue=ops.SKINNY_SWIGLU, out=out[:, :n], bias=bias.cuda(),
                        norm_w=norm_w.cuda(), eps=eps, ssq_in=ssq.cuda(), shape=shape)
        rms = (x.double().pow(2).mean(1, keepdim=True) + eps).rsqrt()
        normed = (norm_w * (x.double() * rms).bfloat16()).bfloat16().double()
        both = (normed @ w.double().t() + bias.double()).bfloat16().double()
        gate, up = both[:, :n], both[:, n:]
        # gate and up round to 2^-9 of values of up to about four, and may round the other way; so may the norm's inputs (2^-8)
        assert (out[:, :n].cpu().double() - gate * torch.sigmoid(gate) * up).abs().max() < 0.12
        assert (out[:, n:] == 7.0).all()
