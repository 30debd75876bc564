"""The few-row product where its waves have no block of k, one, two or more: the order in which blocks are asked for goes by that
and by the rows."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("k", [32, 128, 480, 576, 640, 1024, 1152, 2048, 2080, 3200, 4608])
def test_blocks_of_a_wave(k, shape):
    from dli_amd.kernels import ops

    n = 80
    gen = torch.Generator().manual_seed(k + shape)
    w = torch.randn(2 * n, k, generator=gen).mul_(k ** -0.5).bfloat16()
    norm_w, eps = 1 + 0.1 * torch.randn(k, generator=gen), 1e-5
    for tiled in (False, True) if k % 128 == 0 else (False,):
        one, both = (ops.tile_weights(m.contiguous().cuda()) if tiled else None for m in (w[:n], w))
        for rows in (1, 3, 4, 5, 16):
            x = torch.randn(rows, k, generator=gen).bfloat16()
            want = x.double() @ w[:n].double().t()
            args = dict(shape=shape, w_tiled=one)
            out = torch.full((rows, n), 7.0, device="cuda")
            ops.skinny_gemm(x.cuda(), w[:n].contiguous().cuda(), epilogue=ops.SKINNY_F32, out=out, **args)
            # 32-bit sums of k products of about k^-1/2 each
            assert (out.cpu().double() - want).abs().max() < 2e-5
            old = torch.randn(rows, n, generator=gen).bfloat16()
            stream = old.cuda()
            ssq = ops.skinny_gemm(x.cuda(), w[:n].contiguous().cuda(), epilogue=ops.SKINNY_RESIDUAL, stream=stream, **args)
            summed = old.double() + want.bfloat16().double()
            assert (stream.cpu().double() - summed).abs().max() < 0.04   # two roundings to 2^-9 of values up to about six
            assert torch.allclose(ssq.sum(0).cpu().double(), stream.cpu().double().pow(2).sum(1), rtol=1e-5)
            act = torch.empty(rows, n, dtype=torch.bfloat16, device="cuda")
            sums = x.float().pow(2).sum(1)[None].contiguous().cuda()
            ops.skinny_gemm(x.cuda(), w.cuda(), epilogue=ops.SKINNY_SWIGLU, out=act, norm_w=norm_w.cuda(), eps=eps, ssq_in=sums,
                            shape=shape, w_tiled=both)
            rms = (x.double().pow(2).mean(1, keepdim=True) + eps).rsqrt()
            normed = (norm_w * (x.double() * rms).bfloat16()).bfloat16().double()
            gate, up = (normed @ m.double().t() for m in (w[:n], w[n:]))
            # as in the test of the gated product behind a norm, without its row of large values
            assert (act.cpu().double() - gate * torch.sigmoid(gate) * up).abs().max() < 0.12
