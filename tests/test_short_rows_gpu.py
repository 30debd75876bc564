"""Decode products with short rows: the kernel that the plan names, at the edges where it changes."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [32, 448, 480, 576, 640, 672, 1024, 1056])
@pytest.mark.parametrize("n", [16, 100, 576])
def test_short_rows(k, n):
    from dli_amd.kernels import ops

    gen = torch.Generator().manual_seed(k + n)
    norm_w, eps = 1 + 0.1 * torch.randn(k, generator=gen), 1e-5
    for rows in (1, 3, 4):
        x = torch.randn(rows, k, generator=gen).bfloat16()
        w = torch.randn(2 * n, k, generator=gen).mul_(k ** -0.5).bfloat16()
        old = torch.randn(rows, n, generator=gen).bfloat16()
        xd, wd = x.cuda(), w.cuda()
        ssq = x.float().pow(2).sum(1).view(1, rows).cuda()
        normed = (norm_w * (x.double() * (x.double().pow(2).mean(1, keepdim=True) + eps).rsqrt()).bfloat16()).bfloat16().double()
        both = normed @ w.double().t()
        kw = dict(norm_w=norm_w.cuda(), eps=eps, ssq_in=ssq)
        # results of up to about four (a gated product of eight) round to 2^-9, and the norm's inputs may round the other way (2^-8)
        out32 = torch.empty(rows, n, device="cuda")
        ops.skinny_gemm(xd, wd[:n], epilogue=ops.SKINNY_F32, out=out32, **kw)
        assert (out32.cpu().double() - both[:, :n]).abs().max() < 2e-2
        out = torch.empty(rows, n, dtype=torch.bfloat16, device="cuda") if n % 8 == 0 else torch.empty(rows, n + 4, dtype=torch.bfloat16, device="cuda")[:, :n]
        ops.skinny_gemm(xd, wd[:n], epilogue=ops.SKINNY_STORE, out=out, **kw)
        assert (out.cpu().double() - both[:, :n]).abs().max() < 3e-2
        ops.skinny_gemm(xd, wd, epilogue=ops.SKINNY_SWIGLU, out=out, **kw)
        gate = both[:, :n].bfloat16().double()
        assert (out.cpu().double() - gate * torch.sigmoid(gate) * both[:, n:]).abs().max() < 0.12
        stream = old.cuda()
        parts = ops.skinny_gemm(xd, wd[:n], epilogue=ops.SKINNY_RESIDUAL, stream=stream)
        want = old.double() + (x.double() @ w[:n].double().t()).bfloat16().double()
        assert (stream.cpu().double() - want).abs().max() < 3e-2
        assert parts.shape[0] == ops.skinny_gemm_plan(rows, n, k, ops.SKINNY_RESIDUAL, xd.device)[2]
        total = stream.cpu().double().pow(2).sum(1)
        assert ((parts.sum(0).cpu().double() - total).abs() <= 1e-4 * total).all()


@pytest.mark.parametrize("m", [1, 4, 5, 16])
@pytest.mark.parametrize("qh,kvh,d,k,bs,shape", [(9, 3, 64, 576, 16, None), (2, 1, 16, 32, 16, 0), (15, 5, 64, 960, 16, 4),
                                                 (4, 4, 32, 1056, 8, 1), (3, 1, 64, 160, 16, 2), (3, 1, 64, 224, 16, 3)])
def test_the_rotating_product_takes_a_last_block_that_is_not_whole(m, qh, kvh, d, k, bs, shape):
    import test_kernels_gpu as kernels

    from dli_amd.kernels import ops

    kernels.test_skinny_gemm_qkv_with_rotation_and_cache_write(ops, m, qh, kvh, d, k, bs, shape)
