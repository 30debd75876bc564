"""The 32-bit few-row products that read w by way of LDS: the bits of the kernel that reads it word by word, and of the norm's,
product's and activation's kernels one after the other."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


# k: one half of a run, a last run of one half, several segments a wave, two and four runs a segment with and without a rest;
# columns: part of a tile, and tiles enough for 4, 8 and 16 waves each
@pytest.mark.parametrize("m", [1, 5, 16])
@pytest.mark.parametrize("n,k", [(15, 64), (17, 192), (600, 576), (20000, 320), (4500, 1088), (33, 2048), (90, 4160), (48, 8192)])
def test_through_lds_and_word_by_word(m, n, k):
    from dli_amd.kernels import ops

    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, w = torch.randn(m, k, device="cuda", generator=g), torch.randn(n, k, device="cuda", generator=g)
    odd = torch.empty(n, k + 1, device="cuda")[:, :k].copy_(w)   # rows that begin at no whole load
    got, want = (torch.full((m + 1, n), 7.0, device="cuda") for _ in range(2))
    ops.gemm_f32(a, w, got[:m])
    ops.gemm_f32(a, odd, want[:m])
    assert torch.equal(got, want) and (got[m] == 7).all()
    bound = (128 + k / 128 + 2) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)   # a run's terms, then the runs' sums
    assert ((got[:m].double() - a.double() @ w.double().T).abs() <= bound).all()


# rows that a wave takes one of, and several; rows of less than 512 values, of a rest behind them, of two waves' halves, and more
@pytest.mark.parametrize("m,inter,k", [(1, 8, 64), (16, 1000, 448), (5, 36, 512), (16, 1536, 576), (9, 20, 960), (16, 3000, 1024), (2, 4100, 1088),
                                       (16, 30, 1024)])
def test_norm_ahead_of_the_weights(m, inter, k):
    from dli_amd.kernels import ops

    g = torch.Generator(device="cuda").manual_seed(m + inter + k)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)
    x, w, norm_w, bias = r(m, k), r(2 * inter, k) / k ** 0.5, 1 + 0.1 * r(k), r(2 * inter)
    normed, both, want, got = torch.empty_like(x), r(m, 2 * inter), r(m, inter), torch.full((m + 1, inter), 7.0, device="cuda")
    ops.rms_norm(x, norm_w, 1e-5, normed)
    ops.gemm_f32(normed, w, both, bias=bias)
    ops.silu_mul(both, want)
    ops.gemm_f32_swiglu(x, w, got[:m], norm_w, 1e-5, bias=bias)
    assert torch.equal(got[:m], want) and (got[m] == 7).all()


# rows and columns: parts of tiles of 64 x 64 and 128 x 64, one and several a unit; k: fewer blocks than stages, as many, a segment of
# several runs with a rest
@pytest.mark.parametrize("m,n,k", [(17, 40000, 32), (130, 20000, 64), (300, 9001, 96), (65, 17000, 128), (511, 3072, 576), (193, 2800, 1024),
                                   (960, 960, 2080), (1000, 1400, 4192), (700, 8200, 160)])
def test_tiles_with_loads_ahead(m, n, k):
    from dli_amd.kernels import ops

    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, w = torch.randn(m, k, device="cuda", generator=g), torch.randn(n, k, device="cuda", generator=g)
    bias, whole = torch.randn(n, device="cuda", generator=g), torch.full((m + 2, n), 7.0, device="cuda")
    odd = torch.empty(n, k + 1, device="cuda")[:, :k].copy_(w)   # rows that begin at no whole load: tiles without
    want = torch.empty(m, n, device="cuda")
    ops.gemm_f32(a, w, whole[1:-1], bias=bias)
    ops.gemm_f32(a, odd, want, bias=bias)
    assert torch.equal(whole[1:-1], want) and (whole[0] == 7).all() and (whole[-1] == 7).all()
    bound = (128 + k / 128 + 3) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T + bias.double().abs())
    assert ((want.double() - a.double() @ w.double().T - bias.double()).abs() <= bound).all()
