"""The 32-bit few-row products behind a norm: bit for bit what the norm, product and activation kernels give one after the
other, and so for rotated q and k."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from dli_amd.kernels import ops as o
    return o


def _drawn(m, n, k, seed, bias):
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    return r(m, k), r(n, k) / k ** 0.5, 1.0 + 0.1 * r(k), (r(n) if bias else None)


# depths: part of a run, whole runs and a rest, a row of two and of four waves, more than eight segments, two runs a segment
@pytest.mark.parametrize("m,inter,k,bias", [(1, 8, 8, True), (2, 1536, 576, False), (3, 20, 136, True), (16, 100, 1032, False),
                                            (5, 7, 2048, True), (16, 2560, 960, False), (2, 24, 4104, True)])
def test_swiglu_behind_a_norm(ops, m, inter, k, bias):
    x, w, norm_w, b = _drawn(m, 2 * inter, k, m + inter, bias)
    normed, both, want, got = torch.empty_like(x), torch.empty(m, 2 * inter, device="cuda"), torch.empty(m, inter, device="cuda"), \
        torch.full((m + 1, inter), 7.0, device="cuda")
    ops.rms_norm(x, norm_w, 1e-5, normed)
    ops.gemm_f32(normed, w, both, bias=b)
    ops.silu_mul(both, want)
    ops.gemm_f32_swiglu(x, w, got[:m], norm_w, 1e-5, bias=b)
    assert torch.equal(got[:m], want) and bool((got[m] == 7.0).all())


@pytest.mark.parametrize("m,heads,kv,d,k,page,bias", [(1, 1, 1, 16, 64, 16, True), (2, 9, 3, 64, 576, 16, False), (16, 4, 2, 128, 1032, 48, True),
                                                      (7, 15, 5, 64, 960, 16, False), (3, 2, 1, 80, 4104, 1, True)])
def test_qkv_behind_a_norm_rotated(ops, m, heads, kv, d, k, page, bias):
    x, w, norm_w, b = _drawn(m, (heads + 2 * kv) * d, k, m + heads, bias)
    g = torch.Generator().manual_seed(m)
    positions = torch.randint(0, 5000, (m,), generator=g).to(torch.int32).cuda()
    slots = torch.randperm(6 * page, generator=g)[:m].to(torch.int32) if 6 * page >= m else torch.arange(m, dtype=torch.int32)
    slots[m // 2] = -1 if m > 2 else slots[m // 2]
    slots = slots.cuda()
    inv_freq = (1e4 ** (-torch.arange(0, d, 2).double() / d)).float().cuda()
    pages = [torch.full(s, 3.0, device="cuda") for s in ((6, kv, page, d), (6, kv, d, page)) for _ in range(2)]
    normed, qkv, q = torch.empty_like(x), torch.empty(m, w.shape[0], device="cuda"), torch.empty(m, heads * d, device="cuda")
    ops.rms_norm(x, norm_w, 1e-5, normed)
    ops.gemm_f32(normed, w, qkv, bias=b)
    ops.rope_kv_write(qkv, positions, inv_freq, d, slots, pages[0], pages[2], heads, kv, d)
    ops.gemm_f32_qkv_rope(x, w, q, norm_w, 1e-5, positions, inv_freq, slots, pages[1], pages[3], bias=b)
    assert torch.equal(q, qkv[:, :heads * d]) and torch.equal(pages[1], pages[0])
    assert torch.equal(pages[3], pages[2])
