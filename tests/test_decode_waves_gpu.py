"""Single-token attention with four and with eight waves a workgroup (few workgroups and many), and the place of a tile of keys in
pages of every number of tiles."""

from __future__ import annotations

import math

import pytest
import torch

gpu = pytest.mark.gpu


@gpu
@pytest.mark.parametrize("page", [16, 48, 80, 112, 240, 1040])
@pytest.mark.parametrize("qh,kvh,d,requests", [(6, 2, 64, 3), (6, 2, 64, 150), (20, 1, 128, 5), (5, 5, 48, 60)])
def test_waves_and_pages(page, qh, kvh, d, requests):
    import test_kernels_gpu as kernels
    from kernel_refs import ref_paged_attention

    from dli_amd.kernels import ops

    lens = [(1, n) for n in ([1, 16, 17, 127, 128, 129, 513, 576, page, page + 1] * requests)[:requests]]
    q, kp, vp, q_start, kv_len, tables = kernels._paged_case(torch.bfloat16, qh, kvh, d, page, lens, seed=page + d)
    dev = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    scale = 1.0 / math.sqrt(d)
    ref = ref_paged_attention(q, kp, vp, q_start, kv_len, tables, qh, scale, 0)
    for splits in (1, 3):
        part_o = torch.full((requests * qh * splits * d,), float("nan"), device="cuda")
        part_ml = torch.full((requests * qh * splits * 2,), float("nan"), device="cuda")
        out = torch.full(q.shape, 9.0, dtype=torch.bfloat16, device="cuda")
        ops.attention_decode(q.cuda(), kp.cuda(), vp.cuda(), out, dev(kv_len), dev(tables), qh, scale, 0, splits, part_o, part_ml)
        assert (out.cpu().double() - ref).abs().max() < kernels.tol(torch.bfloat16)


@gpu
@pytest.mark.parametrize("page", [16, 48, 80, 112, 240, 1040])
def test_pages_of_the_32_bit_attention(page):
    import test_f32_gpu as f32

    from dli_amd.kernels import ops

    f32.test_attention_f32(ops, 9, 3, 64, page, 0)
    f32.test_attention_f32(ops, 4, 2, 128, page, 45)


@gpu
@pytest.mark.parametrize("page", [48, 112, 1040])
def test_pages_of_a_long_context(page):
    """Tiles of far larger numbers than a short context has, in both attentions of single tokens."""
    import test_kernels_gpu as kernels
    from kernel_refs import ref_paged_attention

    from dli_amd.kernels import ops

    dev = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    lens = [(1, 70003), (1, 65537)]
    q, kp, vp, q_start, kv_len, tables = kernels._paged_case(torch.bfloat16, 2, 1, 64, page, lens, seed=page)
    ref = ref_paged_attention(q, kp, vp, q_start, kv_len, tables, 2, 0.5, 0)
    out = torch.empty(q.shape, dtype=torch.bfloat16, device="cuda")
    ops.attention_decode(q.cuda(), kp.cuda(), vp.cuda(), out, dev(kv_len), dev(tables), 2, 0.5)
    assert (out.cpu().double() - ref).abs().max() < kernels.tol(torch.bfloat16)
    q, kp, vp = q.float(), kp.float(), vp.float()
    ref = ref_paged_attention(q, kp, vp, q_start, kv_len, tables, 2, 0.5, 0)
    out = torch.empty(q.shape, device="cuda")
    ops.attention_generic(q.cuda(), kp.cuda(), vp.cuda(), out, dev(q_start), dev(kv_len), dev(tables), dev([0, 1]), dev([0, 0]), 2, 0.5)
    assert (out.cpu().double() - ref).abs().max() < 2e-5


def test_a_tile_is_in_the_page_that_division_names():
    """What the host hands over (csrc/common.h, page_of_tile): the upper half of the product with the reciprocal is the quotient for every
    tile below 2^32 / tiles (checked about multiples of the page's tiles)."""
    from dli_amd.kernels import ops

    for tiles in [*range(1, 130), 255, 256, 1000, 4097]:
        held, reciprocal = ops.page_of_tile(16 * tiles)
        assert held == tiles
        if tiles == 1:   # (a page a tile: no product)
            continue
        top = (1 << 32) // tiles - 1
        for q in (1, 2, 3, 1000, top // tiles - 1, top // tiles):
            for tile in (q * tiles - 1, q * tiles, q * tiles + 1):
                if tile <= top:
                    assert (tile * reciprocal) >> 32 == tile // tiles, (tile, tiles)
