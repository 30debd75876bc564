"""Decode attention in pairs of key tiles, and the o projection that merges its runs where the width is no whole blocks of 128."""

from __future__ import annotations

import math

import pytest
import torch

from kernel_refs import ref_paged_attention

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from dli_amd.kernels import ops as o

    o.library()
    return o


def _pool(shape, gen, offset):
    """Values in a buffer that begins `offset` elements behind an allocation."""
    n = math.prod(shape)
    flat = torch.empty(n + offset, dtype=torch.bfloat16, device="cuda")
    flat[offset:] = torch.randn(n, generator=gen).bfloat16().cuda()
    return flat[offset:].view(shape)


# a wave's first and second pair of tiles (32 keys), its rounds of two to four pairs, the last tile's edges
@pytest.mark.parametrize("keys", [1, 16, 17, 31, 32, 33, 48, 255, 256, 257, 511, 513, 1024, 1025, 2600])
@pytest.mark.parametrize("qh,kvh,d,bs,splits,window", [(9, 3, 64, 16, 1, 0), (8, 2, 32, 32, 2, 0), (6, 2, 128, 16, 3, 700), (5, 5, 48, 16, 1, 20)])
def test_pairs_of_tiles_at_their_edges(ops, keys, qh, kvh, d, bs, splits, window):
    """One request whose table holds its pages and nothing more, pages that begin 8 bytes behind a multiple of 16, slots past the last
    key not a number; the same bits beside other requests. Probabilities and results are rounded to bfloat16 (2^-9 each), values
    are below 4.5: 1.8e-2."""
    gen = torch.Generator().manual_seed(keys + d)
    pages = -(-keys // bs)
    kp, vp = _pool((pages + 2, kvh, bs, d), gen, 4), _pool((pages + 2, kvh, d, bs), gen, 4)
    table = torch.randperm(pages + 2, generator=gen)[:pages].int()
    rest = pages * bs - keys
    if rest:
        kp[int(table[-1]), :, bs - rest:] = float("nan")
        vp[int(table[-1]), :, :, bs - rest:] = float("nan")
    q = torch.randn(2, qh * d, generator=gen).bfloat16().cuda()
    scale = 1.0 / math.sqrt(d)
    dev = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")

    def run(rows, kv_len, tables):
        po = torch.full((rows * qh * splits * d,), float("nan"), device="cuda")
        ml = torch.full((rows * qh * splits * 2,), float("nan"), device="cuda")
        out = torch.full((rows, qh * d), 9.0, dtype=torch.bfloat16, device="cuda")
        ops.attention_decode(q[:rows], kp, vp, out, dev(kv_len), tables, qh, scale, window, splits, po, ml)
        return out

    one = table[None].cuda()
    got = run(1, [keys], one)
    want = ref_paged_attention(q[:1].cpu(), kp.cpu().nan_to_num(), vp.cpu().nan_to_num(), [0, 1], [keys], one.tolist(), qh, scale, window)
    assert (got.cpu().double() - want).abs().max().item() < 1.8e-2
    wide = torch.cat([one.repeat(2, 1), torch.zeros(2, 3, dtype=torch.int32, device="cuda")], 1).contiguous()
    both = run(2, [keys, 0], wide)
    assert torch.equal(both[:1], got) and not both[1].any()


# k of 18, 30, 17 and 31 steps of 32: waves of single steps only, of a block and none to three steps behind it
@pytest.mark.parametrize("qh,kvh,d,n", [(9, 3, 64, 576), (15, 5, 64, 960), (17, 1, 32, 272), (31, 1, 32, 64)])
@pytest.mark.parametrize("splits", [2, 3, 8, 9, 16])
@pytest.mark.parametrize("rows", [1, 2, 4])
def test_merging_o_projection_of_odd_widths(ops, qh, kvh, d, n, splits, rows):
    """Widths that end inside a block of 128: the bits of the merge kernel and the product that several rows take, and so a row
    alone in its step those of one among others."""
    bs, k = 16, qh * d
    assert k % 128 and ops.skinny_gemm_merged_supports(rows, n, qh, d, splits, torch.device("cuda", 0))
    gen = torch.Generator().manual_seed(n + splits)
    lens = [700, 33, 1, 260][:rows]
    width = -(-lens[0] // bs)
    kp, vp = _pool((4 * width, kvh, bs, d), gen, 0), _pool((4 * width, kvh, d, bs), gen, 0)
    tables = torch.randperm(4 * width, generator=gen).view(4, width)[:rows].int().cuda()
    q = torch.randn(rows, k, generator=gen).bfloat16().cuda()
    kv_len = torch.tensor(lens, dtype=torch.int32, device="cuda")
    w = (torch.randn(n, k, generator=gen) / math.sqrt(k)).bfloat16().cuda()
    base, bias = torch.randn(rows, n, generator=gen).bfloat16().cuda(), torch.randn(n, generator=gen).bfloat16().cuda()
    po = torch.full((rows * qh * splits * d,), float("nan"), device="cuda")
    ml = torch.full((rows * qh * splits * 2,), float("nan"), device="cuda")
    out = torch.empty_like(q)
    ops.attention_decode(q, kp, vp, out, kv_len, tables, qh, 0.125, 0, splits, po, ml)
    got, want = base.clone(), base.clone()
    ssq = ops.skinny_gemm_merged(po, ml, splits, qh, d, ops.tile_weights_in_chunks(w), got, bias=bias)
    ssq_want = ops.skinny_gemm(out, w, epilogue=ops.SKINNY_RESIDUAL, stream=want, bias=bias)
    assert torch.equal(got, want) and torch.equal(ssq, ssq_want)
    # product and bias rounded once, then their sum with the stream: half of the last of eight bits each, and the 32-bit sums
    y, old = out.cpu().double() @ w.cpu().double().T + bias.cpu().double(), base.cpu().double()
    sums = k * 2.0 ** -23 * (out.cpu().double().abs() @ w.cpu().double().abs().T + bias.cpu().double().abs())
    assert ((got.cpu().double() - old - y).abs() <= 2.0 ** -8 * (y.abs() + (y + old).abs()) * 1.01 + sums).all()
