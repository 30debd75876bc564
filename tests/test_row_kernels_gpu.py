"""Row kernels that hold a row's first values in registers, the convolution by runs of rows, and the sort of many experts."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from dli_amd.kernels import ops as module

    return module


@pytest.mark.parametrize("width", [1, 63, 255, 1024, 1025, 2047, 2048, 2050, 4097, 8192, 8200])
def test_norms_at_the_edges_of_what_is_held(ops, width):
    gen = torch.Generator(device="cuda").manual_seed(width)
    draw = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    rows, eps = 3, 1e-5
    n = lambda t: t.double() / (t.double().pow(2).mean(-1, keepdim=True) + eps).sqrt()
    # 32-bit sums and products: some ten roundings of 2^-24 of results of up to about thirty
    close = lambda got, want: float((got.double() - want).abs().max()) < 2e-5
    ys, ws = [draw(rows, width + 3)[:, :width] for _ in range(4)], [draw(width) for _ in range(4)]
    out = torch.empty(rows, width, device="cuda")
    for count in (1, 2, 3, 4):
        ops.branch_norm_mean(ys[:count], ws[:count], eps, out)
        assert close(out, sum(w.double() * n(y) for y, w in zip(ys[:count], ws)) / count), count
    x, second = ys[0].contiguous(), torch.empty_like(out)
    ops.rms_norm_pair(x, ws[0], ws[1], eps, out, second)
    assert close(out, ws[0].double() * n(x)) and close(second, ws[1].double() * n(x))
    for groups in (1, 3):
        if width % groups == 0:
            for delta in (None, ys[1]):
                kept = x.clone()
                ops.group_norm(kept, ws[0], groups, eps, out, delta=delta)
                total = x if delta is None else x + delta
                assert torch.equal(kept, total)
                assert close(out, ws[0].double() * n(total.view(rows, groups, -1)).view(rows, width)), (groups, delta is None)
    coef = draw(4)
    ops.poly_norm(ys[2], coef, eps, out)
    z = ys[2].double()
    want = coef[0].double() * n(z) + coef[1].double() * n(z ** 2) + coef[2].double() * n(z ** 3) + coef[3].double()
    assert float((out.double() - want).abs().max()) < 2e-5 * max(1.0, width ** 0.5 / 10)   # cubes: results of up to sqrt(width)


@pytest.mark.parametrize("dim,vdim,taps,heads,kv_heads", [(64, 64, 4, 32, 2), (128, 48, 3, 96, 4), (40, 100, 1, 80, 2), (16, 130, 2, 28, 4),
                                                          (64, 64, 4, 4, 2), (128, 48, 3, 4, 2)])
def test_runs_of_rows_convolve_alike(ops, dim, vdim, taps, heads, kv_heads):
    """A step of many rows gives the bits of the wave a row (chosen when there are many requests: empty ones are added)."""
    lengths, starts = [1, 7, 530, 3, 491], [0, 9, 0, 1, 2]
    in_runs = lambda entries: bool(ops.library().dli_conv_prepare_in_runs(sum(lengths), entries, heads, kv_heads, dim, vdim, taps))
    assert in_runs(5) == (heads > 4) and not in_runs(45)
    rows, channels = sum(lengths), 2 * kv_heads * dim + heads * vdim
    gen = torch.Generator(device="cuda").manual_seed(dim)
    draw = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    proj, conv_w, a_log, dt_bias = draw(rows, channels + 2 * heads + 5), draw(channels, taps), draw(heads), draw(heads)
    state = draw(8, max(taps - 1, 1) * channels)
    ends = torch.tensor([0] + lengths).cumsum(0).tolist()
    positions = torch.cat([torch.arange(p, p + n) for p, n in zip(starts, lengths)]).int().cuda()
    results = []
    for empty in (0, 40):
        q_start = torch.tensor(ends + [rows] * empty, dtype=torch.int32, device="cuda")
        slots = torch.tensor([6, 2, 0, 5, 1] + [7] * empty, dtype=torch.int32, device="cuda")
        out, kept = torch.zeros(rows, channels + 2 * heads, device="cuda"), state.clone()
        ops.conv_prepare(proj, channels, channels + heads, conv_w, a_log, dt_bias, kept, 0, q_start, positions, slots, out, heads,
                         kv_heads, dim, vdim)
        results.append((out, kept))
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])
    assert results[0][0].isfinite().all() and float(results[0][0].abs().max()) > 0


@pytest.mark.parametrize("experts,rows,top", [(1, 5, 1), (64, 33, 4), (1024, 40, 3), (1025, 700, 2), (2500, 64, 8)])
def test_many_experts_are_sorted(ops, experts, rows, top):
    gen = torch.Generator().manual_seed(experts)
    width = ff = 32
    w = [torch.randn(experts, 32, 32, generator=gen).mul_(32 ** -0.5).bfloat16() for _ in range(3)]
    h = torch.randn(rows, width, generator=gen).bfloat16()
    ids = torch.randint(0, experts + 1, (rows, top), generator=gen, dtype=torch.int32)   # (`experts` itself: no rows)
    z = ops.expert_products(ids.cuda(), h.cuda(), *(t.cuda() for t in w), 7.0, 1.0, 0.0).cpu().view(rows, top, width)
    e = ids.clamp(max=experts - 1).long()
    gate, up = (torch.einsum("rk,rtfk->rtf", h.double(), t.double()[e]) for t in w[:2])
    gate, up = gate.clamp(max=7.0), up.clamp(-7.0, 7.0)
    want = torch.einsum("rtf,rtwf->rtw", (gate * torch.sigmoid(gate) * up).bfloat16().double(), w[2].double()[e])
    real = ids < experts
    # values of the intermediate that round to bfloat16 the other way: 2^-8 of up to about eight, times weights of up to one half
    assert float((z.double() - want)[real].abs().max()) < 2 ** -8 * 8 * 0.75
