"""Attention with changed scores for steps of single tokens on the matrix cores: against 64-bit arithmetic, and against the
vector units' kernel, which pages of eight keys still take."""

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


def run(ops, q, kp, vp, tables, lengths, heads, out32, gate, extra, **changes):
    entries, V = len(lengths), vp.shape[2]
    width = max(map(len, tables))
    rows = torch.full((entries, width), -1, dtype=torch.int32)
    for e, t in enumerate(tables):
        rows[e, :len(t)] = torch.tensor(t, dtype=torch.int32)
    wide = torch.empty(entries, heads * V + extra, dtype=torch.float32 if out32 else torch.bfloat16, device="cuda")
    held = torch.zeros(entries, q.shape[1] + extra, dtype=torch.bfloat16, device="cuda")
    held[:, :q.shape[1]] = q.bfloat16().cuda()
    ops.attention_scored(held[:, :q.shape[1]], kp.cuda(), vp.cuda(), wide[:, :heads * V], i32(range(entries + 1)), i32(lengths), rows.cuda(),
                         None, None, heads, changes.pop("scale"), gate=None if gate is None else gate.cuda(),
                         **{k: t.cuda() if torch.is_tensor(t) else t for k, t in changes.items()})
    return wide[:, :heads * V].cpu().double()


@pytest.mark.parametrize("H,G,D,V", [(4, 2, 16, 16), (8, 8, 64, 64), (6, 2, 48, 128), (34, 2, 80, 32), (3, 1, 128, 112)])
@pytest.mark.parametrize("extra", [0, 4, 1])
def test_single_tokens(ops, H, G, D, V, extra):
    """`extra`: columns beside the queries and the results, so that their rows lie at other strides (1: the vector units' kernel)."""
    gen = torch.Generator().manual_seed(H * 100 + D)
    lengths = [1, 15, 16, 17, 63, 130, 517, 2100]
    q = torch.randn(len(lengths), H * D, dtype=F, generator=gen).bfloat16().double()
    r1, r2 = 0.2 + torch.rand(H, generator=gen), 0.1 + 2 * torch.rand(H, generator=gen)
    gate = torch.randn(len(lengths), H * V, generator=gen)
    sinks = torch.randn(H, generator=gen)
    pages, held = {}, {}
    for ps in (8, 48):
        kps, vps, tables, base = [], [], [], 0
        for e, n in enumerate(lengths):
            k = torch.randn(n, G, D, dtype=F, generator=torch.Generator().manual_seed(e)).bfloat16().double()
            v = torch.randn(n, G, V, dtype=F, generator=torch.Generator().manual_seed(e + 50)).bfloat16().double()
            held[e] = k, v
            kp, vp, table = paged(k, v, ps, torch.bfloat16)
            if ps % 16 == 0 and extra != 1:   # past a request's last key: what no one has written
                off = (n - 1) % ps + 1
                kp[table[-1], :, off:], vp[table[-1], :, :, off:] = float("nan"), float("nan")
            kps.append(kp), vps.append(vp), tables.append([base + t for t in table])
            base += kp.shape[0]
        pages[ps] = torch.cat(kps), torch.cat(vps), tables
    scale = D ** -0.5
    for case in (dict(), dict(sink=True), dict(sinks=sinks), dict(window=37), dict(window=16, keep_first=5, sinks=sinks),
                 dict(window=100, keep_first=70), dict(chunk=64, r1=r1, r2=r2), dict(chunk=50, window=20, sink=True),
                 dict(r1=r1, r2=r2, sink=True)):
        for out32, g in ((True, None), (False, gate), (True, gate)):
            got = {ps: run(ops, q, *pages[ps], lengths, H, out32, g, extra, scale=scale, **case) for ps in pages}
            worst = {ps: 0.0 for ps in pages}
            for e, n in enumerate(lengths):
                k, v = held[e]
                j, p = torch.arange(n), n - 1
                seen = torch.ones(n, dtype=torch.bool)
                if case.get("chunk"):
                    seen &= j >= p // case["chunk"] * case["chunk"]
                if case.get("window"):
                    seen &= (j > p - case["window"]) | (j < case.get("keep_first", 0))
                s = torch.einsum("hgd,nhd->hgn", q[e].view(G, H // G, D), k).reshape(H, n) * scale
                if "r1" in case:
                    s = s - r1.double()[:, None] * torch.log1p(r2.double()[:, None] * (p - j))
                s = s.masked_fill(~seen, float("-inf"))
                extra_score = sinks.double() if "sinks" in case else torch.zeros(H, dtype=F) if case.get("sink") else None
                if extra_score is not None:
                    s = torch.cat([s, extra_score[:, None]], 1)
                w = s.softmax(1)[:, :n].view(G, H // G, n)
                ref = torch.einsum("hgn,nhv->hgv", w, v).reshape(H * V)
                if g is not None:
                    ref = ref * torch.sigmoid(g[e].double())
                for ps in pages:
                    assert got[ps][e].isfinite().all(), (case, out32, ps, n)
                    worst[ps] = max(worst[ps], float((got[ps][e] - ref).abs().max()))
            # 32-bit weights and sums: 2^-24 of scores of up to about ten and of sums of values of up to about four, with some ten
            # roundings each; a bfloat16 result rounds to 2^-9 of up to about four
            limit = 1.5e-5 if out32 else 1.6e-2
            assert worst[8] < limit and worst[48] < limit, (case, out32, worst)
            print(H, D, V, case.keys(), out32, worst)


@pytest.mark.parametrize("n", [1, 40, 700])
def test_infinite_values(ops, n):
    """A value that is infinite makes its component of the result infinite with its sign, as one sum over the weights does, and
    leaves the other components alone; a weight of exactly one is among them (a single key)."""
    H, G, D, ps = 4, 2, 32, 16
    gen = torch.Generator().manual_seed(n)
    q = torch.randn(1, H * D, dtype=F, generator=gen).bfloat16().double()
    k, v = (torch.randn(n, G, D, dtype=F, generator=gen).bfloat16().double() for _ in range(2))
    v[n // 2, 0, 3], v[n // 3, 1, 7], v[n - 1, 1, 7], v[0, 1, 30] = float("inf"), float("-inf"), float("-inf"), float("inf")
    kp, vp, table = paged(k, v, ps, torch.bfloat16)
    got = run(ops, q, kp, vp, [table], [n], H, True, None, 0, scale=D ** -0.5)[0]
    s = torch.einsum("hgd,nhd->hgn", q.view(G, H // G, D), k) * D ** -0.5
    ref = torch.einsum("hgn,nhv->hgv", s.softmax(2), v).reshape(H * D)
    assert not ref.isnan().any() and ref.isinf().sum() == 6
    assert torch.equal(got.isinf(), ref.isinf()) and torch.equal(got[ref.isinf()], ref[ref.isinf()])
    assert (got - ref)[ref.isfinite()].abs().max() < 1.5e-5


def test_splits_and_replays(ops):
    """Few requests over a wide table: the keys are cut, and a captured step gives the same again for other lengths."""
    gen = torch.Generator().manual_seed(5)
    H, G, D, n, ps = 8, 2, 64, 5000, 16
    k, v = (torch.randn(n, G, D, dtype=F, generator=gen).bfloat16().double() for _ in range(2))
    kp, vp, table = paged(k, v, ps, torch.bfloat16)
    q = torch.randn(1, H * D, dtype=F, generator=gen).bfloat16()
    kp, vp, q_gpu = kp.cuda(), vp.cuda(), q.cuda()
    tables, length, starts = i32(table).view(1, -1), i32([n]), i32([0, 1])
    out = torch.empty(1, H * D, device="cuda")
    call = lambda: ops.attention_scored(q_gpu, kp, vp, out, starts, length, tables, None, None, H, 0.125, sink=True)
    call()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for seen in (n, 1, 33, 1024, 4097):
        length.fill_(seen)
        graph.replay()
        got = out.cpu().double()
        s = torch.einsum("hgd,nhd->hgn", q.double().view(G, H // G, D), k[:seen]) * 0.125
        w = torch.cat([s, torch.zeros(G, H // G, 1, dtype=F)], 2).softmax(2)[..., :seen]
        ref = torch.einsum("hgn,nhv->hgv", w, v[:seen]).reshape(1, H * D)
        assert (got - ref).abs().max() < 1.5e-5, seen
        call()
        assert torch.equal(out.cpu().double(), got)
