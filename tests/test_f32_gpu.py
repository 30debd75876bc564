"""The 32-bit path's product and attention on the matrix cores, at the edges of their tiles, runs and splits."""

from __future__ import annotations

import math

import pytest
import torch

from test_kernels_gpu import _paged_case, _tiles, ref_paged_attention

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from dli_amd.kernels import ops as module

    return module


# rows: the few-row kernel's end and the tiles' (32, 64, 128); columns: part of a tile, and enough of them for most rules
# of the dispatch (the test below goes through every one); k: below a load, across a run's half and end, several runs a
# segment (2,048 is 16 runs, 2,100 two a segment)
@pytest.mark.parametrize("m", [1, 16, 17, 33, 130])
@pytest.mark.parametrize("n,k", [(31, 3), (16, 62), (48, 64), (576, 132), (1024, 1536), (700, 1030), (65, 2048), (33, 2100), (40000, 100)])
def test_gemm_f32_edges(ops, m, n, k):
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, w = (torch.randn(r, k, device="cuda", generator=gen) for r in (m, n))
    out = torch.full((m, n), 7.0, device="cuda")
    ops.gemm_f32(a, w, out)
    ref = a.double() @ w.double().T
    # each of k products and sums rounds by 2^-24 of a partial sum: runs of 128 terms, then the runs' sums
    bound = (128 + k / 128 + 2) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)
    assert ((out.double() - ref).abs() <= bound).all()
    one = torch.empty(1, n, device="cuda")   # a row alone, through the few-row kernel: the same bits
    ops.gemm_f32(a[m - 1:], w, one)
    assert torch.equal(one[0], out[m - 1])


# (rows, columns, k, kernel): every kernel of the dispatch with as many segments as its waves take several of, k in whole loads and
# in single values. Few rows with 2 and 4 waves a tile and one segment, 2 to 4, 5 to 8 (8 waves), more (16); tiles of 32 x 32
# with 8 waves (5, 9 and 16 segments of one, two and five runs) and with 4 (2, 5, 9 and 12 segments), of 64 x 64, of 128 x 64
RULES = [(2, 960, 576, 1), (16, 3072, 576, 1), (9, 600, 1023, 1), (2, 576, 1536, 0), (5, 90, 9001, 0), (2, 40000, 576, 2),
         (7, 700, 390, 2), (2, 300, 100, 3), (3, 140000, 300, 3), (100, 100, 576, 4), (498, 192, 1536, 4), (61, 33, 9001, 4),
         (498, 960, 576, 5), (498, 3072, 576, 5), (498, 576, 1536, 5), (300, 1000, 1101, 5), (130, 65, 132, 5), (333, 9000, 576, 6),
         (300, 1000, 100, 6), (300, 30000, 132, 7), (390, 33000, 61, 7)]


@pytest.mark.parametrize("m,n,k,rule", RULES)
def test_gemm_f32_every_kernel(ops, m, n, k, rule):
    """Each kernel against float64, and each of some rows against the row alone: the same bits."""
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:   # (the rule follows the device's compute units)
        assert ops.gemm_f32_rule(m, n, k) == rule
        assert {r[3] for r in RULES} == set(range(8))
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, w = (torch.randn(r, k, device="cuda", generator=gen) for r in (m, n))
    out = torch.full((m, n), 7.0, device="cuda")
    ops.gemm_f32(a, w, out)
    # each of k products and sums rounds by 2^-24 of a partial sum: runs of 128 terms, then the runs' sums
    bound = (128 + k / 128 + 2) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)
    assert ((out.double() - a.double() @ w.double().T).abs() <= bound).all()
    for row in {0, m // 2, m - 1}:
        one = torch.empty(1, n, device="cuda")
        ops.gemm_f32(a[row:row + 1], w, one)
        assert torch.equal(one[0], out[row]), row


def test_gemm_f32_rows_of_wider_matrices(ops):
    """Strides that allow 16-byte loads and strides that do not; a residual that is the result's own buffer."""
    gen = torch.Generator(device="cuda").manual_seed(1)
    for pad in (4, 3):
        a = torch.randn(70, 200 + pad, device="cuda", generator=gen)[:, :200]
        w = torch.randn(90, 200 + pad, device="cuda", generator=gen)[:, :200]
        bias = torch.randn(90, device="cuda", generator=gen)
        wide = torch.randn(70, 90 + pad, device="cuda", generator=gen)
        before, out = wide.clone(), wide[:, :90]
        ops.gemm_f32(a, w, out, bias=bias, residual=out)
        ref = a.double() @ w.double().T + bias.double() + before[:, :90].double()
        assert (out.double() - ref).abs().max() < 200 * 2.0 ** -24 * 200 and torch.equal(wide[:, 90:], before[:, 90:])


@pytest.mark.parametrize("qh,kvh,d,bs,window", [(9, 3, 64, 16, 0), (4, 4, 64, 48, 0), (6, 2, 128, 16, 0), (4, 2, 64, 16, 37), (2, 1, 128, 32, 150)])
def test_attention_f32(ops, qh, kvh, d, bs, window):
    """Single tokens, prompts and portions on a prefix; more blocks than waves and fewer; keys that no request has
    written (NaN behind every request's last key) stay out."""
    lens = [(1, 1), (1, 16), (1, 17), (1, 127), (1, 129), (7, 7), (16, 16), (33, 33), (5, 40), (17, 300), (130, 130), (1, 1030)]
    q, kp, vp, q_start, kv_len, tables = _paged_case(torch.float32, qh, kvh, d, bs, lens, seed=d + bs, poison=True)
    ref = ref_paged_attention(q, kp, vp, q_start, kv_len, tables, qh, d ** -0.5, window)
    for e, (_, kv) in enumerate(lens):
        if kv % bs:
            page = tables[e][kv // bs]
            kp[page, :, kv % bs:] = float("nan")
            vp[page, :, :, kv % bs:] = float("nan")
    rows = ops.attention_generic_tile_rows(d)
    te, tq = _tiles(q_start, rows)
    dev = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    out = torch.full(q.shape, 9.0, device="cuda")
    ops.attention_generic(q.cuda(), kp.cuda(), vp.cuda(), out, dev(q_start), dev(kv_len), dev(tables), dev(te), dev(tq), qh,
                          d ** -0.5, window)
    # scores of d terms, exponentials and sums of up to 1,030 weights: well under 1e-5 of values of about one
    assert (out.cpu().double() - ref).abs().max() < 1e-5
    # the last prompt's last row as a single token: the same blocks for the same waves, the same bits
    e = len(lens) - 2
    last = q_start[e + 1] - 1
    alone = torch.empty(1, q.shape[1], device="cuda")
    ops.attention_generic(q[last:last + 1].cuda(), kp.cuda(), vp.cuda(), alone, dev([0, 1]), dev([kv_len[e]]),
                          dev([tables[e]]), dev([0]), dev([0]), qh, d ** -0.5, window)
    assert torch.equal(alone[0], out[last])


@pytest.mark.parametrize("head_dim", [64, 128])
def test_recorded_steps_have_the_eager_steps_bits(tmp_path, head_dim):
    """Steps of single tokens on the 32-bit path, replayed from graphs against launched one by one: batches that change (padding
    rows), other work and synchronisations between the replays, pages that are handed on."""
    import random

    from dli_amd.engine.core import build_core
    from dli_amd.trace import TraceSession
    from dli_amd.weights import write_random_model

    cfg = {"model_type": "llama", "architectures": ["LlamaForCausalLM"], "hidden_size": 192, "intermediate_size": 320,
           "num_hidden_layers": 2, "num_attention_heads": 3, "num_key_value_heads": 1, "head_dim": head_dim, "vocab_size": 301,
           "rms_norm_eps": 1e-5, "rope_theta": 10000.0, "max_position_embeddings": 512, "tie_word_embeddings": True}
    write_random_model(tmp_path, cfg, seed=3, std=0.1)

    def run(graphs):
        core = build_core(tmp_path, num_pages=40, page_size=16, max_seqs=8, dtype="float32", enable_prefix_caching=False,
                          watermark=0.0)
        if graphs:
            core.step.enable_decode_graphs(8, 640)
            assert core.step.graphs is not None
        s, rng, outs = TraceSession(core), random.Random(4), []
        toks = [[rng.randrange(301) for _ in range(n)] for n in (40, 9, 70, 23, 55)]
        fed, live, pending = {}, [0, 1, 2], [3, 4]
        for r in live:
            outs.append(s.step([{"id": r, "tokens": toks[r][:5], "want": [4]}]).float().cpu())
            fed[r] = 5
        while live:
            chosen = [r for r in live if len(live) == 1 or rng.random() > 0.15]
            if not chosen:
                continue
            entries = [{"id": r, "tokens": [toks[r][fed[r]]], "want": [0]} for r in chosen]
            for r in chosen:
                fed[r] += 1
            end = [r for r in chosen if fed[r] == len(toks[r])]
            outs.append(s.step(entries, end).float().cpu())
            torch.cuda.synchronize()
            for r in end:
                live.remove(r)
                if pending:
                    new = pending.pop(0)
                    outs.append(s.step([{"id": new, "tokens": toks[new][:6], "want": [5]}]).float().cpu())
                    fed[new] = 6
                    live.append(new)
        return outs, core

    eager, _ = run(False)
    replayed, core = run(True)
    assert core.step.graphs.replays > 20 and len(core.step.graphs.captured) >= 2
    assert len(eager) == len(replayed)
    for i, (a, b) in enumerate(zip(eager, replayed)):
        assert torch.equal(a, b), (i, float((a - b).abs().max()))
