"""Matrix-state recurrences whose rows are cut into runs: against the float64 rules and against the token-by-token kernels,
at the edges of runs and batches, continuing from states and starting in slots that held rubbish."""

from __future__ import annotations

import math

import numpy as np
import pytest
import torch

import plain_makodra as M
import plain_miberax as P
import test_makodra_gpu as TM
import test_miberax_gpu as TP

pytestmark = pytest.mark.gpu

D, EPS = 64, 1e-6


@pytest.fixture(scope="module")
def ops():
    from dli_amd.kernels import ops as module

    return module


def i32(values):
    return torch.tensor(np.asarray(values), dtype=torch.int32, device="cuda")


def cut(monkeypatch, ops, workgroups):
    monkeypatch.setattr(ops, "RUNS_WORKGROUPS", workgroups)
    monkeypatch.setattr(ops, "RUNS_FROM_ROWS", 1)   # short entries too


# steps: rows that each of three requests brings (0: not in it): runs of 64 and of other multiples of 16, an entry
# that ends with its run and one row behind it, single tokens beside long portions
STEPS = [[64, 0, 65], [1, 200, 130], [129, 1, 1], [16, 333, 17], [0, 63, 64]]


def no_further_off(got, refs):
    """The runs' distance from the float64 rule against the token-by-token kernel's. Measured with random rows at 8 to 32 heads and
    300 to 4,096 tokens: 0.99 to 1.02 times as far (2-norm; what a run adds is one more sum of 64 terms a value), 1.05 leaves
    room for the few heads here."""
    far = {way: (sum((torch.cat(g) - r).norm() ** 2 for g, r in zip(got[way], refs)) / sum(r.norm() ** 2 for r in refs)).sqrt().item()
           for way in got}
    assert far["runs"] <= 1.05 * far["tokens"], far


def test_rule_of_the_cut(ops):
    assert ops.scan_runs(1, 2048, 32, 2048, True) == (128, 16) and ops.scan_runs(1, 2048, 32, 2048, False) == (64, 32)
    assert ops.scan_runs(3, 134, 4, 127, True) == (0, 0) and ops.scan_runs(64, 64, 32, 1, False) == (0, 0)
    for entries, rows, heads, longest in ((1, 128, 2, 128), (7, 900, 32, 333), (40, 1539, 32, 1500), (16, 6000, 64, 375)):
        run_rows, runs = ops.scan_runs(entries, rows, heads, longest, True)
        assert run_rows % 16 == 0 and run_rows >= 64 and run_rows * runs >= longest > run_rows * (runs - 1)


def test_rule_where_heads_fill_the_device(ops):
    """Where entries' heads fill the device token by token the gated rule is walked so, and from many heads on an entry is one run;
    a short prompt of the rules that are fast token by token is not cut. (Times of both ways beside ``ops.scan_runs``.)"""
    whole = lambda longest: (-(-longest // 16) * 16, 1)
    for entries, heads, longest, want in ((1, 16, 128, (0, 0)), (1, 32, 160, (64, 3)), (8, 16, 200, (0, 0)), (4, 32, 512, (0, 0)),
                                          (12, 16, 400, (0, 0)), (16, 16, 375, (0, 0)), (12, 24, 400, (0, 0)), (16, 32, 375, whole(375)),
                                          (4, 16, 256, (64, 4)), (1, 32, 2048, (128, 16)), (4, 32, 1024, (256, 4))):
        assert ops.scan_runs(entries, entries * longest, heads, longest, True, gated=True) == want, (entries, heads, longest)
    assert ops.scan_runs(1, 128, 32, 128, False) == (0, 0) and ops.scan_runs(4, 576, 16, 144, False) == (64, 3)
    assert ops.scan_runs(12, 4800, 16, 400, True) == whole(400) and ops.scan_runs(4, 2048, 32, 512, True) == (128, 4)


@pytest.mark.parametrize("workgroups", [1024, 12, 1])   # runs of 64 rows, of 176 and the like, and whole entries
@pytest.mark.parametrize("rule", ["delta", "bonus"])
def test_recurrent_scan_in_runs(ops, monkeypatch, rule, workgroups):
    cut(monkeypatch, ops, workgroups)
    H = 3
    c, total = H * D, [sum(s[i] for s in STEPS) for i in range(3)]
    gen = torch.Generator().manual_seed(3)
    data = [{n: torch.randn(t, c, generator=gen) for n in "rkvgwa"} for t in total]
    bonus, norm_w = 0.5 * torch.randn(H, D, generator=gen), 1 + 0.2 * torch.randn(c, generator=gen)
    for d in data:
        if rule == "delta":
            d["w"], d["a"] = torch.exp(-math.exp(-0.5) * torch.sigmoid(d["w"])), torch.sigmoid(d["a"])
        else:
            d["w"] = torch.exp(-torch.exp(2.0 * d["w"]))   # (some keys forget at once: decays of zero)
    refs = []
    for d, n in zip(data, total):
        v = {k: t.double().view(n, H, D) for k, t in d.items()}
        o = (M.delta_rule(v["r"], v["k"], v["v"], v["w"], v["a"]) if rule == "delta" else
             M.bonus_rule(v["r"], v["k"], v["v"], v["w"], bonus.double()))[0]
        g = d["g"].double()
        refs.append(M.rms(o, EPS).reshape(n, c) * norm_w.double() * torch.sigmoid(g) * (1 if rule == "delta" else g))
    states = {way: torch.full((4, c * D + 4), 9.0, device="cuda") for way in ("runs", "tokens")}
    got, at = {way: [[], [], []] for way in states}, [0, 0, 0]
    for step in STEPS:
        who = sorted((i for i in range(3) if step[i]), key=lambda i: step[i] != 1)   # single tokens first, as the engine does
        pick = lambda n: torch.cat([data[i][n][at[i]:at[i] + step[i]] for i in who]).cuda()
        starts = np.cumsum([0] + [step[i] for i in who])
        args = (i32(starts), i32([p for i in who for p in range(at[i], at[i] + step[i])]), i32([3 - i for i in who]))
        kw = dict(a=pick("a")) if rule == "delta" else dict(bonus=bonus.cuda())
        for way, state in states.items():
            out = torch.empty(starts[-1], c, device="cuda")
            ops.recurrent_scan(pick("r"), pick("k"), pick("v"), pick("w"), pick("g"), norm_w.cuda(), EPS, state, *args, out, H, D,
                               ops.RULE_DELTA if rule == "delta" else ops.RULE_BONUS, longest=max(step) if way == "runs" else 0, **kw)
            for i, a, b in zip(who, starts, starts[1:]):
                got[way][i].append(out[a:b].cpu().double())
        at = [a + n for a, n in zip(at, step)]
    off = {way: max((torch.cat(g) - r).abs().max().item() for g, r in zip(got[way], refs)) for way in got}
    # a row divided by its root mean square: rounding of 2^-24 times the terms of a few hundred decayed sums, in both ways
    assert off["runs"] < 2e-4 * max(r.abs().max() for r in refs), off
    no_further_off(got, refs)
    assert (states["runs"] - states["tokens"]).abs().max() < 1e-4 * states["tokens"].abs().max()
    assert (states["runs"][:, c * D:] == 9.0).all() and (states["runs"][0] == 9.0).all()   # nobody else's memory


@pytest.mark.parametrize("workgroups", [1024, 12, 1])
@pytest.mark.parametrize("H,G", [(4, 2), (3, 3)])
def test_gated_delta_in_runs(ops, monkeypatch, H, G, workgroups):
    cut(monkeypatch, ops, workgroups)
    qk, hv, total = G * D, H * D, [sum(s[i] for s in STEPS) for i in range(3)]
    gen = torch.Generator().manual_seed(4)
    width = 2 * qk + hv + 2 * H
    data, refs = [], []
    for n in total:
        q, k = (P.unit(torch.randn(n, G, D, generator=gen).double()) for _ in "qk")
        v, beta = torch.randn(n, H, D, generator=gen).double(), torch.rand(n, H, generator=gen).double()
        g = torch.exp(-torch.rand(n, H, generator=gen).double() ** 4)
        prep = torch.cat([t.reshape(n, -1) for t in (q, k, v, beta, g)], 1).float()
        p = prep.double()
        q, k, v = p[:, :qk].view(n, G, D), p[:, qk:2 * qk].view(n, G, D), p[:, 2 * qk:2 * qk + hv].view(n, H, D)
        rep = H // G
        refs.append(P.gated_delta_rule(q.repeat_interleave(rep, 1), k.repeat_interleave(rep, 1), v, p[:, -2 * H:-H], p[:, -H:]))
        data.append(prep)
    wide = -(-width // 4) * 4 + 4   # rows on 16-byte boundaries (else the token-by-token kernel takes them)
    states = {way: torch.full((4, hv * D + 8), 9.0, device="cuda") for way in ("runs", "tokens")}
    got, at = {way: [[], [], []] for way in states}, [0, 0, 0]
    for step in STEPS:
        who = sorted((i for i in range(3) if step[i]), key=lambda i: step[i] != 1)
        rows = torch.cat([data[i][at[i]:at[i] + step[i]] for i in who])
        prep = torch.empty(rows.shape[0], wide, device="cuda")[:, :width]
        prep.copy_(rows)
        starts = np.cumsum([0] + [step[i] for i in who])
        args = (i32(starts), i32([p for i in who for p in range(at[i], at[i] + step[i])]), i32([3 - i for i in who]))
        for way, state in states.items():
            o = torch.empty(rows.shape[0], hv, device="cuda")
            ops.gated_delta_scan(prep, state, *args, o, H, G, D, D, longest=max(step) if way == "runs" else 0)
            for i, a, b in zip(who, starts, starts[1:]):
                got[way][i].append(o[a:b].cpu().double())
        at = [a + n for a, n in zip(at, step)]
    for way in got:
        for g, r in zip(got[way], refs):
            assert (torch.cat(g).view(r.shape) - r).abs().max() < 2e-5 * max(1.0, r.abs().max()), way
    no_further_off(got, [r.reshape(r.shape[0], -1) for r in refs])
    assert (states["runs"] - states["tokens"]).abs().max() < 2e-5 * states["tokens"].abs().max()
    assert (states["runs"][:, hv * D:] == 9.0).all() and (states["runs"][0] == 9.0).all()


@pytest.mark.parametrize("rule", ["delta", "bonus"])
def test_state_after_runs(ops, rule):
    """The state that sixteen runs of 64 rows leave, with keys that forget slowly and at once: no further from the float64 rule than
    token by token (measured 0.95 to 1.03 times as far; a run's own part is added last, so that what is left of the state before
    it does not round at that part's size: added first it was 1.2 to 2 times as far)."""
    H, n = 4, 1000
    c, gen = H * D, torch.Generator().manual_seed(5)
    r, k, v, g, a = (torch.randn(n, c, generator=gen) for _ in range(5))
    pre = torch.randn(n, c, generator=gen) + 2 * torch.randn(c, generator=gen)
    bonus, heads = torch.randn(H, D, generator=gen), lambda t: t.double().view(n, H, D)
    if rule == "delta":
        w, a = torch.exp(-math.exp(-0.5) * torch.sigmoid(pre)), torch.sigmoid(a)
        S = M.delta_rule(*map(heads, (r, k, v, w, a)))[1]
    else:
        w = torch.exp(-torch.exp(pre - 2))
        S = M.bonus_rule(*map(heads, (r, k, v, w)), bonus.double())[1]
    S = S.transpose(1, 2).reshape(-1)
    far = []
    for longest in (0, n):
        state, out = torch.zeros(1, c * D, device="cuda"), torch.empty(n, c, device="cuda")
        ops.recurrent_scan(r.cuda(), k.cuda(), v.cuda(), w.cuda(), g.cuda(), torch.ones(c, device="cuda"), EPS, state, i32([0, n]),
                           i32(range(n)), i32([0]), out, H, D, ops.RULE_DELTA if rule == "delta" else ops.RULE_BONUS,
                           a=a.cuda() if rule == "delta" else None, bonus=None if rule == "delta" else bonus.cuda(), longest=longest)
        far.append((state[0].cpu().double() - S).norm() / S.norm())
    assert far[1] <= 1.05 * far[0], far


def test_scratch_follows_the_portions(ops):
    """A step's single tokens take no scratch; a step with more entries that bring portions than the scratch may hold is not cut."""
    cut = ops._cut(torch.device("cpu"), 258, 2555, 4, 1500, 255, True)   # 255 single tokens, portions of 1,500, 400 and 400 rows
    run_rows, slots = cut[1], 2300 // cut[1] + 3
    assert cut[0] == 255 and cut[3].shape == (2300, 256) and cut[4].shape == cut[5].shape == (slots, 4, 64, 64)
    assert ops.scan_runs(480, 4000, 32, 2048, True)[0] and not ops.scan_runs(520, 4000, 32, 2048, True)[0]
    assert not ops._cut(torch.device("cpu"), 5, 5, 4, 1, 5, True)[1]


@pytest.mark.parametrize("rule", ["delta", "bonus", "gated"])
@pytest.mark.parametrize("lens,singles", [([1, 1, 1, 200, 2, 70, 129], 3), ([1] * 70 + [5, 300], 70), ([3] * 40 + [150], 0), ([1, 128], 1),
                                          ([3, 0, 5] * 45 + [300, 2] + [4] * 20, 0), ([1] * 3 + [2] * 63 + [200], 3)])
def test_single_tokens_beside_portions(ops, rule, lens, singles):
    """The leading single tokens have the bits that a step of single tokens gives them, the portions those of a step without them,
    near those of token by token; nobody else's state is written. (Entries of many lengths, none among them, and more than a wave
    looks up at once: slots of the launch that hold no run.)"""
    H, n, E = 2, sum(lens), len(lens)
    c, gen = H * D, torch.Generator(device="cuda").manual_seed(n)
    rnd = lambda *shape: torch.randn(*shape, device="cuda", generator=gen)
    r, k, v, g, a, w = (rnd(n, c) for _ in range(6))
    a, w = torch.sigmoid(a), torch.exp(-math.exp(-0.5) * torch.sigmoid(w))
    bonus, norm_w, state0 = rnd(H, D), rnd(c), rnd(E + 2, c * D)
    prep = torch.cat([0.1 * rnd(n, 2 * c), rnd(n, c), torch.rand(n, 2 * H, device="cuda", generator=gen)], 1)
    starts = np.cumsum([0] + lens)
    positions = np.concatenate([np.arange(m) + (7 if i % 3 else 0) for i, m in enumerate(lens)])

    def run(lo, hi, longest, lead):
        rows, state = slice(starts[lo], starts[hi]), state0.clone()
        args = (i32(starts[lo:hi + 1] - starts[lo]), i32(positions[rows]), i32(range(E - 1, -1, -1)[lo:hi]))
        out = torch.full((starts[hi] - starts[lo], c), 9.0, device="cuda")
        if rule == "gated":
            ops.gated_delta_scan(prep[rows], state, *args, out, H, H, D, D, longest=longest, singles=lead)
        else:
            ops.recurrent_scan(r[rows], k[rows], v[rows], w[rows], g[rows], norm_w, EPS, state, *args, out, H, D,
                               ops.RULE_DELTA if rule == "delta" else ops.RULE_BONUS, a=a[rows] if rule == "delta" else None,
                               bonus=None if rule == "delta" else bonus, longest=longest, singles=lead)
        return out, state

    out, state = run(0, E, max(lens), singles)
    by_token, token_state = run(0, E, 0, 0)
    # (an output is divided by its root mean square: a head whose outputs are small there carries the roundings on)
    assert (out - by_token).abs().max() < 2e-4 * by_token.abs().max() and (state - token_state).abs().max() < 2e-5 * token_state.abs().max()
    portions, portion_state = run(singles, E, max(lens), 0)
    assert torch.equal(out[starts[singles]:], portions)
    assert torch.equal(state[:E - singles], portion_state[:E - singles]) and torch.equal(state[E:], state0[E:])
    if singles:
        alone, alone_state = run(0, singles, 0, 0)
        assert torch.equal(out[:starts[singles]], alone) and torch.equal(state[E - singles:E], alone_state[E - singles:E])


WHOLE = {
    "makodra": (TM, M, {"architecture": "Makodra", "vocab": 97, "width": 96, "norm": {"eps": 1e-2}, "logit_softcap": 12.0, "layers": [
        TM.rec("general_delta", 2, 64, 64, rank=10), TM.attn(4, 2, 32, 16, 50, 0.25, True, 0), TM.rec("wkv", 2, 64, 96, rank=8)]}),
    "miberax": (TP, P, {"architecture": "Miberax", "vocab": 97, "width": 96, "norm": {"eps": 1e-5, "groups": 3}, "layers": [
        TP.layer(TP.left(4, 2, 32, 16, 24, 0.2, rot=16), TP.right(4, 2, 64, 64, 3), TP.dense(72)),
        TP.layer(TP.left(2, 2, 48, 48, 70, 0.15, rot=48), TP.right(3, 3, 64, 64, 4), TP.dense(64))]}),
}


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", list(WHOLE))
def test_whole_models_with_long_portions(ops, monkeypatch, tmp_path, name, dtype):
    """Prompts of 200 and 300 tokens alone, beside each other and a single token, and cut in portions: against the plain model. In
    bfloat16 the rows of every layer are cut into runs (also with an odd number of heads or an odd rank, whose rows the parts fill up
    to 16 bytes); in 32-bit they are walked in order, so that every way leaves the same bits."""
    T, plain, cfg = WHOLE[name]
    W = plain.random_weights(cfg, seed=4)
    folder = plain.write_folder(tmp_path / name, cfg, W)
    cuts, rule = [], ops.scan_runs
    monkeypatch.setattr(ops, "scan_runs", lambda *a, **kw: cuts.append(rule(*a, **kw)) or cuts[-1])
    toks = {"a": T.prompt(cfg, 200, 1), "b": T.prompt(cfg, 300, 2), "c": T.prompt(cfg, 6, 3)}
    refs = {i: (T.reference(name, W, cfg, t, dtype) if T is TP else T.reference(W, cfg, t, dtype)) for i, t in toks.items()}
    entry = lambda i, lo, hi: {"id": i, "tokens": toks[i][lo:hi], "want": list(range(hi - lo))}
    s = T.session(folder, dtype, pages=60)
    alone = {i: s.step([entry(i, 0, len(toks[i]))], end=[i]) for i in "ab"}
    s.step([entry("c", 0, 5)])
    both = s.step([entry("a", 0, 200), entry("b", 0, 300), entry("c", 5, 6)], end=["a", "b", "c"])
    ways = {"a": [alone["a"], both[:200]], "b": [alone["b"], both[200:500]]}
    parts = [s.step([entry("b", 0, 130)]), s.step([entry("a", 0, 40), entry("b", 130, 147)]),
             s.step([entry("b", 147, 300), entry("a", 40, 200)], end=["a", "b"])]
    ways["a"].append(torch.cat([parts[1][:40], parts[2][153:]]))
    ways["b"].append(torch.cat([parts[0], parts[1][40:], parts[2][:153]]))
    T.close(both[500:], T.rows_of(refs["c"], slice(5, 6)), dtype, "c")
    for i in "ab":
        for k, got in enumerate(ways[i]):
            T.close(got, refs[i], dtype, (i, k))
            if dtype == "float32":
                assert torch.equal(got, ways[i][0]), (i, k)
    assert (len([c for c in cuts if c[0]]) >= 6) == (dtype == "bfloat16"), cuts
    s.core.manager.check_invariants()
