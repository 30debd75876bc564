"""The gated delta rule's runs, walked sixteen tokens at a time: every remainder of sixteen against 64-bit arithmetic, decays and
write strengths of zero, and what is infinite at a token."""

from __future__ import annotations

import pytest
import torch

import plain_miberax as P
from test_scan_runs_gpu import i32

pytestmark = pytest.mark.gpu
H, G, D = 4, 2, 64


def rows(n, seed):
    gen = torch.Generator().manual_seed(seed)
    q, k = (P.unit(torch.randn(n, G, D, generator=gen).double()) for _ in "qk")
    v, beta, g = torch.randn(n, H * D, generator=gen), torch.rand(n, H, generator=gen), torch.exp(-4 * torch.rand(n, H, generator=gen) ** 4)
    beta[3::7], g[5::11] = 0.0, 0.0   # a token that writes nothing, a state that is forgotten
    return torch.cat([q.reshape(n, -1).float(), k.reshape(n, -1).float(), v, beta, g], 1)


def scan(prep, lens, longest):
    from dli_amd.kernels import ops

    n, width = prep.shape
    held = torch.empty(n, width + 4 - width % 4, device="cuda")[:, :width]
    held.copy_(prep)
    state, out = torch.zeros(len(lens), H * D * D, device="cuda"), torch.empty(n, H * D, device="cuda")
    starts = [sum(lens[:i]) for i in range(len(lens) + 1)]
    ops.gated_delta_scan(held, state, i32(starts), i32([p for m in lens for p in range(m)]), i32(range(len(lens))), out, H, G, D, D,
                         longest=longest)
    return out.cpu(), state.cpu()


@pytest.mark.parametrize("workgroups", [1024, 1])   # runs of 64 rows, whole entries
def test_every_remainder(monkeypatch, workgroups):
    from dli_amd.kernels import ops

    monkeypatch.setattr(ops, "RUNS_WORKGROUPS", workgroups)
    monkeypatch.setattr(ops, "RUNS_FROM_ROWS", 1)
    lens = [*range(1, 34), 64, 65, 127, 400]
    prep = rows(sum(lens), 1)
    monkeypatch.setattr(ops, "scan_runs", lambda *a, **k: (64 if workgroups > 1 else 400, 7 if workgroups > 1 else 1))
    got, state = scan(prep, lens, max(lens))
    plain, plain_state = scan(prep, lens, 0)
    at, far = 0, [[0.0, 0.0], [0.0, 0.0]]
    for m in lens:
        p = prep[at:at + m].double()
        q, k = (p[:, i * G * D:(i + 1) * G * D].view(m, G, D).repeat_interleave(H // G, 1) for i in range(2))
        ref = P.gated_delta_rule(q, k, p[:, 2 * G * D:2 * G * D + H * D].view(m, H, D), p[:, -2 * H:-H], p[:, -H:]).reshape(m, -1)
        for way, o in enumerate((got, plain)):
            far[way][0] += float((o[at:at + m] - ref).norm() ** 2)
            far[way][1] = max(far[way][1], float((o[at:at + m] - ref).abs().max()))
        at += m
    # as far from 64 bits as token by token: 5 % for the draw; no row on its own further than twice the other way's worst
    assert far[0][0] ** 0.5 <= 1.05 * far[1][0] ** 0.5 and far[0][1] <= 2 * far[1][1], far
    # states of up to about four, some ten roundings of 2^-24 each on either way
    assert (state - plain_state).abs().max() < 2e-5


@pytest.mark.parametrize("where", ["v", "k", "g", "beta", "q"])
def test_infinite_inputs_stay_out_of_earlier_tokens(monkeypatch, where):
    from dli_amd.kernels import ops

    monkeypatch.setattr(ops, "RUNS_FROM_ROWS", 1)
    n, t = 150, 70   # the seventh token of a sixteen
    prep = rows(n, 2)
    clean, _ = scan(prep, [n], n)
    column = {"q": 5, "k": G * D + 5, "v": 2 * G * D + D + 9, "beta": -2 * H + 1, "g": -H + 1}[where]
    prep[t, column] = float("inf")
    got, _ = scan(prep, [n], n)
    plain, _ = scan(prep, [n], 0)
    assert torch.equal(got[:t], clean[:t])
    assert torch.equal(got[t].isfinite(), plain[t].isfinite())
    if where == "q":   # and out of the state
        assert torch.equal(got[t + 1:], clean[t + 1:])
