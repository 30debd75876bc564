"""The gated delta rule of a step of single tokens in one kernel: the bits of the three kernels that it stands for."""

import pytest
import torch

pytestmark = pytest.mark.gpu


# heads on one to all q/k heads; one and two runs of 64 lanes in a head of keys or values; value columns that are no whole turn of a
# workgroup, whole turns, the most; no input to keep to the most; values that no four columns divide
@pytest.mark.parametrize("heads,kv_heads,dim,vdim,taps", [
    (32, 8, 64, 64, 4), (4, 4, 16, 4, 1), (6, 2, 32, 20, 3), (16, 1, 64, 16, 2), (3, 1, 128, 64, 4), (2, 1, 128, 128, 4), (8, 1, 64, 64, 4),
    (16, 1, 16, 32, 3), (5, 1, 32, 100, 4), (3, 3, 64, 10, 4), (2, 2, 16, 128, 2)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_same_bits_as_apart(heads, kv_heads, dim, vdim, taps, dtype):
    from dli_amd.kernels import ops

    assert ops.gated_delta_single_takes(heads, kv_heads, dim, vdim, taps)
    n, hv = 7, heads * vdim
    channels, floats = 2 * kv_heads * dim + hv, hv * dim
    positions = torch.tensor([0, 1, 2, 3, 7, 400, 15], dtype=torch.int32, device="cuda")
    slots = torch.tensor([6, 2, 8, 5, 1, 3, 0], dtype=torch.int32, device="cuda")
    g = torch.Generator(device="cuda").manual_seed(taps + dim + vdim)
    draw = lambda *s: torch.randn(*s, device="cuda", generator=g)
    conv_w, a_log, dt_bias, norm_w = draw(channels, taps), draw(heads), draw(heads), draw(hv)
    state = draw(9, floats + 3 + max(taps - 1, 1) * channels)
    b_off, a_off, g_off = channels + hv + 1, channels + hv + 1 + heads, channels
    steps = [draw(n, a_off + heads + 5) for _ in range(3)]
    q_start, results = torch.arange(n + 1, dtype=torch.int32, device="cuda"), []
    for together in (False, True):
        kept, outs = state.clone(), []
        for t, proj in enumerate(steps):
            out = torch.zeros(n, hv + 3, device="cuda", dtype=dtype)[:, :hv]
            if together:
                ops.gated_delta_single(proj, b_off, a_off, g_off, conv_w, a_log, dt_bias, kept, floats + 3, positions + t, slots, norm_w,
                                       1e-6, out, heads, kv_heads, dim, vdim)
            else:
                prep, o = torch.empty(n, channels + 2 * heads, device="cuda"), torch.empty(n, hv, device="cuda")
                ops.conv_prepare(proj, b_off, a_off, conv_w, a_log, dt_bias, kept, floats + 3, q_start, positions + t, slots, prep, heads,
                                 kv_heads, dim, vdim, singles=True)
                ops.gated_delta_scan(prep, kept, q_start, positions + t, slots, o, heads, kv_heads, dim, vdim, singles=n)
                ops.head_norm_gate(o, proj[:, g_off:g_off + hv], norm_w, 1e-6, out, heads, vdim, gate="silu")
            outs.append(out)
        results.append((*outs, kept))
    assert all(torch.equal(one, other) for one, other in zip(*results))
    assert torch.equal(results[1][-1][[4, 7]], state[[4, 7]])   # nobody else's memory


def test_what_it_does_not_take():
    from dli_amd.kernels import ops

    takes = ops.gated_delta_single_takes
    assert not any(takes(*s) for s in [(4, 4, 48, 16, 4), (4, 4, 16, 129, 4), (4, 4, 16, 16, 5), (17, 1, 16, 4, 4), (9, 1, 16, 64, 4),
                                       (3, 1, 128, 128, 4), (3, 2, 16, 16, 4)])
