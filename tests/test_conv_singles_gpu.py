"""The short convolution of a step of single tokens, which leaves the inputs to keep by itself: the same bits as with the kernel
that keeps them afterwards."""

import pytest
import torch

pytestmark = pytest.mark.gpu


# taps: none to keep, known numbers, four at a time with and without a rest, the most
@pytest.mark.parametrize("taps", [1, 2, 3, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("heads,kv_heads,dim,vdim", [(4, 2, 64, 64), (3, 1, 20, 10), (2, 2, 130, 66)])
def test_kept_inputs_of_single_tokens(taps, heads, kv_heads, dim, vdim):
    from dli_amd.kernels import ops

    positions = torch.tensor([0, 1, 2, 3, 7, 400, 15], dtype=torch.int32, device="cuda")
    n, channels, slots = 7, 2 * kv_heads * dim + heads * vdim, torch.tensor([6, 2, 8, 5, 1, 3, 0], dtype=torch.int32, device="cuda")
    g = torch.Generator(device="cuda").manual_seed(taps + dim)
    draw = lambda *s: torch.randn(*s, device="cuda", generator=g)
    conv_w, a_log, dt_bias, state = draw(channels, taps), draw(heads), draw(heads), draw(9, 11 + max(taps - 1, 1) * channels)
    steps = [draw(n, channels + 2 * heads + 5) for _ in range(3)]
    q_start, results = torch.arange(n + 1, dtype=torch.int32, device="cuda"), []
    for singles in (False, True):
        kept, outs = state.clone(), []
        for t, proj in enumerate(steps):
            out = torch.zeros(n, channels + 2 * heads, device="cuda")
            ops.conv_prepare(proj, channels, channels + heads, conv_w, a_log, dt_bias, kept, 11, q_start, positions + t, slots, out, heads,
                             kv_heads, dim, vdim, singles=singles)
            outs.append(out)
        results.append((*outs, kept))
    assert all(torch.equal(one, other) for one, other in zip(*results))
    assert torch.equal(results[1][-1][[4, 7]], state[[4, 7]])   # nobody else's memory
    # entries of several rows: only the flag makes them wrong, whose waves would write what others of their entry still read
    several = torch.tensor([0, 3, 4, 7], dtype=torch.int32, device="cuda")
    call = lambda singles: ops.conv_prepare(steps[0], channels, channels + heads, conv_w, a_log, dt_bias, state, 11, several, positions,
                                            slots[:3].contiguous(), outs[0], heads, kv_heads, dim, vdim, singles=singles)
    call(False)
    with pytest.raises(ops.KernelArgumentError, match="single tokens"):
        call(True)
