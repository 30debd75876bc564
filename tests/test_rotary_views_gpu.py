"""The rotation and cache write with a bias and norm weights that are views of longer vectors: the same bits wherever they begin."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("rows,qh,kv,d,interleaved", [(3, 5, 5, 48, False), (130, 8, 2, 64, False), (200, 4, 4, 96, True)])
def test_a_bias_and_norm_weights_that_begin_anywhere(rows, qh, kv, d, interleaved, dtype):
    from dli_amd.kernels import ops

    dtype, width = getattr(torch, dtype), (qh + 2 * kv) * d
    g = torch.Generator(device="cuda").manual_seed(rows)
    draw = lambda *s: torch.randn(*s, generator=g, device="cuda")
    proj, inv_freq = draw(rows, width), (1e4 ** (-torch.arange(0, 32, 2).double() / 32)).float().cuda()
    vectors = draw(width), 1 + 0.1 * draw(qh * d), 1 + 0.1 * draw(kv * d)
    slots = torch.arange(rows, device="cuda").int()
    results = []
    for off in range(4):
        bias, q_norm, k_norm = (torch.cat([v.new_zeros(off), v, v.new_zeros(4)])[off:off + v.shape[0]] for v in vectors)
        assert bias.data_ptr() % 16 == 4 * off
        q = torch.empty(rows, qh * d, device="cuda", dtype=dtype)
        pages = [torch.zeros(s, device="cuda", dtype=dtype) for s in ((rows // 16 + 1, kv, 16, d), (rows // 16 + 1, kv, d, 16))]
        ops.rotary_cache(proj, 0, qh * d, (qh + kv) * d, slots, inv_freq, 32, interleaved, q, slots, *pages, qh, bias=bias,
                         row_norm=(q_norm, k_norm, 1e-6))
        results.append((q, *pages))
    for other in results[1:]:
        assert all(torch.equal(a, b) for a, b in zip(results[0], other))
