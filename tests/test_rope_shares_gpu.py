"""The rotation with cache writes of many rows, whose heads are dealt over several workgroups."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from dli_amd.kernels import ops as module

    return module


@pytest.mark.parametrize("qh,kvh,d,rd", [(32, 32, 64, 64), (8, 4, 64, 32), (12, 6, 128, 128), (10, 2, 16, 16), (9, 3, 64, 64)])
@pytest.mark.parametrize("n,offset", [(513, 0), (600, 3), (1100, 16)])
def test_rope_kv_write_in_shares_of_heads(ops, qh, kvh, d, rd, n, offset):
    """Rows by the workgroup whose heads are dealt over several (from 513 rows on), against the same rows 300 at a time
    (an item a thread): every value is made alike."""
    gen = torch.Generator(device="cuda").manual_seed(n + qh)
    dtype, bs = torch.bfloat16, 16
    qkv = torch.randn(n, (qh + 2 * kvh) * d, device="cuda", generator=gen).to(dtype)
    positions = torch.arange(7, 7 + n, dtype=torch.int32, device="cuda")
    slots = (torch.arange(n, device="cuda") + offset).int()
    slots[[5, 400]] = -1   # rows without a place in the cache
    inv_freq = torch.rand(rd // 2, device="cuda", generator=gen)
    pages = (n + offset) // bs + 2
    results = []
    for cut in (n, 300):
        rows = qkv.clone()
        kp, vp = torch.full((pages, kvh, bs, d), 3.0, device="cuda", dtype=dtype), torch.full((pages, kvh, d, bs), 3.0, device="cuda", dtype=dtype)
        for a in range(0, n, cut):
            b = min(n, a + cut)
            ops.rope_kv_write(rows[a:b], positions[a:b], inv_freq, rd, slots[a:b].contiguous(), kp, vp, qh, kvh, d)
        results.append((rows[:, :qh * d], kp, vp))
    for one, other in zip(*results):
        assert torch.equal(one, other)


@pytest.mark.parametrize("heads,d", [(22, 128), (46, 64)])
def test_rows_whose_v_fills_the_lds(ops, heads, d):
    test_rope_kv_write_in_shares_of_heads(ops, heads, heads, d, d, 2100, 3)
