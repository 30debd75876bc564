"""Into how many runs a single request's keys are cut where its o projection merges them (no GPU)."""

from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

# ms, a pass of eight steps: (query heads, kv heads, head size, width): keys at the pass's end: runs: time
TIMES = {
    (9, 3, 64, 576): {312: {1: 4.88, 2: 4.87}, 408: {1: 5.09, 2: 4.85}, 520: {1: 5.17, 2: 4.91, 4: 4.95}, 648: {1: 5.53, 2: 5.11, 4: 4.98},
                      808: {2: 5.20, 4: 4.99}, 1008: {2: 5.27, 4: 5.05, 8: 5.11}, 1512: {4: 5.35, 8: 5.18}, 2008: {4: 5.39, 8: 5.19, 16: 5.46},
                      4008: {8: 5.76, 16: 5.54}, 8008: {16: 5.93}},
    (15, 5, 64, 960): {520: {1: 6.63, 2: 6.29}, 1008: {2: 6.67, 4: 6.38}},
    (32, 8, 64, 2048): {312: {1: 5.47, 2: 5.59}, 408: {1: 5.60, 2: 5.51}, 520: {1: 5.61, 2: 5.54}, 1008: {2: 5.76, 4: 5.57},
                        2008: {4: 5.78, 8: 5.64}, 8008: {16: 6.05}},
    (32, 32, 64, 2048): {520: {1: 8.17, 2: 8.03}, 1008: {2: 8.30, 4: 8.10}, 2008: {4: 8.42, 8: 8.40}, 4008: {4: 9.01, 8: 8.86, 16: 9.06},
                         8008: {8: 9.80, 16: 10.06}, 16008: {8: 11.85, 16: 12.26}, 32008: {8: 15.88, 16: 16.36}},
    (24, 8, 128, 3072): {312: {1: 13.04, 2: 13.26}, 520: {1: 13.37, 2: 13.10, 4: 13.20}, 1008: {2: 13.68, 4: 13.21, 8: 13.40},
                         2008: {4: 13.78, 8: 13.56, 16: 14.06}, 4008: {8: 14.07, 16: 14.06}},
}


@pytest.fixture
def plan(monkeypatch):
    """What an attention layer on 256 compute units answers for one request, whether its o projection merges or not."""
    from dli_amd.kernels import ops
    from dli_amd.parts.attention import GQAttention

    monkeypatch.setattr(ops, "_units", lambda device: 256)

    def answer(q_heads, kv_heads, head_dim, width, keys, merges=True, requests=1):
        layer = object.__new__(GQAttention)
        layer.rt = SimpleNamespace(is_bf16=True, device=torch.device("cuda", 0))
        layer.num_heads, layer.num_kv_heads, layer.head_dim, layer.hidden_size = q_heads, kv_heads, head_dim, width
        layer.w_o_merging = torch.empty(0) if merges else None
        return layer.decode_plan(requests, keys)

    return answer


@pytest.mark.parametrize("sizes", TIMES)
def test_runs_follow_the_times(sizes, plan):
    for keys, times in TIMES[sizes].items():
        runs = plan(*sizes, keys)
        assert times[runs] <= 1.015 * min(times.values()), (keys, runs)


def test_runs_within_the_product(plan):
    """Never a number that the layer does not run: up to the product's sixteen its own rule, past them the rule of steps of several
    requests; and that one from the first key on where the product does not merge."""
    from dli_amd.kernels import ops
    from dli_amd.parts.attention_kernels import planned_splits, runs_for_the_product

    for kv_heads in (1, 8, 32, 300):
        last = 0
        for keys in (1, 128, 383, 384, 1000, 10 ** 4, 10 ** 6):
            runs, others = runs_for_the_product(kv_heads, kv_heads, keys, 256), planned_splits(1, kv_heads, kv_heads, 64, keys, 256)
            if runs is not None:
                assert last <= runs <= ops.MERGED_SPLITS and runs & (runs - 1) == 0 and runs * kv_heads <= max(256, kv_heads)
                last = runs
            if 2 <= kv_heads <= 32:
                assert plan(kv_heads, kv_heads, 64, 2048, keys) == (runs or others)
            assert plan(kv_heads, kv_heads, 64, 2048, keys, merges=False) == others
            assert plan(kv_heads, kv_heads, 64, 2048, keys, requests=2) == planned_splits(2, kv_heads, kv_heads, 64, keys, 256)
    assert runs_for_the_product(8, 8, 4223, 256) == 16 and runs_for_the_product(8, 8, 4224, 256) is None
