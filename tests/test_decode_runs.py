"""Into how many runs a single request's keys are cut where its o projection merges them (no GPU)."""

from __future__ import annotations

import pytest

# ms, a pass of eight steps: (query heads, kv heads): keys at the pass's end: runs: time
TIMES = {
    (9, 3): {312: {1: 4.91, 2: 4.92}, 408: {1: 5.19, 2: 5.05}, 520: {1: 5.30, 2: 4.95, 4: 5.00}, 648: {1: 5.56, 2: 5.17, 4: 5.02},
             808: {2: 5.28, 4: 5.00}, 1008: {2: 5.38, 4: 5.02, 8: 5.09}, 1512: {4: 5.38, 8: 5.20}, 2008: {4: 5.47, 8: 5.17, 16: 5.55},
             4008: {8: 5.80, 16: 5.45, 32: 5.84}},
    (32, 8): {312: {1: 5.47, 2: 5.59}, 408: {1: 5.60, 2: 5.51}, 520: {1: 5.66, 2: 5.56}, 1008: {2: 5.76, 4: 5.57},
              2008: {4: 5.78, 8: 5.64}, 8008: {16: 6.07, 32: 5.99, 64: 6.14}},
    (32, 32): {520: {1: 8.24, 2: 8.04}, 1008: {2: 8.35, 4: 8.10}, 4008: {4: 9.08, 8: 8.87, 16: 9.11}},
}


@pytest.mark.parametrize("q_heads,kv_heads", TIMES)
def test_runs_follow_the_times(q_heads, kv_heads):
    from dli_amd.parts.attention_kernels import runs_for_the_product

    for keys, times in TIMES[q_heads, kv_heads].items():
        runs = runs_for_the_product(q_heads, kv_heads, keys, 256)
        assert times[runs] <= 1.015 * min(times.values()), (keys, runs)


def test_runs_within_their_limits():
    from dli_amd.parts.attention_kernels import MAX_SPLITS, runs_for_the_product

    for kv_heads in (1, 8, 40, 300):
        last = 0
        for keys in (1, 128, 383, 384, 1000, 10 ** 4, 10 ** 6):
            runs = runs_for_the_product(kv_heads, kv_heads, keys, 256)
            assert last <= runs <= MAX_SPLITS and runs & (runs - 1) == 0 and runs * kv_heads <= max(256, kv_heads)
            last = runs
