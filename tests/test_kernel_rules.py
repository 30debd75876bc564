"""Rules that choose between two kernels, held to what both took on an MI355X: at none of the measured sizes does the rule name
one that was more than a few percent behind."""

from __future__ import annotations

import pytest

# us, cold, a launch in a replayed graph, at 1, 2, 3, 4, 5, 6, 8, 12 and 16 rows: the general kernel, then the one that normalises
# the rows once a workgroup
ROWS = (1, 2, 3, 4, 5, 6, 8, 12, 16)
NORMED = {
    # q/k/v: (features, width)
    (960, 576, False): ((4.1, 4.2, 4.2, 4.2, 4.2, 4.2, 4.3, 4.4, 4.4), (3.9, 4.5, 4.3, 4.4, 4.9, 5.0, 5.1, 5.8, 6.2)),
    (1600, 960, False): ((4.6, 4.6, 4.6, 4.7, 4.7, 4.7, 4.8, 4.8, 5.0), (4.3, 4.9, 4.7, 4.9, 5.3, 5.5, 5.6, 6.4, 6.7)),
    (3072, 2048, False): ((6.5, 6.4, 6.5, 6.5, 6.5, 6.5, 6.7, 6.9, 7.2), (5.3, 5.8, 5.8, 5.8, 6.5, 6.6, 6.8, 7.8, 8.1)),
    (6144, 2048, False): ((8.9, 9.0, 9.0, 9.1, 8.8, 8.8, 9.0, 9.4, 9.9), (8.7, 9.1, 9.7, 9.2, 9.2, 9.4, 9.8, 11.4, 12.1)),
    (4608, 1536, False): ((6.9, 6.9, 6.9, 7.0, 7.1, 7.1, 7.3, 7.5, 8.0), (7.1, 7.6, 7.6, 7.5, 8.0, 8.1, 8.5, 9.8, 10.6)),
    (5120, 3072, False): ((11.8, 11.9, 12.0, 11.3, 11.4, 11.5, 11.7, 12.2, 13.0), (9.8, 10.4, 11.8, 10.3, 11.8, 12.0, 11.6, 12.2, 13.0)),
    (6144, 4096, False): ((15.9, 15.2, 15.3, 15.5, 15.6, 15.6, 15.9, 16.4, 17.1), (13.8, 14.3, 16.6, 14.6, 17.1, 17.3, 16.1, 16.4, 17.1)),
    (1536, 1024, False): ((4.5, 4.5, 4.6, 4.6, 4.6, 4.7, 4.7, 4.8, 4.9), (4.3, 4.9, 4.7, 4.8, 5.3, 5.4, 5.6, 6.4, 6.7)),
    (3072, 1024, False): ((4.8, 4.8, 4.9, 4.9, 4.9, 4.9, 5.0, 5.1, 5.2), (4.6, 5.2, 4.9, 5.0, 5.5, 5.6, 5.8, 6.6, 6.9)),
    # gate and up, from two rows on (one row takes neither): (features of one half, width)
    (8192, 2048, True): ((15.4, 15.3, 15.3, 15.4, 15.5, 15.8, 16.1, 16.9), (14.8, 16.0, 15.0, 15.9, 16.0, 16.4, 18.1, 19.0)),
    (6144, 1536, True): ((10.3, 10.2, 10.2, 10.1, 10.2, 10.3, 10.5, 10.8), (10.4, 11.3, 10.5, 10.9, 11.1, 11.4, 12.9, 13.5)),
    (8192, 3072, True): ((22.1, 21.4, 21.5, 21.3, 21.6, 21.7, 22.2, 22.9), (21.0, 22.5, 20.4, 22.8, 23.0, 21.5, 23.1, 23.4)),
    (4096, 1024, True): ((6.5, 6.0, 6.1, 6.1, 6.2, 6.2, 6.3, 6.4), (6.7, 6.6, 6.8, 6.2, 6.3, 6.5, 7.2, 7.6)),
}


@pytest.mark.parametrize("n,k,gated", NORMED)
def test_products_behind_a_norm(n, k, gated):
    from dli_amd.kernels import ops

    for rows, general, normed in zip(ROWS[gated:], *NORMED[n, k, gated]):
        named = normed if ops.normed_tiles_ahead(rows, n, k, gated, 256) else general
        assert named <= 1.03 * min(general, normed), (rows, general, normed)


# ms, a pass of eight steps of a model of twelve layers in 32-bit: (gates and ups, width): rows: apart and fused
F32_NORMED = {
    (4096, 512): {1: (3.49, 2.94), 4: (3.86, 3.34), 16: (4.46, 4.20)},
    (8192, 512): {2: (4.39, 3.92), 6: (5.05, 4.58), 8: (5.10, 4.53), 12: (5.62, 5.36), 16: (5.55, 5.42)},
    (6144, 768): {2: (4.93, 4.41), 6: (5.39, 4.99), 8: (5.47, 5.03), 12: (6.04, 5.78), 16: (6.07, 5.82)},
    (5120, 960): {1: (4.95, 4.40), 4: (5.30, 4.90), 16: (6.20, 6.00)},
    (15360, 960): {2: (6.74, 6.56), 6: (7.59, 7.73), 8: (7.66, 7.76), 12: (8.74, 9.29), 16: (8.79, 9.32)},
    (5632, 1024): {1: (4.77, 4.36), 2: (4.86, 4.52), 4: (5.13, 4.85), 6: (5.39, 5.14), 8: (5.39, 5.14), 12: (6.04, 6.01), 16: (6.08, 6.02)},
    (8192, 1024): {2: (5.21, 4.66), 6: (5.77, 5.38), 8: (5.81, 5.41), 12: (6.51, 6.41), 16: (6.55, 6.49)},
    (16384, 1024): {1: (7.09, 6.90), 2: (7.25, 7.15), 4: (7.61, 7.65), 6: (8.20, 8.43), 8: (8.24, 8.49), 12: (9.88, 10.45), 16: (9.96, 10.54)},
    (5888, 1088): {2: (5.37, 5.68), 6: (5.95, 6.45), 8: (5.98, 6.47), 12: (6.99, 7.61), 16: (7.05, 7.66)},
    (6144, 1152): {1: (5.19, 5.19), 4: (5.52, 5.79), 16: (6.87, 7.32)},
    (6912, 1280): {1: (5.45, 5.43), 4: (5.88, 6.03), 16: (7.27, 7.74)},
    (8192, 1536): {1: (5.89, 5.81), 4: (6.27, 6.46), 16: (8.08, 8.58)},
    (16384, 2048): {1: (8.36, 9.20), 4: (8.82, 9.91), 16: (11.55, 13.29)},
}


@pytest.mark.parametrize("n,k", F32_NORMED)
def test_32_bit_products_behind_a_norm(n, k):
    from dli_amd.kernels import ops

    for rows, (apart, fused) in F32_NORMED[n, k].items():
        assert (fused if ops.gemm_f32_normed_ahead(rows, n, k) else apart) <= 1.02 * min(apart, fused), (rows, apart, fused)


# ms, a pass of eight steps from a context on: (query heads, kv heads, head size, requests): keys at the pass's end: two runs and one
ONE_RUN = {
    (9, 3, 64, 1): {520: (5.91, 5.60), 536: (5.92, 5.73), 552: (5.91, 5.77), 568: (5.90, 5.87), 600: (5.92, 5.94), 632: (5.92, 6.08)},
    (32, 8, 64, 1): {520: (5.86, 5.78), 536: (5.87, 5.79), 552: (5.88, 5.84), 568: (5.88, 5.90), 600: (5.87, 5.95), 632: (5.89, 6.02)},
    (32, 8, 64, 8): {520: (7.03, 6.84), 536: (7.03, 6.87), 552: (7.03, 6.91), 568: (7.04, 6.96), 600: (7.01, 7.04), 632: (7.03, 7.10)},
    (15, 5, 64, 8): {520: (8.90, 8.66), 536: (8.90, 8.72), 552: (8.90, 8.73), 568: (8.91, 8.86), 600: (8.90, 9.00), 632: (8.90, 9.12)},
    (9, 3, 64, 16): {520: (8.12, 7.85), 536: (8.14, 7.89), 552: (8.12, 7.92), 568: (8.15, 8.06), 600: (8.13, 8.23), 632: (8.16, 8.29)},
    (32, 8, 32, 8): {536: (3.25, 3.08), 552: (3.23, 3.09), 568: (3.24, 3.10)},
    (16, 8, 80, 4): {536: (3.42, 3.36), 552: (3.43, 3.39), 568: (3.44, 3.44), 584: (3.43, 3.51)},
    (16, 8, 96, 1): {536: (3.31, 3.35), 552: (3.32, 3.38), 568: (3.33, 3.44), 584: (3.31, 3.49)},
    (16, 8, 96, 8): {536: (3.97, 3.93), 552: (3.98, 3.97), 568: (3.99, 4.02), 584: (3.99, 4.09)},
    (16, 2, 128, 1): {536: (3.70, 3.75), 552: (3.71, 3.82), 568: (3.70, 3.88), 584: (3.70, 3.98)},
    (16, 2, 128, 8): {536: (4.60, 4.41), 552: (4.60, 4.48), 568: (4.60, 4.56), 584: (4.61, 4.65)},
    (24, 8, 128, 1): {520: (4.91, 4.76), 552: (4.91, 4.87), 584: (4.90, 5.04), 648: (4.91, 5.16)},
    (24, 8, 128, 4): {520: (5.19, 5.10), 552: (5.17, 5.22), 584: (5.18, 5.36), 648: (5.20, 5.49)},
    (24, 8, 128, 8): {520: (5.53, 5.43), 552: (5.53, 5.56), 584: (5.53, 5.72), 648: (5.55, 5.84)},
    (16, 1, 128, 1): {520: (3.53, 3.63), 552: (3.55, 3.68), 584: (3.58, 3.76), 648: (3.65, 3.82)},
    (16, 1, 128, 2): {536: (4.29, 3.85), 552: (4.28, 3.87), 568: (4.30, 3.95)},
    (16, 1, 128, 4): {536: (4.32, 3.91), 552: (4.32, 3.93), 568: (4.32, 4.00)},
    (16, 1, 128, 16): {520: (5.49, 5.10), 552: (5.52, 5.14)},
    (14, 1, 112, 2): {536: (4.07, 3.63), 552: (4.06, 3.65), 568: (4.06, 3.67)},
}


@pytest.mark.parametrize("q_heads,kv_heads,head_dim,requests", ONE_RUN)
def test_one_run_of_keys_or_two(q_heads, kv_heads, head_dim, requests):
    from dli_amd.parts.attention_kernels import planned_splits

    for keys, (two, one) in ONE_RUN[q_heads, kv_heads, head_dim, requests].items():
        runs = planned_splits(requests, q_heads, kv_heads, head_dim, keys, 256)
        assert runs in (1, 2)
        assert (one if runs == 1 else two) <= 1.03 * min(two, one), (keys, runs, two, one)


def test_waves_of_a_decode_workgroup():
    """Eight where every workgroup has a compute unit to itself and the states of eight waves fit 48 KB, else four."""
    from dli_amd.kernels import ops

    for group in range(1, 40):
        for d in range(16, 144, 16):
            fits = 8 * 4 * d * min(group, 16) <= 48 * 1024   # a state: a float a dimension and head
            assert ops.attention_decode_waves(256, group, d, 256) == (8 if fits else 4)
            assert ops.attention_decode_waves(257, group, d, 256) == 4
    assert ops.attention_decode_waves(1, 12, 128, 256) == 8 and ops.attention_decode_waves(1, 13, 128, 256) == 4


@pytest.mark.parametrize("kv,d,dtype", [(22, 128, "bfloat16"), (46, 64, "bfloat16"), (11, 128, "float32"), (23, 64, "float32")])
def test_rotated_rows_that_just_fit(kv, d, dtype):
    """Eight rows of v beside their angles fill 48 KB of LDS; one kv head more does not fit."""
    import torch

    from dli_amd.kernels import ops

    shares = lambda heads: ops.rope_kv_shares(4096, d, heads, heads, d, getattr(torch, dtype), 256)
    assert 8 * d * 4 + 8 * kv * d * getattr(torch, dtype).itemsize == 48 * 1024
    assert shares(kv) == 1 and shares(kv - 1) == 1 and shares(kv + 1 + kv % 2) == 0


# (rows, heads, q/k heads, key size, value size): us by the three kernels of the gated delta rule's single tokens, and by the one
GATED_SINGLES = {
    (4, 32, 8, 64, 64): (8.3, 5.5), (256, 32, 8, 64, 64): (58.0, 52.3), (256, 32, 32, 64, 64): (64.8, 57.0), (256, 128, 128, 16, 64): (199.3, 185.0),
    (16, 32, 32, 64, 16): (8.6, 5.6), (64, 8, 8, 64, 16): (9.0, 5.6), (256, 8, 8, 16, 16): (12.0, 12.6), (64, 32, 32, 16, 16): (11.7, 12.7),
    (64, 32, 32, 64, 16): (13.3, 15.3), (256, 32, 32, 32, 16): (30.4, 43.1), (256, 32, 32, 128, 16): (63.3, 63.3), (64, 64, 32, 64, 16): (17.7, 16.1),
    (64, 8, 8, 16, 4): (8.1, 5.0), (64, 32, 32, 16, 4): (9.9, 12.3),
    (256, 32, 32, 64, 32): (44.0, 49.5), (256, 64, 32, 16, 16): (40.1, 44.1), (16, 128, 128, 64, 32): (17.3, 15.9), (256, 128, 128, 128, 32): (481.0, 313.0)}


def test_single_tokens_of_the_gated_delta_rule():
    from dli_amd.parts.recurrent import single_kernel_pays

    for sizes, (three, one) in GATED_SINGLES.items():
        chosen = one if single_kernel_pays(*sizes, 4) else three
        assert chosen <= 1.03 * min(three, one), sizes
    assert not single_kernel_pays(4, 32, 8, 48, 64, 4) and not single_kernel_pays(4, 32, 8, 64, 64, 5)   # sizes without such a kernel
