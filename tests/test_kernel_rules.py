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
