"""Portions under a chunked mask as pieces that are causal by themselves."""

import numpy as np
import pytest


@pytest.mark.parametrize("chunk", [16, 48, 64, 1000])
def test_pieces_see_what_the_mask_lets_rows_see(chunk):
    from dli_amd.parts.attention_kernels import chunk_pieces

    rng = np.random.default_rng(chunk)
    for _ in range(50):
        n = int(rng.integers(1, 6))
        new = rng.integers(1, 3 * chunk, n)
        old = np.where(rng.random(n) < 0.5, 0, rng.integers(0, 3 * chunk, n))
        first = int(rng.integers(0, n))
        q_start = np.concatenate([[0], np.cumsum(new)]).astype(np.int32)
        entry, first_key, begin, keys = chunk_pieces(q_start, (old + new).astype(np.int32), first, chunk)
        assert begin[0] == q_start[first] and begin[-1] == q_start[-1] and (np.diff(begin) > 0).all()
        for v in range(entry.size):
            e, rows = entry[v], range(int(begin[v]), int(begin[v + 1]))
            for place, row in enumerate(rows):
                pos = int(old[e]) + row - int(q_start[e])
                low = pos // chunk * chunk
                # the row is causal row `place` of a piece of len(rows) rows over keys[v] keys that begin at first_key[v]
                assert q_start[e] <= row < q_start[e + 1] and first_key[v] == low
                assert first_key[v] + int(keys[v]) - len(rows) + place == pos
