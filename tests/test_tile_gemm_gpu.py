"""Products of many rows whose result is about one 128 x 128 tile a compute unit, at edges of tiles and the rule's ends."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

UNITS = 256


@pytest.mark.parametrize("rows,feats,k,bias,out", [
    (1, 129 * 128, 256, False, "bfloat16"),           # one row, as few blocks of k as stages, one tile above the half
    (128, 256 * 128 - 120, 256, True, "float32"),     # a whole tile of rows, eight features in the last
    (129, 80 * 128 + 8, 320, True, "bfloat16"),       # a row and eight features in their last tiles, five blocks
    (2047, 2048, 2048, True, "bfloat16"),
    (2048, 2048, 2048, False, "float32"),
    (1025, 2944, 2112, True, "bfloat16"),             # bands of eight tiles and of one; a long k
    (1664, 2000, 8192, False, "bfloat16"),
])
def test_product_of_a_tile_a_unit(rows, feats, k, bias, out):
    from dli_amd.kernels import ops

    if torch.cuda.get_device_properties(0).multi_processor_count != UNITS:
        pytest.skip("sizes chosen for 256 compute units")
    assert ops.library().dli_tile_gemm_takes(rows, feats, k, UNITS)
    g = torch.Generator(device="cuda").manual_seed(rows + feats + k)
    draw = lambda *s: torch.randn(*s, device="cuda", generator=g)
    x, w = draw(rows, k + 24).bfloat16()[:, 8:k + 8], (draw(feats, k + 8) * k ** -0.5).bfloat16()[:, :k]   # rows of a wider matrix
    b = draw(feats).bfloat16() if bias else None
    dtype = getattr(torch, out)
    whole = torch.full((rows + 2, feats + 16), -7.0, device="cuda", dtype=dtype)
    got = whole[1:-1, 8:-8]
    assert ops.gemm_bf16(x, w, got, b)
    expected, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    if bias:
        expected, size = expected + b.double(), size + b.double().abs()
    # k + 1 additions in 32 bits, each off by at most 2^-24 of a partial sum no larger than `size` (products of bfloat16 are exact,
    # and the matrix units' own sums may drop a bit more: twice that), and one rounding to the eight bits of
    # a bfloat16, the first of them included: half of the last is at most 2^-8 of the value
    bound = (k + 1) * 2.0 ** -23 * size
    bound = bound + (2.0 ** -8 * (expected.abs() + bound) if out == "bfloat16" else 0)
    assert ((got.double() - expected).abs() <= bound).all()
    assert (whole[0] == -7).all() and (whole[-1] == -7).all() and (whole[:, :8] == -7).all() and (whole[:, -8:] == -7).all()


def test_rows_of_infinities_stay_in_their_rows():
    from dli_amd.kernels import ops

    x, w = torch.randn(1999, 512, device="cuda").bfloat16(), torch.randn(2048, 512, device="cuda").bfloat16()
    out, alone = (torch.empty(1999, 2048, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    assert ops.gemm_bf16(x, w, alone)
    y = x.clone()
    y[1998], y[64, 3] = float("inf"), float("nan")
    assert ops.gemm_bf16(y, w, out)
    kept = torch.ones(1999, dtype=torch.bool, device="cuda")
    kept[[1998, 64]] = False
    assert torch.equal(out[kept], alone[kept]) and out[64].isnan().all() and not out[1998].isfinite().any()
