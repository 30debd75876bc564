"""Which products of many rows the kernel for one tile a compute unit takes: held to what it and the library took on an MI355X."""

from __future__ import annotations

# us, weights from memory, in a replayed graph: (rows, features, k): library and kernel
MEASURED = {
    (2048, 2048, 2048): (24.2, 21.6), (2048, 2048, 8192): (74.3, 67.2), (1464, 2048, 2048): (21.7, 20.1), (1464, 2048, 8192): (58.3, 64.8),
    (1100, 3072, 2048): (23.5, 21.4), (1100, 3072, 3072): (32.3, 30.2), (1100, 3072, 8192): (71.8, 68.2), (700, 5120, 3072): (33.4, 29.8),
    (700, 3072, 2048): (21.8, 19.9), (511, 6144, 2048): (25.5, 21.9), (1200, 2048, 2048): (23.1, 19.6), (1200, 2048, 8192): (63.2, 63.1),
    (1500, 2048, 2048): (21.8, 20.8), (1000, 3072, 3072): (31.0, 30.6), (344, 5504, 1024): (15.1, 12.5), (984, 2304, 1024): (14.9, 12.2),
    (1368, 2048, 1024): (12.9, 12.2), (2008, 1152, 2048): (21.0, 19.8), (984, 2304, 3072): (28.3, 29.5), (2008, 1536, 3072): (27.4, 28.5),
    (984, 3584, 3072): (32.7, 30.6), (984, 2304, 8192): (61.9, 65.4), (2008, 1408, 8192): (56.7, 61.3), (2008, 1792, 8192): (69.3, 64.3),
}


def test_products_of_a_tile_a_unit():
    from dli_amd.kernels import ops

    for (rows, feats, k), (library, here) in MEASURED.items():
        named = here if ops.library().dli_tile_gemm_takes(rows, feats, k, 256) else library
        assert named <= 1.03 * min(library, here), (rows, feats, k)


def test_sizes_it_leaves_to_the_library():
    from dli_amd.kernels import ops

    takes = ops.library().dli_tile_gemm_takes
    assert takes(2048, 2048, 256, 256)
    for rows, feats, k in [(0, 2048, 256), (2048, 0, 256), (2048, 2048, 0), (2048, 2048, 192), (2048, 2048, 288), (2048, 2044, 256),
                           (2049, 2048, 256), (1024, 2048, 256), (2048, 1664 - 8, 4096 - 32)]:
        assert not takes(rows, feats, k, 256)
