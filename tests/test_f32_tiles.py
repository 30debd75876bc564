"""Which 32-bit products of many rows leave tiles of 32 x 32 with four waves for tiles of 64 x 64 with loads ahead: held to what both
took on an MI355X."""

from __future__ import annotations

# us, weights from memory, in a replayed graph: (rows, columns, k): four waves a tile, loads ahead
MEASURED = {
    (192, 2800, 576): (21.0, 17.6), (192, 2800, 960): (26.7, 25.8), (192, 2800, 2048): (48.0, 48.6), (500, 1536, 576): (23.1, 17.6),
    (500, 1536, 2048): (46.7, 48.1), (700, 1280, 960): (31.5, 25.4), (700, 1280, 2048): (57.1, 48.6), (100, 3072, 576): (13.7, 16.9),
    # rows that half fill their last tile of 64
    (24, 12198, 576): (13.8, 16.8), (28, 14961, 2048): (33.4, 48.3), (177, 2716, 768): (18.4, 20.7), (93, 10291, 2048): (63.0, 80.4),
    (91, 12462, 1536): (58.5, 61.2), (163, 5721, 3072): (101.5, 116.9),
    # tiles just past a round of one or two a unit, and well past it
    (556, 1826, 480): (23.7, 22.4), (526, 1871, 480): (20.9, 22.6), (556, 1826, 576): (29.2, 25.7), (746, 1437, 768): (39.3, 34.3),
    (556, 1826, 960): (39.0, 39.8), (501, 2102, 1024): (39.8, 42.4), (188, 6126, 1536): (58.8, 61.4), (556, 1826, 2048): (74.6, 79.8),
    (503, 2228, 3072): (105.2, 115.7), (1004, 1378, 960): (45.9, 40.6), (1017, 1372, 1024): (46.6, 42.4), (1004, 1378, 2048): (84.4, 78.7),
    (362, 4282, 2048): (106.1, 79.6), (739, 1964, 3072): (130.6, 116.9), (757, 2716, 2048): (118.0, 121.7), (757, 2716, 576): (47.6, 40.8),
    (155, 11000, 576): (44.0, 40.2),
}


def test_tiles_of_a_unit():
    from dli_amd.kernels import ops

    for (m, n, k), (few, ahead) in MEASURED.items():
        named = ahead if ops.library().dli_gemm_f32_few_waves_ahead(m, n, k, 256) else few
        assert named <= 1.035 * min(few, ahead), (m, n, k)
