"""Which f32 kernel a size gets (asked of the launcher, no GPU needed)."""
import pytest


@pytest.mark.parametrize("M,N,K,tile,vector", [
    (128, 512, 256, 16, False), (300, 300, 1000, 16, False),       # few tiles: the small ones
    (1111, 1000, 3000, 32, False), (1111, 3000, 1000, 64, False), (2303, 2305, 130, 64, False),
    (2753, 2750, 515, 128, False), (4096, 4096, 4096, 128, False),
    (1071, 2048, 16, 64, False), (1200, 3000, 32, 64, False),      # a short K: many small tiles cost more than they save
    (1071, 2048, 72, 64, False),
    (256, 2048, 32, 32, True), (512, 900, 16, 32, True), (16, 16, 16, 16, True),  # one slice, under a round of 64 x 64 tiles
    (256, 2048, 33, 64, False), (1024, 1024, 32, 64, False),
])
def test_tile_of(gc, M, N, K, tile, vector):
    c, _ = gc.tile_config(M, N, K, a_dtype=gc.F32)
    assert (c.kernel, c.bm, c.bn, c.mfma_m == 0) == (6, tile, tile, vector)
