"""What a K past 8192 costs tiles of 128 rows counts for wide problems only; few rows or columns keep their slices."""
import pytest


@pytest.mark.parametrize("M,N,K,bm,bn,slices", [
    (249, 40, 25096, 128, 128, 99), (208, 128, 35712, 128, 128, 70), (323, 104, 11392, 128, 128, 30), (632, 72, 18688, 128, 128, 37),
    (194, 4480, 14928, 128, 128, 3), (127, 128, 28416, 128, 128, 74),  # fewer than 257 rows or 512 columns
    (1000, 4096, 11008, 256, 128, 2), (720, 1984, 15608, 192, 128, 4), (1000, 4096, 8192, 128, 128, 1)])
@pytest.mark.parametrize("trans_b", [False, True])
def test_choice(gc, M, N, K, bm, bn, slices, trans_b):
    c = gc.tile_config(M, N, K, trans_b=trans_b)[0]
    assert (c.bm, c.bn, c.split_k) == (bm, bn, slices)
