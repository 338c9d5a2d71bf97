"""bf16 problems of half a round to three rounds of 256 x 256 tiles: the tile with the least estimated time; the large one outside
the range that was measured, and by name."""
import pytest


@pytest.mark.parametrize("M,N,K,kernel,bm,bn", [
    (1000, 11008, 4096, 5, 256, 192), (2655, 3520, 3800, 5, 256, 192), (1643, 10048, 1408, 5, 192, 128), (3597, 4672, 128, 5, 128, 128),
    (2048, 11008, 4096, 2, 256, 256), (4096, 11008, 4096, 2, 256, 256), (4096, 4096, 4096, 2, 256, 256), (4096, 4096, 1000, 2, 256, 256),
    (8192, 12288, 128, 2, 256, 256)])
@pytest.mark.parametrize("trans_b", [False, True])
def test_choice(gc, M, N, K, kernel, bm, bn, trans_b):
    c = gc.tile_config(M, N, K, trans_b=trans_b)[0]
    assert (c.kernel, c.bm, c.bn, c.split_k) == (kernel, bm, bn, 1)
    assert c.workgroups == -(-M // bm) * -(-N // bn) and (c.wave_m, c.wave_n) == (bm // 2, bn // 2)
    c = gc.tile_config(M, N, K, trans_b=trans_b, matmul_config=[1, 1, 1, 256, 256, 64, 128, 128, 32])[0]
    assert (c.kernel, c.bm, c.bn) == (2, 256, 256)
