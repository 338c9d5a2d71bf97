"""f32 GEMMs of more tiles than one dimension of a grid holds (2^24 workgroups of 256 threads)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,ta", [(2, (1 << 28) + 5, True),   # 16 x 16 tiles: two rows stored [K,M] are no 16-byte chunk
                                    (1, (1 << 29) + 3, False)])
def test_f32_many_tiles(gc, dev, M, N, ta):
    A = torch.arange(1, M + 1, device=dev, dtype=torch.float32).reshape((1, M) if ta else (M, 1))
    B = torch.empty(1, N, device=dev)
    B[0] = torch.arange(N, device=dev, dtype=torch.int32) & 0xffff
    out = gc.gemm_f32(A, B, trans_a=ta)
    for m in range(M):  # one product per element: exact
        assert torch.equal(out[m], B[0] * float(m + 1))
