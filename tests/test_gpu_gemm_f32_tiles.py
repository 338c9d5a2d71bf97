"""The f32 GEMM's tiles (16, 32, 64 and 128 squared, chosen by size) at their edges, in every operand layout."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# one row/column, less than a 16-byte chunk, one off a tile, K below, at and past a slice and past its steady loop, on
# tiles of 16 and 64 and on the vector kernel (sizes chosen for each tile, ragged and strided: test_gpu_gemm_f32_edges.py)
SHAPES = [(1, 1, 1), (3, 3, 70), (1, 300, 64), (17, 15, 16), (40, 50, 1030), (513, 547, 65), (545, 511, 400),
          (961, 1023, 33), (1023, 1090, 257), (1111, 1501, 31), (2049, 2050, 47), (2048, 2048, 128)]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("ta", [False, True])
@pytest.mark.parametrize("tb", [False, True])
def test_f32_tiles(gc, dev, M, N, K, ta, tb):
    g = torch.Generator(device=dev).manual_seed(M * 7 + N * 3 + K)
    A = torch.randn((K, M) if ta else (M, K), device=dev, generator=g)
    B = torch.randn((N, K) if tb else (K, N), device=dev, generator=g)
    bias = torch.randn(N, device=dev, generator=g)
    out = gc.gemm_f32(A, B, bias, None, ta, tb).double()
    a, b = (A.t() if ta else A).double(), (B.t() if tb else B).double()
    ref, mag = a @ b + bias.double(), a.abs() @ b.abs() + bias.double().abs()
    # K + 1 additions of exact products, each rounded once, in any order: at most (K + 1) half-ulps of the magnitudes
    assert ((out - ref).abs() <= (K + 1) * 2.0 ** -24 * mag).all()


@pytest.mark.parametrize("nb,M,N,K", [(40, 100, 96, 70), (6, 700, 600, 50)])
def test_f32_batch_has_the_bits_of_its_matrices(gc, dev, nb, M, N, K):
    """Batches large enough for another tile than one of their matrices gets alone."""
    g = torch.Generator(device=dev).manual_seed(5)
    A, B = torch.randn(nb, M, K, device=dev, generator=g), torch.randn(nb, K, N, device=dev, generator=g)
    assert torch.equal(gc.gemm_batched(A, B), torch.stack([gc.gemm_f32(A[i], B[i]) for i in range(nb)]))
