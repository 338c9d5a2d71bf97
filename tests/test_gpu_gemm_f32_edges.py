"""Every f32 kernel (16, 32, 64 and 128 squared tiles of the matrix instruction, the vector kernel) at ragged sizes that
are known to take it, with rows longer than the operands and NaN in what lies between."""
import pytest
import torch

pytestmark = pytest.mark.gpu

NAN = float("nan")
# tile, M, N, K: rows and columns one to three off a chunk of four and a tile, K off a slice (64, 32 and 16 deep) and at one
SIZES = [("vector", 301, 259, 29), ("vector", 5, 6, 32), (16, 133, 95, 77), (16, 67, 130, 515), (32, 777, 555, 260),
         (32, 775, 554, 321), (64, 2303, 2305, 130), (64, 1022, 1090, 257), (64, 1201, 1301, 96), (128, 2753, 2750, 515),
         (128, 2750, 2755, 528)]


def _tile(gc, M, N, K, tb=False):
    c = gc.tile_config(M, N, K, a_dtype=gc.F32, trans_b=tb)[0]
    return c.bm if c.mfma_m else "vector"


def _strided(rows, cols, dev, g, pad):
    """rows x cols random values inside rows of cols + pad, NaN behind each row and below the last."""
    full = torch.full((rows + 3, cols + pad), NAN, device=dev)
    full[:rows, :cols] = torch.randn(rows, cols, device=dev, generator=g)
    return full[:rows, :cols]


def _call(gc, A, B, out, bias, act, ta, tb):
    M, N = out.shape
    K = A.shape[0] if ta else A.shape[1]
    gc.check(gc.lib().gcmi_gemm_f32(A.data_ptr(), B.data_ptr(), out.data_ptr(), M, N, K, A.stride(0), B.stride(0), out.stride(0),
                                    int(ta), int(tb), bias.data_ptr(), gc.ACT[act], torch.cuda.current_stream().cuda_stream))


@pytest.mark.parametrize("tile,M,N,K", SIZES)
# every layout of the operands; every activation (the epilogue does not depend on the layout)
@pytest.mark.parametrize("ta,tb,act", [(False, False, None), (False, True, None), (True, False, None), (True, True, None),
                                       (False, False, "relu"), (False, False, "gelu_erf"), (False, False, "sigmoid")])
def test_edges(gc, dev, tile, M, N, K, ta, tb, act):
    assert _tile(gc, M, N, K, tb) == tile
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    pad = 5  # no row but the first is 16-byte aligned
    A = _strided(K, M, dev, g, pad) if ta else _strided(M, K, dev, g, pad)
    B = _strided(N, K, dev, g, pad) if tb else _strided(K, N, dev, g, pad)
    bias = torch.randn(N, device=dev, generator=g)
    full = torch.full((M + 2, N + 3), 7.0, device=dev)
    _call(gc, A, B, full[:M, :N], bias, act, ta, tb)
    a, b = (A.t() if ta else A).double(), (B.t() if tb else B).double()
    ref, mag = a @ b + bias.double(), a.abs() @ b.abs() + bias.double().abs()
    # K + 1 additions of exact products, each rounded once, in any order; no activation here has a slope above 1.13, and its
    # own value is good to a few units in the last place of its range
    tol = 1.13 * (K + 1) * 2.0 ** -24 * mag + (0.0 if act is None else 4e-6)
    f = {None: lambda x: x, "relu": torch.relu, "sigmoid": torch.sigmoid, "gelu_erf": torch.nn.functional.gelu}[act]
    assert ((full[:M, :N].double() - f(ref)).abs() <= tol).all()
    assert (full[M:] == 7.0).all() and (full[:, N:] == 7.0).all()


@pytest.mark.parametrize("tile,M,N,K", [s for i, s in enumerate(SIZES) if s[0] not in [t[0] for t in SIZES[:i]]])
def test_special_values(gc, dev, tile, M, N, K):
    """An infinity, a NaN and denormals reach the results of their own row or column and no other."""
    g = torch.Generator(device=dev).manual_seed(K)
    A, B = torch.randn(M, K, device=dev, generator=g), torch.randn(K, N, device=dev, generator=g).abs() + 0.5
    A[1, K - 1], A[M - 1, 0], B[K - 1, N - 1] = float("inf"), float("-inf"), NAN
    A[3], A[4] = 1e-39, 1e-20  # a row of denormals; a row whose products with column 2 are denormal
    B[:, 2] = 1e-20
    out = torch.empty(M, N, device=dev)
    _call(gc, A, B, out, torch.zeros(N, device=dev), None, False, False)
    assert out[:, N - 1].isnan().all() and not out[:, :N - 1].isnan().any()
    assert (out[1, :N - 1] == float("inf")).all() and (out[M - 1, :N - 1] == float("-inf")).all()
    rows = [r for r in range(M) if r not in (1, M - 1)]
    a, b = A[rows].double(), B[:, :N - 1].double()
    # a denormal product is rounded to a multiple of 2^-149, by at most half of it
    tol = (K + 1) * (2.0 ** -24 * (a.abs() @ b.abs()) + 2.0 ** -149)
    assert ((out[rows, :N - 1].double() - a @ b).abs() <= tol).all()
    assert (out[4, 2] > 0) and (out[3, :2] > 0).all()


def test_batch_of_large_tiles_has_the_bits_of_its_matrices(gc, dev):
    nb, M, N, K = 12, 900, 1000, 131  # one matrix takes 64 x 64 tiles, twelve of them 128 x 128
    assert _tile(gc, M, N, K) == 64
    g = torch.Generator(device=dev).manual_seed(5)
    A, B = torch.randn(nb, M, K, device=dev, generator=g), torch.randn(nb, K, N, device=dev, generator=g)
    assert torch.equal(gc.gemm_batched(A, B), torch.stack([gc.gemm_f32(A[i], B[i]) for i in range(nb)]))


@pytest.mark.parametrize("nb,M,N,K", [(300, 40, 36, 31), (20, 300, 290, 32)])
def test_batch_on_the_vector_kernel(gc, dev, nb, M, N, K):
    assert _tile(gc, M, N, K) == "vector"
    g = torch.Generator(device=dev).manual_seed(6)
    A, B = torch.randn(nb, M, K, device=dev, generator=g), torch.randn(nb, K, N, device=dev, generator=g)
    assert torch.equal(gc.gemm_batched(A, B), torch.stack([gc.gemm_f32(A[i], B[i]) for i in range(nb)]))
