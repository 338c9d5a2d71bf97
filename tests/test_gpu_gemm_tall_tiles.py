"""Tiles of 192 and 256 rows by 128 columns: whole and cut, K in whole groups and with an incomplete one, one pass and K slices,
both layouts of the weights and 8-bit operands, against exact sums and against the 128 x 128 tile by name."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# rows of the tile, M, N, K, slices
SHAPES = [(192, 1237, 4096, 1376, 1), (192, 576, 8200, 520, 1), (192, 305, 11008, 4096, 1), (192, 305, 4096, 11008, 4),
          (256, 483, 11008, 4096, 1), (256, 512, 10888, 2056, 1), (256, 1000, 4096, 11008, 2)]


def _ints(shape, dev, g, dt, lo=-2, hi=3):
    return torch.randint(lo, hi, shape, device=dev, generator=g, dtype=torch.int32).to(dt)


@pytest.mark.parametrize("rows,M,N,K,slices", SHAPES)
@pytest.mark.parametrize("trans_b", [False, True])
def test_bf16_exact_on_integers(gc, dev, rows, M, N, K, slices, trans_b):
    c = gc.tile_config(M, N, K, trans_b=trans_b, out_dtype=gc.F32)[0]
    assert (c.bm, c.bn, c.split_k) == (rows, 128, slices)
    g = torch.Generator(device=dev).manual_seed(M)
    A, W = _ints((M, K), dev, g, torch.bfloat16), _ints((K, N), dev, g, torch.bfloat16)
    B = W.t().contiguous() if trans_b else W
    guard = torch.full((M + 2, N), 7.0, device=dev)
    (gc.gemm_bf16_nt if trans_b else gc.gemm_bf16)(A, B, out_dtype=gc.F32, out=guard[1:M + 1])
    assert torch.equal(guard[1:M + 1], A.float() @ W.float())
    assert (guard[0] == 7.0).all() and (guard[M + 1] == 7.0).all()


@pytest.mark.parametrize("rows,M,N,K", [(192, 1237, 4096, 1376), (256, 483, 11008, 2056)])
def test_the_bits_of_the_128_row_tile(gc, dev, rows, M, N, K):
    """Same products in the same order, same epilogue (bias, GELU, bf16 rounding points)."""
    import ctypes as C
    assert gc.tile_config(M, N, K)[0].bm == rows
    g = torch.Generator(device=dev).manual_seed(N)
    A, B = torch.randn(M, K, device=dev, generator=g).bfloat16(), (torch.randn(K, N, device=dev, generator=g) * 0.05).bfloat16()
    bias = torch.randn(N, device=dev, generator=g).bfloat16()
    out, named = gc.gemm_bf16(A, B, bias, "gelu_erf"), torch.empty(M, N, device=dev, dtype=torch.bfloat16)
    cfg = (C.c_int64 * 9)(1, 1, 1, 128, 128, 64, 64, 64, 32)
    gc.check(gc.lib().gcmi_gemm_bf16_ws(A.data_ptr(), B.data_ptr(), named.data_ptr(), 1, M, N, K, K, N, N, 0, 0, 0, 0, bias.data_ptr(),
                                        gc.BF16, gc.ACT["gelu_erf"], None, 0, gc.BF16, gc.BF16, None, 0, cfg,
                                        C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    assert torch.equal(out, named)


@pytest.mark.parametrize("rows,M,N,K", [(192, 1153, 4448, 1088), (192, 1255, 4288, 2560), (256, 1001, 8192, 4080)])
def test_int8_exact(gc, dev, rows, M, N, K):
    c = gc.tile_config(M, N, K, a_dtype=gc.U8, out_dtype=gc.S32)[0]
    assert (c.bm, c.bn) == (rows, 128)
    g = torch.Generator(device=dev).manual_seed(K)
    A, W = _ints((M, K), dev, g, torch.uint8, 0, 256), _ints((K, N), dev, g, torch.int8, -128, 128)
    out = gc.gemm_int8(A, W, gc.colsum_s8(W), 0, None, None, None, gc.S32)
    assert torch.equal(out.double(), A.double() @ W.double())
