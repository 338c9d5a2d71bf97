"""256 x 192 tiles (waves of 128 x 96, the last 32 columns an epilogue pass of their own): exact sums with NaN behind K and guards
around C, the last tile cut at 8, 56, 72, 128 and 184 of its columns; every epilogue has the bits of the 256 x 256 tile by name."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(1001, 9608, 392), (2655, 3520, 520), (1537, 5640, 648), (1000, 10888, 1032), (1025, 8192, 1288), (769, 10936, 1024), (769, 10944, 400)]


def _run(gc, A, B, out, trans_b, cfg=None, bias=None, act=None, residual=None):
    M, N, K = out.shape[0], out.shape[1], A.shape[1]
    dt = {torch.bfloat16: gc.BF16, torch.float32: gc.F32}
    gc.check(gc.lib().gcmi_gemm_bf16_ws(A.data_ptr(), B.data_ptr(), out.data_ptr(), 1, M, N, K, A.stride(0), B.stride(0), out.stride(0), 0, 0, 0,
                                        trans_b, None if bias is None else bias.data_ptr(), gc.BF16, gc.ACT[act],
                                        None if residual is None else residual.data_ptr(), 0 if residual is None else residual.stride(0),
                                        gc.BF16 if residual is None else dt[residual.dtype], dt[out.dtype], None, 0,
                                        (C.c_int64 * 9)(*cfg) if cfg else None, C.c_void_p(torch.cuda.current_stream().cuda_stream)))


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("trans_b", [0, 1])
def test_exact_on_integers(gc, dev, M, N, K, trans_b):
    c = gc.tile_config(M, N, K, trans_b=bool(trans_b), out_dtype=gc.F32)[0]
    assert (c.kernel, c.bm, c.bn) == (5, 256, 192)
    g = torch.Generator(device=dev).manual_seed(K)
    ints = lambda *s: torch.randint(-2, 3, s, device=dev, generator=g, dtype=torch.int32).to(torch.bfloat16)  # noqa: E731
    A = torch.full((M, K + 64), float("nan"), device=dev, dtype=torch.bfloat16)
    B = torch.full((N, K + 64) if trans_b else (K + 64, N + 8), float("nan"), device=dev, dtype=torch.bfloat16)
    A[:, :K] = ints(M, K)
    Bk = B[:, :K] if trans_b else B[:K, :N]
    Bk.copy_(ints(*Bk.shape))
    out = torch.full((M + 2, N + 8), 7.0, device=dev)
    _run(gc, A[:, :K], B, out[1:M + 1, :N], trans_b)
    assert torch.equal(out[1:M + 1, :N], A[:, :K].float() @ (Bk.t() if trans_b else Bk).float())
    assert (out[0] == 7.0).all() and (out[M + 1] == 7.0).all() and (out[:, N:] == 7.0).all()


@pytest.mark.parametrize("act", [None, "relu", "gelu_erf", "gelu_tanh", "sigmoid"])
@pytest.mark.parametrize("res_dtype", [None, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_the_bits_of_the_large_tile(gc, dev, act, res_dtype, out_dtype):
    for (M, N, K), trans_b in zip(SHAPES[:4], (0, 1, 0, 1)):
        g = torch.Generator(device=dev).manual_seed(N)
        A, B = (torch.randn(s, device=dev, generator=g).bfloat16() for s in ((M, K), (N, K) if trans_b else (K, N)))
        bias = torch.randn(N, device=dev, generator=g).bfloat16()
        res = None if res_dtype is None else torch.randn(M, N, device=dev, generator=g).to(res_dtype)
        one, two = (torch.empty(M, N, device=dev, dtype=out_dtype) for _ in range(2))
        _run(gc, A, B, one, trans_b, bias=bias, act=act, residual=res)
        _run(gc, A, B, two, trans_b, [1, 1, 1, 256, 256, 64, 128, 128, 32], bias, act, res)
        assert torch.equal(one, two), (M, N, K)
