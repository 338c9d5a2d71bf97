"""Tiles of 192 and 256 rows: padded rows, NaN behind K, bias, residual, batches and the epilogues of 8-bit operands (integers: every
sum is exact)."""
import ctypes as C

import pytest
import torch

from test_gpu_gemm_tall_without_workspace import _captured_grids

pytestmark = pytest.mark.gpu


def _ints(shape, dev, g, dt, lo=-2, hi=3):
    return torch.randint(lo, hi, shape, device=dev, generator=g, dtype=torch.int32).to(dt)


def _padded(t, fill):
    """The same values in rows that are 16 elements longer, one row more; `fill` there."""
    full = torch.full((*t.shape[:-2], t.shape[-2] + 1, t.shape[-1] + 16), fill, device=t.device, dtype=t.dtype)
    full[..., :-1, :-16] = t
    return full[..., :-1, :-16]


@pytest.mark.parametrize("rows,M,N,K,nb", [(192, 1237, 4096, 1376, 1), (256, 483, 11008, 2056, 1), (192, 1201, 4104, 1288, 1), (256, 1000, 4096, 11016, 1),
                                           (192, 600, 4096, 1384, 2), (192, 385, 2568, 1288, 4)])
@pytest.mark.parametrize("trans_b", [False, True])
def test_bf16_padded_with_epilogue(gc, dev, rows, M, N, K, nb, trans_b):
    """Bias, ReLU and an f32 residual; one matrix (K slices too) and batches."""
    g = torch.Generator(device=dev).manual_seed(M + N)
    A, W = _ints((nb, M, K), dev, g, torch.bfloat16), _ints((nb, K, N), dev, g, torch.bfloat16)
    Ap, Bp = _padded(A, float("nan")), _padded(W.transpose(1, 2) if trans_b else W, float("nan"))
    bias, res = _ints((N,), dev, g, torch.float32, -9, 10), _padded(_ints((nb, M, N), dev, g, torch.float32, -9, 10), float("nan"))
    guard = torch.full((nb, M + 1, N + 16), 7.0, device=dev)
    n = gc.lib().gcmi_gemm_bf16_workspace_bytes(M, N, K, int(trans_b)) if nb == 1 else 0
    ws = torch.full((max(16, n),), 255, dtype=torch.uint8, device=dev)
    if nb == 1:
        c = gc.tile_config(M, N, K, trans_b=trans_b, out_dtype=gc.F32)[0]
        assert (c.bm, c.bn) == (rows, 128)

    def call(stream):
        gc.check(gc.lib().gcmi_gemm_bf16_ws(Ap.data_ptr(), Bp.data_ptr(), guard.data_ptr(), nb, M, N, K, K + 16, Bp.stride(1), N + 16, Ap.stride(0),
                                            Bp.stride(0), guard.stride(0), int(trans_b), bias.data_ptr(), gc.F32, gc.ACT["relu"], res.data_ptr(),
                                            N + 16, gc.F32, gc.F32, ws.data_ptr(), n, None, stream))

    slices = n // (4 * M * N) if n else 1
    assert _captured_grids(call)[0] == -(-M // rows) * -(-N // 128) * nb * slices
    call(C.c_void_p(torch.cuda.current_stream().cuda_stream))
    for i in range(nb):
        want = torch.relu(A[i].float() @ W[i].float() + bias) + res[i]
        assert torch.equal(guard[i, :M, :N], want), i
    assert (guard[:, M] == 7.0).all() and (guard[:, :, N:] == 7.0).all()


@pytest.mark.parametrize("rows,M,N,K", [(192, 1153, 4448, 1088), (192, 1255, 4288, 2560), (256, 1001, 8192, 4080)])
@pytest.mark.parametrize("a_dtype", [torch.uint8, torch.int8])
def test_int8_epilogues(gc, dev, rows, M, N, K, a_dtype):
    """Every activation and output type: the bits of the 128 x 128 tile by name, whose epilogue it is; bytes behind K that would count."""
    u8 = a_dtype is torch.uint8
    assert gc.tile_config(M, N, K, a_dtype=gc.U8 if u8 else gc.S8)[0].bm == rows
    g = torch.Generator(device=dev).manual_seed(K)
    A = _padded(_ints((M, K), dev, g, a_dtype, 0 if u8 else -128, 256 if u8 else 128), 77)
    W = _padded(_ints((K, N), dev, g, torch.int8, -128, 128), 55)
    cs, zp = gc.colsum_s8(W), 131 if u8 else 3
    scale, bias = (torch.rand(N, device=dev, generator=g) + 0.5) / (60.0 * K ** 0.5), torch.randn(N, device=dev, generator=g)
    named = [1, 1, 1, 128, 128, 64, 64, 64, 32]
    pre = ((A.double() - zp) @ W.double()) * scale.double() + bias.double()
    for act in (None, "relu", "sigmoid", "gelu_erf", "gelu_tanh"):
        for odt in (gc.BF16, gc.F32):
            got = gc.gemm_int8(A, W, cs, zp, scale, bias, act, odt)
            assert torch.equal(got, gc.gemm_int8(A, W, cs, zp, scale, bias, act, odt, matmul_config=named)), (act, odt)
    # exact accumulators: a conversion, a product and a sum in f32
    y = gc.gemm_int8(A, W, cs, zp, scale, bias, "relu", gc.F32)
    assert ((y.double() - torch.relu(pre)).abs() <= 1.13 * 2.0 ** -22 * (pre.abs() + 2 * bias.double().abs()) + 2e-6).all()
    raw = torch.full((M + 2, N), 7, device=dev, dtype=torch.int32)
    gc.gemm_int8(A, W, cs, 0, None, None, None, gc.S32, out=raw[1:M + 1])
    assert torch.equal(raw[1:M + 1].double(), A.double() @ W.double()) and (raw[0] == 7).all() and (raw[M + 1] == 7).all()
