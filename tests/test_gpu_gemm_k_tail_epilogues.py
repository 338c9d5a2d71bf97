"""K tails of the tile GEMMs behind an epilogue, in batches and in K slices (integers: every sum is exact)."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu


def _ints(shape, lo, hi, dev, g, dtype):
    return torch.randint(lo, hi, shape, device=dev, generator=g, dtype=torch.int32).to(dtype)


def _ws(gc, A, B, out, nb, M, N, K, sa, sb, sc, trans_b, bias, act, residual, ws, lda, ldb):
    rc = gc.lib().gcmi_gemm_bf16_ws(A.data_ptr(), B.data_ptr(), out.data_ptr(), nb, M, N, K, lda, ldb, N, sa, sb, sc, int(trans_b),
                                    None if bias is None else bias.data_ptr(), gc.F32, gc.ACT[act],
                                    None if residual is None else residual.data_ptr(), N, gc.F32, gc.F32,
                                    None if ws is None else ws.data_ptr(), 0 if ws is None else ws.numel(), None,
                                    C.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, gc.lib().gcmi_last_error().decode()


@pytest.mark.parametrize("nb,M,N,K", [(3, 300, 264, 136), (2, 40, 2048, 1376), (5, 256, 256, 72), (2, 2100, 4360, 200)])
@pytest.mark.parametrize("trans_b", [False, True])
def test_batches(gc, dev, nb, M, N, K, trans_b):
    """Bias, ReLU and an f32 residual behind each batch; NaN behind every batch's K."""
    g = torch.Generator(device=dev).manual_seed(M + K)
    A = torch.full((nb, M, K + 8), float("nan"), device=dev, dtype=torch.bfloat16)
    B = torch.full((nb, N, K + 8) if trans_b else (nb, K + 8, N), float("nan"), device=dev, dtype=torch.bfloat16)
    A[:, :, :K] = _ints((nb, M, K), -2, 3, dev, g, torch.bfloat16)
    Bk = B[:, :, :K] if trans_b else B[:, :K]
    Bk.copy_(_ints(tuple(Bk.shape), -2, 3, dev, g, torch.bfloat16))
    bias, res = _ints((N,), -9, 10, dev, g, torch.float32), _ints((nb, M, N), -9, 10, dev, g, torch.float32)
    out = torch.empty(nb, M, N, device=dev)
    _ws(gc, A, B, out, nb, M, N, K, M * (K + 8), B[0].numel(), M * N, trans_b, bias, "relu", res, None, K + 8, B.shape[2])
    for i in range(nb):
        x = A[i, :, :K].double() @ (Bk[i].t() if trans_b else Bk[i]).double()
        assert torch.equal(out[i].double(), torch.relu(x + bias.double()) + res[i].double()), i


@pytest.mark.parametrize("M,N,K", [(129, 1024, 8840), (260, 264, 1048), (32, 1096, 10248)])
@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("slices", [True, False])
def test_slices(gc, dev, M, N, K, trans_b, slices):
    """With a workspace K is sliced (the epilogue is the second pass's), without one it is not; the same result."""
    n = gc.lib().gcmi_gemm_bf16_workspace_bytes(M, N, K, int(trans_b))
    assert n > 0
    g = torch.Generator(device=dev).manual_seed(K)
    A = _ints((M, K), -2, 3, dev, g, torch.bfloat16)
    B = _ints((N, K) if trans_b else (K, N), -2, 3, dev, g, torch.bfloat16)
    bias, res = _ints((N,), -9, 10, dev, g, torch.float32), _ints((M, N), -9, 10, dev, g, torch.float32)
    out = torch.empty(M, N, device=dev)
    ws = torch.full((n,), 255, dtype=torch.uint8, device=dev) if slices else None
    _ws(gc, A, B, out, 1, M, N, K, 0, 0, 0, trans_b, bias, "relu", res, ws, K, B.shape[1])
    x = A.double() @ (B.t() if trans_b else B).double()
    assert torch.equal(out.double(), torch.relu(x + bias.double()) + res.double())


@pytest.mark.parametrize("M,N,K", [(300, 272, 80), (2048, 8208, 240), (40, 528, 1072)])
@pytest.mark.parametrize("a_dtype", [torch.uint8, torch.int8])
def test_int8_epilogue(gc, dev, M, N, K, a_dtype):
    """Zero point, scales of powers of two, bias and ReLU; bytes behind K that would count are there."""
    g = torch.Generator(device=dev).manual_seed(K)
    A = torch.full((M, K + 16), 77, device=dev, dtype=a_dtype)
    A[:, :K] = _ints((M, K), 0 if a_dtype is torch.uint8 else -128, 256 if a_dtype is torch.uint8 else 128, dev, g, a_dtype)
    W = torch.full((K + 16, N), 55, device=dev, dtype=torch.int8)
    W[:K] = _ints((K, N), -128, 128, dev, g, torch.int8)
    scale = 2.0 ** torch.randint(-3, 2, (N,), device=dev, generator=g).float()
    bias = _ints((N,), -9, 10, dev, g, torch.float32)
    out = gc.gemm_int8(A[:, :K], W[:K], gc.colsum_s8(W[:K]), 7, scale, bias, "relu", gc.F32)
    x = (A[:, :K].double() - 7) @ W[:K].double()  # below 2^24 in these sizes: exact in f32
    assert x.abs().max() < 2 ** 24
    assert torch.equal(out.double(), torch.relu(x * scale.double() + bias.double()))
