"""K that is no whole number of ring groups (128 bf16 / 256 bytes): the tile kernels fill the ring with the incomplete
group first.  Small integers, so that every product and sum is exact and a single wrong or doubled k shows."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu

# K left over: one 16-byte chunk, one off a k-block of 64 bytes, whole k-blocks, one off a whole group; no whole group at
# all, one, several
BF16_K = [8, 24, 32, 40, 96, 120, 136, 224, 248, 1376]
INT8_K = [16, 48, 64, 80, 192, 240, 272, 448, 496, 1072]


def _ints(shape, lo, hi, dev, g, dtype):
    return torch.randint(lo, hi, shape, device=dev, generator=g, dtype=torch.int32).to(dtype)


def _config(tile):  # MatmulConfig: workgroup tile and the waves' tiles that go with it
    return [1, 1, 1, tile, tile, 64, tile // 2, tile // 2, 32]


@pytest.mark.parametrize("K", BF16_K)
@pytest.mark.parametrize("tile", [256, 128])
@pytest.mark.parametrize("trans_b", [False, True])
def test_bf16_k_tail(gc, dev, K, tile, trans_b):
    M, N, cfg = 300, 264, _config(tile)
    assert gc.tile_config(M, N, K, trans_b=trans_b, matmul_config=cfg)[0].kernel == (2 if tile == 256 else 5)
    g = torch.Generator(device=dev).manual_seed(K)
    # what lies behind K in memory is NaN: rows of the operands are longer than K
    A = torch.full((M, K + 64), float("nan"), device=dev, dtype=torch.bfloat16)
    B = torch.full((N, K + 64) if trans_b else (K + 64, N), float("nan"), device=dev, dtype=torch.bfloat16)
    A[:, :K] = _ints((M, K), -2, 3, dev, g, torch.bfloat16)
    Bk = B[:, :K] if trans_b else B[:K]
    Bk.copy_(_ints(tuple(Bk.shape), -2, 3, dev, g, torch.bfloat16))
    out = torch.empty(M, N, device=dev)
    rc = gc.lib().gcmi_gemm_bf16_ws(A.data_ptr(), B.data_ptr(), out.data_ptr(), 1, M, N, K, A.stride(0), B.stride(0), N, 0, 0, 0,
                                    int(trans_b), None, gc.BF16, gc.ACT[None], None, N, gc.BF16, gc.F32, None, 0,
                                    (C.c_int64 * 9)(*cfg), C.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, gc.lib().gcmi_last_error().decode()
    ref = A[:, :K].double() @ (Bk.t() if trans_b else Bk).double()
    assert torch.equal(out.double(), ref)


@pytest.mark.parametrize("M,N,K", [(129, 1024, 8840), (512, 512, 8168), (260, 264, 1048)])
@pytest.mark.parametrize("trans_b", [False, True])
def test_bf16_k_tail_in_slices(gc, dev, M, N, K, trans_b):
    c = gc.tile_config(M, N, K, trans_b=trans_b)[0]
    assert c.kernel == 3 and c.bm == 128 and c.split_k > 1
    g = torch.Generator(device=dev).manual_seed(K)
    A = _ints((M, K), -2, 3, dev, g, torch.bfloat16)
    B = _ints((N, K) if trans_b else (K, N), -2, 3, dev, g, torch.bfloat16)
    out = (gc.gemm_bf16_nt if trans_b else gc.gemm_bf16)(A, B, out_dtype=gc.F32)
    assert torch.equal(out.double(), A.double() @ (B.t() if trans_b else B).double())


@pytest.mark.parametrize("K", INT8_K)
@pytest.mark.parametrize("M,N", [(300, 272), (2048, 8208)])  # small tiles, large tiles
@pytest.mark.parametrize("a_dtype", [torch.uint8, torch.int8])
def test_int8_k_tail(gc, dev, K, M, N, a_dtype):
    g = torch.Generator(device=dev).manual_seed(K)
    A = _ints((M, K), 0 if a_dtype is torch.uint8 else -128, 256 if a_dtype is torch.uint8 else 128, dev, g, a_dtype)
    W = _ints((K, N), -128, 128, dev, g, torch.int8)
    c = gc.tile_config(M, N, K, a_dtype=gc.U8 if a_dtype is torch.uint8 else gc.S8, out_dtype=gc.F32)[0]
    assert c.kernel == (5 if M == 300 else 2)
    out = gc.gemm_int8(A, W, gc.colsum_s8(W), 0, None, None, None, gc.F32)
    assert torch.equal(out.double(), A.double() @ W.double())
