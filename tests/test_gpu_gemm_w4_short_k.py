"""The 4-wave kernels at every length of K their loops branch on (one and two groups of 128, the first trips of the steady loop,
an incomplete group in front of each), both layouts of the weights, edge tiles, NaN behind K."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [(256, 260, 520, K) for K in (8, 64, 72, 128, 136, 192, 200, 256, 264, 320, 384, 392, 512, 520, 640, 648)]
CASES += [(128, 260, 520, K) for K in (256, 264, 320, 384, 392, 512, 520, 640, 648, 1032)] + [(128, 2100, 2104, K) for K in (264, 640)]
CASES += [(192, 1237, 4096, K) for K in (264, 320, 384, 392, 512, 520, 640)] + [(256128, 1000, 8192, K) for K in (1024, 1032, 1152)]


@pytest.mark.parametrize("tile,M,N,K", CASES)
@pytest.mark.parametrize("trans_b", [0, 1])
def test_exact_on_integers(gc, dev, tile, M, N, K, trans_b):
    cfg = {256: [1, 1, 1, 256, 256, 64, 128, 128, 32], 128: [1, 1, 1, 128, 128, 64, 64, 64, 32]}.get(tile)
    c = gc.tile_config(M, N, K, trans_b=bool(trans_b), out_dtype=gc.F32, matmul_config=cfg)[0]
    assert (c.kernel, c.bm, c.bn) == {256: (2, 256, 256), 128: (5, 128, 128), 192: (5, 192, 128), 256128: (5, 256, 128)}[tile]
    g = torch.Generator(device=dev).manual_seed(K)
    ints = lambda *s: torch.randint(-2, 3, s, device=dev, generator=g, dtype=torch.int32).to(torch.bfloat16)  # noqa: E731
    A = torch.full((M, K + 64), float("nan"), device=dev, dtype=torch.bfloat16)
    B = torch.full((N, K + 64) if trans_b else (K + 64, N), float("nan"), device=dev, dtype=torch.bfloat16)
    A[:, :K] = ints(M, K)
    Bk = B[:, :K] if trans_b else B[:K]
    Bk.copy_(ints(*Bk.shape))
    out = torch.full((M + 1, N), 7.0, device=dev)
    gc.check(gc.lib().gcmi_gemm_bf16_ws(A.data_ptr(), B.data_ptr(), out.data_ptr(), 1, M, N, K, K + 64, B.stride(0), N, 0, 0, 0, trans_b,
                                        None, gc.BF16, 0, None, 0, gc.BF16, gc.F32, None, 0, (C.c_int64 * 9)(*cfg) if cfg else None,
                                        C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    assert torch.equal(out[:M], A[:, :K].float() @ (Bk.t() if trans_b else Bk).float()) and (out[M] == 7.0).all()
