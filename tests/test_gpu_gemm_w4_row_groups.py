"""The 4-wave kernels' epilogue passes over groups of 32 rows outside C: the last tile cut at both sides of every group, each
result the bits that the whole tile gives the same row."""
import pytest
import torch

pytestmark = pytest.mark.gpu

LARGE, SMALL = [1, 1, 1, 256, 256, 64, 128, 128, 32], [1, 1, 1, 128, 128, 64, 64, 64, 32]


@pytest.mark.parametrize("cfg,rows", [(LARGE, 256), (SMALL, 128)])
@pytest.mark.parametrize("act,out", [(None, "BF16"), ("gelu_erf", "BF16"), ("sigmoid", "F32")])
def test_bf16(gc, dev, cfg, rows, act, out):
    import ctypes as C
    g = torch.Generator(device=dev).manual_seed(rows)
    N, K, dt = 264, 1032, torch.bfloat16 if out == "BF16" else torch.float32
    A, B = (torch.randn(s, device=dev, generator=g).bfloat16() for s in ((2 * rows, K), (K, N)))
    bias = torch.randn(N, device=dev, generator=g).bfloat16()

    def run(M):
        full = torch.full((M + 1, N), 7.0, device=dev, dtype=dt)
        assert gc.tile_config(M, N, K, out_dtype=getattr(gc, out), matmul_config=cfg)[0].bm == rows
        gc.check(gc.lib().gcmi_gemm_bf16_ws(A.data_ptr(), B.data_ptr(), full.data_ptr(), 1, M, N, K, K, N, N, 0, 0, 0, 0, bias.data_ptr(), gc.BF16,
                                            gc.ACT[act], None, 0, gc.BF16, getattr(gc, out), None, 0, (C.c_int64 * 9)(*cfg),
                                            C.c_void_p(torch.cuda.current_stream().cuda_stream)))
        assert (full[M] == 7.0).all()
        return full[:M]

    want = run(2 * rows)
    for m in range(0, rows, 32):
        for M in (m, m + 1, m + 31):
            if M > (0 if rows == 256 else 31):
                assert torch.equal(run(M), want[:M]), M
                assert torch.equal(run(rows + M), want[:rows + M]), rows + M


def test_int8(gc, dev):
    g = torch.Generator(device=dev).manual_seed(8)
    N, K = 272, 528
    A = torch.randint(0, 256, (512, K), device=dev, generator=g, dtype=torch.int32).to(torch.uint8)
    W = torch.randint(-128, 128, (K, N), device=dev, generator=g, dtype=torch.int32).to(torch.int8)
    want = (A.cpu().int() @ W.cpu().int()).to(dev)
    for M in (1, 31, 32, 33, 64, 65, 127, 128, 129, 160, 161, 255, 257, 288, 289, 511):
        out = torch.full((M + 1, N), 7, device=dev, dtype=torch.int32)
        gc.gemm_int8(A[:M], W, gc.colsum_s8(W), out=out[:M], matmul_config=LARGE)
        assert torch.equal(out[:M], want[:M]) and (out[M] == 7).all(), M
