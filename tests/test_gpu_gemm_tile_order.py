"""Tiles in pairs on a compute unit, dealt to the XCDs in runs or in the hardware's order: every tile is computed, once.  Exact
whole numbers; either side of 20 columns of tiles, of a K of 1024 bytes and of a number of tiles that 8 divides."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(2056, 2208, 1104), (1693, 2384, 1120), (1693, 2384, 1008), (3309, 1824, 2160), (1600, 2576, 1040),
                                   (1600, 2704, 1040), (4200, 1008, 1024)])
def test_8_bit(gc, dev, M, N, K):
    g = torch.Generator(device=dev).manual_seed(M)
    A = torch.randint(0, 256, (M, K), device=dev, generator=g, dtype=torch.int32).to(torch.uint8)
    W = torch.randint(-127, 128, (K, N), device=dev, generator=g, dtype=torch.int32).to(torch.int8)
    c, _ = gc.tile_config(M, N, K, a_dtype=gc.U8, out_dtype=gc.S32)
    assert (c.kernel, c.bm, c.bn, c.stages) == (5, 128, 128, 4) and c.workgroups > 256
    full = torch.full((M + 1, N), 7, device=dev, dtype=torch.int32)
    gc.gemm_int8(A, W, colsum=gc.colsum_s8(W), out=full[:M])
    assert torch.equal(full[:M].double(), A.double() @ W.double()) and (full[M] == 7).all()


@pytest.mark.parametrize("M,N,K", [(2834, 2400, 832), (2498, 2544, 512), (2834, 2400, 504)])
@pytest.mark.parametrize("nt", [False, True])
def test_bf16(gc, dev, M, N, K, nt):
    g = torch.Generator(device=dev).manual_seed(M)
    A = torch.randint(-3, 4, (M, K), device=dev, generator=g).bfloat16()
    B = torch.randint(-3, 4, (N, K) if nt else (K, N), device=dev, generator=g).bfloat16()
    c, _ = gc.tile_config(M, N, K, trans_b=nt, out_dtype=gc.F32)
    assert (c.kernel, c.bm, c.bn) == (5, 128, 128) and c.workgroups > 256
    out = (gc.gemm_bf16_nt if nt else gc.gemm_bf16)(A, B, out_dtype=gc.F32)
    assert torch.equal(out.double(), A.double() @ (B.double().t() if nt else B.double()))
