"""Calls that are K-sliced only because of tiles of more than 128 rows: they ran in one pass before there were such tiles, so stream
capture and the static scratch array do not refuse them; the others with a K of whole groups are refused as they were."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu


def _plain(gc, A, B, out, trans_b, residual=None):
    (M, K), N, s = A.shape, out.shape[1], C.c_void_p(torch.cuda.current_stream().cuda_stream)
    ops = (A.data_ptr(), B.data_ptr(), out.data_ptr())
    if residual is not None:
        return gc.lib().gcmi_gemm_bf16_residual(*ops, 1, M, N, K, K, B.shape[1], N, 0, 0, 0, trans_b, None, gc.BF16, 0, residual.data_ptr(),
                                                N, gc.F32, gc.F32, s)
    f = gc.lib().gcmi_gemm_bf16_nt if trans_b else gc.lib().gcmi_gemm_bf16
    return f(*ops, M, N, K, K, B.shape[1], N, None, gc.BF16, 0, gc.F32, s)


@pytest.mark.parametrize("M,N,K", [(1000, 4096, 11008), (556, 3392, 6016), (1000, 4096, 12288)])
@pytest.mark.parametrize("trans_b", [0, 1])
@pytest.mark.parametrize("with_residual", [False, True])
def test_captured_in_one_pass(gc, dev, M, N, K, trans_b, with_residual):
    assert gc.lib().gcmi_gemm_bf16_workspace_bytes(M, N, K, trans_b) > 0  # eager calls are sliced
    g = torch.Generator(device=dev).manual_seed(K)
    ints = lambda *s: torch.randint(-2, 3, s, device=dev, generator=g, dtype=torch.int32).to(torch.bfloat16)  # noqa: E731
    A, B = ints(M, K), ints(*((N, K) if trans_b else (K, N)))  # integers: exact in any order
    res = torch.randint(-9, 10, (M, N), device=dev, generator=g).float() if with_residual else None
    want = A.float() @ (B.t() if trans_b else B).float()
    out, other = torch.zeros(M, N, device=dev), torch.zeros(M, N, device=dev)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        graph = torch.cuda.CUDAGraph()
        graph.capture_begin()
        rc = _plain(gc, A, B, out, trans_b, res)
        graph.capture_end()
    assert rc == 0, gc.lib().gcmi_last_error().decode()
    for _ in range(3):  # with eager calls between the replays, through the workspace the graph must not name
        out.zero_()
        assert _plain(gc, -A, B, other, trans_b) == 0
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(other, -want) and torch.equal(out, want if res is None else want + res)


@pytest.mark.parametrize("trans_b", [0, 1])
def test_more_partial_sums_than_the_static_array_holds(gc, dev, trans_b):
    M, N, K = 1000, 4096, 12288
    assert gc.lib().gcmi_gemm_bf16_workspace_bytes(M, N, K, trans_b) > gc.lib().gcmi_noalloc_scratch_bytes()
    g = torch.Generator(device=dev).manual_seed(1)
    ints = lambda *s: torch.randint(-2, 3, s, device=dev, generator=g, dtype=torch.int32).to(torch.bfloat16)  # noqa: E731
    A, B, out = ints(M, K), ints(*((N, K) if trans_b else (K, N))), torch.zeros(M, N, device=dev)
    rc = gc.lib().gcmi_gemm_bf16_noalloc(A.data_ptr(), B.data_ptr(), out.data_ptr(), M, N, K, K, B.shape[1], N, trans_b, None, gc.BF16,
                                         0, gc.F32, C.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, gc.lib().gcmi_last_error().decode()
    assert torch.equal(out, A.float() @ (B.t() if trans_b else B).float())


@pytest.mark.parametrize("M,N,K", [(192, 1024, 4096), (512, 4096, 16384), (1024, 1024, 8192)])
def test_slices_of_128_and_256_row_tiles_are_refused_as_before(gc, dev, M, N, K):
    assert gc.lib().gcmi_gemm_bf16_workspace_bytes(M, N, K, 0) > 0
    A, B, out = (torch.zeros(s, device=dev, dtype=torch.bfloat16) for s in ((M, K), (K, N), (M, N)))
    side, keep = torch.cuda.Stream(), torch.zeros(1, device=dev)
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        graph = torch.cuda.CUDAGraph()
        graph.capture_begin()
        keep.add_(1)
        rc = gc.lib().gcmi_gemm_bf16(A.data_ptr(), B.data_ptr(), out.data_ptr(), M, N, K, K, N, N, None, gc.BF16, 0, gc.BF16,
                                     C.c_void_p(side.cuda_stream))
        graph.capture_end()
    assert rc == 2 and "captured" in gc.lib().gcmi_last_error().decode()
