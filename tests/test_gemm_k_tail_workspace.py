"""A K that is no whole number of ring groups (128 bf16): its slices fit the static array of the entry point that
allocates nothing, and no entry point refuses it under stream capture."""
import ctypes as C

import pytest


def _status(gc, name, A, B, out, trans_b):
    import torch
    M, K = A.shape
    N = out.shape[1]
    s = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    ops = (A.data_ptr(), B.data_ptr(), out.data_ptr(), M, N, K, K, B.shape[1], N)
    if name == "noalloc":
        return gc.lib().gcmi_gemm_bf16_noalloc(*ops, int(trans_b), None, gc.BF16, 0, gc.F32, s)
    return (gc.lib().gcmi_gemm_bf16_nt if trans_b else gc.lib().gcmi_gemm_bf16)(*ops, None, gc.BF16, 0, gc.F32, s)


# at most two workgroups per compute unit and 128 x 128 f32 sums of each
@pytest.mark.parametrize("M,N,K", [(512, 4096, 16376), (300, 4000, 16000 + 8), (1024, 1024, 32760), (32, 1096, 10248),
                                   (192, 4096, 4072)])
@pytest.mark.parametrize("trans_b", [0, 1])
def test_slices_fit_the_static_array(gc, M, N, K, trans_b):
    n = gc.lib().gcmi_gemm_bf16_workspace_bytes(M, N, K, trans_b)
    assert 0 < n <= 32 << 20


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(32, 4096, 1376), (32, 1096, 10248), (64, 4096, 4072), (192, 4096, 4072), (512, 4096, 16376)])
@pytest.mark.parametrize("trans_b", [False, True])
def test_k_tail_under_capture_and_without_allocation(gc, dev, M, N, K, trans_b):
    import torch
    g = torch.Generator(device=dev).manual_seed(K)
    ints = lambda *s: torch.randint(-2, 3, s, device=dev, generator=g).to(torch.bfloat16)  # noqa: E731
    A, B = ints(M, K), ints(*((N, K) if trans_b else (K, N)))  # integers: sums are exact in any order
    want = (A.float() @ (B.t() if trans_b else B).float())
    out = torch.zeros(M, N, device=dev)
    assert _status(gc, "noalloc", A, B, out, trans_b) == 0, gc.lib().gcmi_last_error().decode()
    assert torch.equal(out, want)
    assert _status(gc, "plain", A, B, out.zero_(), trans_b) == 0, gc.lib().gcmi_last_error().decode()
    assert torch.equal(out, want)
    out.zero_()
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        graph = torch.cuda.CUDAGraph()
        graph.capture_begin()
        rc = _status(gc, "plain", A, B, out, trans_b)
        graph.capture_end()
    assert rc == 0, gc.lib().gcmi_last_error().decode()
    for _ in range(3):  # with eager calls between the replays, through the workspace the graph must not name
        out.zero_()
        other = torch.zeros_like(out)
        assert _status(gc, "plain", -A, B, other, trans_b) == 0
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(other, -want)


@pytest.mark.parametrize("M,K,kernel", [(16, 16, 0), (31, 64, 0), (31, 72, 2), (31, 136, 2), (16, 128, 2)])
@pytest.mark.parametrize("trans_b", [False, True])
def test_a_k_of_one_block_under_few_rows(gc, M, K, kernel, trans_b):
    """Where the tile kernels' set-up costs more than the bounds-checked kernel's checks."""
    assert gc.tile_config(M, 1000, K, trans_b=trans_b)[0].kernel == kernel
