"""Calls that taller tiles bring to K slices, with less workspace than those want: what runs is the best of what is left, not the
tall tile that was chosen together with the slices.  The launched grids are read from a captured graph."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu


class _Dim3(C.Structure):
    _fields_ = [(n, C.c_uint32) for n in "xyz"]


class _KernelNode(C.Structure):  # hipKernelNodeParams
    _fields_ = [("block", _Dim3), ("extra", C.c_void_p), ("func", C.c_void_p), ("grid", _Dim3), ("params", C.c_void_p), ("shared", C.c_uint32)]


def _hip():
    """The runtime that this process has loaded."""
    with open("/proc/self/maps") as maps:
        return C.CDLL(next(line.split()[-1] for line in maps if "libamdhip64" in line))


def _captured_grids(call):
    """Workgroups of each kernel that `call(stream)` launches (none of them runs)."""
    hip, side = _hip(), torch.cuda.Stream()
    stream, graph = C.c_void_p(side.cuda_stream), C.c_void_p()
    torch.cuda.synchronize()
    assert hip.hipStreamBeginCapture(stream, 2) == 0  # relaxed
    call(stream)
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
    n = C.c_size_t(0)
    assert hip.hipGraphGetNodes(graph, None, C.byref(n)) == 0
    nodes = (C.c_void_p * max(1, n.value))()
    assert hip.hipGraphGetNodes(graph, nodes, C.byref(n)) == 0
    grids = []
    for node in nodes[:n.value]:
        k = _KernelNode()
        assert hip.hipGraphKernelNodeGetParams(C.c_void_p(node), C.byref(k)) == 0
        grids.append(k.grid.x * k.grid.y * k.grid.z)
    assert hip.hipGraphDestroy(graph) == 0
    return grids


# M, N, K, slices wanted, share of the workspace, slices cut then, workgroups of the GEMM kernel
@pytest.mark.parametrize("M,N,K,wanted,share,slices,blocks", [
    (1000, 4096, 11008, 2, 0.0, 1, 256), (1000, 4096, 11008, 2, 0.5, 1, 256), (305, 4096, 11008, 4, 0.0, 1, 96),
    (305, 4096, 11008, 4, 0.5, 2, 192), (305, 4096, 11000, 4, 0.0, 1, 96), (556, 3392, 6016, 3, 0.0, 1, 135)])
@pytest.mark.parametrize("trans_b", [0, 1])
def test_less_workspace_than_tall_slices_want(gc, dev, M, N, K, wanted, share, slices, blocks, trans_b):
    want = gc.lib().gcmi_gemm_bf16_workspace_bytes(M, N, K, trans_b)
    c = gc.tile_config(M, N, K, trans_b=bool(trans_b))[0]
    assert c.split_k == wanted and c.bm in (192, 256) and c.bn == 128 and want == wanted * M * N * 4
    g = torch.Generator(device=dev).manual_seed(M)
    ints = lambda *s: torch.randint(-2, 3, s, device=dev, generator=g, dtype=torch.int32).to(torch.bfloat16)  # noqa: E731
    A, B, out = ints(M, K), ints(*((N, K) if trans_b else (K, N))), torch.zeros(M, N, device=dev)
    ws = torch.empty(max(16, want), dtype=torch.uint8, device=dev)

    def call(stream):
        gc.check(gc.lib().gcmi_gemm_bf16_ws(A.data_ptr(), B.data_ptr(), out.data_ptr(), 1, M, N, K, K, B.shape[1], N, 0, 0, 0, trans_b,
                                            None, gc.BF16, 0, None, 0, gc.BF16, gc.F32, ws.data_ptr() if share else None,
                                            int(want * share), None, stream))

    grids = _captured_grids(call)
    assert len(grids) == (2 if slices > 1 else 1) and grids[0] == blocks
    call(C.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert torch.equal(out, A.float() @ (B.t() if trans_b else B).float())  # integers: exact in any order
