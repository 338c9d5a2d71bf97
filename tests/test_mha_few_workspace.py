"""The key ranges of attention with few queries follow from the sizes: every entry point that has the scratch memory gives
the same bits, compiled partitions (also replayed from a HIP graph) among them."""
import ctypes as C

import pytest


def test_workspace_query(gc):
    f = gc.lib().gcmi_mha_fwd_workspace_bytes_bh
    n = f(8, 1, 4096, 128, 0)
    assert n > 0 and n % ((128 + 2) * 4 * 8) == 0 and n == f(8, 1, 4096, 128, 1)  # whole ranges, with and without a mask
    assert f(256, 1, 4096, 128, 0) == 0         # one workgroup per head fills the GPU
    assert f(8, 1, 64, 128, 0) == 0             # too few keys to cut
    assert f(8, 256, 4096, 128, 0) == 0 and f(8, 256, 4096, 128, 1) == gc.lib().gcmi_mha_fwd_workspace_bytes(256, 4096, 128, 1) > 0
    assert f(0, 1, 4096, 128, 0) == f(8, 0, 4096, 128, 0) == f(8, 1, 0, 128, 0) == f(8, 1, 4096, 96, 0) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,Sq,Sk,D", [(1, 8, 1, 4096, 128), (2, 4, 5, 2001, 64), (1, 8, 100, 3000, 128)])
@pytest.mark.parametrize("masked", [False, True])
def test_entry_points_agree(gc, ga, dev, B, H, Sq, Sk, D, masked):
    import torch
    g = torch.Generator(device=dev).manual_seed(Sk)
    Q, K, V = (torch.randn(B, H, s, D, device=dev, generator=g).to(torch.bfloat16) for s in (Sq, Sk, Sk))
    mask = torch.randn(Sq, Sk, device=dev, generator=g) if masked else None
    scale = torch.full((1,), D ** -0.5, device=dev)
    n = gc.lib().gcmi_mha_fwd_workspace_bytes_bh(B * H, Sq, Sk, D, int(masked))
    assert n > 0
    want = gc.mha_fwd_bf16(Q, K, V, mask, float(scale.item()))

    def ws_call(nbytes, flags=1, shift=0):
        ws = torch.full((n + 512,), 255, dtype=torch.uint8, device=dev)
        out = torch.zeros_like(Q)
        rc = gc.lib().gcmi_mha_fwd_bf16_ws(Q.data_ptr(), K.data_ptr(), V.data_ptr(), mask.data_ptr() if masked else None, Sk,
                                           out.data_ptr(), B * H, Sq, Sk, D, float(scale.item()), flags, ws.data_ptr() + shift,
                                           nbytes, C.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0, gc.lib().gcmi_last_error().decode()
        return out, ws

    out, ws = ws_call(n)
    assert torch.equal(out, want) and (ws[n:] == 255).all()
    for args in ((n - 1,), (n, 3), (n, 1, 4)):  # too small, read-only, misaligned: taken, and left alone
        whole, ws = ws_call(*args)
        assert (ws == 255).all()
        assert (whole.double() - want.double()).norm() <= 1e-2 * want.double().norm()
    if masked:
        assert gc.mha_mask_classes(mask, Sq, Sk, D) is None
        assert torch.equal(gc.mha_fwd_bf16_classified(Q, K, V, mask, None, float(scale.item())), want)

    # a partition with the same attention: its arena holds the ranges
    comp = ga.Compiler()
    text = ga.mha_json(B, H, Sq, Sk, D, masked, "Multiply")
    st, exe = comp.compile(text)
    assert st == 0, ga.api().dnnl_graph_compiler_last_error().decode()
    got = torch.zeros_like(Q)
    ins = [(0, Q), (1, K), (2, scale)] + ([(3, mask)] if masked else []) + [(4, V)]
    assert exe.execute(ins, [(9, got)]) == 0
    assert torch.equal(got, want)
    exe.close()
    comp.close()


def _unscaled(ga, B, H, Sq, Sk, D):
    """SoftMax(Q K^T) V; no scale tensor, which execute_async would have to read back."""
    s = [B, H, Sq, Sk]
    return ga._graph([
        {"kind": "MatMul", "attrs": {"transpose_b": {"type": "bool", "value": 1}},
         "inputs": [ga._t(0, "bf16", [B, H, Sq, D]), ga._t(1, "bf16", [B, H, Sk, D])], "outputs": [ga._t(3, "f32", s)]},
        {"kind": "SoftMax", "attrs": {"axis": {"type": "s64", "value": -1}}, "inputs": [ga._t(3, "f32", s)],
         "outputs": [ga._t(4, "bf16", s)]},
        {"kind": "MatMul", "inputs": [ga._t(4, "bf16", s), ga._t(2, "bf16", [B, H, Sk, D])],
         "outputs": [ga._t(5, "bf16", [B, H, Sq, D])]}], [0, 1, 2], [5])


def test_unscaled_attention_is_one_step(ga):
    assert "attention" in ga.explain(_unscaled(ga, 1, 8, 1, 4096, 128))[1]


@pytest.mark.gpu
def test_captured_partition(gc, ga, dev):
    import torch
    B, H, Sq, Sk, D = 1, 8, 1, 4096, 128
    comp = ga.Compiler()
    st, exe = comp.compile(_unscaled(ga, B, H, Sq, Sk, D))
    assert st == 0, ga.api().dnnl_graph_compiler_last_error().decode()
    g = torch.Generator(device=dev).manual_seed(1)
    Q, K, V = (torch.randn(B, H, s, D, device=dev, generator=g).to(torch.bfloat16) for s in (Sq, Sk, Sk))
    out = torch.zeros_like(Q)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        call = exe.bind([(0, Q), (1, K), (2, V)], [(5, out)], stream=side.cuda_stream)
        assert call() == 0
        side.synchronize()
        graph.capture_begin()
        rc = call()
        graph.capture_end()
        assert rc == 0
    for k in range(3):
        Q.copy_(0.1 * torch.randn(B, H, Sq, D, device=dev, generator=g))
        out.zero_()
        want = gc.mha_fwd_bf16(Q, K, V, None, 1.0)  # through the library's workspace
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), k
    del graph
    exe.close()
    comp.close()
