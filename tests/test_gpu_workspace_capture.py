"""Calls that use the library's workspace while the stream that used it last is being captured: they are not drawn into
that graph and the graph does not get to know of them; they do without the workspace."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu


def test_last_users_stream_under_capture(gc, dev):
    g = torch.Generator(device=dev).manual_seed(3)
    bf = lambda *s: torch.randn(*s, device=dev, generator=g).to(torch.bfloat16)  # noqa: E731
    Q, K, V = bf(1, 8, 1, 128), bf(1, 8, 4096, 128), bf(1, 8, 4096, 128)            # keys cut over workgroups
    Qp, Kp, Vp = bf(1, 4, 256, 128), bf(1, 4, 256, 128), bf(1, 4, 256, 128)         # mask classes
    mask = torch.triu(torch.full((256, 256), float("-inf"), device=dev), diagonal=1)
    A = torch.randint(-2, 3, (192, 4096), device=dev, generator=g).to(torch.bfloat16)  # K slices; integers: exact sums
    B = torch.randint(-2, 3, (4096, 1024), device=dev, generator=g).to(torch.bfloat16)
    assert gc.lib().gcmi_gemm_bf16_workspace_bytes(192, 1024, 4096, 0) > 0
    want = gc.mha_fwd_bf16(Q, K, V), gc.mha_fwd_bf16(Qp, Kp, Vp, mask), gc.gemm_bf16(A, B, out_dtype=gc.F32)
    outs = [torch.zeros_like(t) for t in want]
    counter = torch.zeros(1, device=dev)
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    assert gc.lib().gcmi_gemm_bf16(None, None, None, 4, 4, 4, 4, 4, 4, None, 2, 0, 2, None) == 2
    text = gc.lib().gcmi_last_error()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s1):
        gc.mha_fwd_bf16(Q, K, V, out=outs[0])  # s1 is the workspace's last user
        s1.synchronize()
        outs[0].zero_()
        s1.synchronize()
        graph.capture_begin(capture_error_mode="relaxed")
        counter.add_(1)
        with torch.cuda.stream(s2):
            gc.mha_fwd_bf16(Q, K, V, out=outs[0])
            gc.mha_fwd_bf16(Qp, Kp, Vp, mask, out=outs[1])
            gc.gemm_bf16(A, B, out_dtype=gc.F32, out=outs[2])
            s2.synchronize()  # eager work: done here, not part of the graph
            eager = [o.to("cpu") for o in outs]
        graph.capture_end()
    assert gc.lib().gcmi_last_error() == text  # doing without is no error
    assert torch.equal(eager[1], want[1].cpu())
    assert torch.equal(eager[2], want[2].cpu())
    assert (eager[0].double() - want[0].cpu().double()).norm() <= 1e-2 * want[0].double().norm().item()
    for o in outs:
        o.zero_()
    torch.cuda.synchronize()
    for _ in range(3):
        graph.replay()
    torch.cuda.synchronize()
    assert counter.item() == 3 and all((o == 0).all() for o in outs)
    # and the other way round: the workspace is shared again once the capture is over
    with torch.cuda.stream(s2):
        again = gc.mha_fwd_bf16(Q, K, V)
    torch.cuda.synchronize()
    assert torch.equal(again, want[0])
