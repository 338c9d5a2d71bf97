"""Which scratch buffer of the library a call gets: streams keep to their own (four per device), and a call whose buffer's
last user is being captured is not drawn into that graph; it does without."""
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
        gc.mha_fwd_bf16(Q, K, V, out=outs[0])
        s1.synchronize()
        for s in [torch.cuda.Stream() for _ in range(3)]:  # the other buffers: s1's is the one used longest ago
            with torch.cuda.stream(s):
                gc.mha_fwd_bf16(Q, K, V, out=outs[0])
                s.synchronize()
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
    # once the capture is over its buffer can be had again
    with torch.cuda.stream(s2):
        again = gc.mha_fwd_bf16(Q, K, V)
    torch.cuda.synchronize()
    assert torch.equal(again, want[0])


def test_two_streams_do_not_wait_for_each_other(gc, dev):
    """A call on a second stream does not queue up behind what the first stream was given after its own call."""
    g = torch.Generator(device=dev).manual_seed(4)
    bf = lambda *s: torch.randn(*s, device=dev, generator=g).to(torch.bfloat16)  # noqa: E731
    Q, K, V = bf(1, 8, 1, 128), bf(1, 8, 4096, 128), bf(1, 8, 4096, 128)
    A = torch.randint(-2, 3, (192, 5640), device=dev, generator=g).to(torch.bfloat16)
    B = torch.randint(-2, 3, (5640, 1024), device=dev, generator=g).to(torch.bfloat16)
    assert gc.lib().gcmi_gemm_bf16_workspace_bytes(192, 1024, 5640, 0) > 0
    want = gc.mha_fwd_bf16(Q, K, V), gc.gemm_bf16(A, B, out_dtype=gc.F32)
    streams = [torch.cuda.Stream() for _ in range(2)]
    outs = [(torch.zeros_like(want[0]), torch.zeros_like(want[1])) for _ in streams]
    torch.cuda.synchronize()
    for s, (o, c) in zip(streams, outs):
        with torch.cuda.stream(s):
            gc.mha_fwd_bf16(Q, K, V, out=o)
            gc.gemm_bf16(A, B, out_dtype=gc.F32, out=c)
            s.synchronize()
            o.zero_()
            c.zero_()
    torch.cuda.synchronize()
    with torch.cuda.stream(streams[0]):
        gc.mha_fwd_bf16(Q, K, V, out=outs[0][0])
        gc.gemm_bf16(A, B, out_dtype=gc.F32, out=outs[0][1])
        torch.cuda._sleep(1 << 29)  # a fraction of a second
        late = torch.cuda.Event()
        late.record()
    with torch.cuda.stream(streams[1]):
        gc.mha_fwd_bf16(Q, K, V, out=outs[1][0])
        gc.gemm_bf16(A, B, out_dtype=gc.F32, out=outs[1][1])
        streams[1].synchronize()
        assert not late.query(), "the second stream's calls waited for the first stream's later work"
    torch.cuda.synchronize()
    for o, c in outs:
        assert torch.equal(o, want[0]) and torch.equal(c, want[1])


def test_more_streams_than_blocks(gc, dev):
    """Beyond the number of buffers the calls are put in order; every result is right whoever shares."""
    g = torch.Generator(device=dev).manual_seed(5)
    bf = lambda *s: torch.randn(*s, device=dev, generator=g).to(torch.bfloat16)  # noqa: E731
    K, V = bf(1, 8, 3000, 128), bf(1, 8, 3000, 128)
    Qs = [bf(1, 8, 1, 128) for _ in range(7)]
    want = [gc.mha_fwd_bf16(q, K, V) for q in Qs]
    streams = [torch.cuda.Stream() for _ in Qs]
    outs = [[torch.zeros_like(q) for q in Qs] for _ in range(6)]
    torch.cuda.synchronize()
    for row in outs:
        for s, q, o in zip(streams, Qs, row):
            with torch.cuda.stream(s):
                gc.mha_fwd_bf16(q, K, V, out=o)
    torch.cuda.synchronize()
    for row in outs:
        for o, w in zip(row, want):
            assert torch.equal(o, w)


def test_null_stream_calls_follow_one_another(gc, dev):
    """Calls on the null stream, from two host threads, share its buffer without waits; other streams in between."""
    import threading
    g = torch.Generator(device=dev).manual_seed(6)
    bf = lambda *s: torch.randn(*s, device=dev, generator=g).to(torch.bfloat16)  # noqa: E731
    K, V = bf(1, 8, 3000, 128), bf(1, 8, 3000, 128)
    Qs = [bf(1, 8, 1, 128) for _ in range(3)]
    want = [gc.mha_fwd_bf16(q, K, V) for q in Qs]
    outs = [[torch.zeros_like(q) for _ in range(40)] for q in Qs]
    side = torch.cuda.Stream()
    torch.cuda.synchronize()

    def calls(i, stream):
        with torch.cuda.stream(stream):
            for o in outs[i]:
                gc.mha_fwd_bf16(Qs[i], K, V, out=o)

    null = torch.cuda.default_stream()
    assert null.cuda_stream == 0
    threads = [threading.Thread(target=calls, args=a) for a in ((0, null), (1, null), (2, side))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for i, w in enumerate(want):
        assert all(torch.equal(o, w) for o in outs[i]), i
