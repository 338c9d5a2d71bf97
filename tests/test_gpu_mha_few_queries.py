"""Attention of fewer than 128 queries: key blocks cut over waves, and over workgroups where heads are few, at the edges
of query tiles (32), key blocks (32), waves (4) and key ranges; against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _reference(Q, K, V, mask, scale):
    S = torch.matmul(Q.double(), K.double().transpose(-1, -2).contiguous()) * scale
    if mask is not None:
        S = S + mask.double()
    P = torch.softmax(S, -1)
    return torch.matmul(P, V.double()), torch.matmul(P, V.double().abs())


def _check(out, ref, mag):
    # a weight is rounded to bf16 (8 significant bits: by at most 2^-8 of itself), so is the result; the scores' f32 sums
    # move a weight by less than 2^-12
    assert ((out.double() - ref).abs() <= (2.0 ** -8 + 2.0 ** -12) * mag + 2.0 ** -8 * ref.abs() + 1e-30).all()


@pytest.mark.parametrize("Sq", [1, 2, 31, 33, 127])
@pytest.mark.parametrize("Sk", [1, 31, 32, 33, 128, 129, 777, 4097])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("masked", [False, True])
def test_few_queries(gc, dev, Sq, Sk, D, masked):
    B, H = (1, 3) if Sk > 200 else (2, 5)
    g = torch.Generator(device=dev).manual_seed(Sq * 31 + Sk)
    Q, K, V = (torch.randn(B, H, s, D, device=dev, generator=g).to(torch.bfloat16) for s in (Sq, Sk, Sk))
    mask = None
    if masked:  # some keys hidden (never the first), the others moved; rows longer than the keys
        mask = torch.randn(Sq, Sk + 3, device=dev, generator=g)
        mask[torch.rand(Sq, Sk + 3, device=dev, generator=g) < 0.3] = float("-inf")
        mask[:, 0] = 0
        mask = mask[:, :Sk]
    out = gc.mha_fwd_bf16(Q, K, V, mask)
    _check(out, *_reference(Q, K, V, mask, D ** -0.5))
    assert torch.equal(out, gc.mha_fwd_bf16(Q, K, V, mask))  # fixed order of the sums


@pytest.mark.parametrize("D", [64, 128])
def test_few_queries_special_rows(gc, dev, D):
    """A row that sees no key is NaN and leaves its neighbours alone; what lies past the last key counts for nothing;
    a scale of zero weighs all keys alike."""
    g = torch.Generator(device=dev).manual_seed(D)
    Q, K, V = (torch.randn(1, 2, s, D, device=dev, generator=g).to(torch.bfloat16) for s in (3, 2049, 2049))
    mask = torch.zeros(3, 2049, device=dev)
    mask[1] = float("-inf")
    mask[2, :2048] = float("-inf")  # the last key alone, in a block of its own
    out = gc.mha_fwd_bf16(Q, K, V, mask)
    assert out[:, :, 1].isnan().all() and not out[:, :, 0].isnan().any()
    assert torch.equal(out[:, :, 2], V[:, :, 2048])
    V[:, :, 2048] = float("inf")
    assert (gc.mha_fwd_bf16(Q, K, V, mask)[:, :, 2] == float("inf")).all()
    V[:, :, 2048] = 1
    _check(gc.mha_fwd_bf16(Q, K, V, None, scale=0.0), *_reference(Q, K, V, None, 0.0))


def test_few_queries_under_capture_and_on_two_streams(gc, dev):
    """Captured calls take no scratch memory (one piece per head); eager calls of two streams share the library's."""
    g = torch.Generator(device=dev).manual_seed(7)
    Q, K, V = (torch.randn(2, 4, s, 128, device=dev, generator=g).to(torch.bfloat16) for s in (1, 3000, 3000))
    ref, mag = _reference(Q, K, V, None, 128 ** -0.5)
    out = torch.zeros_like(Q)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        gc.mha_fwd_bf16(Q, K, V, out=out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        _check(gc.mha_fwd_bf16(Q, K, V), ref, mag)
        torch.cuda.synchronize()
        _check(out, ref, mag)
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    results = []
    for i in range(8):
        with torch.cuda.stream(streams[i % 2]):
            results.append(gc.mha_fwd_bf16(Q, K, V if i % 2 == 0 else -V))
    torch.cuda.synchronize()
    for i, r in enumerate(results):
        _check(r, ref if i % 2 == 0 else -ref, mag)
