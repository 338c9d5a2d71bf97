"""Up to 256 rows of A in one launch (K over the waves of a workgroup): every tile of the kernel at its edges, ends of K
inside a stage, strided operands, every epilogue, special values behind K, and both layouts of the weights."""
import pytest
import torch

pytestmark = pytest.mark.gpu

FEW = 7
# every tile of 16, 32 and 64 rows and columns, whole and cut, one and two rounds of workgroups; K in whole stages (64 bf16,
# 128 bytes), one chunk into and one chunk short of one, and fewer stages than waves
SHAPES = [(1, 640, 576), (3, 1712, 2736), (16, 24, 144), (17, 1000, 1080), (32, 2048, 1016), (33, 520, 1544), (64, 2008, 640),
          (50, 8, 4096), (5, 8200, 264), (31, 9000, 200), (64, 8208, 328), (9, 16400, 160), (20, 17000, 232), (48, 16376, 296), (128, 1288, 200), (97, 3000, 392), (256, 1000, 256), (65, 520, 4088),
          (32, 4096, 1376), (129, 1024, 4072), (140, 264, 1048), (251, 2648, 776)]


def _ints(shape, lo, hi, dev, g, dt):
    return torch.randint(lo, hi, shape, device=dev, generator=g, dtype=torch.int32).to(dt)


def _padded(t, pad, fill):
    """The same values inside rows that are `pad` elements longer, `fill` between and behind them."""
    full = torch.full((t.shape[0] + 1, t.shape[1] + pad), fill, device=t.device, dtype=t.dtype)
    full[:t.shape[0], :t.shape[1]] = t
    return full[:t.shape[0], :t.shape[1]]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("trans_b", [False, True])
def test_bf16_exact_on_integers(gc, dev, M, N, K, trans_b):
    """NaN in what lies behind the rows and the columns of the operands: none of it may be used."""
    assert gc.tile_config(M, N, K, trans_b=trans_b, out_dtype=gc.F32)[0].kernel == FEW
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    A, W = _ints((M, K), -3, 4, dev, g, torch.bfloat16), _ints((K, N), -3, 4, dev, g, torch.bfloat16)
    want = A.float() @ W.float()
    Ap, Wp = _padded(A, 8, float("nan")), _padded(W.t().contiguous() if trans_b else W, 8, float("nan"))
    guard = torch.full((M + 2, N + 4), 7.0, device=dev)
    out = guard[1:M + 1, :N]
    (gc.gemm_bf16_nt if trans_b else gc.gemm_bf16)(Ap, Wp, out_dtype=gc.F32, out=out)
    assert torch.equal(out, want)
    assert (guard[0] == 7.0).all() and (guard[M + 1] == 7.0).all() and (guard[:, N:] == 7.0).all()


@pytest.mark.parametrize("M,N,K", [(3, 1712, 2736), (32, 2048, 1016), (64, 8208, 328), (20, 17000, 232), (32, 4096, 1376), (140, 264, 1048)])
def test_bf16_rounding_points_and_layouts(gc, dev, M, N, K):
    """Bias, activation and residual against float64 rounded where a bf16 graph rounds; [N,K] and [K,N] weights give the same bits."""
    g = torch.Generator(device=dev).manual_seed(N + K)
    A = torch.randn(M, K, device=dev, generator=g).to(torch.bfloat16)
    W = (torch.randn(K, N, device=dev, generator=g) * 0.05).to(torch.bfloat16)
    bias, res = torch.randn(N, device=dev, generator=g).to(torch.bfloat16), torch.randn(M, N, device=dev, generator=g).to(torch.bfloat16)
    acc = A.double() @ W.double()
    r = lambda t: t.to(torch.bfloat16).double()  # noqa: E731
    gelu = lambda t: 0.5 * t * (1.0 + torch.special.erf(t / 2.0 ** 0.5))  # noqa: E731
    want = r(r(gelu(r(r(acc) + bias.double()))) + res.double())
    nn = gc.gemm_bf16_residual(A, W, res, bias=bias, act="gelu_erf")
    mag = torch.maximum(acc.abs(), torch.maximum(want.abs(), res.double().abs())) + 1.0
    assert float(((nn.double() - want).abs() / mag).max()) < 2.0 ** -7
    nt = gc.gemm_bf16_residual(A, W.t().contiguous(), res, trans_b=True, bias=bias, act="gelu_erf")
    assert torch.equal(nn, nt)
    f32 = gc.gemm_bf16(A, W, bias, "sigmoid", gc.F32)
    # K + 1 additions of exact products, each rounded once; the sigmoid's slope is at most a quarter and its own error 1e-6
    tol = 0.25 * (K + 1) * 2.0 ** -24 * (A.double().abs() @ W.double().abs() + bias.double().abs()) + 1e-6
    assert ((f32.double() - torch.sigmoid(acc + bias.double())).abs() <= tol).all()


@pytest.mark.parametrize("nb,M,N,K", [(3, 3, 1712, 2736), (84, 46, 176, 960), (7, 1, 96, 1064), (300, 20, 24, 144), (9, 64, 520, 328)])
@pytest.mark.parametrize("trans_b", [False, True])
def test_bf16_batches_exact_on_integers(gc, dev, nb, M, N, K, trans_b):
    """Matrices of one and several tiles, whole and cut, their workgroups in one run over the XCDs; one B for all, or each its own."""
    g = torch.Generator(device=dev).manual_seed(nb + N)
    A, W = _ints((nb, M, K), -3, 4, dev, g, torch.bfloat16), _ints((nb, K, N), -3, 4, dev, g, torch.bfloat16)
    guard = torch.full((nb * M * N + 64,), 7.0, device=dev, dtype=torch.bfloat16)
    out = guard[32:32 + nb * M * N].view(nb, M, N)
    for B in (W, W[0]):
        gc.gemm_batched(A, (B.transpose(-2, -1) if trans_b else B).contiguous(), trans_b, out=out)
        want = torch.stack([A[i].float() @ (B[i] if B.dim() == 3 else B).float() for i in range(nb)])
        assert torch.equal(out, want.to(torch.bfloat16))
        assert (guard[:32] == 7.0).all() and (guard[-32:] == 7.0).all()


def test_bf16_special_values(gc, dev):
    """An infinity reaches its own row or column as it is, also in the chunks that stand in for what lies behind K."""
    M, N, K = 18, 520, 1032
    A, W = torch.ones(M, K, device=dev, dtype=torch.bfloat16), torch.ones(K, N, device=dev, dtype=torch.bfloat16)
    A[2, K - 1], W[K - 1, 5], W[3, 7] = float("inf"), float("-inf"), float("nan")
    for out in (gc.gemm_bf16(A, W), gc.gemm_bf16_nt(A, W.t().contiguous())):
        assert out[:, 7].isnan().all() and out[2, 5] == float("-inf")
        assert (out[2, [c for c in range(N) if c not in (5, 7)]] == float("inf")).all()
        assert (out[[m for m in range(M) if m != 2], 5] == float("-inf")).all()
        rest = out[[m for m in range(M) if m != 2]][:, [c for c in range(N) if c not in (5, 7)]]
        assert (rest == K).all()


@pytest.mark.parametrize("M,N,K", [(1, 640, 512), (8, 672, 1856), (17, 1008, 1040), (32, 11008, 4096), (64, 4096, 528), (22, 16, 4080),
                                   (40, 9008, 272 + 16), (12, 16400, 400), (64, 16368, 336), (200, 1040, 528), (256, 3008, 304),
                                   (257, 3264, 4096), (700, 1008, 1040), (2048, 512, 528)])
@pytest.mark.parametrize("a_dtype", [torch.uint8, torch.int8])
def test_int8_exact_and_epilogues(gc, dev, M, N, K, a_dtype):
    u8 = a_dtype is torch.uint8
    assert gc.tile_config(M, N, K, a_dtype=gc.U8 if u8 else gc.S8)[0].kernel == FEW
    g = torch.Generator(device=dev).manual_seed(K + N)
    A = _padded(_ints((M, K), 0 if u8 else -128, 256 if u8 else 128, dev, g, a_dtype), 16, 77)
    W = _padded(_ints((K, N), -128, 128, dev, g, torch.int8), 16, 99)
    zp = 131 if u8 else 0
    cs = gc.colsum_s8(W)
    acc = (A.double() - zp) @ W.double()
    raw = torch.full((M + 2, N), 7, device=dev, dtype=torch.int32)
    gc.gemm_int8(A, W, cs, zp, None, None, None, gc.S32, out=raw[1:M + 1])
    assert torch.equal(raw[1:M + 1].double(), A.double() @ W.double()) and (raw[0] == 7).all() and (raw[M + 1] == 7).all()
    scale = (torch.rand(N, device=dev, generator=g) + 0.5) / (60.0 * K ** 0.5)
    bias = torch.randn(N + 1, device=dev, generator=g)[1:]  # not 16-byte aligned
    pre = acc * scale.double() + bias.double()
    f = {None: lambda x: x, "relu": torch.relu, "sigmoid": torch.sigmoid, "gelu_erf": torch.nn.functional.gelu,
         "gelu_tanh": lambda x: torch.nn.functional.gelu(x, approximate="tanh")}
    for act, fn in f.items():
        # the accumulators are exact: a conversion, a product and a sum in f32, and the activation's own error
        y32 = gc.gemm_int8(A, W, cs, zp, scale, bias, act, gc.F32)
        assert ((y32.double() - fn(pre)).abs() <= 1.13 * 2.0 ** -22 * ((acc * scale.double()).abs() + bias.double().abs()) + 2e-6).all()
        y16 = gc.gemm_int8(A, W, cs, zp, scale, bias, act, gc.BF16)
        # one rounding to bf16; the short GELU is good to 2^-11.9
        assert ((y16.double() - fn(pre)).abs() <= 2.0 ** -8 * 1.1 * fn(pre).abs() + 2e-6).all()


def test_int8_special_scales(gc, dev):
    """Scales and biases that leave the range of f32 take the epilogue that looks for NaN."""
    M, N, K = 4, 48, 512
    A, W = torch.full((M, K), 3, device=dev, dtype=torch.uint8), torch.ones(K, N, device=dev, dtype=torch.int8)
    scale, bias = torch.ones(N, device=dev), torch.zeros(N, device=dev)
    scale[0], scale[1], bias[1], bias[2], scale[20] = float("inf"), float("inf"), float("-inf"), float("nan"), 1e38
    out = gc.gemm_int8(A, W, gc.colsum_s8(W), 0, scale, bias, "relu", gc.BF16)
    assert (out[:, 0] == float("inf")).all() and out[:, 1].isnan().all() and out[:, 2].isnan().all()
    assert (out[:, 20] == float("inf")).all() and (out[:, 3:20] == 3 * K).all()
    assert (out[:, 1].view(torch.int16) == 0x7FC0).all() and (out[:, 2].view(torch.int16) == 0x7FC0).all()


@pytest.mark.parametrize("M,N,K", [(64, 64, 65408), (33, 200, 20008), (19, 224, 20032), (7, 256, 16384), (5, 24, 50000)])
@pytest.mark.parametrize("trans_b", [False, True])
def test_a_long_k_with_and_without_the_workspace(gc, dev, M, N, K, trans_b):
    """K slices where another kernel has them and the buffer can be had; in one launch under capture and without a workspace."""
    import ctypes as C
    g = torch.Generator(device=dev).manual_seed(K)
    A, W = _ints((M, K), -2, 3, dev, g, torch.bfloat16), _ints((K, N), -2, 3, dev, g, torch.bfloat16)
    want = A.double() @ W.double()
    B, f = (W.t().contiguous(), gc.gemm_bf16_nt) if trans_b else (W, gc.gemm_bf16)
    assert torch.equal(f(A, B, out_dtype=gc.F32).double(), want)
    out, none = torch.zeros(M, N, device=dev), torch.zeros(M, N, device=dev)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        graph = torch.cuda.CUDAGraph()
        graph.capture_begin()
        f(A, B, out_dtype=gc.F32, out=out)
        graph.capture_end()
    for _ in range(3):
        out.zero_()
        f(-A, B, out_dtype=gc.F32)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.double(), want)
    gc.check(gc.lib().gcmi_gemm_bf16_ws(A.data_ptr(), B.data_ptr(), none.data_ptr(), 1, M, N, K, K, B.shape[1], N, 0, 0, 0, int(trans_b), None,
                                        gc.BF16, 0, None, 0, gc.BF16, gc.F32, None, 0, None,
                                        C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    assert torch.equal(none.double(), want)
