"""silu(x . Wg^T) * (x . Wu^T) as one launch (gemm_gated.hip) against one launch per op, in every form that sizes select."""
import importlib

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mm(gc):
    return importlib.import_module("graph_compiler_amd.mlir_modules")


def _module(mm, T, K, N):
    f = mm._Fn()
    tw = mm.ttype([T, N], "bf16")
    gate = mm._matmul(f, "matmul_transpose_b", "%arg0", [T, K], "%arg1", [N, K], [T, N], "bf16")
    one = mm._splat(f, 1.0, [T, N], "bf16")
    ex = mm._named(f, "exp", [mm._named(f, "negf", [gate], [tw], [T, N], "bf16")], [tw], [T, N], "bf16")
    sig = mm._binary(f, "div", one, mm._binary(f, "add", one, ex, [T, N], "bf16"), [T, N], "bf16")
    silu = mm._binary(f, "mul", sig, gate, [T, N], "bf16")
    up = mm._matmul(f, "matmul_transpose_b", "%arg0", [T, K], "%arg2", [N, K], [T, N], "bf16")
    out = mm._binary(f, "mul", silu, up, [T, N], "bf16")
    args = [mm.ttype([T, K], "bf16"), mm.ttype([N, K], "bf16"), mm.ttype([N, K], "bf16")]
    return mm._module(args, [tw], f, [out])


def _run(ga, text, ins, out):
    comp = ga.Compiler()
    st, exe = comp.compile_mlir(text)
    assert st == 0, ga.api().dnnl_graph_compiler_last_error().decode()
    try:
        assert exe.bind(list(enumerate(ins)), [(len(ins), out)], torch.cuda.current_stream().cuda_stream)() == 0
        torch.cuda.synchronize()
    finally:
        exe.close()
        comp.close()


def _exact(dev, T, K, N, seed):
    """Small integers times a power of two: every sum is exact in f32 in any order, so both ways have the same bits."""
    g = torch.Generator(device=dev).manual_seed(seed)
    r = lambda s, *shape: (torch.randint(-3, 4, shape, device=dev, generator=g) * s).bfloat16()  # noqa: E731
    return [r(1.0, T, K), r(2.0 ** -6, N, K), r(2.0 ** -6, N, K)]


# The kernel each size selects: rows x columns of C per workgroup.  Few rows: 1 to 4 column tiles per product for up to 32 and 64 rows, 1
# and 2 up to 128, whole and cut workgroups, more than one round of them; tiles of 128 to 256 rows by 64 to 128 columns, rows and
# columns off the tile, a K that ends inside a group.
FEW = [(1, 512, 4096, "32x16"), (31, 512, 4108, "32x20"), (32, 640, 11008, "32x44"), (20, 512, 13000, "32x52"), (17, 1024, 2816, "32x12"),
       (40, 1024, 2816, "64x12"), (64, 512, 4100, "64x20"), (64, 512, 16900, "64x36"), (33, 512, 13000, "64x52"), (100, 1024, 2816, "128x12"),
       (65, 512, 4108, "128x20")]
TILES = [(128, 520, 4100, "128x64"), (129, 512, 11008, "192x64"), (200, 1032, 2816, "128x64"), (250, 512, 11008, "256x64"),
         (250, 520, 11008, "256x64"), (257, 512, 11004, "128x64"), (300, 640, 5632, "192x64"), (513, 520, 8200, "192x64"),
         (700, 520, 8204, "256x128"), (1000, 512, 11008, "256x96"), (1000, 1024, 5632, "256x96"), (1000, 520, 11008, "256x96")]


@pytest.mark.parametrize("T,K,N,tile", FEW + TILES)
def test_bits_of_single_ops(ga, mm, dev, monkeypatch, T, K, N, tile):
    text = _module(mm, T, K, N)
    ins = _exact(dev, T, K, N, T + K + N)
    ins[0][0, 3] = float("inf")  # a row of infinities and NaNs, and no other
    full = torch.full((T + 1, N), 7.0, device=dev, dtype=torch.bfloat16)
    fused, single = full[:T], torch.empty(T, N, device=dev, dtype=torch.bfloat16)
    st, plan = ga.explain_mlir(text)
    assert st == 0 and ", %s per workgroup" % tile in plan and ("weight streaming" in plan) == (T <= 100), plan
    _run(ga, text, ins, fused)
    monkeypatch.setenv("GCMI_NO_POINTWISE_FUSION", "1")
    _run(ga, text, ins, single)
    assert "MatMul x2" in plan and "MatMul x2" not in ga.explain_mlir(text)[1]
    assert torch.equal(fused.view(torch.int16), single.view(torch.int16))
    assert (full[T] == 7.0).all() and not fused[1:].isnan().any()


def test_sigmoid_of_every_value(ga, mm, dev, monkeypatch):
    """Identity weights make the gate's sums the operand itself, every finite bf16 value; up's are 1."""
    T, K, N = 128, 640, 4096
    values = torch.arange(65536, device=dev, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    values = torch.where(values.isfinite(), values, torch.zeros_like(values)).view(T, 512)
    ins = [torch.zeros(T, K, device=dev, dtype=torch.bfloat16)] + [torch.zeros(N, K, device=dev, dtype=torch.bfloat16) for _ in range(2)]
    ins[0][:, :512], ins[0][:, K - 1] = values, 1.0
    ins[1][torch.arange(N), torch.arange(N) % 512] = 1.0
    ins[2][:, K - 1] = 1.0
    text = _module(mm, T, K, N)
    fused, single = (torch.empty(T, N, device=dev, dtype=torch.bfloat16) for _ in range(2))
    assert "MatMul x2" in ga.explain_mlir(text)[1]
    _run(ga, text, ins, fused)
    monkeypatch.setenv("GCMI_NO_POINTWISE_FUSION", "1")
    _run(ga, text, ins, single)
    assert torch.equal(fused.view(torch.int16), single.view(torch.int16))


@pytest.mark.parametrize("T,K,N", [(32, 4096, 11008), (200, 2048, 5632)])
def test_error(ga, mm, dev, T, K, N):
    g = torch.Generator(device=dev).manual_seed(3)
    x = torch.randn(T, K, device=dev, generator=g).bfloat16()
    Wg, Wu = ((torch.randn(N, K, device=dev, generator=g) * K ** -0.5).bfloat16() for _ in range(2))
    out = torch.empty(T, N, device=dev, dtype=torch.bfloat16)
    _run(ga, _module(mm, T, K, N), [x, Wg, Wu], out)
    xd, gd, ud = x.double(), Wg.double(), Wu.double()
    gate, up = xd @ gd.t(), xd @ ud.t()
    eg, eu = ((K + 1) * 2.0 ** -24 * (xd.abs() @ w.abs().t()) for w in (gd, ud))  # f32 sums in any order
    silu = gate * torch.sigmoid(gate)
    # five roundings to bf16, half an ulp each: up, sigmoid, silu, the result, and gate, whose error silu passes on by a factor
    # of up to 1 + |gate|; no slope of silu above 1.1
    bound = 1.01 * (2.0 ** -9 * (5 + gate.abs()) * (silu * up).abs() + 1.1 * up.abs() * eg + silu.abs() * eu)
    assert ((out.double() - silu * up).abs() <= bound).all()


def test_operands_off_16_bytes_take_the_separate_steps(ga, mm, dev):
    T, K, N = 32, 512, 4100
    ins = _exact(dev, T, K, N, 1)
    text = _module(mm, T, K, N)
    want, out = (torch.empty(T, N, device=dev, dtype=torch.bfloat16) for _ in range(2))
    _run(ga, text, ins, want)
    off = torch.empty(N * K + 4, device=dev, dtype=torch.bfloat16)[4:].view(N, K)
    off.copy_(ins[2])
    assert off.data_ptr() % 16 == 8
    _run(ga, text, [ins[0], ins[1], off], out)
    assert torch.equal(out, want)
