"""GELU of bf16 for every finite bf16 value, in a GEMM's epilogue (the product with the identity is the value itself) and as an
op of its own."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _values(dev):
    x = torch.arange(65536, device=dev, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    return torch.where(x.isfinite(), x, torch.zeros_like(x)).view(512, 128)


@pytest.mark.parametrize("rows", [512, 16])  # the tile kernels' epilogue, the few-row kernel's
@pytest.mark.parametrize("nt", [False, True])
def test_every_value(gc, dev, rows, nt):
    A, eye = _values(dev), torch.eye(128, device=dev, dtype=torch.bfloat16)
    f = gc.gemm_bf16_nt if nt else gc.gemm_bf16
    got = torch.cat([f(a.contiguous(), eye, act="gelu_erf") for a in A.split(rows)])
    x = A.double()
    true = 0.5 * x * torch.special.erfc(-x * 0.5 ** 0.5)
    near = true.float().to(torch.bfloat16)
    tiny = 13.2 * 2.0 ** -126  # the exponential's results below the smallest normal number are 0: |x| > 13, times x
    near = torch.where(true.abs() < tiny, got, near)
    off = got != near
    # the exponent's polynomial is good to 8.3e-5, which moves a result by up to 2 % of half a unit in the last place (2^-8): the
    # other neighbour of a value that lies between two.  Past |x| = 6 it is good to 4 % of the value, which is below 1e-8 there.
    assert int(off.sum()) <= 100
    assert ((got.double() - true).abs() <= (1.03 * 2.0 ** -8 * (x > -6) + 0.05 * (x <= -6)) * true.abs() + tiny).all()


def test_infinities(gc, dev):
    A = torch.ones(300, 64, device=dev, dtype=torch.bfloat16)
    B = torch.zeros(64, 256, device=dev, dtype=torch.bfloat16)
    B[3, 0], B[3, 1], B[3, 2], B[3, 5] = float("inf"), float("-inf"), float("nan"), 2.0
    out = gc.gemm_bf16(A, B, act="gelu_erf")
    assert (out[:, 0] == float("inf")).all() and out[:, 1:3].isnan().all() and not out[:, 3:].isnan().any()
    assert ((out[:, 5].float() - 1.953125).abs() < 1e-6).all() and (out[:, 6:] == 0).all()


def _graph(ga, kinds, inner=()):
    """x -> kinds[0] -> kinds[1] ...; MatMul has the identity for its second operand, inner results are outputs too"""
    ops, last = [], 0
    for i, kind in enumerate(kinds):
        t = {"dtype": "bf16", "shape": [512, 128]}
        ins = [dict(t, id=last)] + ([{"id": 100, "dtype": "bf16", "shape": [128, 128]}] if kind == "MatMul" else [])
        attrs = {"attrs": {"mode": {"type": "string", "value": "gelu_erf"}}} if kind == "GELU" else {}
        ops.append(dict({"kind": kind, "inputs": ins, "outputs": [dict(t, id=i + 1)]}, **attrs))
        last = i + 1
    matmul = "MatMul" in kinds
    return ga._graph(ops, [0] + [100] * matmul, list(inner) + [last]), [0] + [100] * matmul, list(inner) + [last]


def _run(ga, graph, x, eye):
    text, ins, outs = graph
    comp = ga.Compiler()
    st, exe = comp.compile(text)
    assert st == 0, ga.api().dnnl_graph_compiler_last_error().decode()
    res = [torch.empty_like(x) for _ in outs]
    try:
        call = exe.bind([(i, x if i == 0 else eye) for i in ins], list(zip(outs, res)), torch.cuda.current_stream().cuda_stream)
        assert call() == 0
        torch.cuda.synchronize()
    finally:
        exe.close()
        comp.close()
    return res[-1]


@pytest.mark.parametrize("kinds,inner,env", [
    (["GELU"], (), None), (["MatMul", "GELU"], (1,), None),                                # a step of its own, alone and behind a GEMM
    (["GELU", "Abs"], (), None), (["GELU", "Abs"], (), "GCMI_NO_GENERATED_KERNELS"),  # in a group: generated, interpreted
    (["GELU", "Abs"], (), "GCMI_NO_POINTWISE_FUSION")])
def test_bits_of_the_epilogue(ga, dev, monkeypatch, kinds, inner, env):
    x, eye = _values(dev), torch.eye(128, device=dev, dtype=torch.bfloat16)
    want = _run(ga, _graph(ga, ["MatMul", "GELU"]), x, eye)
    if env:
        monkeypatch.setenv(env, "1")
    got = _run(ga, _graph(ga, kinds, inner), x, eye)
    assert torch.equal(got, want.abs() if "Abs" in kinds else want)  # (the sum of a product makes -0 a 0)
