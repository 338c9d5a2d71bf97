"""Which gates become one step (planner only, no GPU)."""
import importlib

import pytest


@pytest.fixture(scope="module")
def mm(gc):
    return importlib.import_module("graph_compiler_amd.mlir_modules")


def _gate(mm, T=32, K=1024, N=4096, keep=None, tb=True, swap=False):
    f = mm._Fn()
    s, t = [T, N], "bf16"
    ty = mm.ttype(s, t)
    w = [N, K] if tb else [K, N]

    def mul(a, b):
        return mm._binary(f, "mul", b, a, s, t) if swap else mm._binary(f, "mul", a, b, s, t)

    def dot(arg):
        return mm._matmul(f, "matmul_transpose_b" if tb else "matmul", "%arg0", [T, K], arg, w, s, t)

    gate, up = dot("%arg1"), dot("%arg2")
    one = mm._splat(f, 1.0, s, t)
    ex = mm._named(f, "exp", [mm._named(f, "negf", [gate], [ty], s, t)], [ty], s, t)
    sig = mm._binary(f, "div", one, mm._binary(f, "add", one, ex, s, t), s, t)
    out = mul(mul(sig, gate), up)
    res = [out] + ([] if keep is None else [{"gate": gate, "sig": sig, "up": up}[keep]])
    return mm._module([mm.ttype([T, K], t), mm.ttype(w, t), mm.ttype(w, t)], [ty] * len(res), f, res)


@pytest.mark.parametrize("kw,one_step", [
    ({}, True), ({"swap": True}, True), ({"T": 1000}, True), ({"T": 100, "N": 8188}, True), ({"K": 1032}, True),
    ({"keep": "gate"}, False), ({"keep": "up"}, False), ({"keep": "sig"}, False),  # a value that somebody else reads
    ({"tb": False}, False), ({"K": 1020}, False), ({"N": 4098}, False),            # layouts without a kernel
    ({"N": 1024}, False),                                                          # few weights
    ({"T": 360, "K": 5120, "N": 1024}, False),                                     # few tiles, a long K: K slices are ahead
])
def test_gate(ga, mm, kw, one_step):
    st, plan = ga.explain_mlir(_gate(mm, **kw))
    assert st == 0, plan
    assert ("MatMul x2 + Sigmoid+Multiply+Multiply fused" in plan) == one_step, plan
    assert plan.count("gemm_bf16:") == (1 if one_step else 2)
