"""A row kernel that adds the K slices of the GEMM before it gives the bits of the GEMM's second pass and the row kernel of the
library: the second half of a decoder layer, both of whose norms follow a GEMM with a residual."""
import importlib

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mm(gc):
    return importlib.import_module("graph_compiler_amd.mlir_modules")


def _inputs(dev, T, H, F):
    g = torch.Generator(device=dev).manual_seed(T + H + F)
    r = lambda std, *shape: (torch.randn(*shape, device=dev, generator=g) * std).bfloat16()  # noqa: E731
    eps = torch.full((1,), 1e-5, device=dev)
    return [r(1, 1, T, H), r(H ** -0.5, H, H), r(1, 1, T, H), eps, 1 + r(0.1, H), r(H ** -0.5, F, H), r(H ** -0.5, F, H),
            r(F ** -0.5, H, F), eps.clone(), 1 + r(0.1, H)]


def _run(ga, text, ins, T, H):
    full = [torch.full((T + 1, H), 7.0, device=ins[0].device, dtype=torch.bfloat16) for _ in range(2)]
    comp = ga.Compiler()
    st, exe = comp.compile_mlir(text)
    assert st == 0, ga.api().dnnl_graph_compiler_last_error().decode()
    try:
        outs = [(10 + i, f[:T].view(1, T, H)) for i, f in enumerate(full)]
        call = exe.bind(list(enumerate(ins)), outs, torch.cuda.current_stream().cuda_stream)
        for _ in range(2):
            assert call() == 0
        torch.cuda.synchronize()
    finally:
        exe.close()
        comp.close()
    assert all((f[T] == 7.0).all() for f in full)
    return [f[:T].clone() for f in full]


# two rows and more (of one row the residual is a bias to the planner, and the GEMM adds its slices itself), 4 and 8 slices of the weight stream; slices of tiles; a K that ends inside a group; rows off 512 and 1024
# elements, one and several to a workgroup
@pytest.mark.parametrize("T,H,F,special", [(2, 2048, 2560, False), (32, 2048, 5632, True), (32, 4096, 1024, False), (50, 4100, 4096, False),
                                           (100, 2048, 2560, False), (200, 2056, 8200, True), (300, 776, 6152, False),
                                           (520, 1024, 8192, True), (600, 1000, 9000, False), (1024, 512, 12288, False)])
def test_bits(ga, mm, dev, monkeypatch, T, H, F, special):
    text = mm.decoder_mlp_block(T, H, F)
    st, plan = ga.explain_mlir(text)
    assert st == 0 and "K slices of the GEMM before it" in plan, plan
    ins = _inputs(dev, T, H, F)
    if special:  # infinities and a NaN in single rows
        ins[0][0, 0, 0], ins[2][0, T // 2, 5], ins[2][0, T - 1, H - 1] = float("inf"), float("nan"), float("-inf")
    got = _run(ga, text, ins, T, H)
    monkeypatch.setenv("GCMI_NO_GENERATED_KERNELS", "1")
    assert "K slices of the GEMM before it" not in ga.explain_mlir(text)[1]
    want = _run(ga, text, ins, T, H)
    for a, b in zip(got, want):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))


def test_bits_of_one_row(ga, mm, dev, monkeypatch):
    text, ins = mm.decoder_mlp_block(1, 2048, 2560), _inputs(dev, 1, 2048, 2560)
    got = _run(ga, text, ins, 1, 2048)
    monkeypatch.setenv("GCMI_NO_GENERATED_KERNELS", "1")
    for a, b in zip(got, _run(ga, text, ins, 1, 2048)):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))


def test_a_residual_off_16_bytes_takes_the_second_pass(ga, mm, dev):
    T, H, F = 32, 2048, 1024
    text, ins = mm.decoder_mlp_block(T, H, F), _inputs(dev, T, H, F)
    want = _run(ga, text, ins, T, H)
    off = torch.empty(T * H + 4, device=dev, dtype=torch.bfloat16)[4:].view(1, T, H)
    off.copy_(ins[2])
    ins[2] = off
    for a, b in zip(_run(ga, text, ins, T, H), want):
        assert torch.allclose(a.float(), b.float(), rtol=2.0 ** -6, atol=2.0 ** -6)  # another kernel's sums: a rounding or two apart


@pytest.mark.parametrize("which", ["residual", "operand", "weights of the gate"])
def test_operands_off_16_bytes_keep_the_generated_kernels(ga, mm, dev, monkeypatch, which):
    """The norm behind a GEMM that added its slices itself or ran in one pass, the point-wise group of a gate run in parts."""
    T, H, F = 32, 2048, 2048
    text, ins = mm.decoder_mlp_block(T, H, F), _inputs(dev, T, H, F)
    before = ga.generated_kernel_launches()
    _run(ga, text, ins, T, H)
    per_call = ga.generated_kernel_launches() - before
    at = {"residual": 2, "operand": 0, "weights of the gate": 5}[which]
    off = torch.empty(ins[at].numel() + 4, device=dev, dtype=torch.bfloat16)[4:].view(ins[at].shape)
    off.copy_(ins[at])
    ins[at] = off
    before = ga.generated_kernel_launches()
    got = _run(ga, text, ins, T, H)
    assert ga.generated_kernel_launches() - before == per_call + (2 if at == 5 else 0)
    monkeypatch.setenv("GCMI_NO_GENERATED_KERNELS", "1")
    for a, b in zip(got, _run(ga, text, ins, T, H)):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
