"""GPU: the bf16 rounding of generated kernels -- four values at a time with one NaN check per pair, rows loaded ahead of
their use -- gives the library kernels' bits where it can go wrong: NaNs of either sign with payloads at each of the four
places, infinities, denormals, rows of one step and of an incomplete last step."""
import importlib

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _run(ga, text, ins, out):
    comp = ga.Compiler()
    try:
        st, exe = comp.compile_mlir(text)
        assert st == 0, ga.api().dnnl_graph_compiler_last_error().decode()
        try:
            assert exe.execute(list(enumerate(ins)), [(len(ins), out)]) == 0
            torch.cuda.synchronize()
        finally:
            exe.close()
    finally:
        comp.close()
    return out


@pytest.mark.parametrize("kind", ["rmsnorm", "layernorm"])
@pytest.mark.parametrize("rows,hidden", [(3, 128), (600, 132), (5, 1028), (9, 4096), (700, 4100), (2, 8192)])
def test_special_values_generated_equals_library(gc, dev, monkeypatch, kind, rows, hidden):
    ga = importlib.import_module("graph_compiler_amd.graph_api")
    mm = importlib.import_module("graph_compiler_amd.mlir_modules")
    rng = np.random.default_rng(rows * hidden)
    bits = torch.from_numpy(rng.standard_normal((rows, hidden)).astype(np.float32)).bfloat16().view(torch.int16).numpy().view(np.uint16)
    bits[0] = 0x3F80  # a row of ones; row 1 holds one special value at each place of a quad (the row becomes NaN or 0)
    for place, special in enumerate((0xFFA1, 0x7F80, 0x0001, 0x7FC5)):
        bits[1, 4 * (hidden // 8) + place] = special
    x = torch.from_numpy(bits.view(np.int16).copy()).view(torch.bfloat16).to(dev)
    w = (1 + 0.1 * torch.randn(hidden, device=dev)).bfloat16()
    w[1::37] = float("nan")  # an element's own NaN, its row finite
    w[2::41] = -float("inf")
    w[3::43] = 1e-39
    if kind == "rmsnorm":
        text, ins, shape = mm.rmsnorm(rows, hidden), [x[None], torch.full((1,), 1e-5, device=dev), w], (1, rows, hidden)
    else:
        text, ins, shape = mm.layernorm(rows, hidden, "bf16"), [x, w, w.flip(0).contiguous()], (rows, hidden)
    outs = []
    for mode in ("GCMI_GENERATED_KERNELS_REQUIRED", "GCMI_NO_GENERATED_KERNELS"):
        with monkeypatch.context() as m:
            m.setenv(mode, "1")
            before = ga.generated_kernel_launches()
            outs.append(_run(ga, text, ins, torch.full(shape, 7.0, device=dev, dtype=torch.bfloat16)))
            assert (ga.generated_kernel_launches() > before) == (mode == "GCMI_GENERATED_KERNELS_REQUIRED")
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))
    assert torch.isnan(outs[0].view(rows, hidden)[1]).any() and not torch.isnan(outs[0].view(rows, hidden)[0, :1]).any()
