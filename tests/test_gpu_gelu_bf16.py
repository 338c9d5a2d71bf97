"""GELU of a bf16 GEMM's epilogue for every finite bf16 value: the product with the identity is the value itself."""
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
