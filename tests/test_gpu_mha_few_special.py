"""Infinities and NaN among the operands of attention with few queries: in the rows that they belong to, nowhere else."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("BH,Sk", [(2, 2049), (300, 300)])  # keys cut over workgroups, and whole
@pytest.mark.parametrize("D", [64, 128])
def test_special_values(gc, dev, BH, Sk, D):
    g = torch.Generator(device=dev).manual_seed(Sk)
    Q, K, V = (torch.randn(1, BH, s, D, device=dev, generator=g).to(torch.bfloat16) for s in (6, Sk, Sk))
    mask = torch.zeros(6, Sk, device=dev)
    mask[1, 5], mask[2, Sk - 1] = float("inf"), float("nan")
    mask[3, :64], mask[4, 40:] = float("-inf"), float("-inf")
    Q[0, 0, 0, 3], Q[0, BH - 1, 5, 0] = float("nan"), float("inf")
    K[0, 1, Sk - 2, 0] = float("nan")
    out = gc.mha_fwd_bf16(Q, K, V, mask)
    S = torch.matmul(Q.double(), K.double().transpose(-1, -2).contiguous()) * D ** -0.5 + mask.double()
    P = torch.softmax(S, -1)
    ref, mag = torch.matmul(P, V.double()), torch.matmul(P, V.double().abs())
    want = ref.isnan()
    assert want[:, :, 1].all() and want[:, :, 2].all() and want[0, 0, 0].all() and want[0, BH - 1, 5].all()
    # NaN in a key that a mask of -inf hides is NaN all the same; an infinite score weighs as softmax says: NaN
    assert torch.equal(out.isnan(), want)
    ok = ~want
    # a weight is rounded to bf16 (by at most 2^-8 of itself), so is the result; the scores' f32 sums move a weight by less than 2^-12
    assert ((out.double() - ref).abs()[ok] <= ((2.0 ** -8 + 2.0 ** -12) * mag + 2.0 ** -8 * ref.abs() + 1e-30)[ok]).all()
