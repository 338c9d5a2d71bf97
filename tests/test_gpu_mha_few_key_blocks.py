"""Masked attention over one or two key blocks runs without the pass that classifies the mask's tiles: the bits of the calls that
have classes, on both sides of the line and with masks that leave rows, tiles and single entries out; and no key block that
the mask hides from a workgroup is looked at, whichever way it is found."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("H,Sq,Sk", [(3, 128, 64), (3, 130, 129), (3, 200, 256), (3, 256, 256), (3, 256, 257), (3, 385, 385),
                                     (128, 128, 128), (129, 128, 128), (32, 256, 256), (33, 200, 256)])
@pytest.mark.parametrize("kind", ["causal", "zero", "tiles", "values"])
def test_the_bits_of_the_classified_call(gc, dev, D, H, Sq, Sk, kind):
    g = torch.Generator(device=dev).manual_seed(H + Sq + Sk)
    q, k, v = (torch.randn(2, H, s, D, device=dev, generator=g).bfloat16() for s in (Sq, Sk, Sk))
    mask = torch.zeros(Sq, Sk, device=dev)
    if kind == "causal":
        mask = torch.triu(torch.full((Sq, Sk), float("-inf"), device=dev), diagonal=1 + max(0, Sk - Sq))
    elif kind == "tiles":  # whole tiles of -inf, never a whole row
        mask[:, 64:192] = float("-inf")
        mask[:, Sk - 1] = 0.0
    elif kind == "values":
        mask = torch.randn(Sq, Sk, device=dev, generator=g)
        mask[5, 3:] = float("-inf")
    out = gc.mha_fwd_bf16(q, k, v, mask)
    classes = gc.mha_mask_classes(mask, Sq, Sk, D)
    assert classes is not None
    assert torch.equal(out, gc.mha_fwd_bf16_classified(q, k, v, mask, classes))
    assert torch.equal(out, gc.mha_fwd_bf16(q, k, v, mask, skip_masked=False))
    s = q.double() @ k.double().transpose(-1, -2) * D ** -0.5 + mask.double()
    ref = torch.softmax(s, -1) @ v.double()
    # weights and result rounded to bf16 (2^-9 each), the exponentials' own error far below
    mag = torch.softmax(s, -1) @ v.double().abs() + ref.abs()
    assert ((out.double() - ref).abs() <= 2.0 ** -8 * mag + 1e-6).all()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("BH", [3, 300])
@pytest.mark.parametrize("Sq,Sk", [(256, 128), (200, 128), (256, 192), (256, 256), (300, 320)])
@pytest.mark.parametrize("hidden", [0, 1])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_keys_hidden_from_all_rows_may_hold_anything(gc, dev, D, BH, Sq, Sk, hidden, bad):
    """The first workgroup's rows see all keys but one whole block, the others see that block too."""
    g = torch.Generator(device=dev).manual_seed(Sq + Sk)
    q, k, v = (torch.randn(1, BH, s, D, device=dev, generator=g).bfloat16() for s in (Sq, Sk, Sk))
    mask = torch.zeros(Sq, Sk, device=dev)
    mask[:128, 64 * hidden:64 * hidden + 64] = float("-inf")
    mask[3, 64 * (1 - hidden) + 7] = float("-inf")
    clean = gc.mha_fwd_bf16(q, k, v, mask)
    assert clean.isfinite().all()
    k[:, :, 64 * hidden:64 * hidden + 64] = bad
    v[:, :, 64 * hidden:64 * hidden + 64] = bad
    out = gc.mha_fwd_bf16(q, k, v, mask)
    seen = min(128, Sq - 128)  # (a last workgroup that would stick out takes the last 128 rows, here from `seen` on)
    assert torch.equal(out[:, :, :seen], clean[:, :, :seen])
    assert out[:, :, 128:].isnan().all()
    classes = gc.mha_mask_classes(mask, Sq, Sk, D)
    assert torch.equal(out[:, :, :seen], gc.mha_fwd_bf16_classified(q, k, v, mask, classes)[:, :, :seen])
