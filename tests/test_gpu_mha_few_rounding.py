"""Attention of fewer than 128 queries rounds its weights to bf16 relative to the running maximum of whole 64-key blocks,
as the kernel for more queries does: what its waves share among themselves does not show in the results."""
import ctypes as C
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _blockwise(Q, K, V, mask, scale):
    """float64 but for the one rounding that is meant: the weights of a block of 64 keys, relative to the maximum so far."""
    S = torch.matmul(Q.double(), K.double().transpose(-1, -2).contiguous()) * (scale * math.log2(math.e))
    if mask is not None:
        S = S + mask.double() * math.log2(math.e)
    m = torch.full(S.shape[:-1] + (1,), float("-inf"), device=S.device, dtype=torch.float64)
    o, l = torch.zeros(Q.shape, device=S.device, dtype=torch.float64), torch.zeros_like(m)
    for k in range(0, S.shape[-1], 64):
        s = S[..., k:k + 64]
        m_new = torch.maximum(m, s.amax(-1, keepdim=True))
        m_use = torch.where(m_new == float("-inf"), torch.zeros_like(m_new), m_new)
        alpha, p = torch.exp2(m - m_use), torch.exp2(s - m_use)
        l = l * alpha + p.sum(-1, keepdim=True)
        o = o * alpha + torch.matmul(p.to(torch.float32).to(torch.bfloat16).double(), V[..., k:k + 64, :].double())
        m = m_new
    return (o / l).to(torch.float32).to(torch.bfloat16)


@pytest.mark.parametrize("Sq,Sk", [(1, 4096), (1, 4095), (7, 1000), (31, 777), (100, 321), (2, 97), (1, 33)])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("masked", [False, True])
def test_weights_are_rounded_against_the_blockwise_maximum(gc, dev, Sq, Sk, D, masked):
    BH = 24
    g = torch.Generator(device=dev).manual_seed(Sq + Sk)
    Q, K, V = (torch.randn(1, BH, s, D, device=dev, generator=g).to(torch.bfloat16) for s in (Sq, Sk, Sk))
    mask = None
    if masked:
        mask = torch.randn(Sq, Sk, device=dev, generator=g)
        mask[torch.rand(Sq, Sk, device=dev, generator=g) < 0.3] = float("-inf")
        mask[:, Sk // 2] = 0
    out = torch.empty_like(Q)
    # no workspace: the keys of a head stay in one workgroup
    rc = gc.lib().gcmi_mha_fwd_bf16_ws(Q.data_ptr(), K.data_ptr(), V.data_ptr(), None if mask is None else mask.data_ptr(), Sk,
                                       out.data_ptr(), BH, Sq, Sk, D, D ** -0.5, 1, None, 0,
                                       C.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, gc.lib().gcmi_last_error().decode()
    ref = _blockwise(Q, K, V, mask, D ** -0.5)
    # What remains are the f32 sums: about 2^-21 of the sum of magnitudes, which is up to 32 times a result (4096 terms of
    # either sign), so of 2^-8-wide rounding intervals at most 2 * 2^-21 * 32 / 2^-8, under 1 %, end on the other side.
    # Weights rounded against any other maximum differ by up to 2^-8 each: a third of all results and more then differ.
    assert (out != ref).double().mean().item() <= 0.03
