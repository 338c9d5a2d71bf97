"""f32 operands whose rows lie so far apart that a lane's place in a tile is no 32-bit offset, in all four layouts; on the line
the 32-bit form still runs."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu

LINE = (1 << 31) // 60  # 4 * (15 * stride + 15 + 1) reaches 2^31 bytes from here on (a little below, with the other stride's 15)


def _spread(values, ld):
    """The same matrix with rows `ld` elements apart, in memory that is otherwise not written."""
    flat = torch.empty((values.shape[0] - 1) * ld + values.shape[1], device=values.device)
    t = flat.as_strided(values.shape, (ld, 1))
    t.copy_(values)
    return t


@pytest.mark.parametrize("far_a,far_b", [(True, False), (False, True), (True, True)])
@pytest.mark.parametrize("ta", [False, True])
@pytest.mark.parametrize("tb", [False, True])
@pytest.mark.parametrize("ld", [LINE - 64, LINE + 64])
def test_rows_far_apart(gc, dev, far_a, far_b, ta, tb, ld):
    M, N, K = 21, 19, 43  # two tiles each way, a K that ends inside a step
    assert gc.tile_config(M, N, K, a_dtype=gc.F32)[0].bm == 16
    g = torch.Generator(device=dev).manual_seed(M)
    A, B = (torch.randint(-8, 9, s, device=dev, generator=g).float() for s in ((M, K), (K, N)))  # integers: exact sums
    a, b = A.t().contiguous() if ta else A, B.t().contiguous() if tb else B
    if far_a:
        a = _spread(a, ld)
    if far_b:
        b = _spread(b, ld)
    out = torch.full((M + 2, N), 7.0, device=dev)
    gc.check(gc.lib().gcmi_gemm_f32(a.data_ptr(), b.data_ptr(), out[1:].data_ptr(), M, N, K, a.stride(0), b.stride(0), N, int(ta), int(tb),
                                    None, 0, C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    assert torch.equal(out[1:M + 1].double(), A.double() @ B.double())
    assert (out[0] == 7.0).all() and (out[M + 1] == 7.0).all()
