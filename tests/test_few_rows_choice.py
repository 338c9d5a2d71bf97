"""Which GEMMs of few rows take the kernel that cuts K over the waves of a workgroup, and with which tile (asked of the
launcher, no GPU needed)."""
import pytest


@pytest.mark.parametrize("M,N,K,kernel,bm,bn", [
    (1, 640, 576, 7, 16, 16), (31, 4096, 4032, 7, 32, 16), (31, 4200, 4032, 7, 32, 32), (17, 16384, 200, 7, 32, 64),
    (31, 4096, 4096, 4, 32, 64), (31, 1000, 136, 2, 256, 256),          # a stream of weights; a short K
    (46, 192, 2792, 7, 16, 16), (62, 1208, 3432, 7, 32, 16), (64, 4096, 1000, 7, 32, 32), (64, 4096, 4072, 7, 32, 32),
    (32, 4096, 1376, 7, 32, 16), (32, 2048, 1016, 7, 16, 16), (33, 2048, 1024, 7, 16, 32), (128, 1288, 200, 7, 32, 32), (129, 1024, 4072, 7, 32, 32), (140, 264, 1048, 7, 16, 16),
    (31, 4096, 1376, 7, 32, 16), (33, 4096, 1376, 7, 32, 32), (32, 1024, 2816, 7, 16, 16), (128, 4096, 1376, 7, 64, 32), (129, 4096, 1376, 7, 64, 64), (256, 1024, 512, 7, 32, 32),
    (257, 1024, 512, 5, 128, 128), (64, 8208, 328, 7, 64, 64), (64, 8208, 256, 5, 128, 128), (96, 6000, 512, 5, 128, 128), (64, 8208, 520, 7, 64, 64)])
def test_bf16(gc, M, N, K, kernel, bm, bn):
    for tb in (False, True):
        c = gc.tile_config(M, N, K, trans_b=tb)[0]
        assert (c.kernel, c.bm, c.bn) == (kernel, bm, bn)
        if kernel == 7:  # one launch: no partial sums
            assert c.split_k == 1 and gc.lib().gcmi_gemm_bf16_workspace_bytes(M, N, K, int(tb)) == 0


@pytest.mark.parametrize("trans_b,M,N,K,kernel", [
    (0, 176, 192, 5888, 7), (0, 176, 192, 6016, 3), (0, 157, 40, 16384, 7), (0, 157, 40, 16512, 3), (0, 157, 24, 24576, 7), (0, 157, 24, 24704, 3),   # 16 x 16 tiles; few columns
    (0, 32, 3840, 4600, 7), (0, 32, 3840, 4616, 3), (0, 50, 2056, 4344, 7), (0, 50, 2056, 4360, 3), (0, 41, 4400, 4088, 7), (0, 41, 4400, 4104, 3),   # larger ones
    (0, 96, 3848, 3832, 7), (0, 96, 3848, 3848, 3), (0, 97, 6000, 3576, 7), (0, 97, 6000, 3592, 3),
    (0, 26, 512, 6144, 7), (0, 26, 512, 6272, 3), (0, 16, 96, 65408, 7), (0, 1, 16, 1000000, 7),        # below 32 rows; nobody cuts K
    (1, 192, 136, 16384, 7), (1, 192, 136, 16512, 3), (1, 192, 128, 23040, 7), (1, 192, 128, 23168, 3), (1, 121, 640, 13304, 7), (1, 121, 640, 13320, 3),
    (1, 128, 1504, 8824, 7), (1, 128, 1504, 8840, 3), (1, 32, 3840, 10232, 7), (1, 128, 3200, 5112, 7), (1, 128, 3200, 5128, 3),
    (1, 19, 224, 10240, 7), (1, 19, 224, 10304, 4), (1, 19, 216, 40000, 7), (1, 100, 6000, 3960, 7), (1, 100, 6000, 3976, 3),
    (0, 64, 64, 65408, 3), (1, 64, 64, 65408, 3), (0, 128, 64, 65408, 3), (0, 64, 512, 40008, 3), (1, 64, 512, 40008, 3)])
def test_a_long_k_is_left_to_slices(gc, trans_b, M, N, K, kernel):
    """Where another kernel cuts K over workgroups; it then has the workspace that it wants."""
    c = gc.tile_config(M, N, K, trans_b=bool(trans_b))[0]
    assert c.kernel == kernel and (c.split_k > 1) == (kernel != 7)
    assert (gc.lib().gcmi_gemm_bf16_workspace_bytes(M, N, K, trans_b) > 0) == (kernel != 7)


@pytest.mark.parametrize("M,N,K,kernel", [(1, 512, 512, 7), (32, 11008, 4096, 7), (256, 896, 2112, 7), (234, 10816, 3584, 5), (257, 3264, 4096, 7), (257, 3280, 4096, 5),
                                          (2048, 512, 528, 7), (2049, 512, 528, 5), (1024, 1024, 4096, 7), (1024, 1024, 4112, 5), (700, 496, 1024, 5),
                                          (300, 272, 512, 5), (32, 512, 272, 5), (20, 512, 520, 0)])
def test_int8(gc, M, N, K, kernel):
    for dt in (gc.U8, gc.S8):
        assert gc.tile_config(M, N, K, a_dtype=dt)[0].kernel == kernel


def test_a_matmul_config_names_another_kernel(gc):
    cfg = [1, 1, 1, 128, 128, 64, 64, 64, 32]
    assert gc.tile_config(40, 1024, 1024, matmul_config=cfg)[0].kernel == 5
