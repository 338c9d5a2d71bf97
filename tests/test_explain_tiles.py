"""What a plan and the tile descriptor say about a kernel is what runs (planner only, no GPU)."""
import importlib
import re

import pytest

PAIRS, ALONE = "two workgroups per compute unit", "small tiles, 4 waves (one per SIMD)"


# (k-blocks in the ring: four with two workgroups on a compute unit; alone what 160 KiB hold of both operands, in pairs)
@pytest.mark.parametrize("M,N,K,trans_b,u8,tile,stages,words", [
    (2498, 2544, 512, False, False, (128, 128), 4, PAIRS), (1086, 144, 256, False, False, (128, 128), 4, PAIRS),
    (1000, 4096, 4096, True, False, (128, 128), 8, ALONE), (1000, 4096, 4096, False, False, (128, 128), 6, ALONE),
    (1237, 4096, 1376, True, False, (192, 128), 8, ALONE), (1237, 4096, 1376, False, False, (192, 128), 6, ALONE),
    (1000, 11008, 4096, True, False, (256, 192), 4, ALONE), (1000, 11008, 4096, False, False, (256, 192), 4, ALONE),
    (1024, 4096, 4096, False, True, (128, 128), 6, ALONE)])
def test_small_tiles(gc, ga, M, N, K, trans_b, u8, tile, stages, words):
    c, _ = gc.tile_config(M, N, K, trans_b=trans_b, a_dtype=gc.U8 if u8 else gc.BF16)
    assert (c.kernel, c.bm, c.bn, c.kbytes, c.stages) == (5, *tile, 64, stages)
    if not u8 and not trans_b:
        st, plan = ga.explain(ga.gemm_json(M, K, N))
        assert st == 0 and "tile: %s" % words in plan.replace("small tiles, 4 waves, two", "two"), plan


def test_slices_of_small_tiles(gc):
    assert gc.tile_config(129, 4096, 4096, trans_b=True)[0].stages == 8  # one workgroup per compute unit
    c, _ = gc.tile_config(300, 4096, 11008, trans_b=True)
    assert c.kernel == 3 and c.stages in (4, 6, 8)


@pytest.mark.parametrize("T,K,N,tile,stages", [
    (32, 4096, 11008, "32x44", 4), (64, 512, 16384, "64x64", 3), (100, 512, 8192, "128x32", 3), (100, 1024, 2816, "128x12", 4),
    (250, 512, 11008, "256x64", 6), (300, 640, 5632, "192x64", 8), (1000, 4096, 11008, "256x96", 4), (129, 512, 5632, "128x64", 8)])
def test_gate(ga, T, K, N, tile, stages):
    mm = importlib.import_module("graph_compiler_amd.mlir_modules")
    gate = importlib.import_module("test_gated_plan")._gate
    st, plan = ga.explain_mlir(gate(mm, T=T, K=K, N=N))
    line = re.search(r"tile: (.*), (\d+x\d+) per workgroup, (\d+) B of K per stage x (\d+) stages", plan)
    assert st == 0 and line, plan
    streams = T <= 128 and tile.startswith(("32x", "64x", "128x")) and K % 128 == 0 and "streaming" in line[1]
    assert line[1] == ("weight streaming" if streams else "whole tiles, 4 waves (one per SIMD)")
    assert (line[2], int(line[3]), int(line[4])) == (tile, 256 if streams else 64, stages), plan


def test_second_pass_of_a_streamed_weight(ga):
    plans = [ga.explain(ga.gemm_json(M, 4096, N))[1] for M, N in ((32, 4096), (16, 11008))]
    assert "weight streaming + second pass" in plans[0] and "split_k 4" in plans[0]
    assert "weight streaming, " in plans[1] and "second pass" not in plans[1]
