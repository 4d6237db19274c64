"""Tiles whose K tiles are dealt to groups of wavefronts: fewer K tiles than groups, counts that the groups share
unevenly, and a short last K tile.  Bound: close_enough's, the one of every other GEMM test."""
import numpy as np
import pytest

from test_gpu_edges import close_enough
from test_gpu_gemm import F16, BF16
from test_gpu_unaligned import run

pytestmark = pytest.mark.gpu

DEEP_GROUP_TILES = [(64, 64, 32, 32), (128, 64, 64, 32), (64, 128, 32, 64)]


@pytest.mark.parametrize("K", [8, 64, 65, 128, 136, 192, 257, 320, 585])
@pytest.mark.parametrize("tile", DEEP_GROUP_TILES)
def test_deep_tiles(gpu, beamc, oracle, tile, K):
    import ctypes
    L = beamc.lib
    cfg = beamc.TileConfig(*tile, 2, 0).to_c()
    for (M, N), dtype in (((130, 72), F16), ((33, 129), BF16)):
        a, b = beamc.host_uniform((M, K), dtype, 83, 0), beamc.host_uniform((N, K), dtype, 83, 1)
        bt = np.ascontiguousarray(b.T)
        ref = oracle.gemmrc(a, b, dtype)
        out = run(beamc, lambda pa, pb, pc: L.beam_gemmrc(pa, pb, pc, M, N, K, dtype, ctypes.byref(cfg), None), a, b, (M, N), dtype, (0, 0, 0))
        close_enough(oracle, out, ref, K, dtype, f"gemmrc {(M, N, K)}")
        nn = run(beamc, lambda pa, pb, pc: L.beam_matmul_nn(pa, pb, pc, M, N, K, dtype, ctypes.byref(cfg), None), a, bt, (M, N), dtype, (0, 0, 0))
        assert (nn == out).all(), f"[K][N] {(M, N, K)}: differs from [N][K]"
        for slices in (2, 3):
            ws = beamc.DeviceArray((L.beam_splitk_workspace_bytes(M, N, slices),), itemsize=1)
            out = run(beamc, lambda pa, pb, pc: L.beam_gemmrc_splitk(pa, pb, pc, M, N, K, dtype, ctypes.byref(cfg), slices, ws.ptr, ws.nbytes, None),
                      a, b, (M, N), dtype, (0, 0, 0))
            ws.free()
            close_enough(oracle, out, ref, K, dtype, f"split-K {(M, N, K)} in {slices}")


@pytest.mark.parametrize("M,N,K,dtype", [(33, 12225, 2048, F16), (64, 12289, 2112, BF16), (17, 14273, 2048, F16), (64, 14337, 2111, BF16), (33, 16383, 2112, F16)])
def test_one_row_of_tiles_that_nearly_fills_the_chip(gpu, beamc, oracle, M, N, K, dtype):
    """The library's own choice there is the deep pipeline as one group: gemmrc and split-K with one slice where K is a
    multiple of 64, [K][N] from 14273 columns on."""
    L = beamc.lib
    cfg, _ = beamc.default_config(M, N, K)
    assert (cfg.block_m, cfg.block_n, cfg.pipeline) == (64, 64, 2)
    a, b = beamc.host_uniform((M, K), dtype, 84, 0), beamc.host_uniform((N, K), dtype, 84, 1)
    ref = oracle.gemmrc(a, b, dtype)
    for what, bb, call in (("gemmrc", b, lambda pa, pb, pc: L.beam_gemmrc(pa, pb, pc, M, N, K, dtype, None, None)),
                           ("split-K", b, lambda pa, pb, pc: L.beam_gemmrc_splitk(pa, pb, pc, M, N, K, dtype, None, 1, None, 0, None)),
                           ("[K][N]", np.ascontiguousarray(b.T), lambda pa, pb, pc: L.beam_matmul_nn(pa, pb, pc, M, N, K, dtype, None, None))):
        out = run(beamc, call, a, bb, (M, N), dtype, (0, 0, 0))
        close_enough(oracle, out, ref, K, dtype, f"{what} {(M, N, K)}")


@pytest.mark.parametrize("M,N,K,deep", [(1030, 1000, 704, False), (1030, 1000, 768, True), (1030, 1000, 775, True), (2048, 1024, 1100, True),
                                        (1000, 1040, 2047, True)])
def test_one_round_of_half_tiles(gpu, beamc, oracle, M, N, K, deep):
    """Tiles of 64x128 and 128x64 that fill at most one round of workgroups: two K groups from K = 768 on, in both layouts."""
    L = beamc.lib
    cfg, _ = beamc.default_config(M, N, K)
    assert cfg.block_m * cfg.block_n == 128 * 64 and (cfg.pipeline == 2) == deep, cfg
    for dtype in (F16, BF16):
        a, b = beamc.host_uniform((M, K), dtype, 85, 0), beamc.host_uniform((N, K), dtype, 85, 1)
        ref = oracle.gemmrc(a, b, dtype)
        for what, bb, call in (("gemmrc", b, L.beam_gemmrc), ("[K][N]", np.ascontiguousarray(b.T), L.beam_matmul_nn)):
            out = run(beamc, lambda pa, pb, pc: call(pa, pb, pc, M, N, K, dtype, None, None), a, bb, (M, N), dtype, (0, 0, 0))
            close_enough(oracle, out, ref, K, dtype, f"{what} {(M, N, K)}")
