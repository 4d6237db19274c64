"""Tiles whose fills of LDS take whole 128-byte lines of memory (gemm_kernel.h: Form), as calls without a tile reach them: rows
off lines but on 16-byte chunks.  Shapes end inside a tile in both directions; K is one chunk, ends with and just behind a K tile,
has fewer K tiles than groups and slots, and many; rows take every phase (an operand may itself start behind a line).  Operands
lie inside buffers of NaNs.  That the calls reach those tiles is a test of its own.  Bounds: close_enough's."""
import ctypes

import numpy as np
import pytest

from test_gpu_edges import close_enough
from test_gpu_gemm import BF16, F16
from test_gpu_kwave import silu_pair
from test_gpu_ln import check_ln, make_ln_inputs, run_ln
from test_gpu_unaligned import run
from test_host_logic import small_tile

pytestmark = pytest.mark.gpu

KS = [8, 56, 72, 136, 328, 1096, 2008, 3208]
# A shape for each tile, its choice for K from 1096 on
TILES = {(64, 64): (1000, 1000), (96, 64): (2913, 464), (64, 128): (329, 4648), (128, 64): (1271, 1592), (96, 128): (1477, 2024),
         (128, 128): (399, 7968), (160, 128): (633, 6536), (192, 128): (760, 6536)}


def off_lines_tile(beamc, M, N, K, plan="beam_dbg_off_lines_tile"):
    tile, lines = beamc._TileCfg(), ctypes.c_int()
    beamc._check(getattr(beamc.lib, plan)(M, N, K, ctypes.byref(tile), ctypes.byref(lines)))
    return (tile.block_m, tile.block_n), lines.value


def test_calls_reach_the_tiles_that_they_are_named_after(gpu, beamc):
    assert gpu["compute_units"] == 256
    for tile, (M, N) in TILES.items():
        for K in (K for K in KS if K >= 1096):
            assert small_tile(beamc, 0, M, N, K, 1)[0] == 0 and off_lines_tile(beamc, M, N, K) == (tile, 1), (tile, K)


@pytest.mark.parametrize("tile", sorted(TILES))
@pytest.mark.parametrize("K", KS)
def test_gemmrc(gpu, beamc, oracle, tile, K):
    L = beamc.lib
    M, N = TILES[tile]
    dtype, offsets = ((F16, (0, 0, 0)), (BF16, (8, 24, 1)), (F16, (24, 16, 3)), (BF16, (0, 8, 0)))[KS.index(K) % 4]
    a, b = beamc.host_uniform((M, K), dtype, 71, 0), beamc.host_uniform((N, K), dtype, 71, 1)
    out = run(beamc, lambda pa, pb, pc: L.beam_gemmrc(pa, pb, pc, M, N, K, dtype, None, None), a, b, (M, N), dtype, offsets)
    close_enough(oracle, out, oracle.gemmrc(a, b, dtype), K, dtype, f"{tile} {(M, N, K)} at {offsets}")


# GEMM+LayerNorm: a shape for each tile, K off lines and on them; the last two have more tiles than CUs
LN_TILES = {(96, 64): (1064, 1040, 1480), (64, 128): (163, 6232, 2056), (128, 64): (1240, 1592, 2008),
            (96, 128): (449, 4352, 968), (128, 128): (399, 7968, 2056), (160, 128): (795, 5016, 744), (192, 128): (2912, 2008, 1680)}


def test_layernorm_reaches_them(gpu, beamc):
    for tile, shape in LN_TILES.items():
        assert off_lines_tile(beamc, *shape, "beam_dbg_ln_line_tile") == (tile, 1), (tile, shape)


@pytest.mark.parametrize("dtype", [F16, BF16])
@pytest.mark.parametrize("tile", sorted(LN_TILES))
def test_layernorm(gpu, beamc, oracle, tile, dtype):
    M, N, K = LN_TILES[tile]
    for k in (K, (K + 63) // 64 * 64):
        a, b, g, bt = make_ln_inputs(beamc, M, N, k, dtype, 72)
        ref = oracle.gemmrc_ln(a, b, g, bt, 1e-5, dtype)
        for mode in (beamc.LN_AUTO, beamc.LN_FUSED):
            check_ln(oracle, run_ln(beamc, a, b, g, bt, dtype, mode=mode), ref, dtype, f"{tile} {(M, N, k)} mode {mode}")


# [K][N]: shapes that reach each tile, B's rows of whole chunks and not
NN_TILES = [((64, 64), (155, 4720, 360)), ((64, 64), (2086, 368, 2632)), ((64, 128), (655, 2896, 432)), ((96, 64), (714, 1432, 200)),
            ((96, 64), (860, 1229, 2312)), ((96, 64), (215, 5103, 952)), ((96, 128), (2197, 1384, 2120)), ((96, 128), (551, 3597, 4784)),
            ((128, 128), (723, 3752, 376)), ((128, 128), (2472, 1152, 600)), ((160, 128), (1428, 3456, 336)), ((160, 128), (3677, 1242, 1232)),
            ((192, 128), (1296, 4320, 1136)), ((192, 128), (1713, 3017, 1688))]


def nn_tile(beamc, M, N, K):
    named, _ = beamc.default_config(M, N, K)
    named, tile, lines = named.to_c(), beamc._TileCfg(), ctypes.c_int()
    beamc._check(beamc.lib.beam_dbg_nn_off_lines_tile(M, N, K, ctypes.byref(named), ctypes.byref(tile), ctypes.byref(lines)))
    return (tile.block_m, tile.block_n), lines.value


def test_matmul_nn_reaches_them(gpu, beamc):
    for tile, (M, N, K) in NN_TILES:
        assert small_tile(beamc, 1, M, N, K, 1)[0] == 0 and nn_tile(beamc, M, N, K) == (tile, 1), (tile, (M, N, K))


@pytest.mark.parametrize("tile,shape", NN_TILES)
def test_matmul_nn(gpu, beamc, oracle, tile, shape):
    L = beamc.lib
    M, N, K = shape
    for dtype, offsets in ((F16, (0, 0, 0)), (BF16, (8, 3, 1))):
        a, b = beamc.host_uniform((M, K), dtype, 73, 0), beamc.host_uniform((K, N), dtype, 73, 1)
        out = run(beamc, lambda pa, pb, pc: L.beam_matmul_nn(pa, pb, pc, M, N, K, dtype, None, None), a, b, (M, N), dtype, offsets)
        close_enough(oracle, out, oracle.matmul_nn(a, b, dtype), K, dtype, f"[K][N] {tile} {(M, N, K)} at {offsets}")


@pytest.mark.parametrize("M,N,K", [(5681, 57, 2008), (3817, 364, 880), (860, 1229, 2312), (714, 1432, 200)])
def test_infinities_of_b_reach_their_columns_only(gpu, beamc, M, N, K):
    """The rows of B behind the last K tile of the loop, and at both ends of K, meet only their own elements of A."""
    a, b = beamc.host_uniform((M, K), F16, 74, 0), beamc.host_uniform((K, N), F16, 74, 1)
    rows = [0, 63, 64, K // 2, K - 9, K - 8, K - 1]
    for i, k in enumerate(rows):
        a[:, k], b[k, 2 * i] = 0x3C00, 0x7C00  # one, infinity
    out = run(beamc, lambda pa, pb, pc: beamc.lib.beam_matmul_nn(pa, pb, pc, M, N, K, F16, None, None), a, b, (M, N), F16, (0, 0, 0)).view(np.float16)
    cols = [2 * i for i in range(len(rows))]
    assert (out[:, cols] == np.inf).all() and np.isfinite(np.delete(out, cols, axis=1)).all()


@pytest.mark.parametrize("offset", [0, 1, 3])
@pytest.mark.parametrize("M,N,K", [(16500, 57, 616), (16500, 63, 336), (16500, 9, 2008), (16500, 58, 616), (33000, 65, 616), (33000, 127, 1112),
                                   (48000, 121, 2008), (5681, 57, 2008)])
def test_the_row_behind_the_last_that_is_fetched_stays_out(gpu, beamc, M, N, K, offset):
    """All columns in one tile, rows of B not whole chunks: the descriptor of the last K tile ends with row K - 9 (an odd one an element
    further on), inside a K tile, and A's elements behind it are zeros there.  Row K - 8 is infinite where a fetch beyond would begin;
    times those zeros it would be NaN.  B starts on chunks and one and three elements off.  (The last shape has small tiles.)"""
    assert small_tile(beamc, 1, M, N, K, 1)[0] or (N <= nn_tile(beamc, M, N, K)[0][1] and nn_tile(beamc, M, N, K)[1] == 1)
    assert (K - 8) % 64 != 0
    a, b = beamc.host_uniform((M, K), F16, 76, 0), beamc.host_uniform((K, N), F16, 76, 1)
    a[:, K - 8], b[K - 8, :2] = 0x3C00, 0x7C00  # one, infinity
    out = run(beamc, lambda pa, pb, pc: beamc.lib.beam_matmul_nn(pa, pb, pc, M, N, K, F16, None, None), a, b, (M, N), F16, (0, offset, 0)).view(np.float16)
    assert (out[:, :2] == np.inf).all() and np.isfinite(out[:, 2:]).all()


@pytest.mark.parametrize("M,N,K", [(1100, 1000, 1096), (929, 1232, 200), (1478, 2024, 2008)])
def test_infinities_stay_in_their_row_or_column(gpu, beamc, M, N, K):
    a, b = beamc.host_uniform((M, K), F16, 75, 0), beamc.host_uniform((N, K), F16, 75, 1)
    for i, k in enumerate([0, 7, 8, 63, 64, K // 2, K - 1]):
        a[10 * i, k], b[10 * i + 5, k] = 0xFC00, 0x7C00
    out = run(beamc, lambda pa, pb, pc: beamc.lib.beam_gemmrc(pa, pb, pc, M, N, K, F16, None, None), a, b, (M, N), F16, (0, 0, 0)).view(np.float16)
    assert not np.isfinite(out[0:70:10]).any() and not np.isfinite(out[:, 5:75:10]).any()
    assert np.isfinite(np.delete(np.delete(out, range(0, 70, 10), axis=0), range(5, 75, 10), axis=1)).all()


@pytest.mark.parametrize("M,N,K,count", [(566, 3648, 1304, (1 << 20) - 8), (566, 3648, 1304, 1 << 20), (679, 3080, 4880, 4096),
                                         (1602, 2624, 320, 10 << 20), (2176, 2176, 256, 3 << 20), (3072, 3072, 256, 60 << 18)])
def test_silu_job_beside(gpu, beamc, oracle, M, N, K, count):
    """An elementwise job on either side of the lines from which it gets a launch of its own: by whole lines, behind the loop."""
    a, b = beamc.host_uniform((M, K), BF16, 74, 0), beamc.host_uniform((N, K), BF16, 74, 1)
    silu_pair(beamc, oracle, a, b, oracle.gemmrc(a, b, BF16), BF16, count)
