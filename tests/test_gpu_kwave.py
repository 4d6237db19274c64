"""Small workgroup tiles whose K range is dealt out to the wavefronts, as calls without a named tile reach them: every tile,
fewer K tiles than wavefronts (8x64, which is for K from 512 on, apart), K tiles that end inside a chunk, rows on and off 128-byte
lines (both ways of filling LDS), operands at any element's address inside buffers of NaNs.  That the calls reach those tiles is
a test of its own.  Bounds: close_enough's, the one of every other GEMM test."""
import ctypes

import numpy as np
import pytest

from test_gpu_edges import close_enough
from test_gpu_gemm import F16, BF16
from test_gpu_ln import check_ln, make_ln_inputs, run_ln
from test_gpu_unaligned import run
from test_host_logic import small_tile

pytestmark = pytest.mark.gpu

# The smallest tile of which the problem has at most 256: one shape for each, ragged in both directions where it can be.
TILES = {"8x16": (5, 300), "16x16": (41, 100), "16x32": (297, 400), "32x16": (1030, 100), "32x32": (509, 500), "8x64": (3, 8300),
         "16x64": (130, 1750), "32x64": (466, 864), "64x32": (1030, 475), "64x64": (1000, 1003)}
# one chunk, one K tile, fewer K tiles than wavefronts, several for each; from about 640 (64x64) to 2500 (16x16) on, rows off
# 128-byte lines are filled line by line
KS = [8, 9, 64, 71, 200, 513, 1096, 2057, 3208, 3265]


def starts(K):
    """Where the rows of an operand that itself starts on a line start (beam_dbg_small_tile)."""
    return 0 if K % 8 else 2 if K % 64 == 0 else 1


def test_calls_reach_the_tiles_that_they_are_named_after(gpu, beamc):
    for name, (M, N) in TILES.items():
        shape = tuple(map(int, name.split("x")))
        plans = {K: small_tile(beamc, 0, M, N, K, starts(K)) for K in KS}
        assert all(p[:2] == shape for K, p in plans.items() if name != "8x64" or K >= 512), (name, plans)
        assert {p[3] for p in plans.values()} == ({0, 1} if shape[0] > 8 else {0}), (name, plans)  # both ways of filling LDS
    reached = {small_tile(beamc, 1, M, N, K, starts(K)) for M, N in NN for K in KS}
    tiles = {t for t in (tuple(map(int, n.split("x"))) for n in TILES) if t[0] > 8}
    for lines in (0, 1):
        assert {p[:2] for p in reached if p[0] and p[3] == lines} == tiles, reached
    for name, (M, N) in LN_TILES.items():
        plans = {K: small_tile(beamc, 3, M, N, K, starts(K)) for K in (8, 71, 513, 1096, 3208, 3265)}
        shape = (16, 64) if name == "64 column tiles" else tuple(map(int, name.split("x")))
        # (64 x 64 under a short sum is the tiled kernel's)
        assert all(p[:2] == shape for K, p in plans.items() if name != "64x64" or K >= 600), (name, plans)
        assert plans[3208][3] == 1 and plans[3265][3] == 0, (name, plans)


@pytest.mark.parametrize("tile", sorted(TILES))
@pytest.mark.parametrize("K", KS)
def test_gemmrc(gpu, beamc, oracle, tile, K):
    assert gpu["compute_units"] == 256  # the shapes are chosen for that
    L = beamc.lib
    M, N = TILES[tile]
    for dtype, offsets in ((F16, (0, 0, 0)), (BF16, (1, 3, 1)), (F16, (8, 24, 0))):
        a, b = beamc.host_uniform((M, K), dtype, 94, 0), beamc.host_uniform((N, K), dtype, 94, 1)
        out = run(beamc, lambda pa, pb, pc: L.beam_gemmrc(pa, pb, pc, M, N, K, dtype, None, None), a, b, (M, N), dtype, offsets)
        close_enough(oracle, out, oracle.gemmrc(a, b, dtype), K, dtype, f"{tile} {(M, N, K)} at {offsets}")


# [K][N], rows of whole chunks and not
NN = [(41, 9), (60, 69), (466, 35), (87, 998), (1000, 1003), (41, 96), (297, 400), (1030, 104), (509, 504), (130, 1752), (466, 864),
      (1030, 472), (1000, 1000), (1, 4096)]


@pytest.mark.parametrize("M,N", NN)
@pytest.mark.parametrize("K", KS)
def test_matmul_nn(gpu, beamc, oracle, M, N, K):
    L = beamc.lib
    for dtype, offsets in ((F16, (0, 0, 0)), (BF16, (3, 1, 1))):
        a, b = beamc.host_uniform((M, K), dtype, 95, 0), beamc.host_uniform((K, N), dtype, 95, 1)
        out = run(beamc, lambda pa, pb, pc: L.beam_matmul_nn(pa, pb, pc, M, N, K, dtype, None, None), a, b, (M, N), dtype, offsets)
        close_enough(oracle, out, oracle.matmul_nn(a, b, dtype), K, dtype, f"[K][N] {(M, N, K)} at {offsets}")


# Full tiles of 64 x 64 whose rows of C are whole chunks: the tiled kernels' under a short sum, on both sides of every line
@pytest.mark.parametrize("K", [8, 256, 383, 384, 385, 1024, 1025, 1032, 1280, 1281, 1344, 1984, 2047])
@pytest.mark.parametrize("M,N", [(1000, 1000), (130, 5000)])
def test_full_tiles_under_a_short_sum(gpu, beamc, oracle, M, N, K):
    L = beamc.lib
    for dtype, offsets in ((F16, (0, 0, 0)), (BF16, (3, 1, 1))):
        a, b, bt = (beamc.host_uniform(s, dtype, 92, i) for i, s in enumerate(((M, K), (N, K), (K, N))))
        out = run(beamc, lambda pa, pb, pc: L.beam_gemmrc(pa, pb, pc, M, N, K, dtype, None, None), a, b, (M, N), dtype, offsets)
        close_enough(oracle, out, oracle.gemmrc(a, b, dtype), K, dtype, f"{(M, N, K)} at {offsets}")
        out = run(beamc, lambda pa, pb, pc: L.beam_matmul_nn(pa, pb, pc, M, N, K, dtype, None, None), a, bt, (M, N), dtype, offsets)
        close_enough(oracle, out, oracle.matmul_nn(a, bt, dtype), K, dtype, f"[K][N] {(M, N, K)} at {offsets}")


@pytest.mark.parametrize("M,N,K", [(16, 16, 4096), (41, 100, 8184), (300, 24, 4951), (500, 500, 4096)])
def test_split_k_of_a_short_sum(gpu, beamc, oracle, M, N, K):
    """Left to the library, a sum below 8192 over few outputs runs without slices, and needs no workspace."""
    L = beamc.lib
    assert L.beam_splitk_effective(M, N, K, None, 0) == 1 and L.beam_splitk_effective(M, N, K, None, 4) > 1
    for dtype, offsets in ((F16, (0, 0, 0)), (BF16, (3, 1, 1))):
        a, b = beamc.host_uniform((M, K), dtype, 93, 0), beamc.host_uniform((N, K), dtype, 93, 1)
        out = run(beamc, lambda pa, pb, pc: L.beam_gemmrc_splitk(pa, pb, pc, M, N, K, dtype, None, 0, None, 0, None), a, b, (M, N), dtype, offsets)
        close_enough(oracle, out, oracle.gemmrc(a, b, dtype), K, dtype, f"{(M, N, K)} at {offsets}")


@pytest.mark.parametrize("M,N,K", [(1024, 1024, 2048), (64, 16384, 1024)])
def test_split_k_needs_no_workspace_wherever_rows_start(gpu, beamc, oracle, M, N, K):
    """Rows on lines run on the tiled kernels there, rows off them in small tiles; the caller is told one slice for both."""
    L = beamc.lib
    assert L.beam_splitk_effective(M, N, K, None, 0) == 1
    assert small_tile(beamc, 2, M, N, K, 2)[0] == 0 and small_tile(beamc, 2, M, N, K, 1)[:2] == (64, 64)
    a, b = beamc.host_uniform((M, K), F16, 93, 0), beamc.host_uniform((N, K), F16, 93, 1)
    for offsets in ((0, 0, 0), (8, 24, 0)):
        out = run(beamc, lambda pa, pb, pc: L.beam_gemmrc_splitk(pa, pb, pc, M, N, K, F16, None, 0, None, 0, None), a, b, (M, N), F16, offsets)
        close_enough(oracle, out, oracle.gemmrc(a, b, F16), K, F16, f"{(M, N, K)} at {offsets}")


def test_infinities_and_nan_stay_in_their_row_or_column(gpu, beamc):
    """Rows that start anywhere: a chunk behind the end of K is a zero for every row."""
    M, N, K = 70, 90, 3001
    L = beamc.lib
    a, b = beamc.host_uniform((M, K), F16, 96, 0), beamc.host_uniform((N, K), F16, 96, 1)
    a[69, 3000], a[68, 0], b[88, 1500] = 0x7E00, 0xFC00, 0x7C00
    out = run(beamc, lambda pa, pb, pc: L.beam_gemmrc(pa, pb, pc, M, N, K, F16, None, None), a, b, (M, N), F16, (0, 0, 0)).view(np.float16)
    assert np.isnan(out[69]).all() and not np.isfinite(out[68]).any() and not np.isfinite(out[:, 88]).any()
    assert np.isfinite(np.delete(out[:68], 88, axis=1)).all()


@pytest.mark.parametrize("N", [88, 90])
def test_infinities_of_b_behind_the_whole_chunks(gpu, beamc, N):
    """[K][N]: a row of B behind K's last whole chunk meets only its own elements of A, never the zeros beside them."""
    M, K = 37, 75
    L = beamc.lib
    a, b = beamc.host_uniform((M, K), F16, 97, 0), beamc.host_uniform((K, N), F16, 97, 1)
    a[:, 73] = 0x3C00  # one
    b[73, 5], b[K - 1, 7], a[:, K - 1] = 0x7C00, 0xFC00, 0x3C00
    out = run(beamc, lambda pa, pb, pc: L.beam_matmul_nn(pa, pb, pc, M, N, K, F16, None, None), a, b, (M, N), F16, (0, 0, 0)).view(np.float16)
    assert (out[:, 5] == np.inf).all() and (out[:, 7] == -np.inf).all()
    assert np.isfinite(np.delete(out, (5, 7), axis=1)).all()


@pytest.mark.parametrize("M,N,K", [(70, 90, 3208), (70, 96, 3272), (300, 700, 2008), (466, 864, 1096), (1000, 1003, 1160)])
def test_infinities_by_whole_lines(gpu, beamc, M, N, K):
    """A fill of whole lines brings chunks of two K tiles, and each wavefront has a part of K in one piece: elements at both ends
    of K, on both sides of a line and of a wavefront's part reach every output of their row or column and no other."""
    L = beamc.lib
    assert small_tile(beamc, 0, M, N, K, 1)[3] == 1 and small_tile(beamc, 1, M, N, K, 1)[3] == 1
    waves, tiles = small_tile(beamc, 0, M, N, K, 1)[2], -(-K // 64)
    parts = {64 * (w * tiles // waves) for w in range(1, waves)}
    ks = sorted(k for k in {0, 7, 8, 63, 64, K - 65, K - 64, K - 9, K - 8, K - 1} | parts | {k - 1 for k in parts} if 0 <= k < K)
    a, b, bt = (beamc.host_uniform(s, F16, 96, i) for i, s in enumerate(((M, K), (N, K), (K, N))))
    rows, cols = sorted({0, M // 2, M - 1}), sorted({1, N // 2, N - 1})
    for k in ks:
        a1, b1, bt1 = a.copy(), b.copy(), bt.copy()
        a1[rows, k], b1[cols, k], bt1[k, cols] = 0x7E00, 0x7E00, 0x7E00  # NaN
        want = np.zeros((M, N), bool)
        want[rows, :] = want[:, cols] = True
        for offsets in ((0, 0, 0), (8, 24, 0)):
            for f, second in ((L.beam_gemmrc, b1), (L.beam_matmul_nn, bt1)):
                out = run(beamc, lambda pa, pb, pc: f(pa, pb, pc, M, N, K, F16, None, None), a1, second, (M, N), F16, offsets).view(np.float16)
                assert (np.isnan(out) == want).all() and np.isfinite(out[~want]).all(), (k, offsets)


@pytest.mark.parametrize("N", [9, 10, 15, 88, 90, 92, 1003])
@pytest.mark.parametrize("K", [9, 64, 75, 128, 200, 1032, 2000])
def test_infinities_in_the_last_rows_of_b(gpu, beamc, N, K):
    """[K][N]: a row of B behind the whole chunks meets only its own elements of A, never the zeros beside them.  With
    N % 8 != 0 the last row of B is always one of those (8 * ((K - 1) / 8) is the first), else those of K % 8."""
    M, L = 37, beamc.lib
    first = 8 * ((K - 1) // 8)
    rows = sorted({first, min(first + 1, K - 1), K - 1})
    a = beamc.host_uniform((M, K), F16, 97, 0)
    a[:, first:] = 0x3C00  # one
    for row in rows:
        for cols in ([0], [1], [2], [3], [4], [5], [6], [7], [N - 1], [0, 5, N - 1]):
            b = beamc.host_uniform((K, N), F16, 97, 1)
            b[row, cols] = 0x7C00
            for offsets in ((0, 0, 0), (1, 3, 1)):
                out = run(beamc, lambda pa, pb, pc: L.beam_matmul_nn(pa, pb, pc, M, N, K, F16, None, None), a, b, (M, N), F16, offsets).view(np.float16)
                assert (out[:, cols] == np.inf).all(), (row, cols, offsets)
                assert np.isfinite(np.delete(out, cols, axis=1)).all(), (row, cols, offsets)


# The elementwise job rides in workgroups of its own behind the tiles'.  Counts: a tail only, one access of one thread, ragged,
# more than one round of the accesses of every such workgroup.
@pytest.mark.parametrize("tile", ["8x16", "16x16", "32x32", "64x64"])
def test_silu_job(gpu, beamc, tile):
    L = beamc.lib
    M, N = TILES[tile]
    # (K above 512 for the large tile: under a shorter sum the job runs in the tiled kernel's K loop, test_silu_job_in_the_loop,
    # whose sums are added in another order than beam_gemmrc's)
    for K, dtype in ((520 if tile == "64x64" else 200, F16), (2600, BF16)):
        da, db = (beamc.DeviceArray.from_numpy(beamc.host_uniform(s, dtype, 97, i), dtype) for i, s in enumerate(((M, K), (N, K))))
        want, got = beamc.DeviceArray((M, N), dtype), beamc.DeviceArray((M, N), dtype)
        beamc._check(L.beam_gemmrc(da.ptr, db.ptr, want.ptr, M, N, K, dtype, None, None))
        for count in (0, 5, 8, 4099, 300007, (1 << 22) + 3):
            dx = beamc.DeviceArray.from_numpy(beamc.host_normal((max(count, 1) + 64,), dtype, 97, 2, 0.0, 2.5), dtype)
            y, alone = (beamc.DeviceArray((max(count, 1) + 64,), dtype) for _ in range(2))
            for d in (got, y, alone):
                d.fill_bytes(0xEE)
            beamc._check(L.beam_silu(dx.ptr, alone.ptr, count, dtype, None))
            beamc._check(L.beam_parallel_gemmrc_silu(da.ptr, db.ptr, got.ptr, M, N, K, dx.ptr, y.ptr, count, dtype, None, None))
            assert (got.to_numpy() == want.to_numpy()).all(), (tile, K, count)
            assert (y.to_numpy() == alone.to_numpy()).all(), (tile, K, count)  # the guard behind the array included
            for d in (dx, y, alone):
                d.free()
        for d in (da, db, want, got):
            d.free()


# ... or, in the largest tiles under a short sum, in the tiled kernel's K loop; a long job beside large tiles gets a launch of its
# own.  Counts on both sides of each line (512 x 1024: a pass of the grid is 2^18 elements, 1000 x 1003: 2^19).
@pytest.mark.parametrize("M,N", [(512, 1024), (1000, 1003), (1030, 472)])
@pytest.mark.parametrize("K", [8, 71, 256, 264, 512, 520])
def test_silu_job_in_the_loop(gpu, beamc, oracle, M, N, K):
    for dtype in (F16, BF16):
        a, b = beamc.host_uniform((M, K), dtype, 90, 0), beamc.host_uniform((N, K), dtype, 90, 1)
        ref = oracle.gemmrc(a, b, dtype)
        for count in (0, 5, (1 << 16) - 8, 1 << 16, 1 << 19, (1 << 19) + 8, (1 << 20) + 3, (1 << 20) + 8, (1 << 21) + 8):
            silu_pair(beamc, oracle, a, b, ref, dtype, count)


@pytest.mark.parametrize("M,N,K", [(256, 256, 200), (297, 400, 71), (509, 500, 200), (1000, 1003, 1096)])
def test_silu_long_job(gpu, beamc, oracle, M, N, K):
    a, b = beamc.host_uniform((M, K), F16, 91, 0), beamc.host_uniform((N, K), F16, 91, 1)
    ref = oracle.gemmrc(a, b, F16)
    for count in (1 << 23, (1 << 23) + 8, 1 << 24, (1 << 24) + 5):
        silu_pair(beamc, oracle, a, b, ref, F16, count)


def silu_pair(beamc, oracle, a, b, ref, dtype, count):
    L = beamc.lib
    (M, K), N = a.shape, b.shape[0]
    da, db = beamc.DeviceArray.from_numpy(a, dtype), beamc.DeviceArray.from_numpy(b, dtype)
    dx = beamc.DeviceArray.from_numpy(beamc.host_normal((count + 64,), dtype, 97, 2, 0.0, 2.5), dtype)
    c, y, alone = (beamc.DeviceArray(s, dtype) for s in ((M, N), (count + 64,), (count + 64,)))
    for d in (c, y, alone):
        d.fill_bytes(0xEE)
    beamc._check(L.beam_silu(dx.ptr, alone.ptr, count, dtype, None))
    beamc._check(L.beam_parallel_gemmrc_silu(da.ptr, db.ptr, c.ptr, M, N, K, dx.ptr, y.ptr, count, dtype, None, None))
    close_enough(oracle, c.to_numpy(), ref, K, dtype, f"{(M, N, K)} beside {count} elements")
    assert (y.to_numpy() == alone.to_numpy()).all(), (M, N, K, count)  # the guard behind the array included
    for d in (da, db, dx, c, y, alone):
        d.free()


LN_TILES = {"16x16": (41, 100), "16x32": (297, 400), "32x16": (1030, 100), "32x32": (509, 500), "16x64": (130, 1750), "32x64": (466, 864),
            "64x32": (1030, 475), "64x64": (1000, 1003), "64 column tiles": (60, 4096)}


@pytest.mark.parametrize("tile", sorted(LN_TILES))
@pytest.mark.parametrize("K", [8, 71, 513, 1096, 3265])
def test_layer_norm(gpu, beamc, oracle, tile, K):
    """One kernel (the caller's choice, so it is no fallback), columns that end inside a tile, statistics of up to 64 tiles."""
    M, N = LN_TILES[tile]
    for dtype in (F16, BF16):
        a, b, g, bt = make_ln_inputs(beamc, M, N, K, dtype, 98)
        got = run_ln(beamc, a, b, g, bt, dtype, mode=beamc.LN_FUSED)
        check_ln(oracle, got, oracle.gemmrc_ln(a, b, g, bt, 1e-5, dtype), dtype, f"{tile} {(M, N, K)} dtype {dtype}")


@pytest.mark.parametrize("tile", sorted(LN_TILES))
def test_layer_norm_by_whole_lines(gpu, beamc, oracle, tile):
    test_layer_norm(gpu, beamc, oracle, tile, 3208)


@pytest.mark.parametrize("M,N", [(41, 100), (1030, 475), (60, 4096)])
def test_layer_norm_gives_up_and_recovers(gpu, beamc, M, N):
    """With every wait forced to give up the kernel ends normally, its rows are NaN and the default call repeats as two passes;
    the next call is right again, with no reset in between."""
    K = 264
    a, b, g, bt = make_ln_inputs(beamc, M, N, K, F16, 99)
    good, two_pass = (run_ln(beamc, a, b, g, bt, F16, mode=m) for m in (beamc.LN_FUSED, beamc.LN_TWOPASS))
    d = [beamc.DeviceArray.from_numpy(x) for x in (a, b, g, bt)]
    y = beamc.DeviceArray((M, N))
    try:
        assert beamc.lib.beam_set_ln_spin_limit(-1) == 0
        beamc.gemmrc_ln(d[0], d[1], y, d[2], d[3], mode=beamc.LN_FUSED, check=False)
        beamc.sync()
        assert beamc.gemmrc_ln_timed_out() and np.isnan(y.to_numpy().view(np.float16)).all()
        assert beamc.gemmrc_ln(d[0], d[1], y, d[2], d[3]) is True
        assert (y.to_numpy() == two_pass).all()
    finally:
        beamc.lib.beam_set_ln_spin_limit(beamc.DEFAULT_SPIN_LIMIT)
    assert beamc.gemmrc_ln(d[0], d[1], y, d[2], d[3]) is False
    assert (y.to_numpy() == good).all()
    for t in d + [y]:
        t.free()


@pytest.mark.parametrize("M,N", [(1030, 475), (500, 1024), (60, 4096)])
def test_layer_norm_launches_share_the_device(gpu, beamc, M, N):
    """Two streams with launches that wait for their own workgroups: short bands, which stay on an XCD, and long ones."""
    K, L = 520, beamc.lib
    streams = []
    for _ in range(2):
        s = ctypes.c_void_p()
        beamc._check(L.beam_stream_create(ctypes.byref(s)))
        streams.append(s)
    sets = []
    for i in range(2):
        d = [beamc.DeviceArray.from_numpy(x) for x in make_ln_inputs(beamc, M, N, K, F16, 72 + i)]
        sets.append((d, beamc.DeviceArray((M, N)), beamc.DeviceArray((L.beam_gemmrc_ln_workspace_bytes_for(M, N, K, None, beamc.LN_FUSED),), itemsize=1)))

    def launch(i, stream):
        d, y, ws = sets[i]
        beamc._check(L.beam_gemmrc_ln_ex(d[0].ptr, d[1].ptr, d[2].ptr, d[3].ptr, ctypes.c_float(1e-5), y.ptr, M, N, K, F16, None, beamc.LN_FUSED,
                                         ws.ptr, ws.nbytes, stream))

    want = []
    for i in range(2):
        launch(i, None)
        beamc.sync()
        want.append(sets[i][1].to_numpy().copy())
    for rep in range(20):
        for _ in range(4):
            for i in range(2):
                launch(i, streams[i])
        for i in range(2):
            flag = ctypes.c_int(1)
            beamc._check(L.beam_gemmrc_ln_timed_out(sets[i][2].ptr, streams[i], ctypes.byref(flag)))
            assert flag.value == 0 and (sets[i][1].to_numpy() == want[i]).all(), (i, rep)
    for s in streams:
        beamc._check(L.beam_stream_destroy(s))
    for d, y, ws in sets:
        for t in d + [y, ws]:
            t.free()
