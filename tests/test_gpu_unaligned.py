"""Rows that do not start on 16 bytes: K not a multiple of 8, [K][N] with N not a multiple of 8, operands and outputs
at any element's address, on the tiled kernels.  Every operand lies inside a larger buffer of NaNs: an element read
from beside a row, or beyond a matrix, that reached an output would show.  Every output lies inside a larger buffer
too, which must stay as it was around it."""
import ctypes

import numpy as np
import pytest

from test_gpu_edges import close_enough
from test_gpu_gemm import F16, BF16, all_configs, assert_close
from test_gpu_ln import check_ln, make_ln_inputs

pytestmark = pytest.mark.gpu

PAD = 16
NAN = 0xFFFF


class Embedded:
    """`bits` on the device, `off` elements past a 16-byte boundary, NaNs (or a guard pattern) in front and behind."""

    def __init__(self, beamc, shape, dtype, off, bits=None):
        self.beamc, self.shape, self.n, self.off = beamc, shape, int(np.prod(shape)), off
        host = np.full(self.n + 2 * PAD, NAN, np.uint16)
        if bits is not None:
            host[off:off + self.n] = bits.ravel()
        self.buf = beamc.DeviceArray.from_numpy(host, dtype)
        self.ptr = self.buf.ptr + 2 * off

    def result(self):
        out = self.buf.to_numpy()
        assert (out[:self.off] == NAN).all() and (out[self.off + self.n:] == NAN).all(), "written outside the output"
        return out[self.off:self.off + self.n].reshape(self.shape)


def run(beamc, call, a, b, shape, dtype, offs):
    da, db, c = Embedded(beamc, a.shape, dtype, offs[0], a), Embedded(beamc, b.shape, dtype, offs[1], b), Embedded(beamc, shape, dtype, offs[2])
    beamc._check(call(da.ptr, db.ptr, c.ptr))
    out = c.result()
    for x in (da, db, c):
        x.buf.free()
    return out


# K around one chunk of 8, one K tile of 64 and several of them; M and N around the smallest tile
@pytest.mark.parametrize("K", [8, 9, 15, 57, 63, 65, 71, 127, 129, 1001])
@pytest.mark.parametrize("dtype", [F16, BF16])
def test_any_k(gpu, beamc, oracle, K, dtype):
    L = beamc.lib
    for M, N, offs in ((65, 63, (0, 0, 0)), (1, 9, (1, 3, 5)), (130, 257, (7, 2, 1))):
        a, b = beamc.host_uniform((M, K), dtype, 71, 0), beamc.host_uniform((N, K), dtype, 71, 1)
        out = run(beamc, lambda pa, pb, pc: L.beam_gemmrc(pa, pb, pc, M, N, K, dtype, None, None), a, b, (M, N), dtype, offs)
        close_enough(oracle, out, oracle.gemmrc(a, b, dtype), K, dtype, f"gemmrc {(M, N, K)} at {offs}")
        # slices whose last one ends in a short tile, with and without room for them
        for slices, room in ((3, True), (3, False)):
            ws = beamc.DeviceArray((max(L.beam_splitk_workspace_bytes(M, N, 3), 256),), itemsize=1)
            out = run(beamc, lambda pa, pb, pc: L.beam_gemmrc_splitk(pa, pb, pc, M, N, K, dtype, None, slices, ws.ptr if room else None,
                                                                     ws.nbytes if room else 0, None), a, b, (M, N), dtype,
                      offs if K % 8 or room else (1, 0, 0))
            ws.free()
            close_enough(oracle, out, oracle.gemmrc(a, b, dtype), K, dtype, f"split-K {(M, N, K)} room {room}")


# N a multiple of 4, as the one-launch form asks for: 1, 2 and 4 outputs per thread of a reducing workgroup
@pytest.mark.parametrize("M,N", [(65, 72), (400, 460), (640, 700)])
@pytest.mark.parametrize("offs", [(0, 0, 1), (1, 0, 2), (0, 3, 3)])
def test_split_k_outputs_at_any_address(gpu, beamc, oracle, M, N, offs):
    """Both forms of the reduction store vectors of C at any element's address; same bits either way."""
    K, slices = 392, 3
    L = beamc.lib
    ws = beamc.DeviceArray((L.beam_splitk_workspace_bytes(M, N, slices),), itemsize=1)
    for dtype in (F16, BF16):
        a, b = beamc.host_uniform((M, K), dtype, 82, 0), beamc.host_uniform((N, K), dtype, 82, 1)
        ref = oracle.gemmrc(a, b, dtype)
        for pipeline in (0, 2):
            cfg = beamc.TileConfig(64, 64, 32, 32, pipeline, 0).to_c()
            outs = []
            for two in (False, True):
                beamc.set_splitk_two_launches(two)
                try:
                    outs.append(run(beamc, lambda pa, pb, pc: L.beam_gemmrc_splitk(pa, pb, pc, M, N, K, dtype, ctypes.byref(cfg), slices, ws.ptr,
                                                                                   ws.nbytes, None), a, b, (M, N), dtype, offs))
                finally:
                    beamc.set_splitk_two_launches(False)
            close_enough(oracle, outs[0], ref, K, dtype, f"pipeline {pipeline} at {offs}")
            assert (outs[0] == outs[1]).all()
    ws.free()


@pytest.mark.parametrize("shape,offs", [((65, 72, 321), (0, 0, 0)), ((65, 72, 320), (0, 1, 0))])
def test_split_k_workspace_off_16_bytes(gpu, beamc, oracle, shape, offs):
    """Unaligned rows never needed a workspace: one that is off 16 bytes is left alone."""
    M, N, K = shape
    L = beamc.lib
    a, b = beamc.host_uniform((M, K), F16, 81, 0), beamc.host_uniform((N, K), F16, 81, 1)
    ws = beamc.DeviceArray((L.beam_splitk_workspace_bytes(M, N, 3) + 256,), itemsize=1)
    ws.fill_bytes(0xEE)
    for at in (2, 8):
        out = run(beamc, lambda pa, pb, pc: L.beam_gemmrc_splitk(pa, pb, pc, M, N, K, F16, None, 3, ws.ptr + at, ws.nbytes - at, None), a, b,
                  (M, N), F16, offs)
        close_enough(oracle, out, oracle.gemmrc(a, b, F16), K, F16, f"workspace at {at}")
    assert (ws.to_numpy(np.uint8) == 0xEE).all()
    ws.free()


# N around one chunk, around the tiles' widths, and a last K tile that is whole (64, 128) or short
@pytest.mark.parametrize("N", [8, 9, 63, 65, 127, 129, 255, 257, 1001])
@pytest.mark.parametrize("dtype", [F16, BF16])
def test_any_n_kmajor(gpu, beamc, oracle, N, dtype):
    L = beamc.lib
    for M, K, offs in ((65, 64, (0, 0, 0)), (3, 9, (1, 1, 1)), (130, 128, (0, 5, 3)), (129, 331, (0, 0, 0))):
        a, b = beamc.host_uniform((M, K), dtype, 72, 0), beamc.host_uniform((K, N), dtype, 72, 1)
        out = run(beamc, lambda pa, pb, pc: L.beam_matmul_nn(pa, pb, pc, M, N, K, dtype, None, None), a, b, (M, N), dtype, offs)
        close_enough(oracle, out, oracle.matmul_nn(a, b, dtype), K, dtype, f"matmul {(M, N, K)} at {offs}")


def test_every_tile(gpu, beamc, oracle):
    """Every compiled tile and LDS depth, both layouts: several tiles each way, a short K tile behind several whole ones."""
    M, N, K = 515, 773, 459
    L = beamc.lib
    a, b, bt = beamc.host_uniform((M, K), F16, 73, 0), beamc.host_uniform((N, K), F16, 73, 1), beamc.host_uniform((K, N), F16, 73, 1)
    ref, ref_nn = oracle.gemmrc(a, b, F16), oracle.matmul_nn(a, bt, F16)
    for cfg in all_configs(beamc):
        c = cfg.to_c()
        out = run(beamc, lambda pa, pb, pc: L.beam_gemmrc(pa, pb, pc, M, N, K, F16, ctypes.byref(c), None), a, b, (M, N), F16, (0, 3, 1))
        assert_close(oracle, out, ref, K, F16, f"gemmrc {cfg.name}")
        out = run(beamc, lambda pa, pb, pc: L.beam_matmul_nn(pa, pb, pc, M, N, K, F16, ctypes.byref(c), None), a, bt, (M, N), F16, (0, 3, 1))
        assert_close(oracle, out, ref_nn, K, F16, f"matmul {cfg.name}")


# N around a chunk of 8 and around the largest tile; K a multiple of 64, which is what the 4-wavefront kernel asks of K
@pytest.mark.parametrize("N", [257, 513, 1001, 1004])
def test_every_tile_kmajor_whole_k_tiles(gpu, beamc, oracle, N):
    """[K][N] with N not a multiple of 8 in every compiled tile and LDS depth, C on a 16-byte boundary: no kernel that
    stores whole chunks may take it."""
    M, K = 300, 192
    L = beamc.lib
    a, b = beamc.host_uniform((M, K), F16, 76, 0), beamc.host_uniform((K, N), F16, 76, 1)
    ref = oracle.matmul_nn(a, b, F16)
    for cfg in all_configs(beamc):
        c = cfg.to_c()
        out = run(beamc, lambda pa, pb, pc: L.beam_matmul_nn(pa, pb, pc, M, N, K, F16, ctypes.byref(c), None), a, b, (M, N), F16, (0, 0, 0))
        assert_close(oracle, out, ref, K, F16, f"matmul {cfg.name} N={N}")


# the persistent kernels: more tiles than CUs, K a multiple of 64, operands off a 16-byte boundary
@pytest.mark.parametrize("wave_n", [64, 128])
def test_walking_kernels_at_any_address(gpu, beamc, oracle, wave_n):
    M, N, K = 4200, 4200, 192
    L = beamc.lib
    a, b = beamc.host_uniform((M, K), F16, 74, 0), beamc.host_uniform((N, K), F16, 74, 1)
    c = beamc.TileConfig(256, 256, 128, wave_n).to_c()
    out = run(beamc, lambda pa, pb, pc: L.beam_gemmrc(pa, pb, pc, M, N, K, F16, ctypes.byref(c), None), a, b, (M, N), F16, (1, 3, 0))
    assert_close(oracle, out, oracle.gemmrc(a, b, F16), K, F16, f"256x256, wavefronts 128x{wave_n}")


# N a multiple of 4 and of 8: the vector path of the normalisation pass, Y at any element's address
@pytest.mark.parametrize("shape", [(65, 72, 64), (130, 260, 72), (33, 1028, 200)])
@pytest.mark.parametrize("offs", [(0, 0, 1), (1, 0, 2), (0, 3, 3)])
def test_layer_norm_outputs_at_any_address(gpu, beamc, oracle, shape, offs):
    M, N, K = shape
    L = beamc.lib
    for dtype in (F16, BF16):
        a, b, g, bt = make_ln_inputs(beamc, M, N, K, dtype, 85)
        ref = oracle.gemmrc_ln(a, b, g, bt, 1e-5, dtype)
        dg, dbt = beamc.DeviceArray.from_numpy(g, dtype), beamc.DeviceArray.from_numpy(bt, dtype)
        ws = beamc.DeviceArray((L.beam_gemmrc_ln_workspace_bytes_ex(M, N, None, beamc.LN_AUTO),), itemsize=1)
        for mode in (beamc.LN_TWOPASS, beamc.LN_FUSED):
            out = run(beamc, lambda pa, pb, pc: L.beam_gemmrc_ln_ex(pa, pb, dg.ptr, dbt.ptr, 1e-5, pc, M, N, K, dtype, None, mode, ws.ptr,
                                                                    ws.nbytes, None), a, b, (M, N), dtype, offs)
            check_ln(oracle, out, ref, dtype, f"LayerNorm {shape} mode {mode} at {offs}")
        for v in (dg, dbt, ws):
            v.free()


def test_walking_kernels_at_any_address_kmajor_and_layer_norm(gpu, beamc, oracle):
    """The 4-wavefront kernel's [K][N] and LayerNorm forms with A and B off 16 bytes: one tile per workgroup and, with more
    tiles than CUs, several."""
    L = beamc.lib
    c = beamc.TileConfig(256, 256, 128, 128).to_c()
    for M, N, K in ((300, 520, 192), (4200, 4200, 192)):
        a, b, g, bt = make_ln_inputs(beamc, M, N, K, F16, 86)
        bk = np.ascontiguousarray(b.T)
        out = run(beamc, lambda pa, pb, pc: L.beam_matmul_nn(pa, pb, pc, M, N, K, F16, ctypes.byref(c), None), a, bk, (M, N), F16, (1, 3, 0))
        assert_close(oracle, out, oracle.matmul_nn(a, bk, F16), K, F16, f"[K][N] {(M, N, K)}")
        dg, dbt = beamc.DeviceArray.from_numpy(g, F16), beamc.DeviceArray.from_numpy(bt, F16)
        ws = beamc.DeviceArray((L.beam_gemmrc_ln_workspace_bytes_for(M, N, K, ctypes.byref(c), beamc.LN_FUSED),), itemsize=1)
        out = run(beamc, lambda pa, pb, pc: L.beam_gemmrc_ln_ex(pa, pb, dg.ptr, dbt.ptr, 1e-5, pc, M, N, K, F16, ctypes.byref(c), beamc.LN_FUSED,
                                                                ws.ptr, ws.nbytes, None), a, b, (M, N), F16, (1, 3, 0))
        check_ln(oracle, out, oracle.gemmrc_ln(a, b, g, bt, 1e-5, F16), F16, f"LayerNorm {(M, N, K)}")
        for v in (dg, dbt, ws):
            v.free()


# K a multiple of 8 and not, a short K tile alone and behind whole ones; the job shorter than, and longer than, the K loop
@pytest.mark.parametrize("K,offs", [(63, (0, 0, 0)), (137, (0, 0, 0)), (200, (1, 0, 3)), (459, (3, 1, 1))])
@pytest.mark.parametrize("pipeline", [0, 1])
def test_side_job(gpu, beamc, oracle, K, offs, pipeline):
    """Every tile carries the SiLU job beside rows at any element's address."""
    M, N = 300, 200
    L = beamc.lib
    a, b = beamc.host_uniform((M, K), F16, 87, 0), beamc.host_uniform((N, K), F16, 87, 1)
    ref = oracle.gemmrc(a, b, F16)
    for count in (5, 4099, 100003):
        x = beamc.host_normal((count,), F16, 87, 2, 0.0, 2.0)
        dx, want = beamc.DeviceArray.from_numpy(x, F16), beamc.DeviceArray((count,), F16)
        beamc.silu(dx, want)
        y = Embedded(beamc, (count,), F16, 8)
        for t in beamc.list_configs():
            cfg = beamc.TileConfig(t.block_m, t.block_n, t.wave_m, t.wave_n, pipeline, 0).to_c()
            beamc._check(L.beam_memset(y.ptr, 0xEE, 2 * count))
            out = run(beamc, lambda pa, pb, pc: L.beam_parallel_gemmrc_silu(pa, pb, pc, M, N, K, dx.ptr, y.ptr, count, F16, ctypes.byref(cfg), None),
                      a, b, (M, N), F16, offs)
            close_enough(oracle, out, ref, K, F16, f"{t.name} beside {count}")
            assert (y.result() == want.to_numpy()).all(), (t.name, count)
        for v in (dx, want, y.buf):
            v.free()


@pytest.mark.parametrize("shape", [(65, 63, 9), (130, 257, 71), (33, 1001, 331), (300, 515, 129)])
@pytest.mark.parametrize("dtype", [F16, BF16])
def test_layer_norm(gpu, beamc, oracle, shape, dtype):
    M, N, K = shape
    L = beamc.lib
    a, b, g, bt = make_ln_inputs(beamc, M, N, K, dtype, 75)
    ref = oracle.gemmrc_ln(a, b, g, bt, 1e-5, dtype)
    dg, dbt = beamc.DeviceArray.from_numpy(g, dtype), beamc.DeviceArray.from_numpy(bt, dtype)
    for mode in (beamc.LN_AUTO, beamc.LN_TWOPASS):
        ws = beamc.DeviceArray((L.beam_gemmrc_ln_workspace_bytes_for(M, N, K, None, mode),), itemsize=1)
        out = run(beamc, lambda pa, pb, pc: L.beam_gemmrc_ln_ex(pa, pb, dg.ptr, dbt.ptr, 1e-5, pc, M, N, K, dtype, None, mode, ws.ptr,
                                                                ws.nbytes, None), a, b, (M, N), dtype, (1, 0, 3))
        check_ln(oracle, out, ref, dtype, f"LayerNorm {shape} mode {mode}")
        ws.free()
    dg.free()
    dbt.free()


@pytest.mark.parametrize("shape,offs", [((130, 3, 65), (0, 0, 0)), ((130, 257, 71), (0, 0, 0)), ((130, 257, 72), (1, 0, 0)), ((65, 72, 64), (0, 0, 3))])
def test_layer_norm_workspace_of_the_plain_kernels(gpu, beamc, oracle, shape, offs):
    """Unaligned rows need M * N fp32 values on a 16-byte boundary and no more, whatever the mode."""
    M, N, K = shape
    L = beamc.lib
    a, b, g, bt = make_ln_inputs(beamc, M, N, K, F16, 80)
    ref = oracle.gemmrc_ln(a, b, g, bt, 1e-5, F16)
    dg, dbt = beamc.DeviceArray.from_numpy(g, F16), beamc.DeviceArray.from_numpy(bt, F16)
    room = (M * N * 4 + 255) // 256 * 256
    ws = beamc.DeviceArray((room + 16 + 256,), itemsize=1)
    for mode in (beamc.LN_AUTO, beamc.LN_TWOPASS, beamc.LN_FUSED):
        for at in (0, 16):
            ws.fill_bytes(0xEE)
            out = run(beamc, lambda pa, pb, pc: L.beam_gemmrc_ln_ex(pa, pb, dg.ptr, dbt.ptr, 1e-5, pc, M, N, K, F16, None, mode, ws.ptr + at,
                                                                    room, None), a, b, (M, N), F16, offs)
            check_ln(oracle, out, ref, F16, f"mode {mode}, workspace at {at}")
            assert (ws.to_numpy(np.uint8)[room + at:] == 0xEE).all(), "written beyond the workspace"
    out = run(beamc, lambda pa, pb, pc: L.beam_gemmrc_ln_checked(pa, pb, dg.ptr, dbt.ptr, 1e-5, pc, M, N, K, F16, None, ws.ptr + 16, room, None,
                                                                 None), a, b, (M, N), F16, offs)
    check_ln(oracle, out, ref, F16, "checked")
    for v in (dg, dbt, ws):
        v.free()


@pytest.mark.parametrize("offs", [(1, 0, 0), (0, 3, 0), (0, 0, 1), (4, 4, 2)])
def test_layer_norm_one_kernel_form_where_it_does_not_apply(gpu, beamc, oracle, offs):
    """More than 64 column tiles: BEAM_LN_FUSED is refused on aligned operands and computed (by the plain kernels) on
    others, through the C entry point and the Python operator."""
    M, N, K = 20, 64 * 64 + 8, 64
    L = beamc.lib
    tile = beamc.TileConfig(64, 64, 32, 32)
    cfg = tile.to_c()
    a, b, g, bt = make_ln_inputs(beamc, M, N, K, F16, 77)
    ref = oracle.gemmrc_ln(a, b, g, bt, 1e-5, F16)
    dg, dbt = beamc.DeviceArray.from_numpy(g, F16), beamc.DeviceArray.from_numpy(bt, F16)
    ws = beamc.DeviceArray((L.beam_gemmrc_ln_workspace_bytes_ex(M, N, ctypes.byref(cfg), beamc.LN_FUSED),), itemsize=1)

    def call(pa, pb, pc):
        return L.beam_gemmrc_ln_ex(pa, pb, dg.ptr, dbt.ptr, 1e-5, pc, M, N, K, F16, ctypes.byref(cfg), beamc.LN_FUSED, ws.ptr, ws.nbytes, None)

    check_ln(oracle, run(beamc, call, a, b, (M, N), F16, offs), ref, F16, f"LN_FUSED at {offs}")
    da, db, c = Embedded(beamc, a.shape, F16, 0, a), Embedded(beamc, b.shape, F16, 0, b), Embedded(beamc, (M, N), F16, 0)
    assert call(da.ptr, db.ptr, c.ptr) == 2
    views = []
    for x, off in zip((da, db, c), offs):  # the same buffers, seen `off` elements further on (inputs: other values)
        v = beamc.DeviceArray.__new__(beamc.DeviceArray)
        v.shape, v.dtype, v.itemsize, v.nbytes, v.ptr = x.shape, F16, 2, 2 * x.n, x.ptr + 2 * off
        views.append(v)
    beamc._check(L.beam_memcpy_h2d(views[0].ptr, a.ctypes.data, a.nbytes))
    beamc._check(L.beam_memcpy_h2d(views[1].ptr, b.ctypes.data, b.nbytes))
    beamc.gemmrc_ln(*views, dg, dbt, config=tile, mode=beamc.LN_FUSED)
    c.off = offs[2]
    check_ln(oracle, c.result(), ref, F16, f"gemmrc_ln, LN_FUSED at {offs}")
    for v in views:
        v.ptr = 0
    for x in (da.buf, db.buf, c.buf, dg, dbt, ws):
        x.free()


@pytest.mark.parametrize("shape,offs", [((65, 72, 65), (0, 0, 0)), ((130, 72, 64), (1, 0, 0)), ((65, 200, 192), (0, 2, 0)), ((65, 72, 64), (0, 0, 3))])
@pytest.mark.parametrize("tile", [(64, 64, 32, 32), (128, 128, 64, 64)])
def test_side_job_beside_the_deep_pipeline(gpu, beamc, oracle, tile, shape, offs):
    """The deep pipeline carries no side job: refused on aligned rows (test_gpu_silu), computed in two launches on others."""
    M, N, K = shape
    L = beamc.lib
    cfg = beamc.TileConfig(*tile, 2, 0).to_c()
    a, b = beamc.host_uniform((M, K), BF16, 79, 0), beamc.host_uniform((N, K), BF16, 79, 1)
    dx = beamc.DeviceArray.from_numpy(beamc.host_normal((3001,), BF16, 79, 2, 0.0, 2.0), BF16)
    dy, dy2 = beamc.DeviceArray((3001,), BF16), beamc.DeviceArray((3001,), BF16)
    beamc.silu(dx, dy2)
    out = run(beamc, lambda pa, pb, pc: L.beam_parallel_gemmrc_silu(pa, pb, pc, M, N, K, dx.ptr, dy.ptr, 3001, BF16, ctypes.byref(cfg), None),
              a, b, (M, N), BF16, offs)
    close_enough(oracle, out, oracle.gemmrc(a, b, BF16), K, BF16, f"{shape} at {offs}")
    assert (dy.to_numpy() == dy2.to_numpy()).all()
    for v in (dx, dy, dy2):
        v.free()


@pytest.mark.parametrize("tile", [(96, 64, 32, 32, 0, 0), (128, 128, 64, 64, 7, 0)])
@pytest.mark.parametrize("shape,offs", [((65, 72, 65), (0, 0, 0)), ((65, 72, 64), (1, 0, 0)), ((65, 72, 64), (0, 2, 0)), ((65, 72, 64), (0, 0, 3))])
def test_tile_that_is_not_compiled(gpu, beamc, oracle, tile, shape, offs):
    """Rows off 16 bytes are computed whatever tile is named, by every entry point that takes one; aligned ones are
    refused with it."""
    M, N, K = shape
    L = beamc.lib
    cfg = beamc._TileCfg(*tile)
    cp = ctypes.byref(cfg)
    a, b, g, bt = make_ln_inputs(beamc, M, N, K, F16, 78)
    bk = np.ascontiguousarray(b.T)
    x = beamc.host_normal((1000,), F16, 78, 9, 0.0, 2.0)
    dg, dbt, dx = (beamc.DeviceArray.from_numpy(v, F16) for v in (g, bt, x))
    dy, dy2 = beamc.DeviceArray((1000,), F16), beamc.DeviceArray((1000,), F16)
    beamc.silu(dx, dy2)
    ws = beamc.DeviceArray((1 << 20,), itemsize=1)
    ref, ref_nn, ref_ln = oracle.gemmrc(a, b, F16), oracle.matmul_nn(a, bk, F16), oracle.gemmrc_ln(a, b, g, bt, 1e-5, F16)
    calls = {
        "gemmrc": (b, lambda pa, pb, pc: L.beam_gemmrc(pa, pb, pc, M, N, K, F16, cp, None)),
        "matmul": (bk, lambda pa, pb, pc: L.beam_matmul_nn(pa, pb, pc, M, N, K, F16, cp, None)),
        "split-K": (b, lambda pa, pb, pc: L.beam_gemmrc_splitk(pa, pb, pc, M, N, K, F16, cp, 2, ws.ptr, ws.nbytes, None)),
        "split-K, no workspace": (b, lambda pa, pb, pc: L.beam_gemmrc_splitk_noalloc(pa, pb, pc, M, N, K, F16, cp, 2, None)),
        "with SiLU": (b, lambda pa, pb, pc: L.beam_parallel_gemmrc_silu(pa, pb, pc, M, N, K, dx.ptr, dy.ptr, 1000, F16, cp, None)),
        "LayerNorm": (b, lambda pa, pb, pc: L.beam_gemmrc_ln_ex(pa, pb, dg.ptr, dbt.ptr, 1e-5, pc, M, N, K, F16, cp, beamc.LN_AUTO, ws.ptr,
                                                                ws.nbytes, None)),
    }
    for what, (bb, call) in calls.items():
        out = run(beamc, call, a, bb, (M, N), F16, offs)
        if what == "LayerNorm":
            check_ln(oracle, out, ref_ln, F16, what)
        else:
            close_enough(oracle, out, ref_nn if what == "matmul" else ref, K, F16, what)
        if K % 8 == 0:
            da, db, c = Embedded(beamc, a.shape, F16, 0, a), Embedded(beamc, bb.shape, F16, 0, bb), Embedded(beamc, (M, N), F16, 0)
            assert call(da.ptr, db.ptr, c.ptr) == 2, what
            for v in (da, db, c):
                v.buf.free()
    assert (dy.to_numpy() == dy2.to_numpy()).all()
    if K % 8 != 0:
        assert L.beam_splitk_effective(M, N, K, cp, 2) == 1
        assert L.beam_gemmrc_ln_workspace_bytes_for(M, N, K, cp, beamc.LN_AUTO) >= M * N * 4
    for v in (dg, dbt, dx, dy, dy2, ws):
        v.free()
