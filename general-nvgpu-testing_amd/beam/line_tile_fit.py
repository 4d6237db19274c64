"""The cost models that choose among all tiles, those whose fills take whole 128-byte lines included (csrc/capi.hip:
off_lines_tile, nn_off_lines_tile, ln_line_tile), their timings and their fits.

`line_tile_timings.json` holds microseconds per call of every candidate on drawn shapes, fp16, four sets of operands in turn,
best of two rounds, one MI355X, when these tiles came: beam_gemmrc on rows off lines (280 shapes), beam_matmul_nn with A's rows
off lines and B's rows whole chunks (120) and not (90), the one-kernel GEMM+LayerNorm on rows off lines (200) and on them (160).
Columns that are no candidate are forms that were measured and not built.  A candidate's constants are TFLOP/s per CU (alone, and
for tiles of which a CU holds several with a full CU), microseconds per round of workgroups and per launch: least squares on
the logarithm, a shape's weight falling with how far the tile is behind the best one there.

    python -m beam.line_tile_fit          the library's pick per table: how far behind the best tile, how far ahead of before
    python -m beam.line_tile_fit --fit    the constants, as they are compiled in
"""
import ctypes
import json
import math
import os
import re
import sys

CUS = 256
TIMINGS = os.path.join(os.path.dirname(os.path.abspath(__file__)), "line_tile_timings.json")
TABLES = ("gemmrc", "nn_whole", "nn_odd", "ln_off", "ln_on")


def load():
    """table -> (columns, [(M, N, K, us of the call before these tiles came, {column: us})])"""
    raw = json.load(open(TIMINGS))
    return {name: (t["tiles"], [(*row[:4], {c: us for c, us in zip(t["tiles"], row[4:]) if us is not None}) for row in t["shapes"]])
            for name, t in raw.items()}


def block(column):
    return tuple(int(x) for x in re.match(r"(\d+)x(\d+)", column).groups())


def workgroups_on_a_cu(column):
    return 1 if "_deep" in column or "_lines" in column else {(128, 128): 2, (128, 64): 2, (64, 128): 2, (64, 64): 4}.get(block(column), 1)


def model(table, column, M, N, K):
    """(constants) -> microseconds"""
    bm, bn = block(column)
    tiles_m, tiles_n = -(-M // bm), -(-N // bn)
    mflop = 2e-6 * bm * bn * (-(-K // 64) * 64)
    if table.startswith("ln"):
        rounds = -(-tiles_m // max(1, CUS // tiles_n))
        # the statistics of a wide band, which every workgroup reads (for the other tiles too the picks are no better)
        wide = 0.00125 * bm * max(0, tiles_n - 20) if column.endswith("x64_lines") else 0
        return lambda p: p[2] + rounds * (p[1] + wide + mflop / p[0])
    occ, load = workgroups_on_a_cu(column), -(-tiles_m * tiles_n // CUS)
    share = 0 if occ == 1 else (min(load, occ) - 1) / (occ - 1)
    return lambda p: -(-load // occ) * p[2] + load * mflop / (p[0] + (p[1] - p[0]) * share) + p[3]


def fit(table, column, rows):
    from scipy.optimize import least_squares
    terms = [(model(table, column, M, N, K), t[column], min(t.values())) for M, N, K, _, t in rows if column in t]
    start, low, high = (([4, 5, 2], [0.5, 0.2, 0], [12, 25, 6]) if table.startswith("ln") else
                        ([3, 3.5, 2, 1.5], [0.3, 0.3, 0.1, 0], [12, 12, 15, 4]))
    p = least_squares(lambda p: [math.log(max(us(p), 0.1) / t) * best / t for us, t, best in terms], start, bounds=(low, high)).x
    p = [float(x) for x in p]
    return p if table.startswith("ln") or workgroups_on_a_cu(column) > 1 else [p[0], p[0], p[2], p[3]]


def pick(table, M, N, K):
    """The column that the library takes (None: not one of these, the call runs in small tiles).  Needs no GPU."""
    from . import _C
    L, tile, lines = _C.lib, _C._TileCfg(), ctypes.c_int()
    small = [ctypes.c_int() for _ in range(4)]
    op = 3 if table.startswith("ln") else 1 if table.startswith("nn") else 0
    _C._check(L.beam_dbg_small_tile(op, M, N, K, 2 if K % 64 == 0 else 1, *map(ctypes.byref, small)))
    if small[0].value:
        return None
    if op == 1:
        # what beam_matmul_nn has made of the default tile by then
        named = _C.default_config(M, N, K)[0]
        tiles = lambda bm, bn: -(-M // bm) * -(-N // bn)
        kind = (named.block_m, named.block_n, named.wave_m, named.wave_n)
        if kind == (128, 128, 64, 64):
            named = _C.TileConfig(128, 128, 64, 32, named.pipeline, 0)
        elif kind == (64, 128, 32, 64) and tiles(128, 64) <= tiles(64, 128) and (named.pipeline != 2 or K % 64 == 0):
            named = _C.TileConfig(128, 64, 64, 32, named.pipeline, 0)
        named = named.to_c()
        _C._check(L.beam_dbg_nn_off_lines_tile(M, N, K, ctypes.byref(named), ctypes.byref(tile), ctypes.byref(lines)))
    else:
        _C._check((L.beam_dbg_ln_line_tile if op else L.beam_dbg_off_lines_tile)(M, N, K, ctypes.byref(tile), ctypes.byref(lines)))
    name = f"{tile.block_m}x{tile.block_n}"
    return name + "_lines" if lines.value else f"{name}_w{tile.wave_m}x{tile.wave_n}" + ("_deep" if tile.pipeline == 2 else "")


def regret(table, rows):
    """(geometric mean and worst of the pick's time to the best candidate's, mean of the time before to the pick's, shapes)"""
    behind, ahead = [], []
    for M, N, K, before, t in rows:
        column = pick(table, M, N, K)
        if column is None:
            continue
        behind.append(t[column] / min(us for c, us in t.items() if "_not_built" not in c))
        ahead.append(before / t[column])
    mean = lambda v: math.exp(sum(map(math.log, v)) / len(v))
    return mean(behind), max(behind), mean(ahead), len(behind)


def main(argv):
    for table, (columns, rows) in load().items():
        if argv[:1] == ["--fit"]:
            for c in columns:
                if "_not_built" not in c:
                    print(f"{table:9s} {c:24s}", *(f"{x:.2f}" for x in fit(table, c, rows)))
        else:
            from . import _C
            _C.lib.beam_dbg_assume_compute_units(CUS)  # (without a GPU; refused where one has been probed)
            print(table, "pick / best %.3f, worst %.3f; before / pick %.3f; %d shapes" % regret(table, rows))
    return 0


if __name__ == "__main__":
    sys.exit(main(sys.argv[1:]))
