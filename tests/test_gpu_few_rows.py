"""gemmrc of at most 64 rows without a named tile: the three forms of the kernel for few rows, every row group and its edges,
fewer K tiles than wavefronts, last K tiles of several lengths, columns that end inside a block, operands at any element's
address.  Bound: close_enough's, the one of every other GEMM test."""
import numpy as np
import pytest

from test_gpu_edges import close_enough
from test_gpu_gemm import F16, BF16
from test_gpu_unaligned import run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 7, 8, 9, 16, 17, 31, 32, 33, 48, 64])
@pytest.mark.parametrize("K", [8, 56, 64, 72, 192, 520, 1096, 4104])
def test_few_rows(gpu, beamc, oracle, M, K):
    L = beamc.lib
    for N, dtype, offsets in ((1, F16, (0, 0, 0)), (16, BF16, (0, 0, 0)), (37, F16, (1, 3, 1)), (130, BF16, (0, 1, 2))):
        a, b = beamc.host_uniform((M, K), dtype, 91, 0), beamc.host_uniform((N, K), dtype, 91, 1)
        out = run(beamc, lambda pa, pb, pc: L.beam_gemmrc(pa, pb, pc, M, N, K, dtype, None, None), a, b, (M, N), dtype, offsets)
        close_enough(oracle, out, oracle.gemmrc(a, b, dtype), K, dtype, f"{(M, N, K)}")


# More columns than 16 for every one of the 256 CUs.  4097: one column in the last block; 4131: part of a block of 16, of 32 and
# of 64; 5120: whole blocks; 8192: the last number of columns that the form for a long K takes
@pytest.mark.parametrize("M,N,K,form", [(M, N, K, "wide") for M in (1, 8, 9, 16) for N, K in ((4097, 520), (4131, 1096), (5120, 512), (8200, 2056), (4131, 4096))] +
                                       [(M, N, K, "deep") for M in (1, 8, 9, 16) for N, K in ((4097, 4104), (4131, 4168), (8192, 4104))] +
                                       [(M, N, K, "wide") for M in (17, 32) for N, K in ((4097, 1024), (4131, 2040), (8192, 1096))])
def test_few_rows_of_many_columns(gpu, beamc, oracle, M, N, K, form):
    assert gpu["compute_units"] == 256  # the columns above are chosen for that
    L = beamc.lib
    for dtype, offsets in ((F16, (0, 0, 0)), (BF16, (1, 3, 1))):
        a, b = beamc.host_uniform((M, K), dtype, 93, 0), beamc.host_uniform((N, K), dtype, 93, 1)
        out = run(beamc, lambda pa, pb, pc: L.beam_gemmrc(pa, pb, pc, M, N, K, dtype, None, None), a, b, (M, N), dtype, offsets)
        close_enough(oracle, out, oracle.gemmrc(a, b, dtype), K, dtype, f"{form} {(M, N, K)}")


def test_few_rows_keep_to_their_rows(gpu, beamc):
    """Infinities and NaN stay in the row or column that holds them, also with a short last K tile."""
    M, N, K = 19, 41, 200
    L = beamc.lib
    a, b = beamc.host_uniform((M, K), F16, 92, 0), beamc.host_uniform((N, K), F16, 92, 1)
    a[18, 199], b[40, 7] = 0x7E00, 0x7C00  # NaN, infinity
    out = run(beamc, lambda pa, pb, pc: L.beam_gemmrc(pa, pb, pc, M, N, K, F16, None, None), a, b, (M, N), F16, (0, 0, 0))
    out = out.view(np.float16)
    assert np.isnan(out[18]).all() and not np.isfinite(out[:, 40]).any()
    assert np.isfinite(out[:18, :40]).all()
