"""How 16-bit output leaves a tiled kernel depends on where C's rows start and on how much is written (capi.hip: store_kind).
Every kind writes the same values: rows on and off 64-byte sectors, a C that starts off one, tiles cut by both edges, the
kernels that store through LDS and the one that stores from its accumulators, several rounds of workgroups.  C lies between
guard elements.  Bound: the GEMM bound used everywhere, 1e-2 * sqrt(K / 1024) * RMS (bf16: in excess of |ref| / 256)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# (M, N, K, tile, elements in front of C): what the output takes
CASES = [
    ((300, 328, 72), (64, 64, 32, 32), 0),         # 64 columns, rows off sectors: cached
    ((300, 331, 136), (128, 64, 64, 32), 0),       # ... odd rows
    ((257, 264, 320), (256, 256, 128, 128), 0),    # gemm_w4.h, 8 columns behind a tile: cached
    ((512, 512, 192), (256, 256, 128, 128), 8),    # ... whole tiles, C 16 bytes behind a sector
    ((512, 512, 192), (256, 256, 128, 128), 0),    # ... on sectors: through
    ((3100, 3400, 64), (128, 128, 64, 64), 0),     # 21 MB off sectors: cached
    ((3100, 3400, 72), (192, 256, 96, 64), 1),     # ... C off 4 bytes
    ((3000, 3400, 64), (128, 128, 64, 64), 0),     # 20.4 MB in decimal, below the line: through
    ((4104, 4352, 72), (256, 256, 128, 64), 0),    # 17 x 17 tiles, on sectors, several rounds: cached
]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape,tile,lead", CASES)
@pytest.mark.parametrize("layout", ["nk", "kn"])
def test_every_kind_writes_the_product(gpu, beamc, shape, tile, lead, layout, dtype):
    M, N, K = shape
    gen = torch.Generator(device="cuda").manual_seed(1)
    a = torch.randn(M, K, generator=gen, device="cuda", dtype=dtype)
    b = torch.randn(N, K, generator=gen, device="cuda", dtype=dtype)
    guard = 512
    room = torch.full((lead + M * N + 2 * guard,), 7.0, device="cuda", dtype=dtype)
    c = room[guard + lead:guard + lead + M * N].view(M, N)
    config = beamc.TileConfig(*tile)
    if layout == "nk":
        beamc.gemmrc(a, b, c, config=config)
    else:
        beamc.matmul(a, b.t().contiguous(), c, config=config)
    ref = a.float() @ b.float().t()
    excess = (c.float() - ref).abs() - (ref.abs() / 256 if dtype == torch.bfloat16 else 0)
    assert excess.max().item() <= 1e-2 * (K / 1024) ** 0.5 * ref.square().mean().sqrt().item()
    assert bool((room[:guard + lead] == 7.0).all()) and bool((room[guard + lead + M * N:] == 7.0).all()), "wrote outside C"


@pytest.mark.parametrize("shape,tile", [((520, 520, 256), (256, 256, 128, 128)), ((300, 264, 200), (128, 128, 64, 64)),
                                        ((3100, 3400, 128), (256, 256, 128, 64))])
def test_layernorm_output(gpu, beamc, shape, tile):
    """Rows off sectors: cached in the kernel of gemm_w4.h and from 20 MB on.  Bound: 2e-3 on fp16 results below 8."""
    M, N, K = shape
    gen = torch.Generator(device="cuda").manual_seed(2)
    a = torch.randn(M, K, generator=gen, device="cuda", dtype=torch.float16)
    b = (torch.randn(N, K, generator=gen, device="cuda") * K ** -0.5).half()
    gamma = (1 + 0.1 * torch.randn(N, generator=gen, device="cuda")).half()
    beta = (0.1 * torch.randn(N, generator=gen, device="cuda")).half()
    y = torch.empty(M, N, device="cuda", dtype=torch.float16)
    beamc.gemmrc_ln(a, b, y, gamma, beta, config=beamc.TileConfig(*tile), mode=beamc.LN_FUSED)
    ref = torch.nn.functional.layer_norm(a.float() @ b.float().t(), (N,), gamma.float(), beta.float(), 1e-5)
    assert (y.float() - ref).abs().max().item() <= max(2e-3, ref.abs().max().item() * 2.0 ** -11 + 2e-4)
