"""The tiled int8 GEMM in both tile sizes at the edges of its tiles, steps and
pieces: int32 sums equal torch's on the CPU exactly, whatever the split."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("small", ["1", "100000"])  # 128- and 64-row tiles
@pytest.mark.parametrize("m,n,k,pieces", [(64, 1, 128, 1), (65, 63, 384, 1), (127, 65, 1152, 3),
                                          (129, 130, 256, 2), (200, 257, 1280, 4), (320, 192, 640, 0)])
def test_i8_tiles_exact(gpu, small, m, n, k, pieces, monkeypatch):
    import sparkq

    print(f"[case] i8 tiles small={small} m={m} n={n} k={k} pieces={pieces}", flush=True)
    monkeypatch.setenv("SPARKQ_I8_GEMM_SMALL", small)
    if pieces:
        monkeypatch.setenv("SPARKQ_I8_GEMM_SPLITS", str(pieces))
    gen = torch.Generator().manual_seed(m + n + k)
    a, b = (torch.randint(-128, 128, (r, k), generator=gen, dtype=torch.int8) for r in (m, n))
    y = sparkq.int8_matmul_int32(a.to(gpu), b.to(gpu)).cpu()
    assert torch.equal(y, a.to(torch.int32) @ b.to(torch.int32).T)


@pytest.mark.parametrize("m,n,k", [
    (1020, 960, 2048), (512, 2048, 4096), (1000, 1020, 1024), (64, 16448, 2048),  # 240, 256, 256, 257 tiles
    (448, 4672, 2048), (512, 4096, 2048), (1216, 1728, 2048), (640, 4000, 8192),  # 511, 512, 513, 630
    (2048, 2048, 2048), (2048, 2176, 2048), (4096, 2048, 2048),  # 256, 272 and 512 tiles of 128 rows
])
def test_i8_planned_exact(gpu, m, n, k):
    """The planner's own tiles and pieces around one and two tiles per CU."""
    import sparkq

    print(f"[case] i8 plan m={m} n={n} k={k}", flush=True)
    gen = torch.Generator().manual_seed(m + n + k)
    a, b = (torch.randint(-128, 128, (r, k), generator=gen, dtype=torch.int8) for r in (m, n))
    y = sparkq.int8_matmul_int32(a.to(gpu), b.to(gpu)).cpu()
    assert torch.equal(y.double(), a.double() @ b.double().T)


@pytest.mark.parametrize("k", [128, 256, 384, 3968, 4096])
def test_i8_large_tiles_short_and_long_rows(gpu, k):
    """128-row tiles with loads one step ahead (fewer than 32 steps of 128 in
    less than two rounds) and two, down to a single step."""
    import sparkq

    m, n = 2100, 2050
    print(f"[case] i8 steps ahead k={k}", flush=True)
    gen = torch.Generator().manual_seed(k)
    a, b = (torch.randint(-128, 128, (r, k), generator=gen, dtype=torch.int8) for r in (m, n))
    y = sparkq.int8_matmul_int32(a.to(gpu), b.to(gpu)).cpu()
    assert torch.equal(y.double(), a.double() @ b.double().T)
