"""accumulate_uz_scalar: tables the kernels lay out as a dense grid of near
rows (whole windows, half-planes whose grid has empty cells, one row, one
column) and tables they take row by row (sparse, a repeated row, rows beyond
the LDS halo), at image sizes around the 64 x 32 tile, against the oracle."""
import pytest
import torch

import oracle
from helpers import assert_bound, out_ulp_for, rtol_for
from neural_shift_cuda_amd.workloads import halfplane_rows

pytestmark = pytest.mark.gpu


def _window(r0, r1, c0, c1):
    return [(dx, dy) for dx in range(r0, r1 + 1) for dy in range(c0, c1 + 1)]


TABLES = {
    "window": _window(-5, 5, -5, 5),
    "widest": _window(-8, 8, -8, 8),
    "half": [r[:2] for r in halfplane_rows(4)],
    "one": [(3, -2)],
    "column": _window(-8, 8, 8, 8),
    "row": _window(-7, -7, -8, 5),
    "sparse": [(dx, dy) for dx in range(-8, 9, 4) for dy in range(-8, 9, 4)],
    "repeated": _window(-2, 2, -2, 2) + [(1, 1), (1, 1)],
    "near and far": _window(-1, 1, -2, 2) + [(9, 0), (0, -9), (40, 3), (-1000003, 17)],
    "far": [(9, 9), (-70, 31)],
}


@pytest.mark.parametrize("table", list(TABLES))
@pytest.mark.parametrize("shape", [(2, 2, 33, 65), (1, 1, 32, 64), (1, 2, 5, 7), (1, 1, 70, 130)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32, torch.float64])
def test_scalar_tables(dtype, shape, table):
    from neural_shift_cuda import accumulate_uz_scalar
    rows = TABLES[table]
    B, C, H, W = shape
    g = torch.Generator().manual_seed(len(rows))
    acc = torch.float64 if dtype == torch.float64 else torch.float32
    sh = torch.tensor(rows, dtype=torch.int64)
    x = torch.randn(shape, generator=g).to(dtype)
    w = torch.rand(len(rows), B, C, generator=g).to(dtype)
    gU, gZ = (torch.randn(shape, generator=g).to(acc) for _ in range(2))
    xd, wd = x.cuda().requires_grad_(True), w.cuda().requires_grad_(True)
    U, Z = accumulate_uz_scalar(xd, wd, sh.cuda())
    gx, gw = torch.autograd.grad([U, Z], [xd, wd], [gU.cuda(), gZ.cuda()])
    Uo, Zo = oracle.accumulate_uz_scalar(x, w, sh)
    Us, Zs = oracle.accumulate_uz_scalar(x.abs(), w.abs(), sh)
    gxo, gwo = oracle.accumulate_uz_scalar_bwd(x, w, gU, gZ, sh)
    gxs, gws = oracle.accumulate_uz_scalar_bwd(x.abs(), w.abs(), gU.abs(), gZ.abs(), sh)
    rt, ulp = rtol_for(dtype), out_ulp_for(dtype)
    assert_bound(U, Uo, Us, rt, "U")
    assert_bound(Z, Zo, Zs, rt, "Z")
    assert_bound(gx, gxo, gxs, rt, "grad_x", ulp)
    assert_bound(gw, gwo, gws, rt, "grad_w", ulp)


def test_empty_cells_take_no_part():
    """An infinite pixel reaches only the outputs whose rows read it."""
    from neural_shift_cuda import accumulate_uz_scalar
    rows = [(0, 0), (0, 1), (1, 0), (2, 1), (2, 2)]  # 5 of 9 cells
    x = torch.rand(1, 1, 40, 70)
    x[0, 0, 20, 30] = float("inf")
    w = torch.ones(len(rows), 1, 1)
    U, _ = accumulate_uz_scalar(x.cuda(), w.cuda(), torch.tensor(rows).cuda())
    want = torch.zeros(40, 70, dtype=torch.bool)
    for dx, dy in rows:
        want[20 - dx, 30 - dy] = True
    assert torch.equal(torch.isinf(U.cpu()[0, 0]), want) and not torch.isnan(U).any()
