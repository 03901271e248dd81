"""accumulate_uz_scalar on tables that are no grid: many rows beyond the halo,
sparse and repeated rows in numbers that do not divide the batches, mixtures,
tables of a few rows; infinite pixels on part tiles; and the error of the
weight gradient's sums."""
import random

import pytest
import torch

import oracle
from helpers import assert_bound, out_ulp_for, rtol_for
from neural_shift_cuda_amd import _C

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _random(n, reach, seed):
    r = random.Random(seed)
    return [(r.randint(-reach, reach), r.randint(-reach, reach)) for _ in range(n)]


TABLES = {
    "far 101": _random(101, 200, 1),
    "far 5": [(9, 0), (-9, 8), (0, 17), (100, -100), (-33, 12)],
    "sparse 62": random.Random(2).sample([(a, b) for a in range(-8, 9) for b in range(-8, 9)], 62),
    "repeated 27": [(a, b) for a in range(-2, 3) for b in range(-2, 3)] + [(1, 0), (1, 0)],
    "mixed 150": _random(150, 14, 3),
    "grid and far": [(a, b) for a in range(-3, 4) for b in range(-3, 4)] + _random(30, 90, 4),
    "four": [(0, 0), (0, 1), (1, 0), (1, 1)],
    "two": [(-8, 8), (9, 9)],
}


def _check(dtype, shape, rows, seed):
    B, C, H, W = shape
    g = torch.Generator().manual_seed(seed)
    acc = torch.float64 if dtype == torch.float64 else torch.float32
    sh = torch.tensor(rows, dtype=torch.int64)
    x = torch.randn(shape, generator=g).to(dtype)
    w = torch.rand(len(rows), B, C, generator=g).to(dtype)
    gU, gZ = (torch.randn(shape, generator=g).to(acc) for _ in range(2))
    U, Z = _C.accumulate_uz_scalar_forward(x.to(DEV), w.to(DEV), sh.to(DEV))
    gx, gw = _C.accumulate_uz_scalar_backward(x.to(DEV), w.to(DEV), gU.to(DEV), gZ.to(DEV),
                                              sh.to(DEV))
    Uo, Zo = oracle.accumulate_uz_scalar(x, w, sh)
    Us, Zs = oracle.accumulate_uz_scalar(x.abs(), w.abs(), sh)
    gxo, gwo = oracle.accumulate_uz_scalar_bwd(x, w, gU, gZ, sh)
    gxs, gws = oracle.accumulate_uz_scalar_bwd(x.abs(), w.abs(), gU.abs(), gZ.abs(), sh)
    rt, ulp = rtol_for(dtype), out_ulp_for(dtype)
    assert_bound(U, Uo, Us, rt, "U")
    assert_bound(Z, Zo, Zs, rt, "Z")
    assert_bound(gx, gxo, gxs, rt, "grad_x", ulp)
    assert_bound(gw, gwo, gws, rt, "grad_w", ulp)


@pytest.mark.parametrize("table", list(TABLES))
@pytest.mark.parametrize("shape", [(2, 1, 33, 65), (1, 2, 64, 128), (1, 1, 5, 7), (1, 1, 31, 200)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float64])
def test_rows(dtype, shape, table):
    print("[case] scalar rows", dtype, shape, table, flush=True)
    _check(dtype, shape, TABLES[table], len(table))


@pytest.mark.parametrize("S", [64, 65, 1024])
def test_list_lengths(S):
    """Tables at the edges of the 64-row steps that list their rows."""
    print("[case] scalar list", S, flush=True)
    _check(torch.float32, (1, 1, 40, 70), _random(S, 12, S), S)


def test_infinite_pixel_on_part_tiles():
    """A row beyond the halo multiplies no lane outside the image with the
    pixel that lane reads (0 x inf)."""
    x = torch.rand(1, 1, 40, 70)
    x[0, 0, 20, 30] = float("inf")
    rows = torch.tensor([(12, 3), (-15, 40), (9, -9)])
    g = torch.rand(1, 1, 40, 70) + 0.5
    _, gw = _C.accumulate_uz_scalar_backward(x.to(DEV), torch.ones(3, 1, 1, device=DEV), g.to(DEV),
                                             g.to(DEV), rows.to(DEV))
    assert torch.isposinf(gw).all()


def _waves_of_four(gu, x):
    """The sums of N x 32 x 64 products as eight waves form them, a lane
    adding four pixels: lane sums, a tree over the 64 lanes, the waves in order."""
    n = gu.shape[0]
    gu, x = (t.view(n, 8, 4, 4, 16).double() for t in (gu, x))
    acc = torch.zeros(n, 8, 4, 16)
    for k in range(4):
        acc = (gu[:, :, :, k] * x[:, :, :, k] + acc.double()).float()
    acc = acc.view(n, 8, 64)
    while acc.shape[-1] > 1:
        acc = acc[..., 0::2] + acc[..., 1::2]
    t = torch.zeros(n)
    for i in range(8):
        t = t + acc[:, i, 0]
    return t


@pytest.mark.parametrize("rows", [[(a, b) for a in range(-1, 2) for b in range(-1, 2)],
                                  [(-7, 3), (0, 0), (5, -6)], [(12, 9), (-13, 0), (0, 40)]],
                         ids=["grid", "near", "far"])
def test_weight_gradient_error(rows):
    """Root mean square error against 64 bits, of one tile per plane: no more
    than 1.1 times that of eight waves of four-pixel lanes (measured in
    simulation 0.97; one chain over a lane's 32 rows gives 1.28, and 3000 sums
    determine the ratio to about 0.02)."""
    planes = 3000 // len(rows)
    g = torch.Generator().manual_seed(5)
    x, gu = torch.rand(planes, 1, 32, 64, generator=g), torch.randn(planes, 1, 32, 64, generator=g)
    sh = torch.tensor(rows)
    _, gw = _C.accumulate_uz_scalar_backward(
        x.to(DEV), torch.ones(len(rows), planes, 1, device=DEV), gu.to(DEV),
        torch.zeros_like(gu).to(DEV), sh.to(DEV))
    err, ref = [], []
    for s, (dx, dy) in enumerate(rows):
        v = torch.roll(x, (-dx, -dy), (-2, -1))
        exact = (gu.double() * v.double()).sum((1, 2, 3))
        err.append(gw[s, :, 0].cpu().double() - exact)
        ref.append(_waves_of_four(gu[:, 0], v[:, 0]).double() - exact)
    err, ref = torch.cat(err), torch.cat(ref)
    assert err.square().mean().sqrt() <= 1.1 * ref.square().mean().sqrt()
