"""The normalized forward's own check of the weight contract (weights_ok): one
weight outside it, anywhere, is reported, and every weight inside it passes --
on the scatter kernels, the gather kernels (image too small for tiles) and for
rows beyond the LDS border, with and without the forward box."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DTYPES = [torch.float16, torch.bfloat16, torch.float32, torch.float64]
INF, NAN = float("inf"), float("nan")


def _forward(w, shape, rows, log, box):
    from neural_shift_cuda_amd import _C
    B, C, H, W = shape
    sh = torch.tensor([(dx, dy, inv | (4 if box else 0)) for dx, dy, inv in rows], device="cuda")
    x = torch.rand(shape, device="cuda").to(w.dtype)
    ok = torch.ones((), dtype=torch.int32, device="cuda")
    _C.normalized_accumulate_uz_forward(x, w, sh, log, row_codes=box, weights_ok=ok)
    return int(ok.item())


# scatter tiles with partial last ones; gather (one tile)
@pytest.mark.parametrize("shape", [(1, 2, 75, 150), (2, 1, 20, 21)])
@pytest.mark.parametrize("box", [False, True])
@pytest.mark.parametrize("log", [False, True])
@pytest.mark.parametrize("dtype", DTYPES)
def test_weight_check(dtype, log, box, shape):
    B, C, H, W = shape
    rows = [(0, 0, 0), (2, -1, 1), (-3, 3, 0), (1, 11, 1)]  # the last beyond the 8-pixel border
    S = len(rows)
    g = torch.Generator().manual_seed(3)
    w = torch.rand(S * B, C, H, W, generator=g).to(dtype).cuda()
    big, tiny = torch.finfo(dtype).max, torch.finfo(dtype).smallest_normal / 4
    good = [big, tiny, 0.0, -0.0] + ([-big, -INF] if log else [])
    for i, v in enumerate(good):
        w[i % (S * B), 0, i, W - 1 - i] = v
    assert _forward(w, shape, rows, log, box) != 0
    bad = [NAN, INF] + ([] if log else [-INF, -1.0, -tiny])
    # corners (dropped by the box for some row), a tile's edge, the middle
    places = [(0, 0), (H - 1, W - 1), (H // 2, W // 2), (min(32, H - 1), 3)]
    for i, v in enumerate(bad):
        for p in range(S * B):
            h, c = places[(i + p) % len(places)]
            wb = w.clone()
            wb[p, C - 1, h, c] = v
            assert _forward(wb, shape, rows, log, box) == 0, (v, p, h, c)


def test_validate_leaves_results_alone():
    from neural_shift_cuda import normalized_accumulate_uz
    g = torch.Generator().manual_seed(4)
    sh = torch.tensor([(0, 0, 0), (1, 2, 1), (-2, 1, 1)], device="cuda")
    x = torch.rand(1, 1, 70, 140, generator=g).cuda()
    w = torch.rand(3, 1, 70, 140, generator=g).cuda()
    a = normalized_accumulate_uz(x, w, sh, return_log_degree=True, validate=True)
    b = normalized_accumulate_uz(x, w, sh, return_log_degree=True, validate=False)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
