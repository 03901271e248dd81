"""periodic_inverse / box_forward applied as the kernels decode the table
(`rules`) against the same rules written into the table (row codes): the same
bits, for every has_inverse value, on scatter tiles, gather kernels, wide
borders and rows beyond them; and through the public ops for tables of another
type or layout."""
import pytest
import torch

from neural_shift_cuda_amd.workloads import halfplane_rows

pytestmark = pytest.mark.gpu

RULES = [(False, False), (True, False), (False, True), (True, True)]
ROWS = {
    "flags": [(0, 0, 0), (1, 2, 1), (-2, 1, 2), (3, -3, 5), (0, 4, -1), (2, 0, 7), (1, -1, 4)],
    "wide": [(0, 0, 0), (11, -2, 1), (3, 12, 3), (1, 1, 0)],
    "far": [(0, 1, 1), (30, 2, 1), (-3, 47, 0), (2, 2, 9)],
}


@pytest.mark.parametrize("shape", [(1, 2, 70, 140), (2, 1, 20, 21)])
@pytest.mark.parametrize("rows", list(ROWS))
@pytest.mark.parametrize("periodic,box", RULES)
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32, torch.float64])
def test_rules_equal_row_codes(dtype, periodic, box, rows, shape):
    from neural_shift_cuda_amd import _C
    from neural_shift_cuda_amd.ops import _mirror_table
    g = torch.Generator().manual_seed(1)
    sh = torch.tensor(ROWS[rows]).cuda()
    B, C, H, W = shape
    S = len(ROWS[rows])
    x = torch.rand(shape, generator=g).to(dtype).cuda()
    w = torch.rand(S * B, C, H, W, generator=g).to(dtype).cuda()
    acc = _C._acc_dtype(dtype)
    gU, gZ = (torch.rand(shape, generator=g).to(acc).cuda() for _ in range(2))
    table, codes = _mirror_table(sh, periodic, box)
    rules = (_C.NSH_PERIODIC_INVERSE if periodic else 0) | (_C.NSH_BOX_FORWARD if box else 0)

    def same(a, b):
        assert all(torch.equal(p, q) for p, q in zip(a, b))

    same(_C.accumulate_uz_forward(x, w, table, row_codes=codes),
         _C.accumulate_uz_forward(x, w, sh, rules=rules))
    same(_C.accumulate_uz_backward(x, w, gU, gZ, table, row_codes=codes),
         _C.accumulate_uz_backward(x, w, gU, gZ, sh, rules=rules))
    for log in (False, True):
        a = _C.normalized_accumulate_uz_forward(x, w, table, log, row_codes=codes)
        same(a, _C.normalized_accumulate_uz_forward(x, w, sh, log, rules=rules))
        same(_C.normalized_accumulate_uz_backward(x, w, *a, gU, gZ, table, log, row_codes=codes),
             _C.normalized_accumulate_uz_backward(x, w, *a, gU, gZ, sh, log, rules=rules))


@pytest.mark.parametrize("form", ["int32", "columns", "host"])
def test_other_tables(form):
    from neural_shift_cuda import accumulate_uz, normalized_accumulate_uz
    rows = halfplane_rows(3)
    sh = torch.tensor(rows).cuda()
    other = {"int32": lambda: sh.to(torch.int32), "host": lambda: sh.cpu(),
             "columns": lambda: sh.t().contiguous().t()}[form]()
    x = torch.rand(1, 1, 70, 140).cuda()
    w = torch.rand(len(rows), 1, 70, 140).cuda()
    for fn in (accumulate_uz, lambda *a, **k: (normalized_accumulate_uz(*a, **k),)):
        for periodic, box in RULES:
            a = fn(x, w, sh, periodic_inverse=periodic, box_forward=box)
            b = fn(x, w, other, periodic_inverse=periodic, box_forward=box)
            assert all(torch.equal(p, q) for p, q in zip(a, b))
