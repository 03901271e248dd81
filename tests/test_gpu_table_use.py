"""How the ops use a caller's shift table: the normalized op learns nothing by
waiting for the device, and a differentiable call with row rules keeps a table
of its own."""
import pytest
import torch

from neural_shift_cuda import accumulate_uz, normalized_accumulate_uz
from neural_shift_cuda_amd import _C
from neural_shift_cuda_amd.workloads import halfplane_shifts, window_shifts

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _inputs(S, dtype=torch.float32, H=40, W=72):
    g = torch.Generator().manual_seed(S)
    x = torch.rand(1, 1, H, W, generator=g).to(dtype).to(DEV)
    w = (torch.rand(S, 1, H, W, generator=g) + 0.1).to(dtype).to(DEV)
    return x.requires_grad_(True), w.requires_grad_(True)


TABLES = {
    "half9": halfplane_shifts(9),
    "half10": halfplane_shifts(10),
    "window7": window_shifts(7),
    "odd count": halfplane_shifts(10)[:200],
    "small": halfplane_shifts(3),
}


@pytest.mark.parametrize("table", list(TABLES))
@pytest.mark.parametrize("index", [torch.int64, torch.int32])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_normalized_does_not_wait(table, index, dtype):
    """New device tables, as a caller makes them per call: forward, weight
    check and backward without a synchronisation."""
    sh = TABLES[table].to(device=DEV, dtype=index)
    x, w = _inputs(sh.size(0), dtype)
    normalized_accumulate_uz(x, w, sh.clone()).sum().backward()  # libraries, workspaces
    fresh = sh.clone()
    torch.cuda.synchronize()
    torch.cuda.set_sync_debug_mode("error")
    try:
        D = normalized_accumulate_uz(x, w, fresh, validate=True)
        torch.autograd.grad(D, [x, w], torch.ones_like(D))
    finally:
        torch.cuda.set_sync_debug_mode("default")


def test_fp64_forward_does_not_wait():
    sh = halfplane_shifts(4).to(device=DEV, dtype=torch.int32)
    x, w = _inputs(sh.size(0), torch.float64)
    with torch.no_grad():
        normalized_accumulate_uz(x, w, sh.clone())
        fresh = sh.clone()
        torch.cuda.synchronize()
        torch.cuda.set_sync_debug_mode("error")
        try:
            normalized_accumulate_uz(x, w, fresh)
        finally:
            torch.cuda.set_sync_debug_mode("default")


def test_hint_of_an_unread_table():
    for R in range(9, 17):
        assert _C._norm_halo_flag(halfplane_shifts(R).to(DEV), torch.float32) == _C.NSH_WIDE_HALO
    for t in (window_shifts(7), window_shifts(8), halfplane_shifts(10)[:200]):
        assert _C._norm_halo_flag(t.to(DEV), torch.float32) == 0
    known = halfplane_shifts(10)[20:].to(DEV)  # a count of nothing, read for another op
    assert _C._norm_halo_flag(known, torch.float32) == 0
    assert _C.table_radius(known) == 10
    assert _C._norm_halo_flag(known, torch.float32) == _C.NSH_WIDE_HALO


@pytest.mark.parametrize("op", [accumulate_uz, normalized_accumulate_uz])
@pytest.mark.parametrize("rules", [dict(periodic_inverse=True), dict(box_forward=True)])
def test_table_rewritten_before_the_backward(op, rules):
    """The gradients are those of the table the forward saw."""
    want = []
    for rewrite in (False, True):
        sh = halfplane_shifts(3).to(DEV)
        x, w = _inputs(sh.size(0))
        out = op(x, w, sh, **rules)
        out = out[0] if isinstance(out, tuple) else out
        if rewrite:
            sh.zero_()
        want.append(torch.autograd.grad(out, [x, w], torch.ones_like(out)))
    for a, b in zip(*want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("op", [accumulate_uz, normalized_accumulate_uz])
def test_rewritten_table_is_reported_without_rules(op):
    sh = halfplane_shifts(3).to(DEV)
    x, w = _inputs(sh.size(0))
    out = op(x, w, sh)
    out = out[0] if isinstance(out, tuple) else out
    sh.zero_()
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(out, [x, w], torch.ones_like(out))
