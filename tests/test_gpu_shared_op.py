"""normalized_accumulate_uz with channel-shared weights through autograd at
sizes whose backward forms the weights' own gradient in one pass
(B * H * W >= ops._ONE_PASS_PIXELS), with the row rules, one upstream
gradient only, and types that fall back to the per-channel kernels; against
the oracle, its weight gradient summed over the channels.  The x gradient is
within the same bound; it equals the broadcast weights' bit for bit only where
the per-channel kernels run."""
import sys

import pytest
import torch

import oracle
import test_periodic_inverse as periodic
from helpers import assert_bound, normalized_bwd_cond, out_ulp_for, rtol_for
from neural_shift_cuda import normalized_accumulate_uz
from neural_shift_cuda_amd import _C, ops
from neural_shift_cuda_amd.workloads import halfplane_shifts
from test_shared_weights import DEV, _channel_rounding, _inputs

pytestmark = pytest.mark.gpu

NEAR = halfplane_shifts(2)
FAR = torch.tensor([(0, 0, 0), (1, -2, 1), (0, 3, 1), (4, 11, 1), (-2, 1, 1)])


def _run(shape, dtype, sh, log, upstream, **rules):
    B, C, H, W = shape
    x, w, gD, gL = _inputs(B, C, H, W, sh.size(0), dtype, 3, positive=not log)
    xd, wd = x.to(DEV).requires_grad_(True), w.to(DEV).requires_grad_(True)
    out = normalized_accumulate_uz(xd, wd, sh.to(DEV), log_weights=log, return_log_degree=True,
                                   shared_weights=True, **rules)
    grads = {"both": (gD, gL), "D": (gD, None), "log_C": (None, gL)}[upstream]
    used = [(o, g.to(DEV)) for o, g in zip(out, grads) if g is not None]
    gx, gw = torch.autograd.grad([o for o, _ in used], [xd, wd], [g for _, g in used])
    zero = torch.zeros_like(gD)
    return x, w, *(zero if g is None else g for g in grads), gx, gw


CASES = [
    ((2, 3, 130, 131), torch.float32, NEAR, "both", {}),
    ((2, 3, 130, 131), torch.float32, NEAR, "D", {}),
    ((2, 3, 130, 131), torch.float32, NEAR, "log_C", {}),
    ((1, 2, 182, 181), torch.bfloat16, NEAR, "both", {}),
    ((2, 3, 129, 128), torch.float32, FAR, "both", dict(periodic_inverse=True)),
    ((1, 3, 180, 190), torch.float16, FAR, "both", dict(periodic_inverse=True)),
    ((2, 2, 130, 131), torch.float32, NEAR, "both", dict(periodic_inverse=True)),
    ((1, 3, 181, 182), torch.float64, NEAR, "both", {}),        # per channel
    ((1, 4, 181, 182), torch.float32, NEAR, "both", {}),        # per channel
]


@pytest.mark.parametrize("shape,dtype,sh,upstream,rules", CASES, ids=str)
@pytest.mark.parametrize("log", [False, True])
def test_gradients(monkeypatch, shape, dtype, sh, upstream, rules, log):
    print("[case] shared op", shape, dtype, upstream, rules, log, flush=True)
    sys.stdout.flush()
    B, C, H, W = shape
    assert B * H * W >= ops._ONE_PASS_PIXELS
    served = []
    one_pass = _C.normalized_accumulate_uz_backward_shared
    monkeypatch.setattr(_C, "normalized_accumulate_uz_backward_shared",
                        lambda *a, **k: served.append(one_pass(*a, **k)) or served[-1])
    x, w, gD, gL, gx, gw = _run(shape, dtype, sh, log, upstream, **rules)
    assert [s is not None for s in served] == [dtype != torch.float64 and C in (2, 3)]
    assert gw.shape == w.shape
    wx = w.expand(-1, C, -1, -1).contiguous()
    if rules:  # the circular mirrors as rows of their own
        te, we, pos, mirror = periodic._explicit(sh, wx, B)
        fold = lambda t: periodic._fold(t, sh, pos, mirror, B)  # noqa: E731
    else:
        te, we, fold = sh, wx, lambda t: t  # noqa: E731
    kw = dict(log_weights=log)
    Do, Lo = oracle.normalized(x, we, te, policy="gpu", **kw)
    Ds, _ = oracle.normalized(x.abs(), we, te, policy="gpu", **kw)
    gxo, gwo = oracle.normalized_bwd(x, we, Do, Lo, gD, gL, te, **kw)
    gxs, gws = oracle.normalized_bwd(x.abs(), we, -Ds, Lo, gD.abs(), gL.abs(), te, **kw)
    gxc, gwc = normalized_bwd_cond(x, we, Lo, gD, gL, Ds, te, acc_dtype=dtype, **kw)
    rt, ou = rtol_for(dtype), out_ulp_for(dtype)
    assert_bound(gx, gxo, gxs, rt, "grad_x", ou, extra=gxc)
    gsc = fold(gws).sum(1, keepdim=True)
    # per channel, each channel's gradient is rounded before the sum
    extra = fold(gwc).sum(1, keepdim=True) + ou * gsc + _channel_rounding(dtype, C)
    assert_bound(gw, fold(gwo).sum(1, keepdim=True), gsc, rt, "grad_w", 2 * ou, extra=extra)


@pytest.mark.parametrize("shape", [(1, 3, 181, 180), (1, 3, 182, 182)])
def test_x_gradient_on_either_side_of_the_line(shape):
    """Bitwise the broadcast weights' below the line; above it the sums run in
    another order, each term the same."""
    sh = halfplane_shifts(3)
    B, C, H, W = shape
    x, w, gD, gL, gx, _ = _run(shape, torch.float32, sh, False, "both")
    xe = x.to(DEV).requires_grad_(True)
    we = w.to(DEV).expand(-1, C, -1, -1).contiguous()
    out = normalized_accumulate_uz(xe, we, sh.to(DEV), return_log_degree=True)
    ge, = torch.autograd.grad(out, [xe], [gD.to(DEV), gL.to(DEV)])
    if B * H * W < ops._ONE_PASS_PIXELS:
        assert torch.equal(gx, ge)
        return
    # f gD summed over the table in another order: each sum within rtol of the
    # sum of its terms' magnitudes, the x gradient for |gD|
    xa = x.to(DEV).requires_grad_(True)
    D = normalized_accumulate_uz(xa, we, sh.to(DEV))
    scale, = torch.autograd.grad(D, [xa], [gD.abs().to(DEV)])
    assert_bound(gx, ge.double(), scale.double(), rtol_for(torch.float32), "grad_x")
