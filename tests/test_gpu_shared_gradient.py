"""The one-pass backward of channel-shared normalized weights against the
oracle: the weights' gradient is the oracle's summed over the channels.  Sizes
at the edges of the 64 x 16 tiles (part tiles, the smallest image), rows
beyond the 8-pixel border, every channel count it serves, and the row rules."""
import pytest
import torch

import oracle
from helpers import assert_bound, normalized_bwd_cond, out_ulp_for, rtol_for
from neural_shift_cuda_amd import _C
from neural_shift_cuda_amd.workloads import halfplane_shifts, window_shifts
from test_shared_weights import DEV, HAS_GPU, _channel_rounding, _inputs

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not HAS_GPU, reason="needs a GPU")]

CASES = [
    ((2, 3, 48, 192), torch.float32, halfplane_shifts(3), False, False),
    ((1, 3, 41, 135), torch.float32, halfplane_shifts(5), True, True),
    ((1, 2, 32, 32), torch.float32, window_shifts(2), False, True),
    ((1, 3, 67, 73), torch.float32, halfplane_shifts(8)[::5], True, False),
    ((2, 3, 50, 65), torch.float16, halfplane_shifts(6)[::3], True, True),
    ((1, 2, 33, 129), torch.bfloat16, halfplane_shifts(4), False, True),
    ((1, 3, 45, 130), torch.float32, halfplane_shifts(11)[::6], False, True),
    ((1, 3, 45, 131), torch.float16, halfplane_shifts(10)[::5], True, False),
]


@pytest.mark.parametrize("shape,dtype,table,log_weights,box", CASES)
def test_one_pass_shared_gradient(shape, dtype, table, log_weights, box):
    print(f"\ncase: shared gradient {shape} {dtype} S={table.size(0)} log={log_weights} box={box}",
          flush=True)
    B, C, H, W = shape
    x, w, gD, gL = _inputs(B, C, H, W, table.size(0), dtype, 3, positive=not log_weights)
    rules = _C.NSH_BOX_FORWARD if box else 0
    sh = table.to(DEV)
    D, L = _C.normalized_accumulate_uz_forward(x.to(DEV), w.to(DEV), sh, log_weights,
                                               shared_weights=True, rules=rules)
    got = _C.normalized_accumulate_uz_backward_shared(
        x.to(DEV), w.to(DEV), D, L, gD.to(DEV), gL.to(DEV), sh, log_weights, rules=rules)
    assert got is not None and got[1].shape == w.shape
    wx = w.expand(-1, C, -1, -1).contiguous()
    if box:  # the box is a mask of the weights; a masked weight has no gradient
        hh, ww = torch.arange(H).view(1, H, 1), torch.arange(W).view(1, 1, W)
        dx, dy = table[:, 0].view(-1, 1, 1), table[:, 1].view(-1, 1, 1)
        keep = (hh + dx >= 0) & (hh + dx < H) & (ww + dy >= 0) & (ww + dy < W)
        keep = keep.repeat_interleave(B, 0).unsqueeze(1)
        wx = torch.where(keep, wx, torch.full_like(wx, -float("inf") if log_weights else 0.0))
    kw = dict(log_weights=log_weights)
    Do, Lo = oracle.normalized(x, wx, table, policy="gpu", **kw)
    Ds, _ = oracle.normalized(x.abs(), wx, table, policy="gpu", **kw)
    gxo, gwo = oracle.normalized_bwd(x, wx, Do, Lo, gD, gL, table, **kw)
    gxs, gws = oracle.normalized_bwd(x.abs(), wx, -Ds, Lo, gD.abs(), gL.abs(), table, **kw)
    gxc, gwc = normalized_bwd_cond(x, wx, Lo, gD, gL, Ds, table, acc_dtype=dtype, **kw)
    rt, ou = rtol_for(dtype), out_ulp_for(dtype)
    assert_bound(got[0], gxo, gxs, rt, "grad_x", ou, extra=gxc)
    # one rounding of the sum: within the bound of a rounding per channel
    gsc = gws.sum(1, keepdim=True)
    assert_bound(got[1], gwo.sum(1, keepdim=True), gsc, rt, "grad_w", ou,
                 extra=gwc.sum(1, keepdim=True) + _channel_rounding(dtype, C))


def test_one_pass_shared_gradient_declines():
    """One channel, four, fp64 and small images are left to the per-channel
    kernels: nothing is launched and None is returned."""
    for shape, dtype in [((1, 1, 64, 64), torch.float32), ((1, 4, 64, 64), torch.float32),
                         ((1, 3, 64, 64), torch.float64), ((1, 3, 31, 64), torch.float32)]:
        sh = halfplane_shifts(2)
        x, w, gD, gL = (t.to(DEV) for t in _inputs(*shape, sh.size(0), dtype, 1, positive=True))
        assert _C.normalized_accumulate_uz_backward_shared(
            x, w, gD, gL, gD, gL, sh.to(DEV), False) is None
