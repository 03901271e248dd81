"""normalized_accumulate_uz on the 16-pixel border (NSH_WIDE_HALO): tables of
radius 9..16, tables inside and beyond it under the hint, image sizes around
the 64 x 32 tiles, the hint that the Python layer sets, and a workspace too
small for it; against the oracle and the gather kernels."""
import sys

import pytest
import torch

import test_gpu_normalized_scatter as norm
from helpers import assert_bound
from neural_shift_cuda_amd import _C
from neural_shift_cuda_amd.workloads import halfplane_shifts

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")

TABLES = {
    "reach16": torch.tensor([[0, 0, 0], [16, -16, 1], [-9, 12, 1], [3, 15, 0], [-16, 1, 0],
                             [2, -2, 1]]),
    "reach5": torch.tensor([[0, 0, 0], [5, -1, 1], [-2, 3, 1], [1, 0, 0]]),   # hint too wide
    "reach30": torch.tensor([[0, 0, 1], [30, 2, 1], [-4, 17, 1], [9, -9, 1], [1, 1, 0]]),
    "half10": halfplane_shifts(10),
}
SHAPES = [
    (torch.float32, (1, 2, 96, 128)),
    (torch.float32, (1, 1, 65, 70)),    # last tiles of 1 and 6: they take 16 from the ones before
    (torch.float32, (2, 1, 33, 51)),    # one column of tiles, odd rows: strided backward
    (torch.float16, (1, 2, 64, 130)),
    (torch.bfloat16, (1, 1, 47, 66)),
]


@pytest.mark.parametrize("dtype,shape", SHAPES)
@pytest.mark.parametrize("table", list(TABLES))
@pytest.mark.parametrize("log_weights", [False, True])
def test_wide_border(monkeypatch, dtype, shape, table, log_weights):
    print("[case]", dtype, shape, table, log_weights, flush=True)
    sys.stdout.flush()
    monkeypatch.setattr(_C, "_norm_halo_flag", lambda sh, dt: _C.NSH_WIDE_HALO)
    monkeypatch.setattr(norm, "_table", lambda name: TABLES[name])
    norm.test_normalized_scatter_vs_oracle(dtype, shape, table, log_weights)


def test_hint_follows_the_radius():
    wide, near = halfplane_shifts(10).to(DEV), halfplane_shifts(8).to(DEV)
    far = halfplane_shifts(17).to(DEV)
    assert _C._norm_halo_flag(wide, torch.float32) == _C.NSH_WIDE_HALO
    assert _C._norm_halo_flag(wide, torch.float64) == 0
    assert _C._norm_halo_flag(near, torch.float32) == 0
    assert _C._norm_halo_flag(far, torch.float32) == 0


@pytest.mark.parametrize("box", [False, True])
def test_mixed_heads(box):
    from neural_shift_cuda import normalized_accumulate_uz
    from neural_shift_cuda.ops import normalized_accumulate_uz_mixed
    g = torch.Generator().manual_seed(5)
    sh = halfplane_shifts(9).to(DEV)
    S = sh.size(0)
    x = torch.rand(1, 3, 70, 90, generator=g).to(DEV)
    for heads in (2, 3, 4):
        hw = torch.rand(S, heads, 70, 90, generator=g).to(DEV)
        mix = torch.rand(3, heads, generator=g).to(DEV)
        with torch.no_grad():
            D, L = normalized_accumulate_uz_mixed(x, hw, mix, sh, return_log_degree=True,
                                                  box_forward=box)
            w = (mix.view(1, 3, heads, 1, 1) * hw.unsqueeze(1)).sum(2)
            Do, Lo = normalized_accumulate_uz(x, w, sh, return_log_degree=True, box_forward=box)
        assert_bound(D, Do, Do.abs(), 1e-5, "D")
        assert_bound(L, Lo, Lo.abs(), 1e-5, "log_C")


def test_small_workspace_takes_the_base_tiles():
    """A workspace that holds the 8-pixel border's blocks only: the base tiles
    run, with the same results as without the hint."""
    sh = halfplane_shifts(10).to(DEV)
    S, (B, C, H, W) = sh.size(0), (1, 1, 130, 260)
    lib, code = _C._lib, 3
    x = torch.rand(B, C, H, W, device=DEV)
    w = torch.rand(S * B, C, H, W, device=DEV)
    st = torch.cuda.current_stream().cuda_stream
    base = lib.nsh_normalized_workspace_bytes(S, B, C, H, W, code, 0)
    assert lib.nsh_normalized_workspace_bytes(S, B, C, H, W, code | _C.NSH_WIDE_HALO, 0) > base > 0
    outs = []
    for flag in (0, _C.NSH_WIDE_HALO):
        ws = torch.empty(base, dtype=torch.uint8, device=DEV)
        D, L = torch.empty_like(x), torch.empty_like(x)
        rc = lib.nsh_normalized_accumulate_uz_forward(
            x.data_ptr(), w.data_ptr(), sh.data_ptr(), S, B, C, H, W, code | flag, 0, D.data_ptr(),
            L.data_ptr(), ws.data_ptr(), base, st)
        assert rc == 0
        outs.append((D, L))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
