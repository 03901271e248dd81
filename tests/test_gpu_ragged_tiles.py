"""Scatter tiles on images that no tile divides: a last row or column of tiles
shorter than the tables' radius takes part of the one before, one tile in a
direction is its own neighbour, and rows that no vector divides (or unaligned
buffers) take the strided backward.  Against the oracle, and scatter against
gather kernels."""
import sys

import pytest
import torch

import test_gpu_normalized_scatter as norm
import test_gpu_scatter as acc
from helpers import assert_bound, out_ulp_for, rtol_for
from neural_shift_cuda_amd import _C
from neural_shift_cuda_amd.workloads import halfplane_shifts, window_shifts

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _say(*what):
    print("[case]", *what, flush=True)
    sys.stdout.flush()


# lanes of 4 pixels (many planes), 2 and 1; remainders 1..7 of the tile in
# either direction; W a multiple of 4, of 2 and odd; single tiles
ACC_SHAPES = [
    (torch.float32, (8, 1, 321, 481)),    # 128 x 32, both ragged, odd
    (torch.float32, (8, 1, 321, 260)),    # rows of whole vectors, ragged columns
    (torch.float32, (10, 1, 257, 390)),   # W % 4 = 2
    (torch.float32, (240, 1, 65, 67)),    # 64 x 32, two columns, the last of 3
    (torch.float32, (512, 1, 39, 51)),    # one column of tiles
    (torch.float32, (500, 1, 32, 64)),    # one tile
    (torch.float32, (2, 1, 33, 35)),      # 1-pixel lanes
    (torch.float16, (64, 1, 130, 131)),
    (torch.bfloat16, (1, 1, 49, 53)),
    (torch.float64, (60, 1, 65, 67)),
    (torch.float64, (1, 1, 33, 32)),
]


@pytest.mark.parametrize("dtype,shape", ACC_SHAPES)
@pytest.mark.parametrize("table", ["half8", "win2", "selfinv"])
def test_accumulate_ragged(dtype, shape, table):
    _say("accumulate", dtype, shape, table)
    sh = acc._table(table)
    sh = sh[::5] if sh.size(0) > 100 else sh  # radius 8 in fewer rows
    assert acc._uses_workspace(dtype, shape, sh.size(0), False)
    assert acc._uses_workspace(dtype, shape, sh.size(0), True)
    acc._run_and_check(dtype, shape, sh, 5)


@pytest.mark.parametrize("shape", [(8, 1, 321, 481), (10, 1, 260, 131)])
@pytest.mark.parametrize("table", [halfplane_shifts(10)[::6], window_shifts(4), torch.tensor(
    [[0, 0, 0], [17, 3, 1], [-2, 20, 1], [30, 1, 1]])], ids=["half10", "win4", "far"])
def test_accumulate_ragged_wide_tables(shape, table):
    _say("accumulate wide", shape, table.size(0))
    acc._run_and_check(torch.float32, shape, table, 6)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32, torch.float64])
def test_accumulate_unaligned_buffers(dtype):
    """Contiguous tensors that start one element into their storage."""
    shape, sh = (20, 1, 200, 264), halfplane_shifts(3)
    B, C, H, W = shape
    S = sh.size(0)
    g = torch.Generator().manual_seed(2)
    a = _C._acc_dtype(dtype)

    def shifted(t):
        out = torch.empty(t.numel() + 1, dtype=t.dtype, device=DEV)[1:].view(t.shape)
        return out.copy_(t)

    x, w = torch.rand(shape, generator=g).to(dtype), torch.rand(S * B, C, H, W, generator=g).to(dtype)
    gU, gZ = torch.rand(shape, generator=g).to(a), torch.rand(shape, generator=g).to(a)
    shd = sh.to(DEV)
    one = _C.accumulate_uz_forward(x.to(DEV), w.to(DEV), shd)
    two = _C.accumulate_uz_forward(shifted(x), shifted(w), shd)
    assert all(torch.equal(p, q) for p, q in zip(one, two))
    one = _C.accumulate_uz_backward(x.to(DEV), w.to(DEV), gU.to(DEV), gZ.to(DEV), shd)
    two = _C.accumulate_uz_backward(shifted(x), shifted(w), shifted(gU), shifted(gZ), shd)
    # every term is positive; the same sums, fused differently
    for p, q in zip(one, two):
        assert_bound(q, p, p, rtol_for(dtype), "strided against contiguous", out_ulp_for(dtype))


NORM_SHAPES = [
    (torch.float32, (2, 2, 65, 257)),     # 128 x 32
    (torch.float32, (1, 1, 97, 134)),
    (torch.float32, (3, 1, 65, 67)),      # one 128-wide column
    (torch.float32, (3, 1, 37, 64)),      # 64-wide tiles, one column
    (torch.float32, (2, 2, 70, 45)),
    (torch.float16, (2, 1, 66, 69)),
    (torch.bfloat16, (1, 2, 33, 40)),
    (torch.float64, (1, 1, 33, 65)),
    (torch.float64, (2, 1, 49, 34)),
]


@pytest.mark.parametrize("dtype,shape", NORM_SHAPES)
@pytest.mark.parametrize("table", ["half8", "win2", "selfinv", "far"])
@pytest.mark.parametrize("log_weights", [False, True])
def test_normalized_ragged(dtype, shape, table, log_weights):
    _say("normalized", dtype, shape, table, log_weights)
    assert norm._uses_scatter(shape, dtype, norm._table(table).size(0))
    norm.test_normalized_scatter_vs_oracle(dtype, shape, table, log_weights)


def test_normalized_mixed_heads_on_narrow_images():
    """Head mixing in the forward on an image the 64-wide tiles serve."""
    from neural_shift_cuda import normalized_accumulate_uz
    from neural_shift_cuda.ops import normalized_accumulate_uz_mixed
    g = torch.Generator().manual_seed(9)
    sh = halfplane_shifts(4)
    S = sh.size(0)
    x = torch.rand(2, 3, 41, 50, generator=g).to(DEV)
    hw = torch.rand(S * 2, 2, 41, 50, generator=g).to(DEV)
    mix = torch.rand(3, 2, generator=g).to(DEV)
    with torch.no_grad():
        D, L = normalized_accumulate_uz_mixed(x, hw, mix, sh.to(DEV), return_log_degree=True)
        w = (mix.view(1, 3, 2, 1, 1) * hw.unsqueeze(1)).sum(2)
        Do, Lo = normalized_accumulate_uz(x, w, sh.to(DEV), return_log_degree=True)
    assert_bound(D, Do, Do.abs(), 1e-5, "D")
    assert_bound(L, Lo, Lo.abs(), 1e-5, "log_C")


@pytest.mark.parametrize("dtype,H,W", [(torch.float32, 2300, 2300), (torch.float16, 2240, 2304),
                                       (torch.float32, 4001, 4009)])
def test_noalloc_forward_beyond_the_preferred_tiles(dtype, H, W):
    """The preferred tiles' workspace exceeds the static scratch: the wide
    tiles that fit it, or the gather kernels for ragged images."""
    import ctypes
    _say("noalloc", dtype, H, W)
    lib = ctypes.CDLL(_C.LIBRARY_PATH)
    P, I64, I = ctypes.c_void_p, ctypes.c_int64, ctypes.c_int
    lib.nsh_accumulate_uz_forward_noalloc.argtypes = [P, P, P] + [I64] * 5 + [I, P, P, P]
    lib.nsh_accumulate_uz_workspace_bytes.argtypes = [I64] * 5 + [I, I]
    lib.nsh_accumulate_uz_workspace_bytes.restype = I64
    code = 3 if dtype == torch.float32 else 1
    sh = torch.tensor([[0, 0, 1], [3, -2, 1]], device=DEV)
    assert lib.nsh_accumulate_uz_workspace_bytes(2, 1, 1, H, W, code, 0) > (32 << 20)
    x = torch.rand(1, 1, H, W, device=DEV).to(dtype)
    w = torch.rand(2, 1, H, W, device=DEV).to(dtype)
    U, Z = torch.empty(1, 1, H, W, device=DEV), torch.empty(1, 1, H, W, device=DEV)
    rc = lib.nsh_accumulate_uz_forward_noalloc(
        x.data_ptr(), w.data_ptr(), sh.data_ptr(), 2, 1, 1, H, W, code, U.data_ptr(),
        Z.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    U2, Z2 = _C.accumulate_uz_forward(x, w, sh)
    # sums of at most four terms in [0, 1): orders differ by a few ulp of 4
    torch.testing.assert_close(U, U2, rtol=0, atol=2e-6)
    torch.testing.assert_close(Z, Z2, rtol=0, atol=2e-6)
