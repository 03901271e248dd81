"""Which shapes nsh_accumulate_uz_forward_noalloc takes: those whose tiles fit
its static scratch, images of one tile row or column and images ending 1..7
pixels past whole 16s at any batch size (gather kernels), and tables
hinted beyond 8 pixels whose wider border's tiles do not fit."""
from __future__ import annotations

import ctypes
import sys

import pytest
import torch

from neural_shift_cuda_amd import _C

F16, BF16, F32, F64 = 1, 2, 3, 4
WIDE, WIDER = _C.NSH_WIDE_HALO, _C.NSH_WIDER_HALO

# S, B, C, H, W, dtype
SERVED = [
    (121, 256, 1, 32, 704, F16),
    (5, 64, 3, 512, 64, F32),
    (5, 512, 3, 64, 64, F32),
    (2, 2048, 1, 64, 64, F32),
    (2, 4096, 1, 32, 32, F32),
    (25, 154, 1, 219, 32, F64),
    (61, 997, 2, 2416, 32, F16),
    (225, 1771, 1, 40, 64, F16 | WIDE),
    (225, 234, 1, 6620, 48, F16 | _C.NSH_SHARED_WEIGHTS),
    (5, 3809, 2, 1216, 48, BF16 | WIDE),
    (1013, 1, 3, 3680, 128, F16 | WIDER),
    (225, 1, 3, 1280, 768, BF16 | WIDE),
    (225, 2, 1, 2856, 458, F16 | WIDE),
    (225, 4, 1, 681, 555, F32 | WIDER),
    (85, 235, 1, 60, 268, F16 | _C.NSH_NARROW_HALO),
    (113, 7, 2, 1088, 304, F32),
    (85, 1, 1, 8191, 8193, F32),
]
REFUSED = [
    (85, 1, 1, 8192, 8192, F32),
    (113, 8, 1, 2048, 2048, F16),
    (5, 600, 3, 96, 128, F32),
    (225, 16, 1, 1024, 1024, F64),
]


def _lib():
    lib = ctypes.CDLL(_C.LIBRARY_PATH)
    P, I64, I = ctypes.c_void_p, ctypes.c_int64, ctypes.c_int
    lib.nsh_accumulate_uz_forward_noalloc.argtypes = [P, P, P] + [I64] * 5 + [I, P, P, P]
    lib.nsh_accumulate_uz_forward_noalloc.restype = I
    lib.nsh_last_error.restype = ctypes.c_char_p
    return lib


def _refuses(shape):
    """Whether the call ends at the scratch check.  Its operands are host
    memory, never read: without a GPU an accepted call ends at the device
    query or the launch."""
    lib = _lib()
    buf = ctypes.create_string_buffer(4096)
    p = (ctypes.addressof(buf) + 255) // 256 * 256
    *dims, dtype = shape
    rc = lib.nsh_accumulate_uz_forward_noalloc(p, p, p, *dims, dtype, p, p, None)
    assert rc != 0
    return rc == 1 and b"static scratch" in lib.nsh_last_error()


@pytest.mark.skipif(torch.cuda.is_available(), reason="an accepted call would launch")
@pytest.mark.parametrize("shape", SERVED + REFUSED, ids=str)
def test_shapes_served_and_refused(shape):
    assert _refuses(shape) == (shape in REFUSED)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(2048, 1, 64, 64), (4096, 1, 32, 32), (96, 1, 16, 4096)],
                         ids=str)
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_batches_of_single_tiles(shape, dtype):
    B, C, H, W = shape
    print("[case] noalloc", dtype, shape, flush=True)
    sys.stdout.flush()
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(H + W)
    sh = torch.tensor([[0, 0, 1], [3, -2, 1]], device=dev)
    x = torch.rand(shape, generator=g, device=dev).to(dtype)
    w = torch.rand((2 * B, C, H, W), generator=g, device=dev).to(dtype)
    U, Z = torch.empty(shape, device=dev), torch.empty(shape, device=dev)
    lib = _lib()
    rc = lib.nsh_accumulate_uz_forward_noalloc(
        x.data_ptr(), w.data_ptr(), sh.data_ptr(), 2, B, C, H, W,
        F32 if dtype == torch.float32 else F16, U.data_ptr(), Z.data_ptr(),
        torch.cuda.current_stream().cuda_stream)
    assert rc == 0, lib.nsh_last_error().decode()
    U2, Z2 = _C.accumulate_uz_forward(x, w, sh)
    # sums of at most four terms in [0, 1): orders differ by a few ulp of 4
    torch.testing.assert_close(U, U2, rtol=0, atol=2e-6)
    torch.testing.assert_close(Z, Z2, rtol=0, atol=2e-6)
