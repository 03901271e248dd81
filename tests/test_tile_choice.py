"""Which tiles the accumulate_uz passes take, read off the workspace each
shape asks for: the choice must not send a shape to lanes or kernels that
measured slower (the figures are beside the rules in csrc/accumulate.hip)."""
from __future__ import annotations

import os

import pytest

from neural_shift_cuda_amd import _C

pytestmark = pytest.mark.skipif(not os.path.exists(_C.LIBRARY_PATH), reason="library not built")

F16, BF16, F32, F64 = 1, 2, 3, 4
WIDE = _C.NSH_WIDE_HALO
FWD, BWD = 0, 1


def _bytes(S, B, C, H, W, dtype, backward):
    return int(_C._lib.nsh_accumulate_uz_workspace_bytes(S, B, C, H, W, dtype, backward))


def _tiles(B, C, H, W, dtype, backward, TW, TH, halo=8):
    """Workspace of TW x TH tiles."""
    size = 8 if dtype & 7 == F64 else 4
    tiles = B * C * -(-H // TH) * -(-W // TW)
    spill = 2 * halo * (TW + 2 * halo) + 2 * halo * TH
    def align(n):
        return -(-n // 256) * 256
    part = align(B * C * H * W * 4) if backward and dtype & 7 in (F16, BF16) else 0
    return 256 + align((1 if backward else 2) * tiles * spill * size) + part


# S, (B, C, H, W), dtype, pass, tile (None: the gather kernels)
CASES = [
    # tables hinted beyond 8 pixels on tiles without a wider border
    (181, (4, 1, 280, 391), F64 | WIDE, FWD, None),
    (181, (4, 1, 280, 391), F64 | WIDE, BWD, None),
    (221, (1, 3, 953, 97), F16 | WIDE, BWD, None),
    (181, (1, 1, 592, 592), F64 | WIDE, BWD, (32, 16)),
    # a few rows on many badly filled tiles
    (5, (154, 1, 259, 100), F32, FWD, None),
    (5, (3, 1, 660, 660), F64, FWD, None),
    (5, (8, 1, 1148, 383), F32, BWD, (128, 32)),
]


@pytest.mark.parametrize("S,shape,dtype,backward,tile", CASES, ids=str)
def test_tiles(S, shape, dtype, backward, tile):
    got = _bytes(S, *shape, dtype, backward)
    assert got == (0 if tile is None else _tiles(*shape, dtype, backward, *tile))
