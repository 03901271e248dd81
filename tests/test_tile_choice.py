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
    # the fp32 backward on rows of whole 16s: 1-pixel lanes while three
    # workgroups per compute unit hold them, then 2-pixel ones
    (25, (1, 1, 512, 512), F32, BWD, (16, 32)),
    (113, (16, 1, 128, 128), F32, BWD, (16, 32)),
    (81, (16, 1, 144, 144), F32, BWD, (16, 32)),
    (81, (16, 1, 160, 160), F32, BWD, (32, 32)),
    (81, (4, 1, 384, 384), F32, BWD, (32, 32)),
    (121, (8, 1, 352, 352), F32, BWD, (32, 32)),
    (121, (34, 1, 361, 80), F32, BWD, (32, 32)),
    (81, (8, 1, 304, 304), F32, BWD, (64, 32)),
    # other rows, and two columns of 64 where 128-wide tiles idle half of one
    (81, (3, 1, 387, 386), F32, BWD, (32, 32)),
    (49, (298, 1, 100, 134), F32, BWD, (64, 32)),
    (61, (8, 1, 352, 352), F16, BWD, (32, 32)),
    (85, (192, 1, 48, 96), F16, BWD, (32, 32)),
    (41, (2, 1, 820, 520), F16, BWD, (64, 32)),
    (81, (8, 1, 304, 304), F16, BWD, (64, 32)),
    # fp64: 1-pixel lanes below four workgroups per compute unit
    (25, (17, 1, 100, 140), F64, FWD, (32, 16)),
    (5, (3, 1, 361, 230), F64, BWD, (32, 16)),
    # tables hinted beyond 8 pixels on tiles without a wider border
    (181, (4, 1, 280, 391), F64 | WIDE, FWD, None),
    (181, (4, 1, 280, 391), F64 | WIDE, BWD, None),
    (221, (1, 3, 953, 97), F16 | WIDE, BWD, None),
    (181, (1, 1, 592, 592), F64 | WIDE, BWD, (32, 16)),
    # and on those with one
    (181, (4, 1, 368, 384), F32 | WIDE, FWD, (128, 32, 16)),
    (181, (2, 1, 1251, 148), F32 | WIDE, BWD, (64, 32, 24)),
    # a few rows on many badly filled tiles
    (5, (154, 1, 259, 100), F32, FWD, None),
    (5, (3, 1, 660, 660), F64, FWD, None),
    (5, (8, 1, 1148, 383), F32, BWD, (128, 32)),
]


@pytest.mark.parametrize("S,shape,dtype,backward,tile", CASES, ids=str)
def test_tiles(S, shape, dtype, backward, tile):
    got = _bytes(S, *shape, dtype, backward)
    assert got == (0 if tile is None else _tiles(*shape, dtype, backward, *tile))
