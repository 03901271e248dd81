"""Register spills of the built kernels, from the code objects' metadata."""
from __future__ import annotations

import os
import re
import struct

import msgpack
import pytest

from neural_shift_cuda_amd import _C

pytestmark = pytest.mark.skipif(not os.path.exists(_C.LIBRARY_PATH), reason="library not built")


def _kernels():
    """name -> metadata of every kernel in the library's gfx950 code objects."""
    data = open(_C.LIBRARY_PATH, "rb").read()
    out, at = {}, data.find(b"\x7fELF", 4)
    while at >= 0:
        machine = struct.unpack_from("<H", data, at + 18)[0]
        if machine == 224:  # EM_AMDGPU
            phoff, = struct.unpack_from("<Q", data, at + 32)
            phsize, phnum = struct.unpack_from("<HH", data, at + 54)
            for i in range(phnum):
                kind, _, off, _, _, size = struct.unpack_from("<IIQQQQ", data,
                                                              at + phoff + i * phsize)
                if kind != 4:  # PT_NOTE
                    continue
                p, end = at + off, at + off + size
                while p + 12 <= end:
                    namesz, descsz, note = struct.unpack_from("<III", data, p)
                    desc = p + 12 + (namesz + 3) // 4 * 4
                    if note == 32 and data[p + 12:p + 18] == b"AMDGPU":
                        meta = msgpack.unpackb(data[desc:desc + descsz], raw=False,
                                               strict_map_key=False)
                        out.update({k[".name"]: k for k in meta["amdhsa.kernels"]})
                    p = desc + (descsz + 3) // 4 * 4
        at = data.find(b"\x7fELF", at + 4)
    return out


def test_head_mixing_forward_does_not_spill():
    mixed = {n: k for n, k in _kernels().items()
             if re.search(r"normalized_fwd_scatter_kernelI.*ELb0ELi\dELi[234]ELi\d+EEE", n)}
    assert len(mixed) >= 12  # four types, two to four heads
    spilled = {n: k[".vgpr_spill_count"] for n, k in mixed.items() if k[".vgpr_spill_count"]}
    assert not spilled
