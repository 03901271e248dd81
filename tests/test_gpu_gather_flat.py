"""16-bit gathers on rows that take no vector: planes written as flat runs of
16-byte vectors with single elements at either end, bit for bit the oracle's."""
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


# planes smaller than a vector, ends of 0..7 elements, more than one chunk
@pytest.mark.parametrize("shape", [(1, 1, 1, 1), (2, 3, 1, 5), (1, 2, 3, 3), (2, 1, 7, 9),
                                   (1, 3, 33, 65), (2, 2, 129, 131)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("pair", [False, True])
def test_flat_gather(pair, dtype, shape):
    from neural_shift_cuda import pair_gather, shift_gather
    g = torch.Generator().manual_seed(1)
    x = torch.randn(shape, generator=g).to(dtype)
    sh = torch.tensor([(0, 0), (1, -2), (-3, 4), (5, 0), (0, 131), (-1000, 7)])
    fn, ref = (pair_gather, oracle.pair_gather) if pair else (shift_gather, oracle.shift_gather)
    out, mask = fn(x.cuda(), sh.cuda())
    want, want_mask = ref(x, sh)
    assert torch.equal(out.cpu(), want) and torch.equal(mask.cpu(), want_mask)


def test_flat_gather_unaligned_output():
    """Every alignment of the output's first plane."""
    from neural_shift_cuda_amd import _C
    B, C, H, W = 1, 2, 5, 7
    sh = torch.tensor([(1, 1), (0, -2)]).cuda()
    x = torch.randn(B, C, H, W).half().cuda()
    want = _C.shift_gather_forward(x, sh)[0]
    n = want.numel()
    for off in range(8):
        buf = torch.zeros(n + 16, dtype=torch.float16, device="cuda")
        out = buf[off:off + n]
        rc = _C._lib.nsh_shift_gather_forward(
            x.data_ptr(), sh.data_ptr(), 2, 2, B, C, H, W, 1, out.data_ptr(), None,
            torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        assert torch.equal(out, want.flatten())
        assert not buf[:off].any() and not buf[off + n:].any()
