"""Which kernels the normalized passes take (gather kernels for rows of no
4-vectors on few workgroups and for tables of a few rows), told by bitwise
equality with the gather kernels, and the tiles on shapes and tables that the
rule leaves to them: odd rows on many planes, the weight check, the row rules,
and accumulate_uz's gather form inside its launch."""
import sys

import pytest
import torch

import test_gpu_normalized_scatter as norm
import test_gpu_row_rules as rules
import test_gpu_scatter as acc
import test_gpu_weight_check as check
from neural_shift_cuda_amd import _C
from neural_shift_cuda_amd.workloads import halfplane_rows, halfplane_shifts, window_shifts

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _say(*what):
    print("[case]", *what, flush=True)
    sys.stdout.flush()


def _passes(dtype, shape, sh, log, seed=3):
    """The op's outputs and gradients, and those of the gather kernels."""
    x, w, gD, gL, D, L, gx, gw = norm._run(dtype, shape, sh, log, seed)
    got = (D.detach(), L.detach(), gx, gw)
    return got, norm._gather_path(x.to(DEV), w.to(DEV), sh, log, gD.to(DEV), gL.to(DEV))


# (dtype, shape, table): both passes on the gather kernels
GATHER = [
    (torch.float32, (1, 1, 137, 73), halfplane_shifts(4)),
    (torch.float32, (1, 1, 133, 133), window_shifts(5)),
    (torch.float32, (2, 1, 90, 250), halfplane_shifts(5)),
    (torch.float16, (2, 1, 90, 131), halfplane_shifts(5)),
    (torch.bfloat16, (1, 1, 150, 150), halfplane_shifts(3)),
]


@pytest.mark.parametrize("dtype,shape,table", GATHER)
@pytest.mark.parametrize("log", [False, True])
def test_few_workgroups_take_the_gather_kernels(dtype, shape, table, log):
    _say("gather", dtype, shape, table.size(0), log)
    got, gather = _passes(dtype, shape, table, log)
    assert all(torch.equal(a, b) for a, b in zip(got, gather))


# forwards of tables of a few rows
@pytest.mark.parametrize("dtype,shape,R", [(torch.float64, (12, 1, 35, 154), 1),
                                           (torch.float64, (2, 1, 201, 195), 3),
                                           (torch.float32, (1, 1, 96, 128), 1),
                                           (torch.float32, (20, 1, 48, 129), 3),
                                           (torch.bfloat16, (16, 1, 60, 45), 2)])
@pytest.mark.parametrize("log", [False, True])
def test_few_rows_take_the_gather_forward(dtype, shape, R, log):
    _say("gather forward", dtype, shape, R, log)
    got, gather = _passes(dtype, shape, halfplane_shifts(R), log)
    assert all(torch.equal(a, b) for a, b in zip(got[:2], gather[:2]))


# 16 rows up to 8 pixels, mirrors, a self-inverse row and one beyond the border
MANY = torch.tensor([r for r in halfplane_rows(8)[::10]][:14] + [(0, 0, 1), (3, 11, 1)])
TABLES = {"many": MANY, "win2": window_shifts(2), "half3": halfplane_shifts(3)}


@pytest.mark.parametrize("dtype,shape", [
    (torch.float32, (110, 1, 65, 67)),   # odd rows on more workgroups than the rule holds
    (torch.float32, (40, 1, 97, 134)),   # W % 4 = 2
    (torch.float32, (140, 1, 37, 51)),   # 64-wide tiles, one column
    (torch.float16, (60, 1, 66, 69)),
    (torch.bfloat16, (70, 1, 70, 70)),
    (torch.float64, (2, 1, 49, 66)),
])
@pytest.mark.parametrize("table", list(TABLES))
@pytest.mark.parametrize("log_weights", [False, True])
def test_odd_rows_on_tiles(monkeypatch, dtype, shape, table, log_weights):
    _say("tiles", dtype, shape, table, log_weights)
    monkeypatch.setattr(norm, "_table", lambda name: TABLES[name])
    norm.test_normalized_scatter_vs_oracle(dtype, shape, table, log_weights)


@pytest.mark.parametrize("box", [False, True])
@pytest.mark.parametrize("log", [False, True])
@pytest.mark.parametrize("dtype", check.DTYPES)
def test_weight_check_on_tiles(monkeypatch, dtype, log, box):
    """The check inside the scatter forward: the rows of test_weight_check and
    as many more that make the table one the tiles take."""
    more = [(a, b, 0) for a in (-1, 1) for b in (-4, -2, 0, 2, 4, 6)]
    forward = check._forward

    def padded(w, shape, rows, log, box):
        one = torch.zeros_like(w[:1]).expand(len(more) * shape[0], *w.shape[1:])
        return forward(torch.cat([w, one]), shape, rows + more, log, box)

    monkeypatch.setattr(check, "_forward", padded)
    check.test_weight_check(dtype, log, box, (1, 2, 75, 152))


@pytest.mark.parametrize("periodic,box", rules.RULES)
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32, torch.float64])
def test_rules_on_tiles(monkeypatch, dtype, periodic, box):
    monkeypatch.setitem(rules.ROWS, "many", [tuple(r) for r in MANY.tolist()])
    rules.test_rules_equal_row_codes(dtype, periodic, box, "many", (1, 2, 70, 140))


@pytest.mark.parametrize("dtype,shape", [(torch.float32, (8, 1, 321, 481)),
                                         (torch.float16, (2, 1, 470, 135)),
                                         (torch.float64, (4, 1, 118, 119))])
def test_gather_form_inside_the_launch(monkeypatch, dtype, shape):
    """Tables beyond every border whose radius the library is not told."""
    _say("far tables", dtype, shape)
    monkeypatch.setattr(_C, "table_radius", lambda sh: None)
    sh = torch.tensor([[0, 0, 0], [17, 3, 1], [-2, 20, 1], [30, 1, 1]])
    assert acc._uses_workspace(dtype, shape, sh.size(0), False)
    acc._run_and_check(dtype, shape, sh, 6)
