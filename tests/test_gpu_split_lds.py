"""fp32 cells on the bf16 matrix cores in LDS (rollout_split16, split_wide): infinities, NaN and values that
round to an infinite bf16 value as on fp32 MFMA, with one and several rows per workgroup and the bad
cell in the first, a middle and the last, partly filled, pass; the C = 16 cell's error over many cells."""

import pytest
import torch

from cells import oracle_cell
from ncas_amd.inference import rollout_steps
from oracle import nca_oracle as O
from test_gpu_split import DEV, _path, _run, _state

pytestmark = pytest.mark.gpu


def _step_in_place(md, x, g4, cl, masks):
    """One step in place: on boards that fit it, the LDS kernel (the per-step one would need a workspace)."""
    xd = x.to(DEV)
    with torch.no_grad():
        y, _, _ = rollout_steps(md, xd, g4.to(DEV), cl.to(DEV), 1, masks=masks, out=xd)
    return y


@pytest.mark.parametrize("name,shape,rows", [("maze_c16", (11, 12), 2), ("maze_c16", (11, 12), 700),
                                             ("maze_hard_c32", (11, 12), 3), ("maze_hard_c32", (5, 6), 3),
                                             ("maze_hard_c32", (7, 7), 3), ("maze_hard_c32", (5, 6), 700),
                                             ("sudoku_c64", (9, 9), 3), ("sudoku_c64", (7, 7), 3),
                                             ("sudoku_c64", (4, 5), 3), ("sudoku_c64", (4, 5), 600)])
@pytest.mark.parametrize("bad", [float("inf"), -float("inf"), float("nan"), 3.4e38, 1e-40])
def test_infinities_and_nan_as_fp32(name, shape, rows, bad):
    m, md, x, g4, cl = _state(name, rows, shape, 6)
    H, W = shape
    x[0, 7, 0, 0] = bad
    x[rows // 2, 7, H // 2, W // 2] = bad
    x[rows - 1, 7, H - 1, W - 1] = bad
    g4[:] = False
    masks = torch.ones((1, rows, 1, *shape), dtype=torch.uint8).to(DEV)
    y = _step_in_place(md, x, g4, cl, masks)
    with _path(2):
        y0, _, _ = _run(md, x, g4, cl, 1, masks=masks)
    assert torch.equal(y.isnan(), y0.isnan()) and torch.equal(y.isinf(), y0.isinf())
    ok = y0.isfinite()
    # a dot product's error goes with the sum of its terms' magnitudes, up to 256 terms of 2^-24 each:
    # beside a huge value that is the size of the cell's largest channel, not of one where terms cancel
    scale = torch.where(ok, y0.abs(), 0.0).amax(1, keepdim=True).clamp_min(1.0).expand_as(y0)
    assert ((y - y0)[ok].abs() <= 256 * 2.0**-24 * scale[ok]).all()


@pytest.mark.parametrize("shape,rows", [((13, 13), 64), ((40, 37), 8)])
@pytest.mark.parametrize("in_place", [False, True])
def test_c16_error_of_many_cells(shape, rows, in_place):
    """Over many cells the error against float64 is below the fp32 kernels', step by step and in LDS."""
    m, md, x, g4, cl = _state("maze_c16", rows, shape, 9)
    masks = torch.ones((1, rows, 1, *shape), dtype=torch.uint8)
    ref = O.step(oracle_cell(m), x.double(), g4, cl.double(), masks[0].float(), "fp64")
    y = _step_in_place(md, x, g4, cl, masks.to(DEV)) if in_place else _run(md, x, g4, cl, 1, masks=masks.to(DEV))[0]
    with _path(2):
        y0, _, _ = _run(md, x, g4, cl, 1, masks=masks.to(DEV))
    err, err0 = (y.cpu().double() - ref).norm().item(), (y0.cpu().double() - ref).norm().item()
    print(shape, err / ref.norm().item(), err0 / ref.norm().item())
    assert err <= err0
