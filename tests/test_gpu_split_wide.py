"""fp32 cells with C = 32 and C = 64 on the bf16 matrix cores (nca_split_wide.h): steps against float64,
where the error must not exceed 1.4 times that of the fp32 MFMA kernels on the same inputs, and over
many cells that error itself, fused rollouts against chained steps, and infinities and NaN against
those kernels."""

import pytest
import torch

from cells import oracle_cell
from oracle import nca_oracle as O
from test_gpu_split import DEV, _path, _run, _state

pytestmark = pytest.mark.gpu

# boards whose cells leave passes of 96 with a remainder or fill them, in LDS and (C = 32, from 16 rows
# of 20 cells) step by step
C32 = [(1, 1), (3, 5), (8, 12), (13, 13), (15, 15), (7, 31), (20, 21), (30, 30), (1, 200)]
C64 = [(1, 1), (3, 5), (9, 9), (9, 10)]
CASES = [("maze_hard_c32", s) for s in C32] + [("sudoku_c64", s) for s in C64]


@pytest.mark.parametrize("name,shape", CASES)
@pytest.mark.parametrize("padding", ["wall", "zero", "wrap"])
def test_step_error_against_float64(name, shape, padding):
    m, md, x, g4, cl = _state(name, 3, shape, 2, padding=padding)
    masks = torch.ones((1, 3, 1, *shape), dtype=torch.uint8)
    ref = O.step(oracle_cell(m), x.double(), g4, cl.double(), masks[0].float(), "fp64")
    y, _, _ = _run(md, x, g4, cl, 1, masks=masks.to(DEV))
    with _path(2):
        y0, _, _ = _run(md, x, g4, cl, 1, masks=masks.to(DEV))
    err, err0 = (y.cpu().double() - ref).norm(), (y0.cpu().double() - ref).norm()
    # one step's roundings: 40 % above the fp32 kernel's error covers the smallest boards' scatter
    assert err <= 1.4 * err0 + 1e-7 * ref.norm() / (ref.numel() ** 0.5), (err.item(), err0.item())


@pytest.mark.parametrize("name,shape,rows", [("maze_hard_c32", (13, 13), 3), ("maze_hard_c32", (5, 6), 700),
                                             ("maze_hard_c32", (15, 15), 259), ("maze_hard_c32", (24, 25), 5),
                                             ("sudoku_c64", (9, 9), 3), ("sudoku_c64", (9, 9), 259),
                                             ("sudoku_c64", (4, 5), 600)])
@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("padding", ["wall", "wrap"])
def test_fused_equals_chained(name, shape, rows, gated, padding):
    m, md, x, g4, cl = _state(name, rows, shape, 4, padding=padding)
    kw = dict(p_fire=0.8, p_low=0.2, tau=0.6) if gated else dict(p_fire=0.6)
    y, conf, fired = _run(md, x, g4, cl, 5, **kw)
    cur, total = x, 0
    for t in range(5):
        cur, c1, f1 = _run(md, cur, g4, cl, 1, step0=t, **kw)
        total = total + f1
    assert torch.equal(y, cur) and torch.equal(conf, c1) and torch.equal(fired, total)


@pytest.mark.parametrize("name,shape", [("maze_hard_c32", (11, 12)), ("maze_hard_c32", (22, 23)), ("sudoku_c64", (9, 9))])
@pytest.mark.parametrize("bad", [float("inf"), -float("inf"), float("nan"), 3.4e38, 1e-40])
def test_infinities_and_nan_as_fp32(name, shape, bad):
    m, md, x, g4, cl = _state(name, 2, shape, 6)
    x[0, 7, 5, 5] = bad
    g4[:] = False
    masks = torch.ones((1, 2, 1, *shape), dtype=torch.uint8).to(DEV)
    y, _, _ = _run(md, x, g4, cl, 1, masks=masks)
    with _path(2):
        y0, _, _ = _run(md, x, g4, cl, 1, masks=masks)
    assert torch.equal(y.isnan(), y0.isnan()) and torch.equal(y.isinf(), y0.isinf())
    ok = y0.isfinite()
    # a dot product's error goes with the sum of its terms' magnitudes, up to 256 terms of 2^-24 each:
    # beside a huge value that is the size of the cell's largest channel, not of one where terms cancel
    scale = torch.where(ok, y0.abs(), 0.0).amax(1, keepdim=True).clamp_min(1.0).expand_as(y0)
    assert ((y - y0)[ok].abs() <= 256 * 2.0**-24 * scale[ok]).all()


@pytest.mark.parametrize("name,shape,rows", [("maze_hard_c32", (30, 30), 8), ("maze_hard_c32", (13, 13), 16), ("sudoku_c64", (9, 9), 32)])
def test_error_of_many_cells(name, shape, rows):
    """Over many cells the error against float64 is below the fp32 kernels'."""
    m, md, x, g4, cl = _state(name, rows, shape, 9)
    masks = torch.ones((1, rows, 1, *shape), dtype=torch.uint8)
    ref = O.step(oracle_cell(m), x.double(), g4, cl.double(), masks[0].float(), "fp64")
    y, _, _ = _run(md, x, g4, cl, 1, masks=masks.to(DEV))
    with _path(2):
        y0, _, _ = _run(md, x, g4, cl, 1, masks=masks.to(DEV))
    err, err0 = (y.cpu().double() - ref).norm().item(), (y0.cpu().double() - ref).norm().item()
    print(name, shape, err / ref.norm().item(), err0 / ref.norm().item())
    assert err <= err0
