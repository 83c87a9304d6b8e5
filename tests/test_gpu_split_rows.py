"""fp32 cells on the bf16 matrix cores (nca_split.h): a row's result is its own. Boards that share tiles,
passes or workgroups with a board of infinities or NaN keep their bits, and fused rollouts with such
a board equal chained steps."""

import pytest
import torch

from cells import make_model
from ncas_amd.inference import rollout_steps
from ncas_amd.step import make_step
from test_gpu_split import DEV, _run, _state

pytestmark = pytest.mark.gpu

# several rows per workgroup in LDS, and boards that run step by step; rows whose tiles and passes
# cross from one board into the next
CASES = [("maze_c16", (13, 13), 515), ("maze_c16", (5, 7), 600), ("maze_c16", (33, 35), 3),
         ("maze_hard_c32", (5, 7), 700), ("maze_hard_c32", (13, 13), 3), ("maze_hard_c32", (24, 25), 5),
         ("sudoku_c64", (9, 9), 515), ("sudoku_c64", (4, 5), 600)]


def _same(a, b):
    return torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(), b.nan_to_num())


@pytest.mark.parametrize("name,shape,rows", CASES)
@pytest.mark.parametrize("bad", [float("inf"), float("nan"), 3.4e38])
@pytest.mark.parametrize("gated", [False, True])
def test_a_board_does_not_change_its_neighbours(name, shape, rows, bad, gated):
    m, md, x, g4, cl = _state(name, rows, shape, 4)
    kw = dict(p_fire=0.8, p_low=0.2, tau=0.6) if gated else dict(p_fire=0.6)
    xb = x.clone()
    rb = rows // 2
    xb[rb, m.cfg.channels - 1, -1, -1] = bad  # the board's last cell: beside the next board's first
    xb[rb, m.cfg.channels - 1, 0, 0] = bad
    others = torch.arange(rows) != rb
    for n in (1, 3):
        y, conf, fired = _run(md, x, g4, cl, n, **kw)
        yb, confb, firedb = _run(md, xb, g4, cl, n, **kw)
        assert not torch.equal(yb[rb], y[rb])  # (3.4e38, finite in fp32 and infinite in bf16, may stay finite)
        assert torch.equal(yb[others], y[others]) and torch.equal(confb[others], conf[others])
        assert torch.equal(firedb[others], fired[others])
    cur, total = xb, 0
    for t in range(3):
        cur, c1, f1 = _run(md, cur, g4, cl, 1, step0=t, **kw)
        total = total + f1
    assert _same(yb, cur) and _same(confb, c1) and torch.equal(firedb, total)


@pytest.mark.parametrize("name,shape", [("maze_c16", (201, 201)), ("maze_hard_c32", (30, 30))])
def test_rows_beyond_2_gib(name, shape):
    """A state of more than 2 GiB runs on the kernels that its rows run on alone: the same bits, with
    drawn, injected and float fire masks, noise, and fired counts."""
    m = make_model(name).to(DEV)
    C, c_in = m.cfg.channels, m.cfg.c_in
    rows = 2**31 // (4 * C * shape[0] * shape[1]) + 9
    g = torch.Generator(DEV).manual_seed(8)
    x = torch.randn((rows, C, *shape), generator=g, device=DEV) * 0.3
    given4 = torch.rand((rows, 1, *shape), generator=g, device=DEV) < 0.3
    clamp = torch.randn((rows, c_in, *shape), generator=g, device=DEV)
    masks = (torch.rand((2, rows, 1, *shape), generator=g, device=DEV) < 0.6).to(torch.uint8)
    fire = masks[0].float() * 0.5
    noise = torch.randn((rows, C, *shape), generator=g, device=DEV)
    step = make_step(m)
    parts = [slice(0, 2), slice(rows // 2 - 1, rows // 2 + 2), slice(rows - 3, rows)]
    with torch.no_grad():
        for n in (1, 2):
            for kw in (dict(p_fire=0.8, p_low=0.2, tau=0.6), dict(masks=masks[:n])):
                y, conf, fired = rollout_steps(m, x, given4, clamp, n, seed=5, want_fired=True, **kw)
                for s in parts:
                    ks = dict(masks=masks[:n, s]) if "masks" in kw else dict(kw, row0=s.start)
                    ys, cs, fs = rollout_steps(m, x[s], given4[s], clamp[s], n, seed=5, want_fired=True, **ks)
                    assert torch.equal(y[s], ys) and torch.equal(conf[s], cs) and torch.equal(fired[s], fs)
        y = step(x, given4, clamp, fire, noise)
        for s in parts:
            assert torch.equal(y[s], step(x[s], given4[s], clamp[s], fire[s], noise[s]))


@pytest.mark.parametrize("name", ["maze_c16", "maze_hard_c32", "sudoku_c64"])
@pytest.mark.parametrize("shape", [(1, 1), (4, 4), (1, 17), (5, 6), (4, 8), (3, 11), (7, 7), (8, 8), (5, 13), (9, 9)])
@pytest.mark.parametrize("rows", [3, 515])
def test_a_row_alone_is_the_row_among_others(name, shape, rows):
    """Boards about the sizes where the kernel (16 cells) and the cells of a pass (32, 64) change: a row's bits
    are the same alone, among others, and step by step, with and without the outputs that decide
    where a single step runs."""
    m, md, x, g4, cl = _state(name, rows, shape, 4)
    kw = dict(p_fire=0.8, p_low=0.2, tau=0.6)
    y, conf, fired = _run(md, x, g4, cl, 3, **kw)
    for r in (0, rows - 1):
        with torch.no_grad():
            yr, cr, fr = rollout_steps(md, x[r:r + 1].to(DEV), g4[r:r + 1].to(DEV), cl[r:r + 1].to(DEV), 3, seed=5,
                                       row0=3 + r, want_fired=True, **kw)
        assert torch.equal(y[r:r + 1], yr) and torch.equal(conf[r:r + 1], cr) and torch.equal(fired[r:r + 1], fr)
    for outputs in (False, True):
        cur = x.to(DEV)
        for t in range(3):
            with torch.no_grad():
                cur, _, _ = rollout_steps(md, cur, g4.to(DEV), cl.to(DEV), 1, seed=5, row0=3, step0=t, want_conf=outputs,
                                          want_fired=outputs, **kw)
        assert torch.equal(y, cur)
