"""fp32 C = 16 cells on the bf16 matrix cores (nca_split.h): steps against float64, where the error of
boards of any size must not exceed 1.4 times that of the fp32 MFMA kernels on the same inputs
(test_gpu_split_lds.py: over many cells, that error itself), fused rollouts against chained
steps, and infinities and NaN against those kernels."""

import copy

import pytest
import torch

from cells import boards_for, initial_state, make_model, oracle_cell
from ncas_amd import _lib
from ncas_amd.inference import rollout_steps
from oracle import nca_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


class _path:
    """Kernel path for the duration of a block: 1 is the generic resident kernel, 2 the per-step one."""

    def __init__(self, path):
        self.path = path

    def __enter__(self):
        assert _lib.load().nca_set_kernel_path(self.path) == 0

    def __exit__(self, *exc):
        _lib.load().nca_set_kernel_path(0)


def _state(name, rows, shape, seed, sigma=0.3, **overrides):
    m = make_model(name, seed)
    for k, v in overrides.items():
        setattr(m.cfg, k, v)
    g = torch.Generator().manual_seed(seed)
    C = m.cfg.channels
    x = torch.randn((rows, C, *shape), generator=g) * sigma
    given4 = torch.rand((rows, 1, *shape), generator=g) < 0.3
    clamp = torch.randn((rows, m.cfg.c_in, *shape), generator=g)
    return m, copy.deepcopy(m).to(DEV), x, given4, clamp


def _run(md, x, g4, cl, n, **kw):
    with torch.no_grad():
        return rollout_steps(md, x.to(DEV), g4.to(DEV), cl.to(DEV), n, seed=5, row0=3, want_fired=True, **kw)


@pytest.mark.parametrize("name", ["maze_c16", "ref_maze_ood"])
@pytest.mark.parametrize("shape", [(13, 13), (1, 1), (3, 5), (25, 25), (7, 31), (40, 37), (1, 200)])
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
    # (the sums' own error is 0.6 of it over many cells)
    assert err <= 1.4 * err0 + 1e-7 * ref.norm() / (ref.numel() ** 0.5), (err.item(), err0.item())


@pytest.mark.parametrize("shape", [(13, 13), (9, 14), (25, 25), (33, 35)])
@pytest.mark.parametrize("gated", [False, True])
def test_fused_equals_chained(shape, gated):
    """The LDS-resident rollout (boards up to 25x25) and the per-step kernel give the same bits, also
    with several rows per workgroup."""
    rows = 3 if shape != (13, 13) else 515
    m, md, x, g4, cl = _state("maze_c16", rows, shape, 4)
    kw = dict(p_fire=0.8, p_low=0.2, tau=0.6) if gated else dict(p_fire=0.6)
    y, conf, fired = _run(md, x, g4, cl, 5, **kw)
    cur, total = x, 0
    for t in range(5):
        cur, c1, f1 = _run(md, cur, g4, cl, 1, step0=t, **kw)
        total = total + f1
    assert torch.equal(y, cur) and torch.equal(conf, c1) and torch.equal(fired, total)


@pytest.mark.parametrize("bad", [float("inf"), -float("inf"), float("nan"), 3.4e38, 1e-40])
def test_infinities_and_nan_as_fp32(bad):
    """Tiles with a NaN among their sums run on fp32 MFMA: the same infinities and NaN in the same
    places as the fp32 kernels, also for values that round to an infinite bf16 value."""
    m, md, x, g4, cl = _state("maze_c16", 2, (11, 12), 6)
    x[0, 7, 5, 5] = bad
    g4[:] = False
    masks = torch.ones((1, 2, 1, 11, 12), dtype=torch.uint8).to(DEV)
    y, _, _ = _run(md, x, g4, cl, 1, masks=masks)
    with _path(2):
        y0, _, _ = _run(md, x, g4, cl, 1, masks=masks)
    assert torch.equal(y.isnan(), y0.isnan()) and torch.equal(y.isinf(), y0.isinf())
    ok = y0.isfinite()
    assert ((y - y0)[ok].abs() <= 1e-5 * y0[ok].abs().clamp_min(1.0)).all()
