"""The BPTT backward of cells outside the bf16 C = 32 path (nca_bptt_step.h) where one launch's
workgroups own several tiles and the weight gradients are summed over several groups of steps: against
the fp64 autograd oracle, with a loss mask, sparse weights and a cotangent of the last state."""

import ctypes

import pytest
import torch

from ncas_amd import _lib
from ncas_amd.step import step_vjp
from oracle import nca_oracle as O
from test_gpu_bptt import DEV, NAMES, _case, _gpu_chunk, _rel, oracle_cell

pytestmark = pytest.mark.gpu

# the cells the path takes, with the tolerances of test_gpu_bptt.py
CELLS_TOL = [("maze_c16", "fp32", 1e-4), ("maze_c16", "bf16", 1e-2), ("maze_hard_c32", "fp32", 1e-4),
             ("sudoku_c64", "fp32", 1e-4), ("sudoku_c64", "bf16", 1e-2)]


def _workspace_for(monkeypatch, steps):
    """Workspaces are sized for `steps` steps, whatever the chunk: the backward's groups hold that many."""
    L = _lib.load()
    whole = L.nca_bptt_workspace_bytes
    monkeypatch.setattr(L, "nca_bptt_workspace_bytes", lambda cell, B, H, W, n: whole(cell, B, H, W, steps))
    return whole


@pytest.mark.parametrize("name,precision,tol", CELLS_TOL)
@pytest.mark.parametrize("group", [1, 3])
def test_a_workspace_of_fewer_steps_is_enough(name, precision, tol, group, monkeypatch):
    """The backward takes any workspace that holds one step: its groups are as long as fit (7 steps in
    groups of 3, 3 and 1, or of 1)."""
    m, md, x, g4, cl, masks, targets = _case(name, steps=7)
    weights = [0.5, 0.0, 1.0, 0.0, 0.0, 2.0, 1.0]
    ref = _gpu_chunk(md, x, g4, cl, targets, weights, precision, masks=masks.to(DEV))
    whole = _workspace_for(monkeypatch, group)
    B, _, H, W = x.shape
    desc = md.packed(precision, DEV).desc
    assert whole(ctypes.byref(desc), B, H, W, group) < whole(ctypes.byref(desc), B, H, W, 7)
    res = _gpu_chunk(md, x, g4, cl, targets, weights, precision, masks=masks.to(DEV))
    assert torch.equal(res.grad_x0, ref.grad_x0) and torch.equal(res.loss, ref.loss)
    for k in ("kernels", "head_w", "head_b"):
        assert torch.equal(res.grads[k], ref.grads[k]), k
    for k in ("w1", "b1", "w2", "b2"):  # fp32 sums over the same cells in another order
        assert _rel(res.grads[k], ref.grads[k]) <= 1e-6, (k, _rel(res.grads[k], ref.grads[k]))


@pytest.mark.parametrize("name,precision,tol", CELLS_TOL)
def test_many_cells_and_groups_match_oracle(name, precision, tol, monkeypatch):
    """More than 512 tiles of 32 cells, the last one partly filled, and groups of 3 and 1 steps."""
    rows = {"maze_c16": 103, "maze_hard_c32": 209, "sudoku_c64": 209}[name]
    m, md, x, g4, cl, masks, targets = _case(name, n_boards=rows, k=1, steps=4)
    M = targets.numel()
    assert M > 512 * 32 and M % 32 != 0
    weights = [1.0, 0.0, 0.5, 1.0]
    g = torch.Generator().manual_seed(9)
    lm = (torch.rand(targets.shape, generator=g) < 0.8).float()
    cot = torch.randn(x.shape, generator=g) * (1.0 / M)
    _workspace_for(monkeypatch, 3)
    res = _gpu_chunk(md, x, g4, cl, targets, weights, precision, masks=masks.to(DEV), loss_mask=lm.to(DEV),
                     grad_final=cot.to(DEV))
    kw = dict(grad_round=True) if precision == "bf16" else {}
    loss, ref = O.bptt_chunk(oracle_cell(m), x, g4, cl, masks.double(), targets, weights, precision, loss_mask=lm,
                             grad_x0=True, final_cotangent=cot.double(), **kw)
    loss -= float((cot.double() * res.x.cpu().double()).sum())  # the oracle's scalar has the cotangent's term
    assert abs(float(res.loss) - loss) <= (1e-5 if precision == "fp32" else 1e-4) * abs(loss)
    for k in NAMES:
        assert _rel(res.grads[k], ref[k]) <= tol, (k, _rel(res.grads[k], ref[k]))
    if precision == "fp32":
        assert _rel(res.grad_x0, ref["x0"]) <= tol


def test_bf16_c32_beyond_32_bit_offsets():
    """From 2^23 cells a bf16 C = 32 batch runs on back_step<32, 256, true>, as the fused MLP kernel holds 32-bit
    offsets: the gradients of a step are those of the batch's two halves."""
    m, md, x, g4, cl, masks, targets = _case("maze_hard_c32")
    H = W = 30
    rows = 2**23 // (H * W) + 3
    g = torch.Generator(DEV).manual_seed(11)
    x = torch.randn((rows, 32, H, W), generator=g, device=DEV) * 0.3
    cot = torch.randn((rows, 32, H, W), generator=g, device=DEV)
    given4 = torch.rand((rows, 1, H, W), generator=g, device=DEV) < 0.3
    fire = (torch.rand((rows, 1, H, W), generator=g, device=DEV) < 0.6).float()
    gx, gp = step_vjp(md, x, given4, fire, cot, "bf16")
    half = rows // 2
    a = step_vjp(md, x[:half], given4[:half], fire[:half], cot[:half], "bf16")
    b = step_vjp(md, x[half:], given4[half:], fire[half:], cot[half:], "bf16")

    def rel(p, q):  # (on the GPU: 3e8 values)
        return float((p - q).norm() / q.norm())

    # the same bf16 operands; a sum in another order rounds g_z to the neighbouring bf16 value now and then
    assert rel(gx[:half], a[0]) <= 1e-3 and rel(gx[half:], b[0]) <= 1e-3
    for k in range(5):
        assert rel(gp[k], a[1][k] + b[1][k]) <= 1e-3, k
