"""nca_bptt_forward in one launch: state t of the chunk equals a t-step rollout bit for bit, on the kernels
that record every step (the streamed bf16 C = 64 kernel, the fp32 kernels in LDS) and for an odd
number of boards, whose last workgroup is partly empty."""

import ctypes

import pytest
import torch

from ncas_amd import _lib
from ncas_amd.inference import rollout_steps
from ncas_amd.rng import fire_desc
from test_gpu_split import DEV, _state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("masks", [False, True])
@pytest.mark.parametrize("name,precision,shape,rows", [
    ("sudoku_c64", "bf16", (9, 9), 5), ("sudoku_c64", "bf16", (1, 3), 31), ("sudoku_c64", "bf16", (1, 1), 83),
    ("sudoku_c64", "bf16", (10, 9), 3), ("sudoku_c64", "fp32", (9, 9), 3), ("maze_hard_c32", "fp32", (13, 13), 3),
    ("maze_hard_c32", "fp32", (4, 5), 523), ("maze_hard_c32", "fp32", (20, 22), 3)])
def test_recorded_states_are_rollout_states(name, precision, shape, rows, masks):
    m, md, x, g4, cl = _state(name, rows, shape, 3)
    n, C = 5, m.cfg.channels
    xd, gd, cd = x.to(DEV), g4.to(DEV), cl.to(DEV)
    m8 = None
    if masks:
        g = torch.Generator().manual_seed(7)
        m8 = (torch.rand((n, rows, 1, *shape), generator=g) < 0.5).to(torch.uint8).to(DEV)
    fd = fire_desc(11, 0.7, None, None, True, 2, 3, None, m8)
    pk = md.packed(precision, torch.device(DEV))
    states = torch.full((n + 1, rows, C, *shape), float("nan"), device=DEV)
    g8 = gd.to(torch.uint8).contiguous()
    L = _lib.load()
    _lib.check(L.nca_bptt_forward(ctypes.byref(pk.desc), pk.buf.data_ptr(), rows, *shape, xd.data_ptr(), g8.data_ptr(),
                                  cd.data_ptr(), ctypes.byref(fd), n, states.data_ptr(), _lib.stream_of(torch.device(DEV))),
               "nca_bptt_forward")
    assert torch.equal(states[0], xd)
    kw = dict(seed=11, p_fire=0.7, row0=2, step0=3)
    with torch.no_grad():
        for t in range(1, n + 1):
            y, _, _ = rollout_steps(md, xd, gd, cd, t, precision=precision, **(dict(masks=m8[:t]) if masks else kw))
            assert torch.equal(states[t], y), t
