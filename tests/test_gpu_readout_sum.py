"""The board confidence of large boards: the wave's block-wise sum (`ordered_sum`) equals the sum of
the cells' confidences one after another, bit for bit, where blocks end in a tie, leave a binade,
or hold equal values, zeros or NaN."""

import numpy as np
import pytest
import torch

from cells import make_model

pytestmark = pytest.mark.gpu


def _sequential_mean(conf_cell):
    c = conf_cell.cpu().numpy().reshape(conf_cell.shape[0], -1)
    s = np.cumsum(c, axis=1, dtype=np.float32)[:, -1]  # fp32 additions in cell order
    return s / np.float32(c.shape[1])


@pytest.mark.parametrize("shape", [(201, 201), (64, 32), (45, 45), (46, 45), (1, 1089), (13, 5)])
@pytest.mark.parametrize("scale", [0.0, 1e-3, 1.0, 30.0])
def test_board_confidence_is_the_ordered_sum(shape, scale):
    from ncas_amd.readout import readout

    m = make_model("maze_c16").cuda()
    g = torch.Generator().manual_seed(1)
    x = (torch.randn((3, 16, *shape), generator=g) * scale).cuda()
    conf, board, _ = readout(m, x)
    assert np.array_equal(board.cpu().numpy(), _sequential_mean(conf))


def test_board_confidence_with_nan_and_few_bits():
    from ncas_amd.readout import readout

    m = make_model("maze_c16").cuda()
    with torch.no_grad():  # confidences 1 / (1 + exp(-k / 8)) of few distinct values
        m.head.weight.zero_()
        m.head.weight[0, 0] = 1.0
        m.head.bias.zero_()
    g = torch.Generator().manual_seed(2)
    x = (torch.randint(-9, 10, (2, 16, 150, 151), generator=g) / 8).cuda()
    x[1, :, 70, 3] = float("nan")
    conf, board, _ = readout(m, x)
    ref = _sequential_mean(conf)
    assert board[0].item() == ref[0]
    assert np.isnan(ref[1]) and torch.isnan(board[1])


def test_rollout_confidence_equals_readout():
    from ncas_amd.inference import rollout_steps
    from ncas_amd.readout import readout

    m = make_model("maze_c16").cuda()
    g = torch.Generator().manual_seed(3)
    x = torch.randn((2, 16, 97, 61), generator=g).cuda()
    given4 = torch.zeros((2, 1, 97, 61), dtype=torch.bool).cuda()
    clamp = torch.zeros((2, 4, 97, 61)).cuda()
    with torch.no_grad():
        for precision in ("fp32", "bf16"):
            for n in (1, 2, 3):
                y, conf, _ = rollout_steps(m, x, given4, clamp, n, precision=precision)
                assert torch.equal(conf, readout(m, y)[1])


def test_many_rows_equal_few():
    """Boards of several kilocells are read out in two launches or, from some hundred rows, in one: the
    same bits."""
    from ncas_amd.readout import readout

    m = make_model("maze_c16").cuda()
    g = torch.Generator("cuda").manual_seed(4)
    x = torch.randn((515, 16, 46, 45), generator=g, device="cuda")
    conf, board, cls = readout(m, x)
    for r in (0, 514):
        c1, b1, k1 = readout(m, x[r:r + 1])
        assert torch.equal(conf[r:r + 1], c1) and torch.equal(board[r:r + 1], b1) and torch.equal(cls[r:r + 1], k1)
    assert np.array_equal(board.cpu().numpy(), _sequential_mean(conf))
