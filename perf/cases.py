"""The work this framework is used for, as cases that can be timed and checked: single steps,
fused rollouts and training passes of the five cells' shapes, in fp32 and bf16.

A case is a dict of plain values:

* `op`: "step" (one step through `make_step`), "rollout" (`rollout_steps`), "chunk" (forward and
  backward of a BPTT chunk, `bptt_chunk`) or "iteration" (`Engine.train_iteration`);
* `preset`: the cell (`ncas_amd.model.PRESETS`); `precision`: "fp32" or "bf16";
* `boards`, `k`: boards and trials per board (rows = boards * k); `height`, `width`: the grid;
* `depth`: steps of the rollout, or of the chunk;
* `gated`: confidence-gated firing (p_fire 0.8, 0.2 above confidence 0.9) instead of uniform.

`listed()` gives the fixed ones, `draw(rng)` one more of the same ranges; `prepare` makes a
case's inputs on the GPU from a seed, `run` is one pass through the public entry points, `work`
prices it, `exact` restates it in 64 bits with plain torch and `tolerance` says how far two
correct implementations may lie apart.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from ncas_amd.inference import rollout_steps
from ncas_amd.model import build_model
from ncas_amd.step import make_step
from ncas_amd.tasks import maze_boards, sudoku_boards
from ncas_amd.train import Engine, bptt_chunk

P_GATED, P_LOW, TAU = 0.8, 0.2, 0.9

# (scale, decay) of the cell's weights per preset: dynamics that keep moving and stay bounded
DYNAMICS = {"maze_c16": (1.5, 0.8), "maze_hard_c32": (1.8, 0.8), "sudoku_c64": (1.3, 0.6),
            "maze_ood": (1.4, 0.8), "maze_hard": (1.5, 0.8)}


# ------------------------------------------------------------------------------ the cases
def _case(op, preset, precision, boards, k, height, width, depth, gated=False, name=None):
    c = dict(op=op, preset=preset, precision=precision, boards=boards, k=k, height=height,
             width=width, depth=depth, gated=gated)
    return c if name is None else dict(c, name=name)


def listed() -> list[dict]:
    return [
        # one step of the step protocol on the smoke batch, as a caller's own loop takes it:
        # the smallest call, bound by launches and the host
        _case("step", "maze_c16", "fp32", 8, 1, 13, 13, 1, name="step-maze13-fp32"),
        # the smoke configuration: few small boards, a long rollout
        _case("rollout", "maze_c16", "fp32", 8, 1, 13, 13, 300, name="rollout-maze13-fp32"),
        # inference on large mazes, in both precisions (a part of the 13,000 steps that such a
        # maze takes to solve)
        _case("rollout", "maze_c16", "bf16", 16, 1, 201, 201, 128, name="rollout-maze201-bf16"),
        _case("rollout", "maze_c16", "fp32", 16, 1, 201, 201, 32, name="rollout-maze201-fp32"),
        # K trials per Sudoku board for conf@K: the headline evaluation in bf16, and a smaller
        # evaluation batch in fp32 (the default precision of a rollout)
        _case("rollout", "sudoku_c64", "bf16", 256, 128, 9, 9, 256, name="rollout-sudoku9-bf16"),
        _case("rollout", "sudoku_c64", "fp32", 64, 32, 9, 9, 64, name="rollout-sudoku9-fp32"),
        # hard mazes with confidence-gated firing and K trials, in both precisions
        _case("rollout", "maze_hard_c32", "bf16", 128, 64, 30, 30, 200, True,
              name="rollout-hardmaze30-bf16"),
        _case("rollout", "maze_hard_c32", "fp32", 32, 16, 30, 30, 32, True,
              name="rollout-hardmaze30-fp32"),
        # training: forward and backward of the BPTT chunk of the hard-maze configuration, the
        # same of the small maze in fp32 (training without amp) and of the Sudoku cell in bf16
        _case("chunk", "maze_hard_c32", "bf16", 64, 1, 30, 30, 32, name="chunk-hardmaze30-bf16"),
        _case("chunk", "maze_c16", "fp32", 64, 1, 13, 13, 32, name="chunk-maze13-fp32"),
        _case("chunk", "sudoku_c64", "bf16", 128, 1, 9, 9, 32, name="chunk-sudoku9-bf16"),
        # a training iteration of the embedding-head maze cell: the MSE loss, step by step through
        # the differentiable step (the trainer's default loss)
        _case("iteration", "maze_ood", "fp32", 64, 1, 13, 13, 16, name="iteration-mazeood13-fp32"),
    ]


# What a drawn case may cost, in FLOPs: well under the largest listed case (1.2e14) also where the
# work runs far from the matrix cores' rate.
_DRAW_FLOPS = {"step": 4e10, "rollout": 2e12, "chunk": 1e12, "iteration": 1e11}


def _log_int(rng, lo: float, hi: float) -> int:
    return max(1, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng) -> dict:
    """One more case: op, cell and precision at random, the grid between 5 and 201 (up to 31 for
    the wide cells, Sudoku boards 9x9), rows and depth over their logarithm."""
    op = rng.choice(["step", "rollout", "rollout", "rollout", "chunk", "chunk", "iteration"])
    if op == "iteration":
        preset, precision = rng.choice(["maze_ood", "maze_hard"]), "fp32"
    else:
        presets = ["maze_c16", "maze_hard_c32", "sudoku_c64"]
        preset = rng.choice(presets if op == "chunk" else presets * 2 + ["maze_ood", "maze_hard"])
        precision = rng.choice(["fp32", "bf16"])
    if preset == "sudoku_c64":
        height = width = 9
    else:
        big = 201 if preset in ("maze_c16", "maze_ood") and op == "rollout" else 31
        height = _log_int(rng, 5, big)
        width = height if rng.random() < 0.6 else _log_int(rng, 5, big)
    k = rng.choice([1, 1, 8, 32]) if op == "rollout" else 1
    boards = _log_int(rng, 4, 256)
    depth = 1 if op == "step" else _log_int(rng, 4, 200 if op == "rollout" else 32)
    gated = op == "rollout" and preset == "maze_hard_c32" and rng.random() < 0.5
    case = _case(op, preset, precision, boards, k, height, width, depth, gated)
    while work(case)["flops"] > _DRAW_FLOPS[op] and (case["boards"] > 1 or case["depth"] > 1):
        if case["boards"] > 4 or case["depth"] == 1:
            case["boards"] = max(1, case["boards"] // 2)
        else:
            case["depth"] = max(1, case["depth"] // 2)
    return case


# ------------------------------------------------------------------------------ the inputs
def _model(case, seed):
    """The cell with synthetic weights of a trained cell's size: random fc1, fc2 and head, and a
    leak dx_c -= decay * x_c through the identity kernel in the first 2C hidden units, which
    bounds the dynamics as training does."""
    m = build_model(case["preset"])
    scale, decay = DYNAMICS[case["preset"]]
    g = torch.Generator().manual_seed(seed)
    C, F, hid = m.cfg.channels, m.perceive.out_dim, m.cfg.hidden
    with torch.no_grad():
        if m.cfg.kernel_init != "fixed":  # learned kernels
            m.perceive.weight.copy_(torch.randn(m.perceive.weight.shape, generator=g) / 3)
        ident = torch.zeros(3, 3)
        ident[1, 1] = 1.0
        m.perceive.weight[0, 0] = ident
        w1 = torch.randn(hid, F, generator=g) * (scale / F**0.5)
        w2 = torch.randn(C, hid, generator=g) * (0.5 * scale / hid**0.5)
        b1 = torch.randn(hid, generator=g) * 0.01
        b2 = torch.randn(C, generator=g) * 0.01
        w1[:2 * C], b1[:2 * C], w2[:, :2 * C] = 0.0, 0.0, 0.0
        c = torch.arange(C)
        w1[2 * c, c], w1[2 * c + 1, c] = 1.0, -1.0
        w2[c, 2 * c], w2[c, 2 * c + 1] = -decay, decay
        m.update.fc1.weight.copy_(w1.reshape(m.update.fc1.weight.shape))
        m.update.fc2.weight.copy_(w2.reshape(m.update.fc2.weight.shape))
        m.update.fc1.bias.copy_(b1)
        m.update.fc2.bias.copy_(b2)
        if m.cfg.head == "mlp":
            # confident enough that gated firing meets cells on both sides of its threshold
            std = 4.0 if case["gated"] else 1.0
            m.head.weight.copy_(torch.randn(m.head.weight.shape, generator=g) * std / m.cfg.c_out**0.5)
            m.head.bias.copy_(torch.randn(m.head.bias.shape, generator=g) * 0.1)
    return m


def _boards(case, seed):
    """(inputs, targets, given) token boards: Sudoku grids with 17 to 30 clues, or mazes with 10 %
    extra openings, cut to the grid where it is not square."""
    n, h, w = case["boards"], case["height"], case["width"]
    if case["preset"] == "sudoku_c64":
        b = sudoku_boards(n, seed)
        return b.inputs, b.targets, b.given
    b = maze_boards(n, max(h, w, 5), seed, extra_openings=0.10)
    inputs, targets, given = (np.ascontiguousarray(a[:, :h, :w]) for a in (b.inputs, b.targets, b.given))
    if case["preset"] in ("maze_ood", "maze_hard"):
        # these cells' vocabularies: empty 0, path 1, wall 2, endpoints 3 (or start 3, goal 4)
        to = np.array([0, 2, 3, 3, 1] if case["preset"] == "maze_ood" else [0, 2, 3, 4, 1])
        inputs, targets = to[inputs], to[targets]
        given = inputs >= 2
    return inputs, targets, given


def _inputs(case, seed) -> dict:
    dev = torch.device("cuda", torch.cuda.current_device())
    model = _model(case, seed).to(dev)
    inputs, targets, given = (np.repeat(a, case["k"], 0) for a in _boards(case, seed))
    inputs = torch.from_numpy(inputs).to(dev)
    given4 = torch.from_numpy(given).to(dev)[:, None]
    g = torch.Generator(device=dev).manual_seed(seed)
    B, H, W = inputs.shape
    # states in the middle of a rollout: every channel in use, clamped at given cells
    x = torch.randn((B, model.cfg.channels, H, W), generator=g, device=dev).mul_(0.3)
    clamp = model.clamp_values(inputs)
    x[:, model.cfg.in_slice] = torch.where(given4, clamp, x[:, model.cfg.in_slice])
    s = dict(case=case, model=model, x=x, given4=given4, clamp=clamp, seed=seed)
    rng = np.random.default_rng(seed)
    if case["op"] == "step":
        s["fire"] = (torch.rand((B, 1, H, W), generator=g, device=dev) < model.cfg.fire_rate).float()
    if case["op"] in ("chunk", "iteration"):
        s["targets"] = torch.from_numpy(targets).to(dev)
        s["seeds"] = rng.integers(0, 2**62, size=case["depth"], dtype=np.int64)
        s["weights"] = np.ones(case["depth"], np.float32)
    return s


def prepare(case, seed) -> dict:
    s = _inputs(case, seed)
    model = s["model"]
    if case["op"] == "step":
        s["step"] = make_step(model)
    elif case["op"] == "chunk":
        s["classes"] = model.output_index(s["targets"], torch.int32)
    elif case["op"] == "iteration":
        s["engine"] = Engine(model, None, {"rollout": case["depth"], "chunk": case["depth"],
                                           "loss": "mse", "perturb": False}, s["x"].device)
        s["batch"] = {"x": s["x"], "given4": s["given4"], "clamp": s["clamp"], "targets": s["targets"]}
    return s


def run(s):
    case, model = s["case"], s["model"]
    if case["op"] == "step":
        with torch.no_grad(), torch.autocast("cuda", torch.bfloat16, enabled=case["precision"] == "bf16"):
            return s["step"](s["x"], s["given4"], s["clamp"], s["fire"], None, None, None)
    if case["op"] == "rollout":
        gate = dict(p_fire=P_GATED, p_low=P_LOW, tau=TAU) if case["gated"] else {}
        with torch.no_grad():
            x, conf, fired = rollout_steps(model, s["x"], s["given4"], s["clamp"], case["depth"],
                                           seed=s["seed"], precision=case["precision"],
                                           want_conf=True, want_fired=True, **gate)
        return {"x": x, "conf": conf, "fired": fired}
    if case["op"] == "chunk":
        r = bptt_chunk(model, s["x"], s["given4"], s["clamp"], s["classes"], s["weights"],
                       step_seeds=s["seeds"], precision=case["precision"])
        return {"x": r.x, "loss": r.loss, **r.grads}
    for p in model.parameters():
        p.grad = None
    x, loss, _ = s["engine"].train_iteration(s["batch"], s["seeds"], 0, s["weights"], None)
    return {"x": x, "loss": loss, **{n: p.grad for n, p in model.named_parameters()}}


# ------------------------------------------------------------------------------ the price
def work(case) -> dict:
    """FLOPs: 2 (36 C + F hidden + hidden C) per cell and step for the forward (the multiplies and
    adds of the perception and the MLP), twice that again for the backward. Bytes: state, given
    mask and clamp values read once, state (and the gradients' size of weights) written once."""
    cfg = build_model(case["preset"]).cfg
    C, hid = cfg.channels, cfg.hidden
    cells = case["boards"] * case["k"] * case["height"] * case["width"]
    per = 2 * (36 * C + 4 * C * hid + hid * C)
    weights = 4 * (36 + 5 * C * hid + hid + C)
    train = case["op"] in ("chunk", "iteration")
    nbytes = cells * (8 * C + 4 * cfg.c_in + 1 + (4 if case["op"] == "step" else 0)) + weights
    if train:
        nbytes += cells * 4 + weights
    return {"bytes": nbytes, "flops": cells * case["depth"] * per * (3 if train else 1)}


# ------------------------------------------------------------------------------ the result in 64 bits
def _uniforms(seed, step, row, hw):
    """u of every cell of the rows numbered `row` at a step, (rows, hw) float64: Philox4x32-10
    (Salmon et al., SC'11) on the counter (cell >> 2, step, row, 0) with the key `seed`, word
    cell & 3, its top 24 bits."""
    mask, rows, dev = 0xFFFFFFFF, len(row), row.device

    def mulhilo(a, b):  # 32 x 32 bits in int64 without overflow
        lo, hi = a * (b & 0xFFFF), a * (b >> 16)
        mid = hi + (lo >> 16)
        return mid >> 16, ((mid << 16) | (lo & 0xFFFF)) & mask

    nq = (hw + 3) // 4
    c0 = torch.arange(nq, device=dev).expand(rows, nq)
    c2 = row[:, None].expand(rows, nq)
    c1 = torch.full_like(c0, step & mask)
    c3 = torch.zeros_like(c0)
    k0, k1 = seed & mask, (seed >> 32) & mask
    for _ in range(10):
        h0, l0 = mulhilo(c0, 0xD2511F53)
        h1, l1 = mulhilo(c2, 0xCD9E8D57)
        c0, c1, c2, c3 = h1 ^ c1 ^ k0, l1, h0 ^ c3 ^ k1, l0
        k0, k1 = (k0 + 0x9E3779B9) & mask, (k1 + 0xBB67AE85) & mask
    w = torch.stack([c0, c1, c2, c3], -1).reshape(rows, 4 * nq)[:, :hw]
    return (w >> 8).double() * 2.0**-24


class _Cell:
    """The cell's step in float64 on cells-last tensors (rows, H, W, C)."""

    def __init__(self, model, case):
        cfg = model.cfg
        self.cfg, self.case = cfg, case
        d = lambda t: t.detach().double()  # noqa: E731
        self.params = {"kernels": d(model.perceive.weight).reshape(4, 9),
                       "w1": d(model.update.fc1.weight).reshape(cfg.hidden, -1),
                       "b1": d(model.update.fc1.bias),
                       "w2": d(model.update.fc2.weight).reshape(cfg.channels, -1),
                       "b2": d(model.update.fc2.bias)}
        if cfg.head == "mlp":
            self.params["head_w"] = d(model.head.weight).reshape(len(cfg.output_tokens), -1)
            self.params["head_b"] = d(model.head.bias)
        self.pad_vec = d(model.pad_vec)
        self.model = model

    def step(self, x, given, clamp, fire):
        """x + fire * MLP(perception of x), the input slice of given cells at the clamp values."""
        cfg, p = self.cfg, self.params
        B, H, W, C = x.shape
        if cfg.padding == "wrap":
            xp = torch.cat([x[:, -1:], x, x[:, :1]], 1)
            xp = torch.cat([xp[:, :, -1:], xp, xp[:, :, :1]], 2)
        else:
            v = self.pad_vec if cfg.padding == "wall" else torch.zeros_like(self.pad_vec)
            xp = v.expand(B, H + 2, W + 2, C).clone()
            xp[:, 1:-1, 1:-1] = x
        taps = [xp[:, i:i + H, j:j + W] for i in range(3) for j in range(3)]
        z = torch.cat([sum(p["kernels"][k, t] * taps[t] for t in range(9)) for k in range(4)], -1)
        h = torch.relu(z @ p["w1"].T + p["b1"])
        u = x + fire[..., None] * (h @ p["w2"].T + p["b2"])
        sl = cfg.in_slice
        u_in = torch.where(given[..., None], clamp, u[..., sl])
        return torch.cat([u[..., :sl.start], u_in, u[..., sl.stop:]], -1)

    def logits(self, x):
        return x[..., self.cfg.out_slice] @ self.params["head_w"].T + self.params["head_b"]

    def confidence(self, x):
        if self.cfg.head == "l2":
            d2 = (x[..., self.cfg.out_slice][..., None, :] - self.model.out_embed.double()).square().sum(-1)
            return (1 / (1 + (d2 + 1e-8).sqrt())).amax(-1)
        return torch.softmax(self.logits(x), -1).amax(-1)


def exact(case, seed):
    cells = case["boards"] * case["k"] * case["height"] * case["width"]
    if cells * case["depth"] > 2e9:
        return None
    s = _inputs(case, seed)
    model, cell = s["model"], _Cell(s["model"], case)
    rows, H, W = s["x"].shape[0], case["height"], case["width"]
    dev = s["x"].device
    given = s["given4"][:, 0]

    def cells_last(t, lo, hi):
        return t[lo:hi].permute(0, 2, 3, 1).double()

    if case["op"] == "step":
        with torch.no_grad():
            y = cell.step(cells_last(s["x"], 0, rows), given, cells_last(s["clamp"], 0, rows),
                          s["fire"][:, 0].double())
        return y.permute(0, 3, 1, 2).contiguous()
    if case["op"] == "rollout":
        out = torch.empty(s["x"].shape, dtype=torch.float64, device=dev)
        conf = torch.empty(rows, dtype=torch.float64, device=dev)
        fired = torch.empty(rows, dtype=torch.int32, device=dev)
        part = max(1, 400_000 // (H * W))  # rows at a time, to bound the memory
        p_low, p_high = (P_LOW, P_GATED) if case["gated"] else (None, model.cfg.fire_rate)
        # the thresholds in 32 bits, as the entry point takes them
        p_high = float(np.float32(p_high))
        with torch.no_grad():
            for lo in range(0, rows, part):
                hi = min(rows, lo + part)
                x, cl, gv = cells_last(s["x"], lo, hi), cells_last(s["clamp"], lo, hi), given[lo:hi]
                n = torch.zeros(hi - lo, dtype=torch.int64, device=dev)
                row = torch.arange(lo, hi, device=dev)
                for t in range(case["depth"]):
                    u = _uniforms(int(seed), t, row, H * W).view(hi - lo, H, W)
                    p = torch.full_like(u, p_high)
                    if p_low is not None:
                        sure = (cell.confidence(x) > float(np.float32(TAU))) | gv
                        p = torch.where(sure, float(np.float32(p_low)), p)
                    f = u < p
                    n += f.flatten(1).sum(1)
                    x = cell.step(x, gv, cl, f.double())
                out[lo:hi] = x.permute(0, 3, 1, 2)
                conf[lo:hi] = cell.confidence(x).flatten(1).mean(1)
                fired[lo:hi] = n.int()
        return {"x": out, "conf": conf, "fired": fired}
    # training: autograd through the chunk
    for p in cell.params.values():
        p.requires_grad_(True)
    x, cl = cells_last(s["x"], 0, rows), cells_last(s["clamp"], 0, rows)
    p = float(np.float32(model.cfg.fire_rate))
    all_rows = torch.arange(rows, device=dev)
    loss = 0.0
    for t in range(case["depth"]):
        f = (_uniforms(int(s["seeds"][t]), t, all_rows, H * W) < p).double().view(rows, H, W)
        x = cell.step(x, given, cl, f)
        if case["op"] == "chunk":
            cls = model.output_index(s["targets"])
            lg = torch.log_softmax(cell.logits(x), -1)
            loss = loss - lg.gather(-1, cls[..., None]).mean()
        else:
            e = model.target_embedding(s["targets"]).permute(0, 2, 3, 1).double()
            loss = loss + (x[..., model.cfg.out_slice] - e).square().sum(-1).mean()
    loss = loss / case["depth"]
    loss.backward()
    out = {"x": x.detach().permute(0, 3, 1, 2).contiguous(), "loss": loss.detach()}
    names = ({"kernels": model.perceive.weight, "w1": model.update.fc1.weight,
              "b1": model.update.fc1.bias, "w2": model.update.fc2.weight,
              "b2": model.update.fc2.bias})
    if cell.cfg.head == "mlp":
        names.update(head_w=model.head.weight, head_b=model.head.bias)
    if case["op"] == "chunk":
        for n, q in names.items():
            out[n] = cell.params[n].grad.reshape(q.shape)
        return out
    by_id = {id(q): cell.params[n].grad.reshape(q.shape) for n, q in names.items()}
    out.update({n: by_id[id(q)] for n, q in model.named_parameters()})
    return out


def tolerance(case) -> dict:
    """About four times the relative error against `exact` that was measured over the ranges of
    `draw`: fp32 steps 1e-7 and rollouts 4e-7 (the board confidence, a sum over the cells in one
    order, 4e-6), bf16 steps 3e-3, rollouts 1.3e-2 and chunk gradients 1e-2. The gradients of an
    fp32 chunk reach 8e-5, where one hidden unit's input lies within an fp32 rounding of zero and
    its ReLU passes the gradient or not. Gated firing compares a confidence with a threshold: a
    cell whose confidence lies within the rounding of it fires or not, which moves that cell's
    state by its whole update and the fired count of its row by one."""
    bf16 = case["precision"] == "bf16"
    if case["op"] == "step":
        return {"rel": 1.2e-2 if bf16 else 1e-6}
    if case["op"] == "rollout":
        if case["gated"]:
            return {"rel": 5e-2, "differ": 0.95} if bf16 else {"rel": 2e-3, "differ": 0.02}
        return {"rel": 5e-2 if bf16 else 1.5e-5}
    if case["op"] == "chunk":
        return {"rel": 4e-2 if bf16 else 3e-4}
    return {"rel": 2e-4}
