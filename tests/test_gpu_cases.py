"""The measured cases (perf/cases.py) at small sizes: what `run` returns lies within `tolerance` of
`exact`, and the fired counts of gated bf16 rollouts, whose single values may differ, within what
independent draws of the same gate would show."""

import math

import pytest
import torch

from perf import cases as P

pytestmark = pytest.mark.gpu


def _small(c):
    c = dict(c, boards=min(c["boards"], 6), k=min(c["k"], 2), depth=min(c["depth"], 6))
    return dict(c, height=min(c["height"], 45), width=min(c["width"], 45))


def _flat(o):
    return o if isinstance(o, dict) else {"out": o}


@pytest.mark.parametrize("case", [_small(c) for c in P.listed()], ids=lambda c: c["name"])
def test_run_is_within_tolerance_of_exact(case):
    out = {k: v.clone() if torch.is_tensor(v) else v for k, v in _flat(P.run(P.prepare(case, 3))).items()}
    ref, tol = _flat(P.exact(case, 3)), P.tolerance(case)
    assert out.keys() == ref.keys()
    for k, e in ref.items():
        if e is None:
            continue
        v = torch.as_tensor(out[k]).double().cpu().flatten()
        e = torch.as_tensor(e).double().cpu().flatten()
        if k != "fired":
            assert float((v - e).norm()) <= tol["rel"] * float(e.norm()), k
            continue
        assert float((v != e).double().mean()) <= tol.get("differ", 0.0)
        # two draws of the same gate differ by a binomial scatter: 5 sigma of the difference of two
        # totals (p (1 - p) <= 1/4); another gate or mask moves the total by a share of all cells
        n = case["height"] * case["width"] * case["depth"] * len(v)
        assert abs(float(v.sum() - e.sum())) <= 5 * math.sqrt(2 * n / 4)
