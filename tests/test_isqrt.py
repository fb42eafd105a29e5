"""M^(-1/2) by polynomial iteration (letkf_isqrt.h): the step table on the CPU,
and the core entry at the edges of its tiles and of its condition classes
against the oracle's eigensolve."""
import os
import re
from fractions import Fraction

import numpy as np
import pytest

SRC = os.path.join(os.path.dirname(__file__), "..", "dida-thhpca-sc23_amd", "csrc",
                   "letkf_isqrt.h")
TOL = 1e-10  # the repository's bar for the FP64 forms


def _plans():
    text = open(SRC).read()
    body = re.search(r"kIsqrtPlan\[kIsqrtPlans\] = \{(.*?)\n\};", text, re.S).group(1)
    body = re.sub(r"//.*", "", body)
    tree = eval("[" + body.replace("{", "[").replace("}", "]") + "]")  # numbers only
    limit = float(re.search(r"kIsqrtMaxKappa = ([0-9.]+)", text).group(1))
    count = int(re.search(r"kIsqrtPlans = (\d+)", text).group(1))
    assert len(tree) == count
    return tree, limit


def test_plans_reach_rounding_over_their_whole_interval():
    """x -> x p(x^2) over every step of a plan, in exact arithmetic on the
    table's doubles, ends within 2^-52 of 1 for x in [kappa^-1/2, 1]."""
    plans, limit = _plans()
    assert [p[0] for p in plans] == sorted(p[0] for p in plans) and plans[-1][0] == limit
    for kappa, nstep, steps in plans:
        assert len(steps) == nstep and all(s[0] in (2, 3, 5) for s in steps)
        assert steps[0][0] > 2  # the first step's T^2 is formed for the norm in any case
        lo = 1.0 / kappa ** 0.5
        worst = 0.0
        for x0 in np.linspace(lo, 1.0, 101):
            x = Fraction(float(x0))
            for nc, c in steps:
                t = x * x
                x = x * sum(Fraction(c[j]) * t ** j for j in range(nc))
                x = Fraction(int(x * 2 ** 90), 2 ** 90)  # keep the fractions short
            worst = max(worst, abs(float(x - 1)))
        assert worst < 2.0 ** -52, (kappa, worst)


def _rel(a, b):
    """The measure of the core entry's other parity tests (test_gpu_core.py)."""
    return np.abs(a - b).max() / max(1.0, np.abs(b).max())


def _problem(rng, k, p, kappa, rho=1.1):
    """Obs of one analysis scaled so that M's condition number is kappa."""
    y = rng.normal(size=(p, k)) * np.exp(rng.uniform(-1.0, 1.0, (p, 1)))
    y -= y.mean(axis=1, keepdims=True)
    c = y.T @ y
    top = np.linalg.eigvalsh(c)[-1]
    y *= np.sqrt((kappa - 1.0) * (k - 1) / rho / top)
    return y, np.ones(p, np.float32), rng.normal(size=p), np.ones(p), rho


# 2..64 at the edges of the 16-row tiles; condition numbers inside the classes,
# at the iteration's limit and above it (where the Jacobi takes over)
@pytest.mark.gpu
@pytest.mark.parametrize("k", [2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64])
def test_core_over_condition_numbers(cuda, dl, oracle, k):
    rng = np.random.default_rng(k)
    kappas = [1.001, 1.9, 3.0, 7.0, 15.0, 30.0, 60.0, 120.0, 250.0, 900.0, 2000.0, 4000.0, 4.0e4]
    max_obs = 133
    hx = np.zeros((len(kappas), max_obs, k))
    nb = np.zeros(len(kappas), np.int32)
    dep = np.zeros((len(kappas), max_obs))
    for j, kappa in enumerate(kappas):
        p = (1, 31, 32, 33, 63, 64, 65, 96, 97, 127, 128, 129, 133)[j]
        y, _, d, _, rho = _problem(rng, k, p, kappa)
        hx[j, :p], dep[j, :p], nb[j] = y, d, p
    ri, rl = np.ones((len(kappas), max_obs), np.float32), np.ones((len(kappas), max_obs))
    print(f"isqrt core k={k}", flush=True)
    trans, wbar = dl.letkf_core_batch(nb, hx, ri, dep, rl, rho)
    for j, kappa in enumerate(kappas):
        p = nb[j]
        t_o, w_o, _ = oracle.letkf_core(hx[j, :p], ri[j, :p], dep[j, :p], rl[j, :p], rho)
        assert _rel(trans[j], t_o) < TOL, (k, kappa)
        assert _rel(wbar[j], w_o) < TOL, (k, kappa)
