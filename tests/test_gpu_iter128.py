"""The iteration kernel of 65 to 128 members (letkf_iter128.hip) at the edges of
its tiles of 16 members, stages of 16 obs and groups of 64 analyses, over its
condition classes, above them (the marked analyses of the Jacobi) and with an obs
that is not finite.  Bar: 1e-10 against the oracle, as the other core tests.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = 1e-10


def _rel(a, b):
    return np.abs(a - b).max() / max(1.0, np.abs(b).max())


@pytest.mark.parametrize("k", [65, 79, 80, 81, 96, 97, 112, 113, 127, 128])
def test_core_over_tiles_and_condition_numbers(cuda, dl, oracle, k):
    rng = np.random.default_rng(1000 + k)
    rho = 1.1
    kappas = [1.001, 1.9, 3.0, 7.0, 15.0, 30.0, 60.0, 120.0, 250.0, 900.0, 2000.0, 4000.0, 4.0e4]
    counts = [1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 64, 100, 145]
    max_obs, reps = 145, 5                     # 66 analyses: past one group of 64
    n = len(kappas) * reps + 1
    hx = np.zeros((n, max_obs, k))
    dep = np.zeros((n, max_obs))
    nb = np.zeros(n, np.int32)                 # the last analysis has no obs
    for j in range(n - 1):
        p, kappa = counts[(j + j // len(kappas)) % len(counts)], kappas[j % len(kappas)]
        y = rng.normal(size=(p, k)) * np.exp(rng.uniform(-1.0, 1.0, (p, 1)))
        y -= y.mean(axis=1, keepdims=True)
        y *= np.sqrt((kappa - 1.0) * (k - 1) / rho / np.linalg.eigvalsh(y.T @ y)[-1])
        hx[j, :p], dep[j, :p], nb[j] = y, rng.normal(size=p), p
    bad = 20
    hx[bad, 0, k - 1] = np.nan
    ri, rl = np.ones((n, max_obs), np.float32), np.ones((n, max_obs))
    print(f"iter128 core k={k}", flush=True)
    trans, wbar = dl.letkf_core_batch(nb, hx, ri, dep, rl, rho)
    for j in range(n):
        if j == bad:
            assert np.isnan(trans[j]).all() and np.isnan(wbar[j]).all()
            continue
        if 13 <= j < n - 1 - 13:
            continue                           # the first and last repeat, and the rest unread
        p = nb[j]
        t_o, w_o, _ = oracle.letkf_core(hx[j, :p], ri[j, :p], dep[j, :p], rl[j, :p], rho)
        assert _rel(trans[j], t_o) < TOL, (k, j)
        assert _rel(wbar[j], w_o) < TOL, (k, j)
