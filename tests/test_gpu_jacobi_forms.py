"""The FP64 Jacobi kernels that callers reach with the Jacobi's own parameters
(here jacobi_tol; FP64 contexts iterate otherwise): the plain forms, the
queue of warm-started chains in both orders, the obs-count buckets, cubes, vertical
localisation, FP32 state and the autotuner.  Each case checks by the sweep counts
that the Jacobi ran.  Bar: 1e-10 against the oracle, as the other FP64 forms.
"""
import numpy as np
import pytest

from test_gpu_sweep import _rel_err, _var_rows

pytestmark = pytest.mark.gpu
TOL = 1e-13             # the Jacobi's tolerance in FP64 when a caller sets none
NZ = 2
LEVELS = ([0, 1, 1 + NZ, 1 + 2 * NZ], [1, NZ, NZ, NZ])


def _data(dl, k, nlat=24, nlon=48, nobs=1500):
    cfg = dl.synth_cfg(nlat, nlon, NZ, k, nobs, seed=0xD1DA0D00 + k + nlon, cluster_frac=0.5,
                       nclusters=2, rscale=(0.5, 3.0))
    return cfg, dl.synth_generate(cfg)


def _engine(dl, torch, cfg, data, ph=None, **over):
    p = dict(nanals=cfg.k, nrow=1 + 3 * NZ, nlat=cfg.nlat, nlon=cfg.nlon, local_dist=900.0,
             inflation_factor=1.05, bin_deg=4.0, form=dl.FORM_BATCHED, gram=dl.GRAM_FP64,
             jacobi_tol=TOL)
    p.update(over)
    params = dl.default_params(**p)
    eng = dl.Engine(params, nobs_max=cfg.nobs)
    eng.set_grid(data["grid_lat"], data["grid_lon"])
    phd = None
    if ph is not None:
        T = lambda x: torch.tensor(np.ascontiguousarray(x), dtype=torch.float64, device="cuda")
        eng.set_levels({"type": 0, "c1": T(np.linspace(0.0, 1.0, NZ + 1)), "ptop": 10.0}, 0,
                       *LEVELS)
        phd = T(ph)
    return params, eng, dl.DeviceObs(data["lat"], data["lon"], data["yb"], data["dep"],
                                     data["rinv"], phd)


def _run(dl, torch, cfg, data, ph=None, f32=False, **over):
    params, eng, obs = _engine(dl, torch, cfg, data, ph, **over)
    xb = data["xb"].float() if f32 else data["xb"]
    xa, axa = torch.empty_like(xb), torch.empty_like(data["axb"])
    eng.sweep(obs, xb, data["axb"], xa, axa)
    st = eng.stats()
    eng.close()
    assert st["status"] == 0 and st["nonconverged"] == 0, st
    return params, xa, axa, st


def _check(oracle, cfg, data, params, xa, axa, ph=None, f32=False):
    h = {key: v.cpu().numpy() for key, v in data.items()}
    if f32:
        h["xb"] = h["xb"].astype(np.float32).astype(np.float64)
    o = oracle.Obs(h["lat"], h["lon"], h["yb"], h["dep"], h["rinv"])
    perm, bs, nb, nl = oracle.bin_obs(o, 4.0, params.obs_polar)
    prm = oracle.params(cfg.k, params.nrow, cfg.nlat, cfg.nlon, params.local_dist,
                        params.inflation_factor, max_obs=params.max_obs)
    bins = (bs, nb, nl, 4.0, perm)
    if ph is not None:
        vc = {"type": 0, "c1": np.linspace(0.0, 1.0, NZ + 1), "ptop": 10.0}
        out = oracle.sweep_vertical(prm, h["grid_lat"], h["grid_lon"], o.permuted(perm), ph[perm],
                                    h["xb"], h["axb"], vc, 0, *LEVELS, params.vert_dist,
                                    params.cube_nz, bool(params.gc_filter_vertical), bins=bins,
                                    cube_n=params.cube_n)
    else:
        out = oracle.sweep_cubes(prm, h["grid_lat"], h["grid_lon"], o.permuted(perm), h["xb"],
                                 h["axb"], params.cube_n, params.overlap, bins=bins)
    assert out["nfail"] == 0
    xa_h, axa_h = xa.double().cpu().numpy(), axa.cpu().numpy()
    for var, rows in _var_rows(NZ).items():
        assert _rel_err(axa_h[:, rows] - h["axb"][:, rows],
                        out["axa"][:, rows] - h["axb"][:, rows]) <= 1e-10, var
        assert _rel_err(xa_h[:, rows], out["xa"][:, rows]) <= (2.0 ** -24 if f32 else 1e-10), var


CASES = {
    # the plain form: one wavefront (padded to 32 and 64) and one workgroup an analysis
    "plain_k20": (20, dict(form=0)),
    "plain_k33": (33, dict(form=0)),
    "plain_k64": (64, dict(form=0)),
    "plain_k40_f32": (40, dict(form=0, f32=True)),
    "plain_k100": (100, dict(form=0)),
    "plain_k128": (128, dict(form=0)),
    "plain_k24_cubes": (24, dict(form=0, cube_n=3, overlap=1)),
    # chains: cold and warm starts, a chain per column and longer ones
    "batched_k20_chain1": (20, dict(chain_len=1)),
    "batched_k20_chain8": (20, dict(chain_len=8)),
    "batched_k64_chain8_grouped": (64, dict(chain_len=8, xcd_tiles=1)),
    "batched_k64_cold": (64, dict(chain_len=8, warm_start=0)),
    "batched_k32": (32, {}),
    "batched_k50_cubes": (50, dict(cube_n=2, overlap=1)),
    "batched_k32_buckets": (32, dict(bucket_chain=[1, 64, 2, 8])),
    "batched_k100": (100, dict(chain_len=7)),
    "vertical_k24": (24, dict(vert_dist=0.8, cube_nz=1)),
    "vertical_k40_hcube2": (40, dict(vert_dist=0.8, cube_nz=2, cube_n=2)),
}


@pytest.mark.parametrize("case", list(CASES))
def test_jacobi_form_matches_oracle(cuda, dl, oracle, case):
    torch = cuda
    k, over = CASES[case]
    over = dict(over)
    f32 = over.pop("f32", False)
    print(f"Jacobi form {case}", flush=True)
    cfg, data = _data(dl, k)
    ph = np.random.default_rng(k).uniform(50.0, 1000.0, cfg.nobs) if "vert_dist" in over else None
    params, xa, axa, st = _run(dl, torch, cfg, data, ph, f32, **over)
    print(f"  mean sweeps {st['sweeps_sum'] / st['nanal']:.2f}", flush=True)
    assert st["max_sweeps_used"] > 4
    _check(oracle, cfg, data, params, xa, axa, ph, f32)


@pytest.mark.parametrize("k", [20, 64])
def test_warm_starts_take_fewer_sweeps(cuda, dl, k):
    torch = cuda
    print(f"warm starts k={k}", flush=True)
    cfg, data = _data(dl, k)
    warm = _run(dl, torch, cfg, data, chain_len=8)[3]
    cold = _run(dl, torch, cfg, data, chain_len=8, warm_start=0)[3]
    iterated = _run(dl, torch, cfg, data, chain_len=8, jacobi_tol=0.0)[3]
    assert iterated["max_sweeps_used"] <= 4
    assert 4 * warm["nanal"] < warm["sweeps_sum"] < cold["sweeps_sum"]


# the queue's order decides which wavefront runs a chain, not its analyses
@pytest.mark.parametrize("nlat,nlon,chain_len", [(24, 48, 7), (30, 5, 64), (9, 17, 1)])
def test_grouped_jacobi_queue_equals_sorted_queue(cuda, dl, nlat, nlon, chain_len):
    torch = cuda
    print(f"Jacobi queue {nlat}x{nlon} chain {chain_len}", flush=True)
    cfg, data = _data(dl, 20, nlat, nlon)
    _, xa, axa, st = _run(dl, torch, cfg, data, chain_len=chain_len, xcd_tiles=0)
    _, xa2, axa2, st2 = _run(dl, torch, cfg, data, chain_len=chain_len, xcd_tiles=1)
    assert st["max_sweeps_used"] > 4 and st["sweeps_sum"] == st2["sweeps_sum"]
    assert torch.equal(xa, xa2) and torch.equal(axa, axa2)


@pytest.mark.parametrize("k", [32, 72])
def test_autotune_of_the_jacobi_times_chains(cuda, dl, oracle, k):
    torch = cuda
    print(f"autotune of chains k={k}", flush=True)
    cfg, data = _data(dl, k)
    params, eng, obs = _engine(dl, torch, cfg, data)
    xa, axa = torch.empty_like(data["xb"]), torch.empty_like(data["axb"])
    t = eng.autotune(obs, data["xb"], data["axb"], xa, axa)
    print(f"  {t}", flush=True)
    st = eng.stats()
    eng.close()
    assert st["status"] == 0 and st["nonconverged"] == 0 and st["max_sweeps_used"] > 4
    assert t["chain_len"] > 0 and t["ncand"] >= 4 + 10      # lengths times queue orders
    assert 0.0 < t["ms_best"] <= t["ms_initial"]
    _check(oracle, cfg, data, params, xa, axa)
