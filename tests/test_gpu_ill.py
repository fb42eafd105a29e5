"""FP64 sweeps whose analyses are above the condition limit of the polynomial
iteration (letkf_isqrt.h), so that the Jacobi of the iterating contexts runs: in
every form of the kernels (columns with the update fused, transforms of cubes,
vertical localisation, runs that start inside the grid, FP32 state, the marked
analyses of 65 to 128 members).

Accurate, dense obs: condition numbers of some 5e3 to 1e5.  Bar: 1e-10 against the
oracle, as the other FP64 sweeps; the rounding of C's entries alone, a few 1e-16 of
its norm, is 1e-11 of the smallest eigenvalues there.
"""
import numpy as np
import pytest

from test_gpu_sweep import _rel_err, _var_rows

pytestmark = pytest.mark.gpu
NZ = 2


def _case(dl, k, scale, nlat=16, nlon=32, nobs=1500):
    cfg = dl.synth_cfg(nlat, nlon, NZ, k, nobs, seed=0xD1DA0A00 + k)
    data = dl.synth_generate(cfg)
    data["rinv"] = (data["rinv"].double() * scale).float()
    return cfg, data


def _sweep(dl, torch, cfg, data, ph=None, capacity=0, f32=False, **over):
    p = dict(nanals=cfg.k, nrow=1 + 3 * NZ, nlat=cfg.nlat, nlon=cfg.nlon, local_dist=1200.0,
             inflation_factor=1.05, bin_deg=4.0)
    p.update(over)
    params = dl.default_params(**p)
    eng = dl.Engine(params, nobs_max=cfg.nobs, capacity=capacity)
    eng.set_grid(data["grid_lat"], data["grid_lon"])
    phd = None
    if ph is not None:
        T = lambda x: torch.tensor(np.ascontiguousarray(x), dtype=torch.float64, device="cuda")
        eng.set_levels({"type": 0, "c1": T(np.linspace(0.0, 1.0, NZ + 1)), "ptop": 10.0}, 0,
                       [0, 1, 1 + NZ, 1 + 2 * NZ], [1, NZ, NZ, NZ])
        phd = T(ph)
    obs = dl.DeviceObs(data["lat"], data["lon"], data["yb"], data["dep"], data["rinv"], phd)
    xb = data["xb"].float() if f32 else data["xb"]
    xa, axa = torch.empty_like(xb), torch.empty_like(data["axb"])
    eng.sweep(obs, xb, data["axb"], xa, axa)
    st = eng.stats(strict=False)
    eng.close()
    return params, xa, axa, st


# name: k, scale of R^-1, engine parameters
CASES = {
    "columns_k20": (20, 1e4, {}),
    "columns_k48": (48, 1e4, {}),
    "columns_k64_rtps": (64, 1e4, dict(rtps=1, rtps_alpha=0.8)),
    "columns_k40_batched": (40, 1e4, dict(form=1)),
    "columns_k33_runs": (33, 1e4, dict(capacity=3)),
    "columns_k40_f32": (40, 1e4, dict(f32=True)),
    "cubes_k16": (16, 1e4, dict(cube_n=3, overlap=1)),
    "cubes_k63_batched": (63, 1e4, dict(cube_n=2, overlap=1, form=1)),
    "vertical_k24": (24, 1e4, dict(form=1, vert_dist=1.0, cube_nz=1)),
    "vertical_k50_hcube2": (50, 1e4, dict(form=1, vert_dist=1.0, cube_nz=2, cube_n=2)),
    "columns_k65": (65, 1e4, {}),
    "columns_k100_batched": (100, 1e4, dict(form=1)),
    "columns_k97_runs": (97, 1e4, dict(capacity=3)),
    "cubes_k128_batched": (128, 1e4, dict(cube_n=2, overlap=1, form=1)),
}


@pytest.mark.parametrize("case", list(CASES))
def test_ill_conditioned_sweep_matches_oracle(cuda, dl, oracle, case):
    torch = cuda
    k, scale, over = CASES[case]
    over = dict(over)
    cfg, data = _case(dl, k, scale)
    vert = "vert_dist" in over
    f32 = over.pop("f32", False)
    ph = np.random.default_rng(k).uniform(50.0, 1000.0, cfg.nobs) if vert else None
    cap = over.pop("capacity", 0)
    print(f"ill-conditioned sweep {case}", flush=True)
    if cap:  # a workspace of a third of the lists
        cap = _sweep(dl, torch, cfg, data, **over)[3]["nobsl_sum"] // cap + 1
    params, xa, axa, st = _sweep(dl, torch, cfg, data, ph, cap, f32, **over)
    mean = st["sweeps_sum"] / st["nanal"]
    print(f"  mean sweeps {mean:.2f}, at most {st['max_sweeps_used']}", flush=True)
    assert st["status"] == 0 and st["nonconverged"] == 0, st
    assert mean > 4.5           # (the iteration takes at most 4 steps)
    h = {key: v.cpu().numpy() for key, v in data.items()}
    if f32:
        h["xb"] = h["xb"].astype(np.float32).astype(np.float64)
    o = oracle.Obs(h["lat"], h["lon"], h["yb"], h["dep"], h["rinv"])
    perm, bs, nb, nl = oracle.bin_obs(o, params.bin_deg, params.obs_polar)
    prm = oracle.params(k, params.nrow, cfg.nlat, cfg.nlon, params.local_dist,
                        params.inflation_factor, max_obs=params.max_obs)
    bins = (bs, nb, nl, params.bin_deg, perm)
    if vert:
        vc = {"type": 0, "c1": np.linspace(0.0, 1.0, NZ + 1), "ptop": 10.0}
        out = oracle.sweep_vertical(prm, h["grid_lat"], h["grid_lon"], o.permuted(perm), ph[perm],
                                    h["xb"], h["axb"], vc, 0, [0, 1, 1 + NZ, 1 + 2 * NZ],
                                    [1, NZ, NZ, NZ], params.vert_dist, params.cube_nz,
                                    bool(params.gc_filter_vertical), bins=bins,
                                    cube_n=params.cube_n)
    else:
        out = oracle.sweep_cubes(prm, h["grid_lat"], h["grid_lon"], o.permuted(perm), h["xb"],
                                 h["axb"], params.cube_n, params.overlap, bins=bins)
    assert out["nfail"] == 0
    if params.rtps:
        full, _, _ = oracle.post(1, h["grid_lat"], cfg.nlat, cfg.nlon, 90.0, 0, 0,
                                 params.rtps_alpha, h["xb"], h["axb"], out["xa"], out["axa"])
        out["xa"] = full - out["axa"][..., None]
    xa_h, axa_h = xa.double().cpu().numpy(), axa.cpu().numpy()
    for var, rows in _var_rows(NZ).items():
        e_inc = _rel_err(axa_h[:, rows] - h["axb"][:, rows], out["axa"][:, rows] - h["axb"][:, rows])
        e_xa = _rel_err(xa_h[:, rows], out["xa"][:, rows])
        print(f"  {var}: increment {e_inc:.2e} Xa' {e_xa:.2e}", flush=True)
        assert e_inc <= 1e-10, var
        # FP32 state: one rounding of each value
        assert e_xa <= (2.0 ** -24 if f32 else 1e-10), var


# The Jacobi in the iteration's kernel runs one wavefront a SIMD above 32 members, that
# of a caller's jacobi_tol two, from M itself: equal sweeps took 11 to 21 % longer.
@pytest.mark.parametrize("k", [24, 48, 64, 100])
def test_ill_conditioned_sweeps_start_from_the_cholesky_factor(cuda, dl, k):
    torch = cuda
    cfg, data = _case(dl, k, 1e4)
    print(f"sweeps of ill-conditioned analyses k={k}", flush=True)
    _, xa, axa, st = _sweep(dl, torch, cfg, data)
    _, xa2, axa2, st2 = _sweep(dl, torch, cfg, data, jacobi_tol=1e-13)
    print(f"  sweeps {st['sweeps_sum']} from L, {st2['sweeps_sum']} from M", flush=True)
    assert st["status"] == 0 and st["max_sweeps_used"] > 4, st
    assert st["sweeps_sum"] < 0.875 * st2["sweeps_sum"]


@pytest.mark.parametrize("form", [0, 1])
@pytest.mark.parametrize("k", [100, 128])
def test_very_ill_conditioned_sweeps_converge(cuda, dl, k, form):
    """Condition numbers of 1e7 and more, where cold sweeps of M itself pass the cap."""
    torch = cuda
    cfg, data = _case(dl, k, 1e6)
    print(f"very ill-conditioned k={k} form={form}", flush=True)
    _, xa, axa, st = _sweep(dl, torch, cfg, data, form=form)
    print(f"  {st['nonconverged']} of {st['nanal']} not converged, mean sweeps "
          f"{st['sweeps_sum'] / st['nanal']:.2f}", flush=True)
    assert st["status"] == 0 and st["nonconverged"] == 0, st
    assert bool(torch.isfinite(xa).all()) and bool(torch.isfinite(axa).all())
