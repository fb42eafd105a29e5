"""The update of columns from the mean of their covering cubes' transforms, at
the sizes where its blocks of columns and tiles of members end: k at and beside
multiples of 16 and of 4, cubes whose starts and ends fall on different columns
(cube_n not a multiple of the step), grids that give a wavefront several columns
and one, FP64 and FP32 state.  Bar: 1e-10 against the oracle, as the FP64 cube
sweeps, and one rounding of Xa' stored in FP32.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rel_err(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


# k, grid, cube_n, overlap, rtps, state in FP32
CASES = [
    (15, 150, 160, 3, 1, 0.0, False),   # segments of one column, blocks of up to two
    (16, 23, 41, 4, 0, 0.8, False),     # one column a wavefront
    (33, 130, 141, 4, 2, 0.8, False),   # blocks of 2 x 2, clipped at the last longitude
    (48, 128, 140, 5, 2, 0.0, False),   # segments of two and one columns
    (63, 23, 41, 5, 2, 0.8, False),
    (64, 131, 130, 2, 0, 0.0, False),   # blocks of 2 x 2, clipped at the last latitude
    # above 64 members: 5 to 8 tiles, their last one from 1 to 16 members wide
    (65, 31, 37, 4, 2, 0.8, False),
    (80, 23, 41, 3, 0, 0.0, True),
    (82, 95, 96, 2, 0, 0.0, True),      # blocks of 2 x 2
    (95, 23, 41, 5, 2, 0.8, True),
    (97, 23, 41, 3, 1, 0.0, False),
    (115, 23, 41, 4, 0, 0.8, True),
    (128, 23, 41, 3, 1, 0.8, False),
]


@pytest.mark.parametrize("k,nlat,nlon,cube_n,overlap,rtps,f32", CASES)
def test_cube_update_blocks(cuda, dl, oracle, k, nlat, nlon, cube_n, overlap, rtps, f32):
    torch = cuda
    print(f"cube update k={k} {nlat}x{nlon} cube {cube_n}/{overlap}", flush=True)
    cfg = dl.synth_cfg(nlat, nlon, 1, k, 400, seed=0xD1DA0900 + k)
    data = dl.synth_generate(cfg)
    if f32:
        data["xb"] = data["xb"].float()
    n = 1 + 3 * cfg.nz
    extra = dict(rtps=1, rtps_alpha=rtps) if rtps else {}
    params = dl.default_params(nanals=k, nrow=n, nlat=nlat, nlon=nlon, local_dist=700.0,
                               inflation_factor=1.05, bin_deg=3.0, cube_n=cube_n,
                               overlap=overlap, form=dl.FORM_BATCHED, gram=dl.GRAM_FP64, **extra)
    eng = dl.Engine(params, nobs_max=cfg.nobs)
    eng.set_grid(data["grid_lat"], data["grid_lon"])
    obs = dl.DeviceObs(data["lat"], data["lon"], data["yb"], data["dep"], data["rinv"])
    xa = torch.full_like(data["xb"], float("nan"))
    axa = torch.full_like(data["axb"], float("nan"))
    eng.sweep(obs, data["xb"], data["axb"], xa, axa)
    assert eng.stats()["status"] == 0
    h = {key: v.cpu().numpy() for key, v in data.items()}
    h["xb"] = h["xb"].astype(np.float64)
    o = oracle.Obs(h["lat"], h["lon"], h["yb"], h["dep"], h["rinv"])
    perm, bin_start, nband, nlonbin = oracle.bin_obs(o, 3.0, params.obs_polar)
    prm = oracle.params(k, n, nlat, nlon, params.local_dist, params.inflation_factor,
                        max_obs=params.max_obs)
    out = oracle.sweep_cubes(prm, h["grid_lat"], h["grid_lon"], o.permuted(perm), h["xb"],
                             h["axb"], cube_n, overlap, bins=(bin_start, nband, nlonbin, 3.0, perm))
    assert out["nfail"] == 0
    exp_xa, exp_axa = out["xa"], out["axa"]
    if rtps:
        full, _, _ = oracle.post(1, h["grid_lat"], nlat, nlon, 90.0, 0, 0, rtps, h["xb"],
                                 h["axb"], exp_xa, exp_axa)
        exp_xa = full - exp_axa[..., None]
    xa_h, axa_h = xa.cpu().numpy(), axa.cpu().numpy()
    for row in range(n):
        inc = exp_axa[:, row] - h["axb"][:, row]
        assert _rel_err(axa_h[:, row] - h["axb"][:, row], inc) <= 1e-10, row
        # FP32 state: one rounding of each value
        assert _rel_err(xa_h[:, row], exp_xa[:, row]) <= (2.0 ** -24 if f32 else 1e-10), row
    eng.close()
