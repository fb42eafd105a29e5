"""A background mean that is not finite: its row of Xa' is NaN and its mean not finite
in every form (the reference forms Xa = trans^T Xb' + xbar_b before it takes the mean,
letkf_compute.F90:261-299), and every other row is that of a clean sweep."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# k, cube_n, overlap, form, rtps, FP32 state: the fused update, the update of blocks of
# columns (up to and above 64 members) and the one of FP32 state up to 64
CASES = [
    (20, 1, 0, 0, 0.0, False),
    (24, 3, 1, 1, 0.0, False),
    (64, 2, 0, 0, 0.8, False),
    (40, 1, 0, 0, 0.0, True),
    (82, 1, 0, 1, 0.0, False),
    (100, 2, 1, 0, 0.8, True),
]


@pytest.mark.parametrize("k,cube_n,overlap,form,rtps,f32", CASES)
def test_nonfinite_background_mean(cuda, dl, k, cube_n, overlap, form, rtps, f32):
    torch = cuda
    print(f"non-finite mean k={k} cube {cube_n}/{overlap}", flush=True)
    cfg = dl.synth_cfg(14, 22, 5, k, 600, seed=0xD1DA0C00 + k)
    data = dl.synth_generate(cfg)
    n = 1 + 3 * cfg.nz
    extra = dict(rtps=1, rtps_alpha=rtps) if rtps else {}
    params = dl.default_params(nanals=k, nrow=n, nlat=cfg.nlat, nlon=cfg.nlon, local_dist=1200.0,
                               inflation_factor=1.05, bin_deg=4.0, cube_n=cube_n,
                               overlap=overlap, form=form, gram=dl.GRAM_FP64, **extra)
    eng = dl.Engine(params, nobs_max=cfg.nobs)
    eng.set_grid(data["grid_lat"], data["grid_lon"])
    obs = dl.DeviceObs(data["lat"], data["lon"], data["yb"], data["dep"], data["rinv"])
    xb = data["xb"].float() if f32 else data["xb"]
    out = []
    axb = data["axb"].clone()
    where = [(0, 0), (17, n - 1), (cfg.nlat * cfg.nlon - 1, 3)]
    for bad in (False, True):
        if bad:
            for (col, row), v in zip(where, (float("nan"), float("inf"), float("-inf"))):
                axb[col, row] = v
        xa, axa = torch.empty_like(xb), torch.empty_like(axb)
        eng.sweep(obs, xb, axb, xa, axa)
        assert eng.stats()["status"] == 0
        out.append((xa.cpu().numpy(), axa.cpu().numpy()))
    eng.close()
    (xa0, axa0), (xa1, axa1) = out
    keep = np.ones(axa0.shape, bool)
    for col, row in where:
        keep[col, row] = False
        assert np.isnan(xa1[col, row]).all(), (col, row)
        assert not np.isfinite(axa1[col, row]), (col, row)
    assert np.array_equal(xa1[keep], xa0[keep]) and np.array_equal(axa1[keep], axa0[keep])
