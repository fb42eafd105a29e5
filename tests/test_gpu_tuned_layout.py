"""A context created with the layout that the autotuner returned runs the sweep that
was tuned: the same solver (FP64 contexts iterate, also above 64 members, where a
chain length asks for the Jacobi) and the same bits."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,form", [(40, 1), (82, 1), (82, 0)])
def test_returned_layout_reproduces_the_tuned_sweep(cuda, dl, k, form):
    torch = cuda
    print(f"tuned layout k={k} form={form}", flush=True)
    cfg = dl.synth_cfg(20, 40, 2, k, 1500, seed=0xD1DA0B00 + k)
    data = dl.synth_generate(cfg)
    obs = dl.DeviceObs(data["lat"], data["lon"], data["yb"], data["dep"], data["rinv"])
    p = dict(nanals=k, nrow=7, nlat=cfg.nlat, nlon=cfg.nlon, local_dist=1200.0,
             inflation_factor=1.05, form=form, gram=dl.GRAM_FP64)

    def engine(**over):
        eng = dl.Engine(dl.default_params(**dict(p, **over)), nobs_max=cfg.nobs)
        eng.set_grid(data["grid_lat"], data["grid_lon"])
        return eng

    eng = engine()
    xa, axa = torch.empty_like(data["xb"]), torch.empty_like(data["axb"])
    t = eng.autotune(obs, data["xb"], data["axb"], xa, axa)
    st = eng.stats()
    eng.close()
    print(f"  {t}", flush=True)
    assert st["status"] == 0 and st["max_sweeps_used"] <= 4      # steps of the iteration
    over = dict(chain_len=t["chain_len"], xcd_tiles=t["xcd_tiles"], bin_deg=t["bin_deg"])
    if t["bucketed"]:
        over["bucket_chain"] = t["bucket_chain"]
    eng = engine(**over)
    xa2, axa2 = torch.empty_like(xa), torch.empty_like(axa)
    eng.sweep(obs, data["xb"], data["axb"], xa2, axa2)
    st2 = eng.stats()
    eng.close()
    assert st2["status"] == 0 and st2["max_sweeps_used"] <= 4, st2
    assert st2["sweeps_sum"] == st["sweeps_sum"]
    assert torch.equal(xa, xa2) and torch.equal(axa, axa2)
