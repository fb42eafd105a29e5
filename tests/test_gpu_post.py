"""dida_letkf_post over member counts at the edges of its lane groups, odd and
even (8- and 16-byte accesses), from arrays at 16-byte and at odd 8-byte
addresses, and in place, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = 1e-13  # sums of at most 260 squares in another order, and one blend


@pytest.mark.parametrize("k", [1, 2, 3, 4, 7, 8, 9, 16, 17, 31, 32, 33, 64, 65, 127, 128, 129, 260])
@pytest.mark.parametrize("shift", [0, 1])
def test_post_member_counts(cuda, dl, oracle, k, shift):
    torch = cuda
    nlat, nlon, nrow = 5, 3, 7
    rng = np.random.default_rng(1000 * shift + k)
    ncol = nlat * nlon
    lat = np.linspace(-80.0, 80.0, nlat).astype(np.float32)
    xb, xa = rng.normal(size=(ncol, nrow, k)), rng.normal(size=(ncol, nrow, k))
    axb, axa = rng.normal(size=(ncol, nrow)), rng.normal(size=(ncol, nrow))

    def dev(x):
        t = torch.empty(x.size + shift, dtype=torch.float64, device="cuda")[shift:]
        t.copy_(torch.from_numpy(x.reshape(-1)))
        return t

    print(f"post k={k} shift={shift}", flush=True)
    d = [dev(x) for x in (xb, axb, xa, axa)]
    out = dev(np.zeros_like(xb))
    sb, sa = dev(np.zeros_like(axb)), dev(np.zeros_like(axb))
    glat = torch.from_numpy(lat).cuda()
    ref, ref_b, ref_a = oracle.post(0, lat, nlat, nlon, 45.0, 0.6, 0.4, 0.0, xb, axb, xa, axa)
    for target in (out, d[2]):  # a buffer of its own, then in place of Xa'
        dl.post(k, nrow, nlat, nlon, glat, 45.0, 0.6, 0.4, *d, target, sb, sa)
        torch.cuda.synchronize()
        for got, want in ((target, ref), (sb, ref_b), (sa, ref_a)):
            want = np.asarray(want).reshape(-1)
            err = np.abs(got.cpu().numpy() - want).max()
            assert err <= TOL * max(1.0, np.abs(want).max()), (k, shift, err)
