"""The host-array cores' packing (ragged obs counts, none, and counts past
max_obs; blocks below and above the small-call limit and over several staging
slots; REAL(8) and REAL(4)): bit-equal to the device-array core on the same
values, also from several threads at once."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _inputs(k, batch, max_obs, seed):
    rng = np.random.default_rng(seed)
    nb = rng.integers(0, max_obs + 1, batch).astype(np.int32)
    nb[rng.integers(0, batch, max(1, batch // 5))] = 0
    nb[0] = max_obs + 3  # clamped to max_obs
    hx = rng.normal(size=(batch, max_obs, k))
    hx -= hx.mean(axis=2, keepdims=True)
    return (nb, hx, rng.uniform(0.5, 2.0, (batch, max_obs)).astype(np.float32),
            rng.normal(size=(batch, max_obs)), rng.uniform(0.0, 1.0, (batch, max_obs)))


def _device(dl, torch, args):
    nb, hx, ri, dep, rl = (torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in args)
    batch, _, k = hx.shape
    trans = torch.empty(batch, k, k, dtype=torch.float64, device="cuda")
    wbar = torch.empty(batch, k, dtype=torch.float64, device="cuda")
    dl.core_batch_dev(nb, hx, ri, dep, rl, trans, wbar, 1.1)
    torch.cuda.synchronize()
    return trans.cpu().numpy().transpose(0, 2, 1), wbar.cpu().numpy()


# (7, 900, 130): 6.6 MB of obs, two slots' worth; (64, 300, 150): 23 MB in, 9.8
# MB out; (100, 9, 40): the workgroup kernel (64 < k <= 128)
@pytest.mark.parametrize("k,batch,max_obs", [(20, 1, 245), (5, 3, 0), (33, 40, 9), (7, 900, 130),
                                             (64, 300, 150), (100, 9, 40)])
def test_host_core_equals_device_core(cuda, dl, k, batch, max_obs):
    torch = cuda
    print(f"host core k={k} batch={batch} max_obs={max_obs}", flush=True)
    args = _inputs(k, batch, max_obs, k + batch)
    t0, w0 = _device(dl, torch, args)
    t1, w1 = dl.letkf_core_batch(*args, 1.1)
    assert np.array_equal(t1, t0) and np.array_equal(w1, w0)
    nb, hx, ri, dep, rl = args
    f32 = [x.astype(np.float32) for x in (hx, dep, rl)]
    wide = (nb, f32[0].astype(np.float64), ri, f32[1].astype(np.float64),
            f32[2].astype(np.float64))
    t0, w0 = _device(dl, torch, wide)
    t1, w1 = dl.letkf_core_batch_r4(nb, f32[0], ri, f32[1], f32[2], 1.1)
    assert np.array_equal(t1, t0.astype(np.float32)) and np.array_equal(w1, w0.astype(np.float32))


def test_host_core_from_threads(cuda, dl):
    torch = cuda
    print("host core from threads", flush=True)
    cases = [_inputs(k, b, p, 7 + k) for k, b, p in ((64, 120, 150), (20, 1, 60), (16, 500, 90))]
    want = [_device(dl, torch, a) for a in cases]
    bad = []

    def work(i):
        for _ in range(4):
            t, w = dl.letkf_core_batch(*cases[i], 1.1)
            if not (np.array_equal(t, want[i][0]) and np.array_equal(w, want[i][1])):
                bad.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(cases))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
