"""The benchmark's roofline record names the kernel that each form runs and counts the
update where that kernel does it."""
import types

import pytest


@pytest.mark.parametrize("head,k,chain_len,f32,kernel,fused", [
    ("plain_fp64", 64, 0, False, "k_letkf_iter ", True),
    ("plain_fp64", 64, 0, True, "k_letkf_iter ", False),
    ("batched_fp64", 20, 8, False, "k_letkf_iter ", True),
    ("batched_fp64", 128, 0, False, "k_letkf_iter128 ", False),
    ("plain_fp64", 65, 0, False, "k_letkf_iter128 ", False),
    ("batched_fp64", 128, 8, False, "k_letkf_chain_f64 ", False),
    ("batched_bf16x3", 64, 8, False, "k_letkf_wave ", True),
    ("batched_fp16x3", 128, 0, True, "k_letkf_chain_f64 ", False),
])
def test_roofline_names_the_kernel(head, k, chain_len, f32, kernel, fused):
    import bench
    cfg = types.SimpleNamespace(k=k, nz=4, nlat=10, nlon=20)
    r = bench.kernel_roofline(cfg, {"nobsl_sum": 5000}, head, 1.0, 2, 1.0, None,
                              chain_len=chain_len, state_f32=f32)
    assert r["kernel"].startswith(kernel)
    n, ncol = 13, 200
    assert r["algorithmic_bytes"]["update"] == (ncol * (2.0 * k * n * 8 + 2.0 * n * 8)
                                                if fused else 0.0)
    row = 8.0 if head.endswith("fp64") else 4.0
    assert r["algorithmic_bytes"]["obs_gathered"] == 5000 * (row * k + 24.0)
    gram = 2.0 * k * k * 5000
    assert r["half_flops"] == (0.0 if head.endswith("fp64") else 3.0 * gram)
