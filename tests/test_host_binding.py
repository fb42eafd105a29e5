"""The host-array binding in a program of numpy alone: it neither needs nor loads torch."""
import os
import subprocess
import sys

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                   "dida-thhpca-sc23_amd")

PROGRAM = """
import sys
sys.path.insert(0, {pkg!r})
if {absent}:
    sys.modules["torch"] = None          # import torch raises ImportError
import numpy as np
import dida_letkf as dl
batch, k = 20, 64                        # 81920 values
t = np.arange(batch * k * k, dtype=np.float64)
want = np.stack([t[b * k * k:(b + 1) * k * k].reshape(k, k).T for b in range(batch)])
got = dl._by_rows(t, batch, k)
assert got.flags.c_contiguous and np.array_equal(got, want)
assert sys.modules.get("torch") is None
import torch                             # present from here on
assert np.array_equal(dl._by_rows(t, batch, k), want)
"""


def _run(absent):
    src = PROGRAM.format(pkg=PKG, absent=absent)
    if absent:
        src = src[:src.index("import torch  ")]
    return subprocess.run([sys.executable, "-c", src], capture_output=True, text=True)


def test_batch_results_without_torch():
    r = _run(True)
    assert r.returncode == 0, r.stderr


def test_batch_results_do_not_load_torch():
    r = _run(False)
    assert r.returncode == 0, r.stderr
