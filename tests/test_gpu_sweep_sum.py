"""GPU: the adjoint's summing sweeps (streaming bands, whole levels by
diagonal) against one sweep at a time, bit for bit, and the sweeps by
diagonal against the oracle."""
import os
import subprocess
import sys

import numpy as np
import pytest

from helpers import bits_equal, oracle_solve
from test_gpu_parity import random_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pd,h,w,n", [
    (1, 5, 3, 4), (2, 64, 65, 1), (1, 100, 90, 2), (2, 129, 200, 7), (1, 300, 261, 25),
    (4, 1023, 1024, 60)])
def test_summing_sweeps_equal_single_sweeps(pd, h, w, n, tmp_path):
    from sweep_sum_child import gradients
    print(f"sweep sum {pd}x{h}x{w} n={n}", flush=True)
    out = str(tmp_path / "one.npz")
    child = os.path.join(os.path.dirname(__file__), "sweep_sum_child.py")
    env = dict(os.environ, SIMPOIS_HIP_GS_FLOW="0", SIMPOIS_HIP_GS_CELLS="0")
    r = subprocess.run([sys.executable, child, *map(str, (pd, h, w, n)), out], env=env,
                       timeout=100)
    assert r.returncode == 0
    one = np.load(out)
    a, b = gradients(pd, h, w, n)
    assert bits_equal(a, one["g"]) and bits_equal(b, one["f"])


@pytest.mark.parametrize("pd,h,w,n", [
    (1, 1, 700, 3), (1, 700, 1, 3), (3, 2, 9, 2), (1, 128, 128, 10), (2, 127, 129, 64),
    (1, 96, 128, 56), (1, 96, 128, 57), (1, 20, 800, 1)])
@pytest.mark.parametrize("withf", [False, True])
@pytest.mark.parametrize("wild", [False, True])
def test_sweeps_by_diagonal_match_raster_sweeps(pd, h, w, n, withf, wild):
    import imscript_amd as m
    g, f = random_case(h + 3 * w + n, pd, h, w, 0.4, withf)
    if wild:
        at = np.flatnonzero(~np.isnan(g))[:3]
        g.reshape(-1)[at] = [np.inf, -np.inf, 3e37][:at.size]
    print(f"by diagonal {pd}x{h}x{w} n={n} f={withf} wild={wild}", flush=True)
    out = m.simpois(g, f, niter=n, scale=1, trace=False)
    assert bits_equal(out, oracle_solve(g, f, 0.25, n, 1, 0)[0])
