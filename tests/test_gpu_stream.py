"""GPU: the streaming Gauss-Seidel sweeps (radius 1) against the oracle's
raster sweeps, bit for bit, where the schedule has its edges: plane heights
around a band of 64 rows, the smallest plane it takes, sweeps around a
block, steps around a phase, several planes, values that need the general
update."""
import numpy as np
import pytest

from helpers import bits_equal, oracle_solve
from test_gpu_parity import random_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pd,h,w,n", [
    (1, 4, 4099, 33), (1, 4099, 4, 9), (1, 63, 301, 1), (1, 64, 300, 10), (2, 65, 299, 11),
    (1, 127, 257, 16), (1, 128, 136, 17), (1, 191, 129, 31), (3, 192, 128, 32),
    (1, 257, 200, 64), (1, 150, 140, 500), (2, 513, 511, 20)])
@pytest.mark.parametrize("withf", [False, True])
@pytest.mark.parametrize("kind", ["small", "step", "wild"])
def test_stream_sweeps_match_raster_sweeps(pd, h, w, n, withf, kind):
    import imscript_amd as m
    g, f = random_case(7 * h + w + n, pd, h, w, 0.4, withf)
    t = 0.25
    if kind == "step":       # a step above 1/4: values need not stay small
        t = 0.3
    if kind == "wild":       # neighbours that the update skips
        rng = np.random.default_rng(h + n)
        known = np.flatnonzero(~np.isnan(g))
        at = rng.choice(known, 12, replace=False)
        g.reshape(-1)[at] = np.array([np.inf, -np.inf, 3e37, -3e37], np.float32)[
            rng.integers(0, 4, 12)]
    print(f"stream {pd}x{h}x{w} n={n} f={withf} {kind}", flush=True)
    out = m.simpois(g, f, tstep=t, niter=n, scale=1, trace=False)
    ref, _ = oracle_solve(g, f, t, n, 1, 0)
    assert bits_equal(out, ref)
