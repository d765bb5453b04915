"""GPU: streaming sweeps of planes of several sizes in one launch, whose
layouts share one allocation, against the oracle's raster sweeps bit for bit."""
import numpy as np
import pytest

from helpers import bits_equal, oracle_solve
from test_gpu_parity import random_case

pytestmark = pytest.mark.gpu

SIZES = [(150, 140), (4, 4200), (257, 64), (129, 400), (4200, 4), (64, 300), (200, 131)]


@pytest.mark.parametrize("n", [10, 33, 150])
@pytest.mark.parametrize("withf", [False, True])
def test_planes_of_several_sizes(n, withf):
    import torch
    import imscript_amd as m
    cases = [random_case(31 * h + w + n, 1, h, w, 0.4, withf) for h, w in SIZES]
    gs = [torch.from_numpy(g).cuda() for g, _ in cases]
    fs = [torch.from_numpy(f).cuda() for _, f in cases] if withf else None
    print(f"stream batch n={n} f={withf}", flush=True)
    outs, _ = m.solve_batch_device(gs, fs, niter=n, tstep=0.25, scale=1, cgit=0)
    for (g, f), o in zip(cases, outs):
        want, _ = oracle_solve(g, f, 0.25, n, 1, 0)
        assert bits_equal(o.cpu().numpy().reshape(want.shape), want), g.shape
