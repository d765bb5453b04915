"""GPU: a choice of the autotuner serves calls of the same code only: with and
without a data term, with steps up to and above 1/4 (the streaming sweeps'
finite tests), with and without the streaming sweeps."""
import numpy as np
import pytest

from helpers import bits_equal, oracle_solve
from test_gpu_parity import random_case

pytestmark = pytest.mark.gpu


def test_choices_are_told_apart(monkeypatch):
    import torch
    import imscript_amd as m
    h, w, n = 237, 331, 23
    g, f = random_case(5, 1, h, w, 0.4, True)
    dg, df = torch.from_numpy(g).cuda(), torch.from_numpy(f).cuda()

    def lines():
        return [ln for ln in m.autotune_report().splitlines()
                if f"T={n} planes=1 px={h * w} " in ln]

    assert not lines()
    print("autotune keys", flush=True)
    seen = 0
    for shape in (None, "0"):
        if shape:
            monkeypatch.setenv("SIMPOIS_HIP_GS_SHAPE", shape)
        for data in (None, df):
            for t in (0.25, 0.3):
                m.plan_cache_clear()
                out, _ = m.solve_device(dg, data, tstep=t, niter=n, scale=1, autotune=1)
                torch.cuda.synchronize()
                want, _ = oracle_solve(g, None if data is None else f, t, n, 1, 0)
                assert bits_equal(out.cpu().numpy(), want)
                # (the tiles have one code for all of them)
                seen += 1 if shape is None or seen == 4 else 0
                assert len(lines()) == seen
    assert sum("stream:" in ln for ln in lines()) == 4
