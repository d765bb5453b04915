"""GPU: the memory of the finite-sweep gradient.  The values that the summing
sweeps keep are at most 1 GiB whatever the planes' shape and the sweeps' count
(longer runs go in groups), and where they do not fit the gradient runs one
sweep at a time; the bits stay those of one sweep at a time."""
import os
import subprocess
import sys

import numpy as np
import pytest

from helpers import bits_equal

pytestmark = pytest.mark.gpu

SHAPES = [(16, 64, 64, 1600), (1, 20000, 4, 300), (8, 512, 512, 150), (2, 40, 3000, 700)]


def _one_at_a_time(shape, out):
    child = os.path.join(os.path.dirname(__file__), "sweep_sum_child.py")
    env = dict(os.environ, SIMPOIS_HIP_GS_FLOW="0", SIMPOIS_HIP_GS_CELLS="0")
    r = subprocess.run([sys.executable, child, *map(str, shape), out], env=env, timeout=110)
    assert r.returncode == 0
    return np.load(out)


@pytest.mark.parametrize("shape", SHAPES)
def test_history_is_bounded(shape, tmp_path):
    import torch
    import imscript_amd as m
    from sweep_sum_child import gradients
    print("gradient memory", shape, flush=True)
    one = _one_at_a_time(shape, str(tmp_path / "one.npz"))
    gradients(1, 8, 8, 1)              # (the plans of the last shape are kept)
    m.plan_cache_clear()
    base = m.device_bytes()
    a, b = gradients(*shape)
    m.plan_cache_clear()
    held = m.device_bytes() - base
    assert bits_equal(a, one["g"]) and bits_equal(b, one["f"])
    # 1 GiB of values, and the layouts of three plans and pyramids
    assert held < (1 << 30) + (1 << 29), held
    torch.cuda.synchronize()


@pytest.mark.parametrize("shape", [(2, 300, 401, 12)])
def test_one_sweep_at_a_time_where_memory_is_short(shape):
    import imscript_amd as m
    from sweep_sum_child import gradients
    print("gradient short of memory", shape, flush=True)
    gradients(1, 8, 8, 1)
    m.plan_cache_clear()
    base = m.device_bytes()
    want = gradients(*shape)
    m.plan_cache_clear()
    held = m.device_bytes() - base
    gradients(1, 8, 8, 1)
    m.plan_cache_clear()
    # (the forward fill, in tiles if need be, comes and goes under the same cap)
    old = m.set_alloc_cap(m.device_bytes() + held - 1)
    try:
        got = gradients(*shape)
    finally:
        m.set_alloc_cap(old)
        m.plan_cache_clear()
    assert m.device_bytes() - base < held
    assert all(bits_equal(x, y) for x, y in zip(got, want))
