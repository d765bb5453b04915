"""GPU: 4-neighbour AMLE of the smallest planes runs in tiles (a launch per
wavefront of them, at most three), larger ones stream (three launches), with
the oracle's bits on both sides of the rule, zeros of both signs included."""
import numpy as np
import pytest

from helpers import bits_equal, oracle_amle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pd,h,w,n,launches", [
    (1, 16, 16, 16, 1), (1, 16, 16, 17, 3), (1, 32, 32, 16, 3), (1, 33, 32, 16, 3),
    (1, 63, 63, 2, 3), (1, 64, 64, 2, 3), (1, 62, 62, 3, 3), (1, 16, 62, 3, 2),
    (3, 90, 12, 16, 2), (3, 33, 65, 16, 3), (2, 4, 4, 1, 1)])
def test_both_sides_of_the_rule(pd, h, w, n, launches):
    import torch
    import imscript_amd as m
    rng = np.random.default_rng(h * 7 + w + n)
    x = np.where(rng.random((pd, h, w)) < 0.5, np.float32(-0.0), np.float32(0.0))
    x[:, ::5, ::3] = rng.uniform(-9, 9, x[:, ::5, ::3].shape)
    x[rng.random(x.shape) < 0.4] = np.nan
    x = x.astype(np.float32)
    print(f"amle small {pd}x{h}x{w} n={n}", flush=True)
    m.profile(True)
    y = m.amle(torch.from_numpy(x).cuda(), 4, n)
    torch.cuda.synchronize()
    assert m.profile_read("amle_tile")[1] == launches
    m.profile(False)
    for l in range(pd):
        assert bits_equal(y[l].cpu().numpy(), oracle_amle(x[l], 4, n, None))
