"""GPU: the streaming 4-neighbour AMLE sweeps against the oracle's raster
sweeps, bit for bit, at the schedule's edges: zeros of both signs (the order
of the scan shows in their sign), infinities, NaN made from them, several
planes, an initial image."""
import numpy as np
import pytest

from helpers import bits_equal, oracle_amle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pd,h,w,n", [
    (1, 4, 300, 21), (1, 301, 4, 7), (2, 63, 65, 10), (1, 64, 129, 20), (1, 65, 64, 33),
    (3, 130, 200, 16), (1, 257, 190, 100)])
@pytest.mark.parametrize("kind", ["plain", "zeros", "signed", "wild"])
@pytest.mark.parametrize("withinit", [False, True])
def test_stream_amle_matches_raster_sweeps(pd, h, w, n, kind, withinit):
    import imscript_amd as sp
    rng = np.random.default_rng(h * 7 + w + n)
    x = rng.uniform(0, 255, (pd, h, w)).astype(np.float32)
    if kind == "zeros":
        x = np.where(x < 120, np.float32(-0.0), np.float32(0.0))
        x[:, ::5, ::7] = 3
    if kind == "signed":
        x -= 127
    if kind == "wild":
        x.reshape(-1)[rng.choice(x.size, 9, replace=False)] = np.repeat(
            np.array([np.inf, -np.inf, 3e38], np.float32), 3)
    hole = rng.random((pd, h, w)) < 0.4
    hole[:, : h // 2, w // 3: 2 * w // 3] = True
    x[hole] = np.nan
    init = rng.uniform(-5, 5, x.shape).astype(np.float32) if withinit else None
    print(f"amle {pd}x{h}x{w} n={n} {kind} init={withinit}", flush=True)
    y = sp.amle(x, 4, n, init=init)
    for l in range(pd):
        with np.errstate(all="ignore"):
            want = oracle_amle(x[l], 4, n, None if init is None else init[l])
        assert bits_equal(y[l], want)
