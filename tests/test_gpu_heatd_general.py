"""GPU: heatd's general tiles (values that are not finite or too large for the
short form) where lane shifts could show: infinities and NaN at the columns
where the waves' tiles meet and at the image border, against the oracle bit for
bit."""
import numpy as np
import pytest

from helpers import bits_equal, oracle_heatd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(36, 52), (48, 64), (90, 105), (101, 157), (37, 400)])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan, 3e38])
@pytest.mark.parametrize("n", [1, 6, 13])
def test_bad_values_at_tile_borders(shape, bad, n):
    import imscript_amd as sp
    rng = np.random.default_rng(shape[0] * 7 + shape[1] + n)
    x = rng.uniform(-100, 100, (2,) + shape).astype(np.float32)
    h, w = shape
    cols = sorted({c for c in (0, 1, 51, 52, 57, 58, 63, 64, 103, 104, w - 2, w - 1) if c < w})
    for k, c in enumerate(cols):          # 52 columns a tile of 6 steps
        x[0, (5 * k + 3) % h, c] = bad
    x[1, 0, 0] = x[1, h - 1, w - 1] = bad
    print(f"heatd general {shape} {bad} n={n}", flush=True)
    with np.errstate(all="ignore"):
        want = oracle_heatd(x, n, np.float32(0.25), None)[0]
    assert bits_equal(sp.heatd(x, n, np.float32(0.25)), want)
