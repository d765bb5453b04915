"""GPU: heatd's short form for tiles of small finite values, and the limit
above which a tile takes the general one, against the oracle bit for bit."""
import numpy as np
import pytest

from helpers import bits_equal, oracle_heatd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [0.25, 1.0, -0.3, 4.0])
@pytest.mark.parametrize("top", [1e-38, 1.0, 1e34, 1e36, 3e37])
@pytest.mark.parametrize("shape", [(36, 52), (48, 64), (101, 157), (37, 400)])
def test_short_and_general_tiles_match_oracle(shape, top, t):
    import imscript_amd as sp
    rng = np.random.default_rng(shape[0] + shape[1])
    x = (rng.uniform(-1, 1, (2,) + shape) * top).astype(np.float32)
    x.reshape(-1)[rng.choice(x.size, 200, replace=False)] = np.float32(-0.0)
    x.reshape(-1)[rng.choice(x.size, 200, replace=False)] = np.float32(0.0)
    print(f"heatd short {shape} top={top} t={t}", flush=True)
    with np.errstate(all="ignore"):
        want = oracle_heatd(x, 13, np.float32(t), None)[0]
    assert bits_equal(sp.heatd(x, 13, np.float32(t)), want)
