"""GPU: SIMPOIS_HIP_AMLE_VARIANT is read at each call, also where the kept
plan has the same size and tile shape: set, the sweeps run in tiles (one
launch); unset or empty, they stream (three)."""
import numpy as np
import pytest

from helpers import bits_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pd,variant", [(1, "6"), (3, "0")])
def test_variant_is_read_at_each_call(pd, variant, monkeypatch):
    import torch
    import imscript_amd as m
    rng = np.random.default_rng(pd)
    x = rng.uniform(0, 255, (pd, 300, 310)).astype(np.float32)
    x[rng.random(x.shape) < 0.4] = np.nan
    x = torch.from_numpy(x).cuda()
    out = torch.empty_like(x)
    print(f"amle variant pd={pd}", flush=True)

    def launches(value):
        if value is None:
            monkeypatch.delenv("SIMPOIS_HIP_AMLE_VARIANT", raising=False)
        else:
            monkeypatch.setenv("SIMPOIS_HIP_AMLE_VARIANT", value)
        m.profile(True)
        m.amle(x, 4, 16, out=out)
        torch.cuda.synchronize()
        n = m.profile_read("amle_tile")[1]
        m.profile(False)
        return n, out.cpu().numpy()

    runs = [launches(v) for v in (None, variant, None, "", variant, "")]
    assert [n for n, _ in runs] == [3, 1, 3, 3, 1, 3]
    assert all(bits_equal(o, runs[0][1]) for _, o in runs)
