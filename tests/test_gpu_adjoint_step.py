"""The finite-sweep gradient follows tstep from call to call: its kept plans
are told apart by the step."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _grad(h, w, tstep):
    import torch
    from imscript_amd.autograd import simpois_fill
    rng = np.random.default_rng(5)
    a = rng.uniform(0, 255, (h, w)).astype(np.float32)
    a[rng.random((h, w)) < 0.5] = np.nan
    g = torch.from_numpy(a).cuda().requires_grad_(True)
    f = torch.zeros(h, w, device="cuda", requires_grad=True)
    simpois_fill(g, f, niter=3, tstep=tstep).sum().backward()
    return f.grad.cpu().numpy()


def test_gradient_after_another_step():
    first = _grad(40, 56, 0.25)
    after = _grad(40, 56, 0.1)       # the same shape, another step
    _grad(24, 32, 0.1)               # another shape: the plans are built anew
    alone = _grad(40, 56, 0.1)
    assert np.array_equal(after.view(np.int32), alone.view(np.int32))
    assert not np.array_equal(first, alone)
