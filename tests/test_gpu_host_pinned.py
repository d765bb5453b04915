"""GPU: the host-array solve on pinned arrays (copied as they are) and on
pageable ones (through pinned chunks), in all pairs of input and output, at
addresses inside an allocation: the device solve's bits."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pin_in", [False, True])
@pytest.mark.parametrize("pin_out", [False, True])
@pytest.mark.parametrize("pin_data", [None, False, True])
def test_pinned_and_pageable_arrays(pin_in, pin_out, pin_data):
    import torch
    from imscript_amd import lib, solve_device
    from imscript_amd._lib import default_params, sp_stats
    pd, h, w = 1, 2049, 2051                     # above the smallest chunked copy
    rng = np.random.default_rng(3)
    g = rng.uniform(0, 255, (pd, h, w)).astype(np.float32)
    g[:, rng.random((h, w)) < 0.3] = np.nan
    f = None if pin_data is None else rng.normal(0, 1, g.shape).astype(np.float32)

    def host(a, pin):
        buf = torch.empty(g.size + 100, pin_memory=pin)[37:37 + g.size].view(g.shape)
        if a is not None:
            buf.copy_(torch.from_numpy(a))
        return buf

    a, o = host(g, pin_in), host(None, pin_out)
    d = None if f is None else host(f, pin_data)
    o.fill_(-1)
    p = default_params(niter=2, scale=2, cgit=0, trace=0, tstep=0.25)
    print(f"host arrays pinned {pin_in} {pin_out} {pin_data}", flush=True)
    rc = lib.sp_solve_host(o.data_ptr(), a.data_ptr(), None if d is None else d.data_ptr(),
                           w, h, pd, ctypes.byref(p), ctypes.byref(sp_stats()))
    assert rc == 0
    want, _ = solve_device(torch.from_numpy(g).cuda(),
                           None if f is None else torch.from_numpy(f).cuda(), niter=2, scale=2)
    assert np.array_equal(o.numpy().view(np.int32), want.cpu().numpy().view(np.int32))
