"""The host-array solve copies large planes in chunks by several threads:
the same bits as the device solve, whatever the remainder, and with calls
from several threads at once (the later ones find no free buffer)."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _planes(pd, h, w, seed):
    rng = np.random.default_rng(seed)
    g = rng.uniform(0, 255, (pd, h, w)).astype(np.float32)
    g[:, rng.random((h, w)) < 0.3] = np.nan
    return g, rng.normal(0, 1, (pd, h, w)).astype(np.float32)


def _device(g, f):
    import torch
    import imscript_amd as m
    df = None if f is None else torch.from_numpy(f).cuda()
    return m.solve_device(torch.from_numpy(g).cuda(), df, niter=2, scale=2)[0].cpu().numpy()


# around the smallest chunked copy (2^22 pixels), whole chunks, remainders
@pytest.mark.parametrize("pd,h,w,data", [(1, 2048, 2047, False), (1, 2048, 2048, True),
                                         (1, 2049, 2049, True), (3, 1537, 2051, False),
                                         (2, 2048, 4096, True)])
def test_host_solve_equals_device_solve(pd, h, w, data):
    import imscript_amd as m
    g, f = _planes(pd, h, w, h + w)
    f = f if data else None
    print(f"host copies {pd}x{h}x{w}", flush=True)
    got = np.asarray(m.simpois(g, f, niter=2, scale=2, trace=False)).reshape(g.shape)
    assert np.array_equal(got.view(np.int32), _device(g, f).view(np.int32))
    m.plan_cache_clear()      # gives the buffers back


def test_host_solves_from_several_threads():
    import imscript_amd as m
    jobs = [_planes(1, 2100 + 7 * k, 2200, k)[0] for k in range(4)]
    outs = [None] * 4

    def work(k):
        outs[k] = np.asarray(m.simpois(jobs[k], None, niter=2, scale=2, trace=False))

    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for g, o in zip(jobs, outs):
        assert np.array_equal(o.reshape(g.shape).view(np.int32), _device(g, None).view(np.int32))
