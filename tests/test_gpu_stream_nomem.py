"""GPU: where the streaming sweeps' scratch does not fit under the allocation
cap, the call runs in tiles, with the same bits, in the memory that tiles
need."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _image(pd, h, w):
    import torch
    rng = np.random.default_rng(h + w)
    x = rng.uniform(0, 255, (pd, h, w)).astype(np.float32)
    x[rng.random(x.shape) < 0.4] = np.nan
    return torch.from_numpy(x).cuda(), torch.from_numpy(
        rng.normal(0, 1, x.shape).astype(np.float32)).cuda()


@pytest.fixture
def cap():
    """Caps the library's memory at what it holds now plus some bytes."""
    import imscript_amd as m
    m.plan_cache_clear()
    old = m.set_alloc_cap(0)
    yield lambda more: m.set_alloc_cap(m.device_bytes() + more if more else 0)
    m.set_alloc_cap(old)
    m.plan_cache_clear()


# the sweeps alone; with solvers whose scratch is allocated on first use
@pytest.mark.parametrize("kw", [
    dict(niter=20, scale=1, cgit=0), dict(niter=30, scale=99, cgit=0),
    dict(niter=12, scale=99, cgit=-1, cg_fp32=1, cg_rel=1e-6, cg_mg=1, plane_stats=True),
    dict(niter=12, scale=2, cgit=5)], ids=["level", "pyramid", "multigrid", "fp64"])
def test_solve_runs_in_tiles(kw, cap, monkeypatch):
    import torch
    import imscript_amd as m
    g, f = _image(2, 500, 620)
    print("no room", kw, flush=True)
    kw = dict(dict(tstep=0.25), **kw)

    def solve():
        base = m.device_bytes()
        out = m.solve_batch_device([g], [f], **kw)[0][0]
        torch.cuda.synchronize()
        return out, m.device_bytes() - base

    want, streamed = solve()
    m.plan_cache_clear()
    monkeypatch.setenv("SIMPOIS_HIP_GS_SHAPE", "0")
    _, tiles = solve()
    m.plan_cache_clear()
    monkeypatch.delenv("SIMPOIS_HIP_GS_SHAPE")
    assert tiles < streamed
    cap(tiles)
    for _ in range(2):           # built, then from the cache
        got, held = solve()
        assert torch.equal(got.view(torch.int32), want.view(torch.int32))
    cap(0)
    m.plan_cache_clear()
    cap(tiles // 4)
    with pytest.raises(m.SimpoisError, match="status 2"):
        solve()


def test_amle_runs_in_tiles(cap, monkeypatch):
    import torch
    import imscript_amd as m
    x, _ = _image(1, 500, 620)
    small = torch.full((1, 8, 8), 3.0, device="cuda")

    def amle(n, capped=0, variant=None):
        m.amle(small, 4, 1)      # (one plan is kept: the small one, always alike)
        base = m.device_bytes()
        cap(capped)
        if variant:
            monkeypatch.setenv("SIMPOIS_HIP_AMLE_VARIANT", variant)
        try:
            out = m.amle(x, 4, n)
            torch.cuda.synchronize()
        finally:
            cap(0)
            monkeypatch.delenv("SIMPOIS_HIP_AMLE_VARIANT", raising=False)
        return out, m.device_bytes() - base

    print("no room, amle", flush=True)
    want, streamed = amle(30)
    _, tiles = amle(30, variant="6")
    assert tiles < streamed
    got, held = amle(30, tiles)
    assert held <= tiles
    assert torch.equal(got.view(torch.int32), want.view(torch.int32))
