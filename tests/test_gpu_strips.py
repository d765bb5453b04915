"""Level 0 of the multigrid by one wave per tile: the same bits as by
work-groups.  A plane alone has too few pixels for the strips; in a batch
with a large plane all planes take them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# tile edges (108 x 44) and remainders, narrow and short planes
EVEN = [(2, 2), (3, 4), (5, 128), (43, 106), (44, 108), (45, 110), (46, 2), (88, 216),
        (89, 218), (133, 330), (64, 1030)]
ODD = [(2, 3), (3, 5), (44, 107), (45, 109), (47, 129), (90, 217), (301, 401), (64, 33)]


def _plane(h, w, seed):
    rng = np.random.default_rng([h, w, seed])
    g = rng.uniform(0, 255, (h, w)).astype(np.float32)
    g[rng.random((h, w)) < 0.6] = np.nan
    if h * w > 2000:
        g[h // 4:h // 2, w // 4:w // 2] = np.nan
        g[h // 2:, :w // 4] = 7.0
    g[0, 0] = 5.0
    return g, rng.normal(0, 0.5, (h, w)).astype(np.float32)


@pytest.mark.parametrize("sizes", [EVEN, ODD + EVEN[::3]], ids=["even", "odd"])
def test_strips_keep_the_bits_of_the_tiles(sizes):
    import torch
    import imscript_amd as m
    planes = [_plane(h, w, 1) for h, w in sizes]
    bad = _plane(70, 118, 2)
    bad[1][np.isnan(bad[0])] = np.inf      # no finite solution
    planes.append(bad)
    big = _plane(2300, 2400, 3)
    dev = [(torch.from_numpy(g).cuda(), torch.from_numpy(f).cuda()) for g, f in planes + [big]]
    kw = dict(niter=0, scale=1, cgit=-1, cg_fp32=1, cg_rel=1e-6, cg_mg=1, plane_stats=True)
    print("strips", sizes, flush=True)
    outs, _, ps = m.solve_batch_device([g for g, _ in dev], [f for _, f in dev], **kw)
    for k in range(len(planes)):
        alone, _, pa = m.solve_batch_device([dev[k][0]], [dev[k][1]], **kw)
        assert pa[0].status == ps[k].status, planes[k][0].shape
        assert pa[0].cg_iters == ps[k].cg_iters, planes[k][0].shape
        if k < len(sizes):
            assert ps[k].status == m.PLANE_CONVERGED
            assert torch.equal(alone[0].view(torch.int32), outs[k].view(torch.int32)), \
                planes[k][0].shape
    assert ps[len(sizes)].status == m.PLANE_NONFINITE
    assert ps[-1].status == m.PLANE_CONVERGED and ps[-1].rel_residual <= 1e-5
    got, want = outs[-1].cpu().numpy(), big[0]
    assert np.array_equal(got[~np.isnan(want)], want[~np.isnan(want)])


@pytest.mark.parametrize("h,w", [(2300, 2400), (2301, 2399)])
def test_strips_solve_the_system(h, w):
    """The fill by strips against the FP64 residual of the system."""
    import torch
    import imscript_amd as m
    g, f = _plane(h, w, 4)
    dg, df = torch.from_numpy(g).cuda(), torch.from_numpy(f).cuda()
    print(f"strips {h}x{w}", flush=True)
    u, st = m.solve_device(dg, df, niter=0, scale=1, cgit=-1, cg_fp32=1, cg_rel=1e-6, cg_mg=1)
    # the residual of an FP32 image: the stop plus its rounding, as elsewhere
    assert m.residual_device(u, dg, df)[0] <= 1e-5
