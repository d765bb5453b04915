"""The gradient's gather by groups of four pixels: the bits of the form that
takes one pixel at a time (an odd offset of the planes selects it), and the
sum it stands for."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,w", [(2, 4), (2, 8), (9, 4), (5, 12), (33, 256), (17, 1028),
                                 (64, 260)])
def test_gather_by_groups(h, w):
    import torch
    from imscript_amd.autograd import _adjoint, _params
    rng = np.random.default_rng(h * 1000 + w)
    g = rng.uniform(0, 255, (h, w)).astype(np.float32)
    g[rng.random((h, w)) < 0.5] = np.nan
    g[0, 0] = 3.0
    v = rng.normal(0, 1, (h, w)).astype(np.float32)

    def place(a, off):
        buf = torch.zeros(h * w + 8, device="cuda")
        t = buf[off:off + h * w].view(1, h, w)
        t[0].copy_(torch.from_numpy(a))
        return t

    print(f"gather {h}x{w}", flush=True)
    res = []
    for off in (0, 1):
        gg, gf = place(v, off), place(v, off)
        _adjoint(place(g, off), place(v, off), gg, gf, _params(1e-6, 0, 1))
        torch.cuda.synchronize()
        res.append((gg[0].cpu().numpy(), gf[0].cpu().numpy()))
    for a, b in zip(*res):
        assert np.array_equal(a.view(np.int32), b.view(np.int32))
    # dL/dg = v + the adjoint solution (-dL/df) of the unknown neighbours,
    # summed in float32 in the order E, S, W, N
    gg, gf = res[0]
    hole = np.isnan(g)
    lam = np.where(hole, -gf, np.float32(0))
    p = np.pad(lam, 1)
    want = v.copy()
    for d in (p[1:-1, 2:], p[2:, 1:-1], p[1:-1, :-2], p[:-2, 1:-1]):
        want = want + d
    assert np.array_equal(gg, np.where(hole, np.float32(0), want))
