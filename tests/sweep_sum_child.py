"""Child process of the GPU test of the finite-sweep adjoint: gradients of
one size and sweep count from seeded data, saved to argv[5].  The environment
that the parent sets (SIMPOIS_HIP_GS_FLOW, SIMPOIS_HIP_GS_CELLS, read when the
library loads) chooses between the summing sweeps and one sweep at a time."""
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))

import numpy as np
import torch

from imscript_amd.autograd import simpois_fill


def gradients(pd, h, w, n):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(pd + h + w + n)
    g = torch.rand(pd, h, w, device="cuda", generator=gen) * 255
    hole = torch.rand(pd, h, w, device="cuda", generator=gen) < 0.3
    hole[:, h // 4: h // 2, w // 3: w // 2] = True
    g[hole] = float("nan")
    f = torch.randn(pd, h, w, device="cuda", generator=gen)
    v = torch.randn(pd, h, w, device="cuda", generator=gen)
    g.requires_grad_(True)
    f.requires_grad_(True)
    simpois_fill(g, f, niter=n).backward(v)
    return g.grad.cpu().numpy(), f.grad.cpu().numpy()


if __name__ == "__main__":
    a, b = gradients(*map(int, sys.argv[1:5]))
    np.savez(sys.argv[5], g=a, f=b)
