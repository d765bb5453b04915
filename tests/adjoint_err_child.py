"""Child process of the GPU test of the finite-sweep gradient's error path:
with SIMPOIS_HIP_GS_FLOW_SPIN=0 (read when the library loads) a band or tile
whose predecessor is not there yet gives up at once, and the gradient must
report it.  Exit status 0 when it did."""
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))

import torch

from imscript_amd.autograd import _adjoint
from imscript_amd._lib import default_params


def gradient(pd, h, w, n):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(h)
    g = torch.rand(pd, h, w, device="cuda", generator=gen) * 255
    g[torch.rand(pd, h, w, device="cuda", generator=gen) < 0.5] = float("nan")
    v = torch.ones_like(g)
    gg, gf = torch.empty_like(g), torch.empty_like(g)
    _adjoint(g, v, gg, gf, default_params(tstep=0.25, niter=n, scale=1, cgit=0, trace=0))


def main():
    for n in (64, 1):
        try:
            gradient(2, 900, 1000, n)
            print(f"gradient of {n} sweeps: no error", flush=True)
            return 1
        except Exception as e:
            print(f"gradient of {n} sweeps: {type(e).__name__}: {e}", flush=True)
            if "dependence wait" not in str(e):
                return 1
    gradient(1, 40, 50, 4)    # a plane without waits: the word was cleared
    return 0


if __name__ == "__main__":
    sys.exit(main())
