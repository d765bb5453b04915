"""Child process of the GPU test of the finite-sweep gradient's error path:
with SIMPOIS_HIP_GS_FLOW_SPIN=0 (read when the library loads) a band or tile
whose predecessor is not there yet gives up at once, and the gradient must
report it.  Exit status 0 when it did."""
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))

import ctypes

import torch

from imscript_amd.autograd import sp_adjoint_image
from imscript_amd._lib import check, default_params, lib, sp_stats


def gradient(n, *shapes):
    """The gradient of n sweeps of some images in one call."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(n)
    arr, keep = (sp_adjoint_image * len(shapes))(), []
    for k, (pd, h, w) in enumerate(shapes):
        g = torch.rand(pd, h, w, device="cuda", generator=gen) * 255
        g[torch.rand(pd, h, w, device="cuda", generator=gen) < 0.5] = float("nan")
        t = [g, torch.ones_like(g), torch.empty_like(g), torch.empty_like(g)]
        arr[k] = sp_adjoint_image(w, h, pd, *[a.data_ptr() for a in t])
        keep.append(t)
    p = default_params(tstep=0.25, niter=n, scale=1, cgit=0, trace=0)
    check(lib.sp_adjoint_batch_device(
        len(shapes), ctypes.cast(arr, ctypes.c_void_p), ctypes.byref(p),
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream), ctypes.byref(sp_stats())))


BIG, SMALL = (2, 900, 1000), (1, 40, 50)    # with waits, without


def main():
    # (of several images, one whose plans the next image's replace)
    for n, shapes in ((64, [BIG]), (1, [BIG]), (10, [BIG, SMALL]), (10, [SMALL, BIG])):
        try:
            gradient(n, *shapes)
            print(f"gradient of {n} sweeps of {shapes}: no error", flush=True)
            return 1
        except Exception as e:
            print(f"gradient of {n} sweeps of {shapes}: {type(e).__name__}: {e}", flush=True)
            if "dependence wait" not in str(e):
                return 1
        gradient(n, SMALL)    # the word was cleared
    return 0


if __name__ == "__main__":
    sys.exit(main())
