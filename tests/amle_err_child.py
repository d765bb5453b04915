"""Child process of the GPU test of AMLE's error path: with
SIMPOIS_HIP_GS_FLOW_SPIN=0 the sweeps of a large plane give up a dependence
wait, and the next call reports it also where it comes at once, with another
size that replaces the kept plan; a call on host arrays reports its own.  Exit
status 0 when they did."""
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))

import torch

import imscript_amd as m


def main():
    x = torch.rand(3, 1500, 1400, device="cuda")
    x[torch.rand_like(x) < 0.7] = float("nan")
    small = torch.rand(1, 20, 20, device="cuda")
    m.amle(small, 4, 1)
    torch.cuda.synchronize()
    m.amle(x, 4, 200)        # still running when the next call comes
    try:
        m.amle(small, 4, 1)
        print("no error", flush=True)
        return 1
    except Exception as e:
        print(f"{type(e).__name__}: {e}", flush=True)
        if "dependence wait" not in str(e):
            return 1
    m.amle(small, 4, 1)      # reported once
    torch.cuda.synchronize()
    try:                     # host arrays: the call is not asynchronous
        m.amle(x.cpu().numpy(), 4, 200)
        print("host arrays: no error", flush=True)
        return 1
    except Exception as e:
        print(f"host arrays: {type(e).__name__}: {e}", flush=True)
        if "dependence wait" not in str(e):
            return 1
    m.amle(small.cpu().numpy(), 4, 1)
    return 0


if __name__ == "__main__":
    sys.exit(main())
