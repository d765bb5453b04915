"""The finite-sweep gradient reports a dependence wait that gave up."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flow", ["stream", "tiles"])
def test_gradient_reports_a_wait_that_gave_up(flow):
    """The wait bound forced to 0 polls, so in a child process; every kernel
    still ends normally.  GS_SHAPE asks for the tiles."""
    env = dict(os.environ, SIMPOIS_HIP_GS_FLOW_SPIN="0")
    env.pop("SIMPOIS_HIP_GS_FLOW", None)
    if flow == "tiles":
        env["SIMPOIS_HIP_GS_SHAPE"] = "0"
    child = os.path.join(os.path.dirname(__file__), "adjoint_err_child.py")
    print("gradient error child", flow, flush=True)
    p = subprocess.run([sys.executable, child], env=env, capture_output=True, timeout=100)
    print(p.stdout.decode(), flush=True)
    assert p.returncode == 0, p.stdout.decode()[-2000:] + p.stderr.decode()[-2000:]
