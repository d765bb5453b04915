"""AMLE reports a dependence wait that gave up also where the next call, of
another size, replaces the plan."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu


def test_a_replaced_plan_reports_its_wait():
    env = dict(os.environ, SIMPOIS_HIP_GS_FLOW_SPIN="0")
    env.pop("SIMPOIS_HIP_GS_FLOW", None)
    child = os.path.join(os.path.dirname(__file__), "amle_err_child.py")
    print("amle error child", flush=True)
    p = subprocess.run([sys.executable, child], env=env, capture_output=True, timeout=100)
    print(p.stdout.decode(), flush=True)
    assert p.returncode == 0, p.stdout.decode()[-2000:] + p.stderr.decode()[-2000:]
