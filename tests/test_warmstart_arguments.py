"""Arguments that the warm-start entry points refuse, before any device call: in
a process of its own, so that a fault in the host code ends that alone."""
import os
import subprocess
import sys

import pytest

import qmin
from conftest import REPO

CALL = """
import ctypes, qmin
lib = qmin.library()
p = ctypes.c_void_p(4096)   # never read
d = [int(v) for v in %r]
rc = lib.qm_ws_conv_wgrad(p, 16, p, 16, 0, d[0], d[1], d[2], 1, p, ctypes.c_longlong(4096), p, None)
print(rc, lib.qm_last_error().decode())
"""


@pytest.mark.parametrize("dims", [(0, 4, 4), (4, 0, 4), (4, 4, 0), (-3, 4, 4)])
def test_weight_gradient_of_an_empty_lattice_is_refused(dims):
    if not os.path.exists(qmin.LIB_PATH):
        pytest.skip("libqmin.so not built (run __graft_entry__.build())")
    env = dict(os.environ, PYTHONPATH=os.path.join(REPO, "open-qmin_amd"))
    p = subprocess.run([sys.executable, "-c", CALL % (dims,)], env=env, capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stderr
    assert p.stdout.startswith("-1 bad weight-gradient argument"), p.stdout
