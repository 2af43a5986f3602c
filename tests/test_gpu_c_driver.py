"""The C ABI driven from plain C (tests/cla_c_driver.c, built by systemds_amd/build.py): block construction from
C arrays, the four products, decompression and counts, each checked inside the driver against long-double
products of the dense matrix it built. This is the call pattern of a JNI shim (systemds_amd/jni/cla_jni.c),
with no Python or C++ between the caller and include/cla_hip.h."""
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu

ALLOC_DRIVER = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cla_alloc_driver")
DRIVER = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cla_c_driver")


@pytest.mark.parametrize("n_rows", [1, 4097, 300007])
def test_c_driver(n_rows):
    assert os.path.exists(DRIVER), "tests/cla_c_driver not built: run __graft_entry__.build()"
    r = subprocess.run([DRIVER, str(n_rows)], capture_output=True, text=True, timeout=170)
    print(r.stdout)
    print(r.stderr)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "C-DRIVER OK" in r.stdout and "FAIL" not in r.stdout


def test_allocation_failures_leave_no_state():
    """Host memory runs out at every place inside cla_mmchain in turn: an error code each time, and no trace of the chain's
    weights in the next X %*% v of the block; likewise inside cla_tsmm of two wide groups, and no trace of the failed call's
    sums in the next t(X) %*% X. A launch fails at every place inside a Y %*% X on decoded rows: no trace in a replay or the next call.
    A device allocation fails at every place inside a first product of a byte-code block: none of the digits' plans makes it fail.
    Profiling that was on before a failed call or prepare is on behind it."""
    assert os.path.exists(ALLOC_DRIVER), "tests/cla_alloc_driver not built: run __graft_entry__.build()"
    r = subprocess.run([ALLOC_DRIVER], capture_output=True, text=True, timeout=110)
    print(r.stdout)
    print(r.stderr)
    assert r.returncode == 0 and "ALLOC-DRIVER OK" in r.stdout, r.stdout + r.stderr
