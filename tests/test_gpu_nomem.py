"""Plans of the force phase and the adjoint on a device without room for the
finer cut of short lists: the coarse cut is taken, as where the caller's cap
rules the finer one out (allocations refused by the test program)."""
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EXE = os.path.join(ROOT, "hacc-coral_amd", "bin", "test_nomem")


def test_coarse_cut_where_memory_is_short():
    print("case plans without room for the finer cut", flush=True)
    r = subprocess.run([EXE], capture_output=True, text=True, timeout=100)
    print(r.stdout, r.stderr, flush=True)
    assert r.returncode == 0
