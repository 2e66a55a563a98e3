"""How a team's blocks agree on their next instance (cuopo_amd/csrc/opo_handoff.h), on the CPU under every
interleaving of their shared-memory operations: one to four blocks, one and two teams, one to three slices, finished
instances at every place in the queue.  No block misses its word, all blocks of a team run the same instances, and
every running instance is run exactly once."""
import os
import shutil
import subprocess

import pytest

from tests.conftest import ROOT

NATIVE = os.path.join(ROOT, "tests", "native")


def test_hand_off_under_every_interleaving():
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    out = os.path.join(NATIVE, "_build", "handoff_check")
    r = subprocess.run(["make", "-C", NATIVE, out], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([out], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
    assert r.stdout.count(": ok") == 11
