"""A download refuses a corrupt resident order (the C++ program writes one into
the engine's device memory; see tests/cpp/order_check.cpp)."""
import os
import subprocess

import pytest

from helpers import announce

pytestmark = pytest.mark.gpu
EXE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "order_check")


def test_corrupt_resident_order_is_refused():
    assert os.path.exists(EXE), "tests/cpp/order_check is not built (run __graft_entry__.build())"
    announce("order check program")
    r = subprocess.run([EXE], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
