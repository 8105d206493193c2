"""The order in which the resident LSTM time loops of a process's networks run on a device (myea_amd/csrc/myea_loop_order.h), with a stand-in for
the device (tests/cpp/loop_order_check.cpp, built by `python -m myea_amd.build`): turns of two networks, a network that joins while another is
about to launch, one that leaves while its loop runs."""
import os
import subprocess

import pytest

BIN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "loop_order_check")


@pytest.mark.parametrize("what", ["turns", "join", "leave-one", "leave-two", "leave-three"])
def test_no_two_loops_beside_each_other(what):
    out = subprocess.run([BIN, what], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout + out.stderr
