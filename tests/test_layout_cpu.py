"""Runs tests/cpp/layout_test (built by __graft_entry__.build()): host checks of
sizes and index arithmetic that kernels rely on."""
import os
import subprocess

import pytest

BIN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "_build", "layout_test")


@pytest.mark.parametrize("part", ["level_slots", "stretch", "deal", "few"])
def test_layout(part):
    assert os.path.exists(BIN), "tests/cpp/_build/layout_test is not built (run __graft_entry__.build())"
    r = subprocess.run([BIN, part], capture_output=True, text=True, timeout=120)
    print(r.stdout[-3000:])
    assert r.returncode == 0 and "LAYOUT OK" in r.stdout
