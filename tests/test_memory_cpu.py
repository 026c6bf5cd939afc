"""Runs tests/cpp/memory_test (built by __graft_entry__.build()): the library's
device memory tables over a stub of the HIP runtime's memory calls."""
import os
import subprocess

import pytest

BIN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "_build", "memory_test")


@pytest.mark.parametrize("part", ["results", "captures", "host_words", "server", "bounds", "threads"])
def test_memory_tables(part):
    assert os.path.exists(BIN), "tests/cpp/_build/memory_test is not built (run __graft_entry__.build())"
    r = subprocess.run([BIN, part], capture_output=True, text=True, timeout=60)
    print(r.stdout[-3000:])
    assert r.returncode == 0 and "MEMORY OK" in r.stdout
