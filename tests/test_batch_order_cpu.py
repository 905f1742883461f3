"""The order in which workgroups take a batch's tile runs (tests/cpp/test_batch_order.cpp)."""
import subprocess

from host_cpp import program


def test_runs_are_taken_longest_first():
    r = subprocess.run([program("test_batch_order")], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
