"""Error paths of the ensemble solve, on the CPU: tests/cpp/ensemble_errors_check links the
library's host code against a HIP runtime that fails one call after the other."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
BIN = os.path.join(HERE, "cpp", "ensemble_errors_check")


def test_a_failing_call_leaves_no_work_unordered():
    assert os.path.exists(BIN), "run __graft_entry__.build() (it builds tests/cpp)"
    p = subprocess.run([BIN], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stdout[-3000:] + p.stderr[-2000:]
    tried = int(p.stdout.split()[-6])
    assert tried > 500 and p.stdout.rstrip().endswith("0 violations")
