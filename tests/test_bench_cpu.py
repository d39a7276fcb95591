"""bench.py's CPU sample of the ensemble without the reference's build: it fails at once, with the library's name."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_ensemble_sample_without_the_reference():
    if os.path.exists(os.path.join(ROOT, "oracle", "_ref", "libfenice_ref.so")):
        pytest.skip("the reference build is present")
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--cpu-worker", "--n", "2", "--cpu-budget", "1", "--workload", "ensemble"],
                       capture_output=True, text=True, timeout=60)
    assert r.returncode != 0 and "libfenice_ref.so" in r.stderr
