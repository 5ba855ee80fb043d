"""A serving round that is refused its memory can be run again
(tests/cpp/serve_retry_test.cpp)."""
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu

BIN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "build", "serve_retry_test")


def test_round_refused_its_memory_runs_again():
    print("[case] serving round without memory", flush=True)
    res = subprocess.run([BIN], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=100)
    assert res.returncode == 0, res.stdout
