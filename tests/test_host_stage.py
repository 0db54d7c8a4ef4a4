"""The staging of blocking reads on the CPU, under sanitizers."""
import os
import subprocess

import pytest

from tests.native import build_native


@pytest.mark.parametrize("sanitize", ["asan", "tsan"])
def test_blocking_reads(sanitize):
    r = subprocess.run([build_native.build("stage_test", sanitize)], capture_output=True, text=True, timeout=300,
                       env=dict(os.environ, ASAN_OPTIONS="detect_leaks=1", TSAN_OPTIONS="halt_on_error=1"))
    assert r.returncode == 0 and "all checks passed" in r.stdout, r.stderr[-3000:]
