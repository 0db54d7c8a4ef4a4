"""The rules that select launches, without a device (CPU only)."""
import subprocess

from tests.native import build_native


def test_launch_rules():
    r = subprocess.run([build_native.build_with_library("rules_test")], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "all checks passed" in r.stdout, r.stderr
