"""Carries from one 64-word chunk of a scan's number to the next, on the CPU
(tests/shim/carry_test.cpp): no family has a centre of more than 64 words of
ones, so scans themselves do not reach them."""
import os
import subprocess

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_carries_cross_chunks():
    r = subprocess.run([os.path.join(REPO, "tests", "shim", "carry_test")], capture_output=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == b"ok", r.stdout
