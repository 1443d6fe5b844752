"""The orbit M2L's host code (orbits of every parity class, operator fragments
of the three kernels) built with g++ under AddressSanitizer and
UndefinedBehaviorSanitizer (tests/asan/Makefile.orbits) and run."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

ASAN = os.path.join(ROOT, "tests", "asan")


@pytest.mark.skipif(shutil.which("g++") is None or shutil.which("make") is None, reason="needs g++ and make")
def test_orbit_host_code_under_asan_ubsan():
    b = subprocess.run(["make", "-s", "-C", ASAN, "-f", "Makefile.orbits"], capture_output=True, text=True, timeout=600)
    assert b.returncode == 0, b.stderr[-4000:]
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=1:abort_on_error=0", UBSAN_OPTIONS="print_stacktrace=1")
    r = subprocess.run([os.path.join(ASAN, "_build", "orbit_checks")], capture_output=True, text=True, timeout=600,
                       env=env)
    assert r.returncode == 0, (r.stdout + r.stderr)[-4000:]
    assert "0 failures" in r.stdout
