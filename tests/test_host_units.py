"""Units of the library's host code on their own (tests/sanitize/sanitize_<unit>.cpp), built with
AddressSanitizer and UndefinedBehaviorSanitizer.  CPU only: no device code is built or run."""
import os
import shutil
import subprocess

import pytest

SAN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "sanitize")

pytestmark = pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include"),
                                reason="needs g++ and the ROCm headers")


def _run(unit, *args):
    target = f"_build/sanitize_{unit}"
    subprocess.run(["make", "-s", "-C", SAN, target], check=True, timeout=600)
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=1:abort_on_error=0:verify_asan_link_order=0",
               UBSAN_OPTIONS="print_stacktrace=1")
    proc = subprocess.run([os.path.join(SAN, target), *args], env=env, capture_output=True, text=True, timeout=600)
    assert proc.returncode == 0, proc.stdout[-2000:] + proc.stderr[-4000:]
    return proc.stdout


def test_tuning_cache():
    assert "checks passed" in _run("tune")


@pytest.mark.parametrize("check", ["refused", "failing", "at_once"])
def test_state_reads(check):
    assert "checks passed" in _run("readback", check)
