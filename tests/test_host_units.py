"""Units of the library's host code on their own (tests/sanitize/sanitize_<unit>.cpp), built with
AddressSanitizer and UndefinedBehaviorSanitizer.  CPU only: no device code is built or run."""
import os
import shutil
import subprocess

import numpy as np
import pytest

import test_gpu_link_forms as forms

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


def test_packed_links():
    assert "checks passed" in _run("links", "pack")


def _width(tmp_path, solid):
    solid.astype(np.int32).tofile(tmp_path / "solid.bin")
    return int(_run("links", "width", *[str(n) for n in solid.shape], str(tmp_path / "solid.bin")).split()[0])


@pytest.mark.parametrize("box", range(3))
def test_boxes_of_the_oracle_comparison_lie_on_both_sides_of_the_width_rule(tmp_path, box):
    """The boxes that test_gpu_link_forms compares with the oracle, drawn as it draws them."""
    boxes = next(m for m in forms.test_large_boxes_match_the_oracle.pytestmark if m.name == "parametrize").args[1]
    shape, porosity = boxes[box]
    solid = np.random.default_rng(11).uniform(size=shape) > porosity
    assert _width(tmp_path, solid) == [8, 8, 16][box]


def test_box_of_faces_and_power_law_has_eight_bit_ranks(tmp_path):
    assert _width(tmp_path, np.random.default_rng(13).uniform(size=(40, 170, 160)) > 0.97) == 8
