"""Reads where scratch memory cannot be had.  A child process loads a small library ahead of the solver's
that refuses allocations of a given size, on the device or page-locked, while told to, and compares
every read with the same read when nothing is refused."""
import os
import shutil
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

REFUSE = r"""
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>
static size_t device_size = 0, pinned_size = 0;
extern "C" void refuse(size_t device, size_t pinned) { device_size = device; pinned_size = pinned; }
extern "C" hipError_t hipMalloc(void **p, size_t n)
{
    static auto real = (hipError_t(*)(void **, size_t))dlsym(RTLD_NEXT, "hipMalloc");
    return n == device_size ? hipErrorOutOfMemory : real(p, n);
}
extern "C" hipError_t hipHostMalloc(void **p, size_t n, unsigned int flags)
{
    static auto real = (hipError_t(*)(void **, size_t, unsigned int))dlsym(RTLD_NEXT, "hipHostMalloc");
    return n == pinned_size ? hipErrorOutOfMemory : real(p, n, flags);
}
"""

CHILD = r"""
import ctypes, importlib.util, os, sys
refuse = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL).refuse
refuse.argtypes = [ctypes.c_size_t, ctypes.c_size_t]
refuse.restype = None
import numpy as np
d = os.path.join(sys.argv[2], "jianhui-lbm_amd")
spec = importlib.util.spec_from_file_location("jianhui_lbm_amd", os.path.join(d, "__init__.py"), submodule_search_locations=[d])
pkg = importlib.util.module_from_spec(spec)
sys.modules["jianhui_lbm_amd"] = pkg
spec.loader.exec_module(pkg)
STAGE, SLOT = 16 << 20, 2 << 20
solid = (np.random.default_rng(9).uniform(size=(31, 33, 35)) < 0.1).astype(np.int32)
for precision in ("fp64", "fp32"):
    print("[gpu] scratch limits", precision, flush=True)
    s = pkg.SinglePhase(solid, 0.1, (1e-4, -2e-4, 3e-4), precision=precision)
    s.init(1.0, (0.01, 0.0, 0.0))
    s.set_power_law(0.05, 0.9)
    s.step(14)
    refuse(STAGE, SLOT)
    nu = s.viscosity()
    try:
        s.state()
        raise SystemExit("state() has had its transfer buffer")
    except pkg.LBMError:
        pass
    refuse(0, SLOT)
    refused = list(s.state()) + [s.viscosity()] + list(s.dense())
    refuse(0, 0)
    had = list(s.state()) + [s.viscosity()] + list(s.dense())
    assert np.array_equal(nu, had[3])
    assert all(np.array_equal(a, b) for a, b in zip(refused, had))
    assert np.isfinite(nu).all() and (nu > 0).all()
print("reads agree")
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_reads_without_scratch_memory(tmp_path):
    src, lib = tmp_path / "refuse.cpp", tmp_path / "librefuse.so"
    src.write_text(REFUSE)
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", str(src), "-o", str(lib),
                    "-L/opt/rocm/lib", "-Wl,--no-as-needed", "-lamdhip64", "-ldl", "-Wl,-rpath,/opt/rocm/lib"], check=True, timeout=120)
    (tmp_path / "child.py").write_text(CHILD)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    proc = subprocess.run([sys.executable, str(tmp_path / "child.py"), str(lib), root], capture_output=True, text=True, timeout=100)
    assert proc.returncode == 0 and "reads agree" in proc.stdout, proc.stdout[-1000:] + proc.stderr[-3000:]
