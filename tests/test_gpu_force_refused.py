"""A count-mode force that is refused for want of memory does not count as a
call (tests/native/force_refused.cpp, built here with the host compiler)."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu


def test_refused_force_does_not_count(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ is not available")
    lib = os.path.join(ROOT, "lgca_amd")
    exe = str(tmp_path / "force_refused")
    r = subprocess.run([gxx, "-O2", "-std=c++17", "-rdynamic", "-I", os.path.join(ROOT, "include"),
                        os.path.join(ROOT, "tests", "native", "force_refused.cpp"), "-o", exe, "-L", lib, "-llgca_hip",
                        "-ldl", f"-Wl,-rpath,{lib}", "-Wl,--allow-shlib-undefined"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    print("[force] refused for want of memory", flush=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "REFUSED CALL PASSED", r.stdout + r.stderr
