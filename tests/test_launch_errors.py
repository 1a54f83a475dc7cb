"""A launch that fails comes back as an error from the transform's launchers: a
program linked to the library whose hipLaunchKernel fails on demand (CPU only,
no kernel runs)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(shutil.which(HIPCC) is None, reason="no hipcc")
def test_failed_launch_is_reported(tmp_path):
    from dida_letkf import _build
    if not os.path.exists(_build.LIB_PATH):
        _build.build()
    exe = tmp_path / "launch_check"
    r = subprocess.run([HIPCC, "-std=c++17", "--offload-arch=" + _build.ARCH, "-I", _build.CSRC,
                        "-o", str(exe), os.path.join(ROOT, "tests", "native", "launch_check.cpp"),
                        "-rdynamic", "-L" + _build.LIB_DIR, "-ldida_letkf",
                        "-Wl,-rpath," + _build.LIB_DIR],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0 and "launch_check ok" in r.stdout, r.stdout + r.stderr
