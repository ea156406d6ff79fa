"""The detector's work-buffer entry points under host-side AddressSanitizer and
UndefinedBehaviorSanitizer, as test_host_sanitizers does for the rest of the C ABI (device code is
compiled as usual and never launched)."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.join(os.path.dirname(__file__), "..")
SAN = ["-Xarch_host", "-fsanitize=address", "-Xarch_host", "-fsanitize=undefined"]


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc not available")
def test_detector_work_under_asan_ubsan(tmp_path):
    exe = str(tmp_path / "driver")
    build = subprocess.run(
        ["hipcc", "--offload-arch=gfx950", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "include"),
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"] + SAN +
        ["-o", exe, os.path.join(ROOT, "giwaxsim_amd", "csrc", "gx_detector.hip"),
         os.path.join(ROOT, "tests", "host", "detector_work_driver.cpp")],
        capture_output=True, text=True, timeout=600)
    assert build.returncode == 0, build.stderr[-3000:]
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=1:halt_on_error=1",
               UBSAN_OPTIONS="halt_on_error=1:print_stacktrace=1")
    run = subprocess.run([exe], capture_output=True, text=True, timeout=120, env=env)
    assert run.returncode == 0, (run.stdout + run.stderr)[-3000:]
    assert "checks passed:" in run.stdout
