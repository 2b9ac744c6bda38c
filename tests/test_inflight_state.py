"""The host state about work in flight (dyc_inflight.hpp: which first-bucket rules a table keeps and
the finds that rely on one) over a stand-in for the HIP runtime, built for the host with ASan and UBSan."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_state_transitions(tmp_path):
    exe = tmp_path / "inflight"
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-pthread", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=undefined", "-I", os.path.join(ROOT, "databases_gpu_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "inflight_check.cpp"), "-o", str(exe)],
                   check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "inflight ok" in r.stdout
