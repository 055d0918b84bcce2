"""The few-token prefill kernel's slices of K on the host (tests/few_token_slices.cpp): with more slices
than its 8-bit arrival count holds no workgroup would be the last, and the output would stay unwritten.
Compiled with g++ here; no GPU involved."""
import os
import shutil
import subprocess

import pytest

from conftest import REPO


@pytest.mark.skipif(not shutil.which("g++"), reason="needs g++")
def test_slices_fit_the_arrival_counter(tmp_path):
    exe = tmp_path / "few_token_slices"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-I", os.path.join(REPO, "tiny-llm_amd", "csrc"),
                    os.path.join(REPO, "tests", "few_token_slices.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and "ok slices" in out.stdout, out.stdout + out.stderr
