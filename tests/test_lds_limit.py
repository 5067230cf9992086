"""The dynamic-LDS limit is raised per device (a host build over a counting stand-in
for the HIP runtime), and every launcher of the kernels goes through it."""
import os
import re
import shutil
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
CSRC = HERE.parent / "tinyinfer_amd" / "csrc"
ROCM = Path(os.environ.get("ROCM_PATH", "/opt/rocm"))


def test_limit_is_raised_once_on_each_device(tmp_path):
    if shutil.which("g++") is None or not (ROCM / "include" / "hip").is_dir():
        pytest.skip("needs g++ and the HIP headers")
    exe = tmp_path / "lds_limit"
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", str(ROCM / "include"),
                    str(HERE / "host" / "lds_limit.cpp"), "-o", str(exe)], check=True)
    subprocess.run([str(exe)], check=True)


def test_no_launcher_raises_the_limit_by_itself():
    for source in CSRC.glob("*.hip"):
        assert not re.search(r"hipFuncSetAttribute", source.read_text()), source.name
