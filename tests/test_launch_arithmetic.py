"""CPU: launch arithmetic that the kernels share with plain C++."""
import os
import subprocess

import pytest

CPP = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp")


@pytest.mark.parametrize("name", ["test_wide_requests", "test_few_offsets", "test_small_division", "test_decode_wide", "test_decode_forms", "test_decode_choice", "test_decode_steps"])
def test_launch_arithmetic(name, tmp_path):
    exe = tmp_path / name
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", str(exe), os.path.join(CPP, name + ".cpp")], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[-2000:]
    assert r.stdout.startswith("OK")
