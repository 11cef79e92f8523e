"""The size rules that pick kernels and tiles (csrc/backend/launch_rules.h),
compiled for the host and checked at the sizes where they change over
(tests/native/launch_rules_tests.cpp)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
GXX = shutil.which("g++")


@pytest.mark.skipif(GXX is None, reason="g++ not available")
def test_launch_rules(tmp_path):
    exe = tmp_path / "launch_rules_tests"
    subprocess.run([GXX, "-std=c++17", "-Wall", "-Werror", "-g", "-fsanitize=undefined", "-fno-sanitize-recover=undefined",
                    f"-I{ROOT / 'tinyinfer_amd' / 'csrc' / 'backend'}",
                    str(ROOT / "tests" / "native" / "launch_rules_tests.cpp"), "-o", str(exe)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0 and run.stdout == "ok\n", run.stderr
