"""Host-side rules of the device backend (csrc/backend), compiled for the host
and checked without a GPU:

- launch_rules.h: the size rules that pick kernels and tiles, at the sizes
  where they change over (tests/native/launch_rules_tests.cpp);
- idle_memory.h: memory that outlives a call, over an allocator that fails on
  request (tests/native/idle_memory_tests.cpp)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
GXX = shutil.which("g++")


@pytest.mark.skipif(GXX is None, reason="g++ not available")
@pytest.mark.parametrize("name", ["launch_rules_tests", "idle_memory_tests"])
def test_backend_rules(tmp_path, name):
    exe = tmp_path / name
    subprocess.run([GXX, "-std=c++17", "-Wall", "-Werror", "-g", "-pthread", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=undefined", f"-I{ROOT / 'tinyinfer_amd' / 'csrc' / 'backend'}",
                    str(ROOT / "tests" / "native" / f"{name}.cpp"), "-o", str(exe)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0 and run.stdout == "ok\n", run.stderr
