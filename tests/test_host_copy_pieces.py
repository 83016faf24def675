"""The cut of a host copy into pieces, on the CPU: tests/native/host_copy_pieces.cpp
against the library's own host_copy.h."""
import pathlib
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parent.parent


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_pieces(tmp_path):
    exe = tmp_path / "host_copy_pieces"
    build = subprocess.run(["g++", "-std=c++17", "-Wall", f"-I{ROOT / 'perks_amd' / 'csrc'}",
                            str(ROOT / "tests" / "native" / "host_copy_pieces.cpp"), "-o", str(exe)],
                           capture_output=True, text=True)
    assert build.returncode == 0, build.stderr[-3000:]
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0 and run.stdout.strip() == "ok", run.stdout + run.stderr
