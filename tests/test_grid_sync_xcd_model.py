"""The grid barrier's per-XCD form, on the CPU.

Builds tests/native/grid_sync_xcd_model.cpp against the library's own
grid_sync.h (host-compiled by hipcc) and runs it: a thread model of the first
barrier's count and the later barriers' two stages, over several spreads of the
workgroups over the XCDs, consecutive launches on the same words and counters
that wrap around.
"""
import pathlib
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parent.parent
HIPCC = shutil.which("hipcc") or ("/opt/rocm/bin/hipcc" if pathlib.Path("/opt/rocm/bin/hipcc").exists() else None)


@pytest.mark.skipif(HIPCC is None, reason="no hipcc")
def test_per_xcd_protocol(tmp_path):
    exe = tmp_path / "grid_sync_xcd_model"
    build = subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-O1", "-std=c++17", "-pthread",
                            f"-I{ROOT / 'include'}", f"-I{ROOT / 'perks_amd' / 'csrc'}",
                            str(ROOT / "tests" / "native" / "grid_sync_xcd_model.cpp"), "-o", str(exe)],
                           capture_output=True, text=True)
    assert build.returncode == 0, build.stderr[-3000:]
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert run.returncode == 0 and run.stdout.strip().endswith("ok"), run.stdout + run.stderr
