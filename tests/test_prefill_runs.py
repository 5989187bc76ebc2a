"""The runs of split prefill launches (bnr::plan_prefill_runs): a host-only
harness built against the library decodes every run of 4000 seeded plans the
way the kernel does, and checks on which side of the line between split and
fp32 launches measured shapes fall (no GPU needed)."""
import os
import shutil
import subprocess

import pytest

from bitnetrs_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_prefill_runs(tmp_path):
    _lib.load()  # the library is built
    lib_dir = os.path.dirname(_lib.LIB_PATH)
    exe = tmp_path / "prefill_runs_check"
    subprocess.run([HIPCC, "-O1", "-std=c++17", "-I", os.path.join(ROOT, "bitnetrs_amd", "csrc"),
                    "-o", str(exe), os.path.join(ROOT, "tests", "native", "prefill_runs_check.cpp"),
                    "-L", lib_dir, "-lbitnet_hip", f"-Wl,-rpath,{lib_dir}"],
                   check=True, capture_output=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.startswith("ok"), out.stdout + out.stderr
