"""Read-backs with host failures (native/readback_host.cpp, no device): an
allocation or a copy that fails ends the call with a status, never the
process, and leaves the staging fit for the next call."""

import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]


def test_host_failures_are_statuses(tmp_path):
    source = ROOT / "cenote_amd" / "csrc"
    program = tmp_path / "readback_host"
    subprocess.run(["g++", "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", f"-I{source}",
                    str(source / "cn_readback.cpp"), str(ROOT / "tests" / "native" / "readback_host.cpp"), "-pthread",
                    "-o", str(program)], check=True)
    run = subprocess.run([str(program)], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, run.stdout + run.stderr
    assert "allocation" in run.stdout and "FAILED" not in run.stdout
