"""The build's flags: a define that varies a constant reaches host and device
code alike, since both read the shared headers."""

import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parents[1] / "cenote_amd" / "csrc"


def test_extra_defines_reach_host_and_device_code(tmp_path):
    lines = subprocess.run(["make", "-n", "-C", str(CSRC), "EXTRA=-DSLOT_GROUP=8u", f"BUILD={tmp_path / 'objects'}",
                            f"OUT={tmp_path / 'library.so'}"], check=True, capture_output=True, text=True).stdout
    compiles = [line for line in lines.splitlines() if " -c " in line]
    sources = sorted(f.name for f in CSRC.iterdir() if f.suffix in (".hip", ".cpp"))
    assert sorted(line.split(" -c ")[1].split()[0] for line in compiles) == sources
    assert all("-DSLOT_GROUP=8u" in line for line in compiles)
