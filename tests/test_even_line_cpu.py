"""The even-share line (which tiles a workgroup takes, how its waves walk them) run on the host.

With the row lengths as they are at the launch, every tile is attended once and every cut row's parts are the ones
its merge reads.  With lengths that change while the launch reads them (a caller that updates them on another
stream), rows may be wrong, but every wave comes to an end, and every read and store stays inside its buffer.
"""

import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_every_walk_ends_in_range(tmp_path):
    exe = tmp_path / "even_line_host"
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", str(ROOT / "flashdec_amd" / "csrc"),
                    str(ROOT / "tests" / "native" / "even_line_host.cpp"), "-o", str(exe)], check=True)
    ran = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert ran.returncode == 0, ran.stderr
