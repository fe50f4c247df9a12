"""The readback kernel marks a chunk as arrived only after every wave's stores of it have completed.  A
missing wait shows as stale pixels too rarely for a test on a GPU, so the order is read from the code the
compiler makes: between the last store of a chunk and the barrier that thread 0's mark follows, each wave
writes back what it stored and waits for it."""
from __future__ import annotations

import re
import shutil
import subprocess
from pathlib import Path

import pytest

from vkscanlinepr_amd import build

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def test_every_wave_waits_for_its_stores_before_the_mark(tmp_path):
    if not Path(HIPCC).exists():
        pytest.skip("hipcc is not installed")
    out = tmp_path / "k_readback.asm"
    r = subprocess.run([HIPCC, *build.HIP_FLAGS, "-x", "hip", "--cuda-device-only", "-S",
                        str(build.CSRC / "k_readback.hip"), "-o", str(out)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    code = [line.split(";")[0].strip() for line in out.read_text().splitlines()]
    at = {k: [i for i, line in enumerate(code) if re.match(k, line)]
          for k in (r"(global|flat)_store", r"s_barrier", r"buffer_wbl2 sc0 sc1", r"s_waitcnt .*vmcnt\(0\)")}
    stores, barriers, writebacks, waits = at.values()
    assert len(barriers) == 1
    pixels, marks = [i for i in stores if i < barriers[0]], [i for i in stores if i > barriers[0]]
    assert pixels and len(marks) == 1
    done = [i for i in writebacks if pixels[-1] < i < barriers[0]]
    assert done and any(done[-1] < i < barriers[0] for i in waits)
