"""The host sources compile for a processor other than x86 (syntax only: the system's headers, as an aarch64
compiler reads them)."""
from __future__ import annotations

import subprocess
from pathlib import Path

import pytest

from vkscanlinepr_amd import build

CLANG = Path("/opt/rocm/llvm/bin/clang++")
SYSTEM = ["/usr/include/c++/11", "/usr/include/x86_64-linux-gnu/c++/11", "/usr/include/x86_64-linux-gnu"]


@pytest.mark.parametrize("name", sorted(p.name for p in build.CSRC.glob("*.cpp")))
def test_host_source_for_aarch64(tmp_path, name):
    if not CLANG.exists() or not all(Path(d).is_dir() for d in SYSTEM):
        pytest.skip("needs ROCm's clang and the system's C++ headers")
    (tmp_path / "gnu").mkdir()
    (tmp_path / "gnu" / "stubs-32.h").touch()  # the x86-64 headers name it for other targets
    r = subprocess.run([str(CLANG), "--target=aarch64-linux-gnu", "-fsyntax-only", "-std=c++17", "-x", "c++",
                        "-D__HIP_PLATFORM_AMD__", f"-I{tmp_path}", "-I/opt/rocm/include", f"-I{build.ROOT / 'include'}",
                        f"-I{build.CSRC}", *(a for d in SYSTEM for a in ("-isystem", d)), str(build.CSRC / name)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
