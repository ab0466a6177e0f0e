"""The copies through pinned slots on the host, over a stand-in for HIP: bytes,
devices, errors and what is given back (tests/native/hostcopy_check.cpp).
Events made on the current device instead of the stream's must fail it."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
NATIVE = ROOT / "tests" / "native"
SRC = ROOT / "pyro_amd" / "csrc"


def _run(tmp_path, text):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    (tmp_path / "hostcopy.hip").write_text(text)
    shutil.copy(SRC / "hostcopy.hpp", tmp_path)
    exe = tmp_path / "hostcopy_check"
    subprocess.run([gxx, "-O1", "-std=c++17", "-pthread", "-I", str(tmp_path), "-I", str(NATIVE / "fake_hip"),
                    str(NATIVE / "hostcopy_check.cpp"), "-o", str(exe)], check=True)
    return subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)


def test_copies(tmp_path):
    r = _run(tmp_path, (SRC / "hostcopy.hip").read_text())
    print(r.stdout)
    assert r.returncode == 0 and r.stdout.strip().endswith("0 wrong"), r.stdout + r.stderr


@pytest.mark.parametrize("old,new", [
    ("hipStreamGetDevice(s, &dev)", "hipGetDevice(&dev)"),
    ("if (cur != dev) note_locked(hipSetDevice(cur));", ""),
    ("const size_t len = std::min(CHUNK, j.bytes - off);", "const size_t len = std::min(CHUNK, j.bytes - off) & ~7ull;"),
])
def test_planted_mistakes(tmp_path, old, new):
    text = (SRC / "hostcopy.hip").read_text()
    assert old in text
    assert _run(tmp_path, text.replace(old, new)).returncode != 0
