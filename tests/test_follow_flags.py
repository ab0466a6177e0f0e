"""What a Poisson handle forms from its solid flags after calls that fail at any
step (pyro_amd/csrc/solve_guard.hpp); an order that keeps the old data for good
must fail the host program."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
SRC = ROOT / "tests" / "native" / "flags_check.cpp"
HDR = ROOT / "pyro_amd" / "csrc" / "solve_guard.hpp"


def _run(tmp_path, text):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    (tmp_path / "solve_guard.hpp").write_text(text)
    exe = tmp_path / "flags_check"
    subprocess.run([gxx, "-O1", "-std=c++17", "-I", str(tmp_path), str(SRC), "-o", str(exe)], check=True)
    return subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)


def test_follow_flags(tmp_path):
    r = _run(tmp_path, HDR.read_text())
    assert r.returncode == 0 and r.stdout.strip().endswith(" 0 wrong"), r.stdout + r.stderr


@pytest.mark.parametrize("old,new", [
    ("  formed = false;\n  bool changed = true;\n  int rc = compare(changed);\n",
     "  bool changed = true;\n  int rc = compare(changed);\n  if (rc) return rc;\n"),
    ("(changed || !was)", "(changed)"),
    ("(changed || !was)", "(true)"),
    ("  formed = rc == 0;\n", "  formed = true;\n"),
])
def test_follow_flags_catches_planted_mistakes(tmp_path, old, new):
    text = HDR.read_text()
    assert old in text
    assert _run(tmp_path, text.replace(old, new)).returncode != 0
