"""When a pressure solve starts the next V-cycle before it knows whether it needs
one (ResidWatch::expects_more, pyro_amd/csrc/solve_guard.hpp): the host program
drives residuals of solves through the rule; always starting must fail it."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
SRC = ROOT / "tests" / "native" / "next_cycle_check.cpp"
HDR = ROOT / "pyro_amd" / "csrc" / "solve_guard.hpp"
RULE = "return last * rate > tol;"


def _run(tmp_path, text):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    (tmp_path / "solve_guard.hpp").write_text(text)
    exe = tmp_path / "next_cycle_check"
    subprocess.run([gxx, "-O1", "-std=c++17", "-I", str(tmp_path), str(SRC), "-o", str(exe)], check=True)
    return subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)


def test_rule(tmp_path):
    r = _run(tmp_path, HDR.read_text())
    print(r.stdout)
    assert r.returncode == 0 and r.stdout.strip().endswith("0 wrong"), r.stdout + r.stderr


@pytest.mark.parametrize("new", ["return true;", "return false;", "return last > tol;"])
def test_rule_catches_planted_mistakes(tmp_path, new):
    text = HDR.read_text()
    assert RULE in text
    assert _run(tmp_path, text.replace(RULE, new)).returncode != 0
