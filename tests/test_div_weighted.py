"""The multigrid tail's division by weighted counts equals IEEE division
(tests/native/div_weighted_check.c, on a stride of the mantissas)."""
import subprocess
from pathlib import Path


def test_corrected_product_equals_division(tmp_path):
    exe = tmp_path / "div_weighted_check"
    src = Path(__file__).resolve().parent / "native" / "div_weighted_check.c"
    subprocess.run(["gcc", "-O3", "-march=x86-64-v3", "-ffp-contract=off", str(src), "-o", str(exe), "-lm"], check=True)
    out = subprocess.run([str(exe), "4099"], stdout=subprocess.PIPE, text=True)
    counts, bad = map(int, out.stdout.split())
    assert counts > 200 and bad == 0, out.stdout
