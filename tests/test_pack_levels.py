"""The INT4 pack's level arithmetic (layer_quant_amd/csrc/int4_pack.hip, pack_levels), checked on the
CPU against the IEEE quotient for every fp32 mantissa next to every half-integer."""
import shutil
import subprocess
from pathlib import Path

import pytest

CHECK = Path(__file__).resolve().parent / "native" / "pack_levels.c"


@pytest.mark.skipif(shutil.which("gcc") is None, reason="needs gcc")
def test_levels_equal_the_ieee_quotients(tmp_path):
    exe = tmp_path / "pack_levels"
    subprocess.run(["gcc", "-O2", "-march=native", "-fopenmp", "-ffp-contract=off", "-o", str(exe),
                    str(CHECK), "-lm"], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=600)
    assert res.returncode == 0 and " bad=0" in res.stdout, res.stdout + res.stderr
