"""Forms of the batched LU and solve kernels that the larger scenarios do not
reach, under the CPU emulation with ASan on a few systems, against the oracle."""
import os
import subprocess
import sys
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
sys.path.insert(0, str(HERE / "emu"))

import build_emu  # noqa: E402


@pytest.mark.timeout(900)
@pytest.mark.parametrize("scenario", ["zero_pivot", "dense_zero_pivot", "ties", "wave", "wide", "plan_variants",
                                      "getrs", "getrs_vbatched"])
def test_form_under_asan(scenario):
    cxx = build_emu.clang()
    if cxx is None or build_emu.asan_runtime(cxx) is None:
        pytest.skip("no clang++ with the ASan runtime")
    build_emu.build()
    env = dict(os.environ, LD_PRELOAD=build_emu.asan_runtime(cxx), ASAN_OPTIONS="detect_leaks=0",
               EMU_WG_WINDOW="5")
    r = subprocess.run([sys.executable, str(HERE / "emu" / "forms.py"), scenario], env=env, capture_output=True,
                       text=True, timeout=880)
    out = r.stdout + r.stderr
    assert "AddressSanitizer" not in out, out[-6000:]
    assert r.returncode == 0, out[-6000:]
    assert "all scenarios passed" in out
