"""The one-workgroup LU, the wave LU and the MFMA solve under the CPU
emulation with ASan: every form the dispatch sends them (square, tall, wide
panels' edges, mixed orders of a plan, more right-hand sides than one strip)."""
import os
import subprocess
import sys
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
sys.path.insert(0, str(HERE / "emu"))

import build_emu  # noqa: E402

SCENARIOS = ["getrf:512:13", "getrf:143:100", "getrf:161:129", "getrf:257:257", "sgesv:60:33", "sgesv:31:17",
             "sgesv:130:40", "vbplan:6", "acc:bf16x3:ir:100:129"]


@pytest.mark.timeout(900)
def test_new_kernels_under_asan():
    cxx = build_emu.clang()
    if cxx is None or build_emu.asan_runtime(cxx) is None:
        pytest.skip("no clang++ with the ASan runtime")
    build_emu.build()
    env = dict(os.environ, LD_PRELOAD=build_emu.asan_runtime(cxx), ASAN_OPTIONS="detect_leaks=0")
    r = subprocess.run([sys.executable, str(HERE / "emu" / "scenarios.py"), *SCENARIOS], env=env,
                       capture_output=True, text=True, timeout=880)
    out = r.stdout + r.stderr
    assert "AddressSanitizer" not in out, out[-6000:]
    assert r.returncode == 0, out[-6000:]
    assert "all scenarios passed" in out
