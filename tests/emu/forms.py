"""Forms of the batched LU kernels that need large batches to be dispatched,
run on a few systems through the entries of forms.cpp under the CPU emulation
with AddressSanitizer (exact-size buffers), against the oracle. One scenario
per argument; exits non-zero on the first failure.

Run as scenarios.py (ASan runtime preloaded):
      python tests/emu/forms.py zero_pivot
"""
import sys
from pathlib import Path

import numpy as np

sys.path.insert(0, str(Path(__file__).resolve().parent))
sys.path.insert(0, str(Path(__file__).resolve().parents[2]))

import oracle  # noqa: E402
from lu_inputs import dominant_with_zeros, getf2_nopiv, zero_columns_with_nan  # noqa: E402
from scenarios import FAILURES, LIB, Buf, check, i32, ptr_array, vp  # noqa: E402

LU_FWD_TOL = 1e3 * np.finfo(np.float64).eps

LIB.emu_lu_wave_d.argtypes = [i32, i32, i32, vp, vp, vp, vp, vp, vp, vp, i32, i32, i32]
LIB.emu_lu_wave_s.argtypes = [i32, i32, i32, vp, vp, vp, i32]
LIB.emu_lu_wg_d.argtypes = [i32, i32, i32, vp, vp, vp, vp, i32, i32, i32]


def run_lu(kernel, A, m, pivot=True):
    """LU of the batch A (batch, n, ld) by one kernel: (LU, ipiv, info)."""
    batch, n, ld = A.shape
    k = min(m, n)
    bA, bP, bI = Buf(A), Buf(np.zeros((batch, k), np.int32)), Buf(np.full(batch, -7, np.int32))
    pA = ptr_array(bA, batch, n * ld * A.itemsize)
    pP = ptr_array(bP, batch, k * 4)
    if kernel == "wave":
        rc = LIB.emu_lu_wave_d((n + 15) // 16, n, ld, None, None, None, pA.ptr, pP.ptr, bI.ptr, None, 0, 0, batch)
    elif kernel == "wave_f32":
        rc = LIB.emu_lu_wave_s((n + 15) // 16, n, ld, pA.ptr, pP.ptr, bI.ptr, batch)
    else:
        rc = LIB.emu_lu_wg_d(m, n, ld, pA.ptr, pP.ptr if pivot else None, bI.ptr, None, 0, 0, batch)
    check(rc == 0, f"{kernel} {m}x{n} rc {rc}")
    return bA.get(), bP.get(), bI.get()


def zero_pivot():
    """A zero pivot sets info and skips the scaling only: every later column,
    in the pivot's own group of columns or not, is updated the same way."""
    rng = np.random.default_rng(3)
    for kernel, n, cols in (("wave", 32, [0]), ("wave", 48, [3, 20]), ("wave", 13, [0]), ("wg", 80, [0]),
                            ("wg", 130, [5, 20, 40]), ("wave_f32", 64, [0, 17]), ("wave_f32", 20, [2])):
        A = zero_columns_with_nan(rng, n, cols)
        LUo, ipo, info_o = oracle.dgetrf(A)
        LU, ip, info = run_lu(kernel, A.astype(np.float32) if kernel == "wave_f32" else A, n)
        check(info[0] == info_o[0], f"zero pivot {kernel} {n}: info {info[0]} {info_o[0]}")
        check(np.array_equal(ip, ipo), f"zero pivot {kernel} {n}: pivots")
        check(np.array_equal(np.isfinite(LU), np.isfinite(LUo)),
              f"zero pivot {kernel} {n}: {np.isfinite(LU).sum()} finite entries, {np.isfinite(LUo).sum()} in the oracle")
    for m, n, zeros in ((80, 80, [0]), (130, 130, [5, 20, 40]), (64, 20, [17])):
        M = dominant_with_zeros(rng, m, n, zeros)
        ref, info_ref = getf2_nopiv(M)
        LU, _, info = run_lu("wg", np.ascontiguousarray(M.T)[None], m, pivot=False)
        err = oracle.lu_forward_error(ref.T[None], LU, m)[0]
        check(info[0] == info_ref and err < LU_FWD_TOL, f"no pivoting {m}x{n}: info {info[0]} {info_ref}, error {err:.1e}")


SCENARIOS = {"zero_pivot": zero_pivot}

if __name__ == "__main__":
    for name in sys.argv[1:]:
        SCENARIOS[name]()
    if FAILURES:
        print("failed:", FAILURES, flush=True)
        sys.exit(1)
    print("all scenarios passed", flush=True)
