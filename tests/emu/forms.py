"""Forms of the batched LU and solve kernels that scenarios.py does not reach
(those that need large batches through the entries of forms.cpp), run on a few
systems under the CPU emulation with AddressSanitizer (exact-size buffers),
against the oracle. One scenario
per argument; exits non-zero on the first failure.

Run as scenarios.py (ASan runtime preloaded):
      python tests/emu/forms.py zero_pivot
"""
import ctypes
import sys
from pathlib import Path

import numpy as np

sys.path.insert(0, str(Path(__file__).resolve().parent))
sys.path.insert(0, str(Path(__file__).resolve().parents[2]))

import oracle  # noqa: E402
from lu_inputs import dominant_with_zeros, getf2_nopiv, tied_pairs, zero_columns_with_nan  # noqa: E402
from scenarios import FAILURES, LIB, Buf, check, i32, ptr_array, queue, vp  # noqa: E402

QUEUE = queue()
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


def run_getrs(prec, n, nrhs, trans, batch=2, pad=0):
    """Solve with the oracle's factors of uniform systems; the backward error
    (FP32: of the system that the rounded factors multiply out to)."""
    rng = np.random.default_rng(n * 5 + nrhs)
    dt = np.float64 if prec == "d" else np.float32
    ld = n + pad
    A, B = rng.uniform(-1, 1, (batch, n, ld)), rng.uniform(-1, 1, (batch, nrhs, ld)).astype(dt)
    LU, piv, _ = oracle.dgetrf(A, m=n)
    bA, bB, bP = Buf(LU.astype(dt)), Buf(B), Buf(piv)
    pA, pB, pP = (ptr_array(b, batch, b.nbytes // batch) for b in (bA, bB, bP))
    fn = getattr(LIB, f"magma_{prec}getrs_batched")
    fn.argtypes = [i32, i32, i32, vp, i32, vp, vp, i32, i32, vp]
    rc = fn(112 if trans else 111, n, nrhs, pA.ptr, ld, pP.ptr, pB.ptr, ld, batch, QUEUE)
    X, eye = bB.get(), np.arange(n)
    check(rc == 0 and np.array_equal(X[:, :, n:], B[:, :, n:]), f"{prec}getrs {n} {nrhs} {trans}: rc {rc} or padding")
    for s in range(batch):
        M = LU[s].astype(dt).astype(np.float64)[:, :n].T
        L, U = np.tril(M, -1), np.triu(M)
        L[eye, eye] = 1.0
        P = L @ U
        for j in reversed(range(n)):                       # undo the interchanges: A = P^T L U
            P[[j, piv[s][j] - 1]] = P[[piv[s][j] - 1, j]]
        x, b = X[s, :, :n].astype(np.float64).T, B[s, :, :n].astype(np.float64).T
        r = np.abs(b - (P.T if trans else P) @ x).max() / (n * np.abs(L).sum(1).max() * np.abs(U).sum(1).max() *
                                                          np.abs(x).max())
        check(r < 30 * np.finfo(dt).eps, f"{prec}getrs n={n} nrhs={nrhs} trans={trans}: {r:.1e}")


def getrs():
    """The solve kernels at the edges of their blocks, with the right-hand
    sides in LDS and in global memory (more than 36 KB of them)."""
    for prec in "ds":
        for n, nrhs, pad in ((3, 6, 0), (17, 3, 1), (33, 5, 0), (64, 2, 0), (65, 4, 2), (100, 17, 0), (150, 40, 1),
                             (257, 1, 0), (290, 4, 3), (300, 40, 0)):
            for trans in (0, 1):
                run_getrs(prec, n, nrhs, trans, batch=1 if n > 128 else 2, pad=pad)


def getrs_vbatched():
    """Mixed orders and right-hand side counts, empty ones among them, both
    directions, where the largest order decides the kernel."""
    rng = np.random.default_rng(8)
    for ns, rs in (([40, 0, 100, 33, 7], [2, 1, 1, 0, 2]), ([8, 3, 5], [8, 1, 4]), ([130, 64, 20], [5, 17, 1])):
        A = [rng.uniform(-1, 1, (1, max(n, 1), max(n, 1))) for n in ns]
        F = [oracle.dgetrf(a) for a in A]
        for trans in (0, 1):
            B = [rng.uniform(-1, 1, (1, max(r, 1), max(n, 1))) for n, r in zip(ns, rs)]
            bA, bP, bB = [Buf(f[0]) for f in F], [Buf(f[1]) for f in F], [Buf(b) for b in B]
            pA, pP, pB = (Buf(np.array([x.ptr for x in y], np.uint64)) for y in (bA, bP, bB))
            dn, dr, ld = Buf(np.array(ns, np.int32)), Buf(np.array(rs, np.int32)), Buf(np.maximum(ns, 1).astype(np.int32))
            fn = LIB.magma_dgetrs_vbatched
            fn.argtypes = [i32, vp, vp, i32, i32, vp, vp, vp, vp, vp, i32, vp]
            rc = fn(112 if trans else 111, dn.ptr, dr.ptr, max(ns), max(rs), pA.ptr, ld.ptr, pP.ptr, pB.ptr, ld.ptr,
                    len(ns), QUEUE)
            check(rc == 0, f"dgetrs_vbatched {ns} rc {rc}")
            for n, r, f, b, x in zip(ns, rs, F, B, bB):
                X = x.get()
                if n == 0 or r == 0:
                    check(np.array_equal(X, b), f"dgetrs_vbatched n={n} nrhs={r}: touched")
                    continue
                ref = oracle.dgetrs(trans, f[0], f[1], b)
                # the oracle solves with the same factors: both errors are of the size n eps times the growth of
                # the triangles, which uniform factors of these orders keep below 1e8
                check(np.abs(X - ref).max() <= 1e-7 * np.abs(ref).max(), f"dgetrs_vbatched n={n} nrhs={r} trans={trans}")


def ties():
    """Candidates that tie, in all bits or in the upper 32: the oracle's pivots."""
    rng = np.random.default_rng(21)
    for kernel, sizes in (("wave", (2, 16, 33, 48)), ("wg", (64, 127, 256, 300)), ("wave_f32", (5, 32, 64))):
        f32 = kernel == "wave_f32"
        for n in sizes:
            for _ in range(3):
                A = tied_pairs(rng, n, 2.0 ** (-20 if f32 else -50))
                LU, ip, info = run_lu(kernel, A.astype(np.float32) if f32 else A, n)
                check(info[0] == 0 and np.array_equal(ip, oracle.dgetrf(A)[1]), f"ties {kernel} {n}")


def wave():
    """The FP64 wave kernel with a map, per-matrix orders and leading dimensions
    (an empty system among them), and fused with up to four right-hand sides."""
    rng = np.random.default_rng(31)
    for nch, ns in ((1, [16, 1, 0, 9]), (2, [17, 32, 20, 31]), (3, [48, 33, 47, 40])):
        lds = [max(n, 1) + k % 3 for k, n in enumerate(ns)]
        A = [rng.uniform(-1, 1, (1, max(n, 1), ld)) for n, ld in zip(ns, lds)]
        bA, bP = [Buf(a) for a in A], [Buf(np.zeros(max(n, 1), np.int32)) for n in ns]
        pA, pP = (Buf(np.array([x.ptr for x in y], np.uint64)) for y in (bA, bP))
        dn, dl, dm = Buf(np.array(ns, np.int32)), Buf(np.array(lds, np.int32)), Buf(np.array([3, 1, 0, 2], np.int32))
        info = Buf(np.zeros(4, np.int32))
        rc = LIB.emu_lu_wave_d(nch, 0, 0, dm.ptr, dn.ptr, dl.ptr, pA.ptr, pP.ptr, info.ptr, None, 0, 0, 4)
        check(rc == 0 and (info.get() == 0).all(), f"wave {ns}: rc {rc} info {info.get()}")
        for n, a, b, p in zip(ns, A, bA, bP):
            if n == 0:
                check(np.array_equal(b.get(), a), "wave: empty system touched")
                continue
            LUo, ipo, _ = oracle.dgetrf(a, m=n)
            check(np.array_equal(p.get(), ipo[0]), f"wave n={n}: pivots")
            check(oracle.lu_forward_error(LUo, b.get(), n)[0] < LU_FWD_TOL, f"wave n={n}: factors")
            check(np.array_equal(b.get()[:, :, n:], a[:, :, n:]), f"wave n={n}: padding touched")
    for n, nrhs, ld in ((1, 1, 1), (16, 4, 17), (17, 3, 17), (32, 1, 32), (48, 4, 50)):
        A, B = rng.uniform(-1, 1, (3, n, ld)), rng.uniform(-1, 1, (3, nrhs, ld))
        bA, bB, bP, bI = Buf(A), Buf(B), Buf(np.zeros((3, n), np.int32)), Buf(np.zeros(3, np.int32))
        pA, pB, pP = (ptr_array(b, 3, b.nbytes // 3) for b in (bA, bB, bP))
        rc = LIB.emu_lu_wave_d((n + 15) // 16, n, ld, None, None, None, pA.ptr, pP.ptr, bI.ptr, pB.ptr, nrhs, ld, 3)
        be = oracle.gesv_backward_error(A, bB.get(), B, n)
        check(rc == 0 and (be < 30 * np.finfo(np.float64).eps).all(), f"wave gesv n={n} nrhs={nrhs}: {be}")


def wide():
    """Wide systems on the one-workgroup kernel."""
    rng = np.random.default_rng(41)
    for m, n in ((20, 50), (33, 40), (64, 100), (130, 145)):
        A = rng.uniform(-1, 1, (1, n, m))
        LU, ip, info = run_lu("wg", A, m)
        LUo, ipo, _ = oracle.dgetrf(A, m=m)
        check(info[0] == 0 and np.array_equal(ip, ipo), f"wide {m}x{n}: pivots")
        check(oracle.lu_forward_error(LUo, LU, m)[0] < LU_FWD_TOL, f"wide {m}x{n}: factors")


def dense_zero_pivot():
    """The same on one matrix (magma_dgetrf_gpu, magma_sgetrf_gpu): an exact
    zero pivot with a NaN below it."""
    rng = np.random.default_rng(12)
    for prec, n, cols in (("d", 300, [0, 40, 130]), ("s", 300, [3])):
        A = zero_columns_with_nan(rng, n, cols)
        LUo, ipo, info_o = oracle.dgetrf(A)
        bA = Buf(A[0] if prec == "d" else A[0].astype(np.float32))
        ipiv, info = (i32 * n)(), i32(-7)
        fn = getattr(LIB, f"magma_{prec}getrf_gpu")
        fn.argtypes = [i32, i32, vp, i32, vp, ctypes.POINTER(i32)]
        rc = fn(n, n, bA.ptr, n, ipiv, ctypes.byref(info))
        P = np.array(ipiv[:], np.int32)
        first = int(np.argmax(P != ipo[0])) if not np.array_equal(P, ipo[0]) else -1
        check(rc >= 0 and info.value == info_o[0], f"dense {prec} zero pivot: rc {rc} info {info.value} {info_o[0]}")
        check(first < 0, f"dense {prec} zero pivot: pivots differ from step {first}")


def plan_variants():
    """The kernel that a plan picks for 65..128 rows by itself: the register
    tile (1) below 1,536 systems and, without right-hand sides, for 69..80 rows
    (up to 76 but for 1,537..2,048 systems); one workgroup per system (6) else."""
    LIB.magma_dgesv_vbatched_plan_create.argtypes = [vp, vp, i32, vp, vp, ctypes.POINTER(vp)]
    LIB.magma_vbatched_plan_bucket.argtypes = [vp, i32, ctypes.POINTER(i32)]
    LIB.magma_vbatched_plan_destroy.argtypes = [vp]
    for n, count, solve, want in ((68, 1536, False, 6), (69, 1536, False, 1), (80, 1536, False, 1), (81, 1536, False, 6),
                                  (68, 1535, False, 1), (76, 1537, False, 6), (76, 2048, False, 6),
                                  (76, 2049, False, 1), (77, 2048, False, 1), (69, 1536, True, 6), (80, 1536, True, 6), (80, 1535, True, 1)):
        hn, hr = np.full(count, n, np.int32), np.ones(count, np.int32)
        plan, info = vp(), (i32 * 5)()
        rc = LIB.magma_dgesv_vbatched_plan_create(hn.ctypes.data, hr.ctypes.data if solve else None, count, None, QUEUE,
                                                  ctypes.byref(plan))
        LIB.magma_vbatched_plan_bucket(plan, 0, info)
        LIB.magma_vbatched_plan_destroy(plan)
        check(rc == 0 and info[2] == count and info[1] == want, f"plan of {count} x {n}, solve {solve}: variant {info[1]}")


SCENARIOS = {f.__name__: f for f in (zero_pivot, dense_zero_pivot, ties, wave, wide, plan_variants, getrs, getrs_vbatched)}

if __name__ == "__main__":
    for name in sys.argv[1:]:
        SCENARIOS[name]()
    if FAILURES:
        print("failed:", FAILURES, flush=True)
        sys.exit(1)
    print("all scenarios passed", flush=True)
