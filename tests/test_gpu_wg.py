"""The one-workgroup batched LU (and LU + solve) on the GPU against the oracle
at the edges of its tiles: block (32 and 16 columns), strip (16 columns),
workgroup size (128, 256, 512 rows), padded leading dimensions, rectangular
shapes, 1 and 16 right-hand sides, exact ties, a zero column, entries that are
not finite."""
import numpy as np
import pytest

from conftest import EPS, TESTER_TOL, uniform_batch

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

LU_FWD_TOL = 1e3 * EPS
VARIANT_WG, VARIANT_BLOCKED = 6, 2


@pytest.fixture(scope="module")
def mb():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from magma_amd import batched
    return batched


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def check(oracle, A, LU, ipiv, info, m, n):
    LUo, ipo, info_o = oracle.dgetrf(A, m=m)
    tie_free = oracle.pivot_margin(A, m) > 1e-10
    assert np.array_equal(info, info_o)
    assert np.array_equal(ipiv[tie_free], ipo[tie_free])
    assert (oracle.lu_forward_error(LUo[tie_free], LU[tie_free], m) < LU_FWD_TOL).all()
    assert (oracle.lu_residual(A, LU, ipiv, m, n) < TESTER_TOL).all()


@pytest.mark.parametrize("m,n,ld", [(129, 129, 129), (143, 143, 150), (159, 159, 159), (161, 161, 161),
                                    (255, 255, 256), (257, 257, 257), (289, 289, 301), (511, 511, 511),
                                    (512, 512, 513), (128, 96, 128), (127, 33, 130), (512, 13, 512), (65, 48, 65)])
def test_getrf_edges(mb, oracle, m, n, ld):
    A = uniform_batch(np.random.default_rng(m * 3 + n), 3, m, ld=ld, cols=n)
    dA = dev(A)
    ipiv, info = mb.dgetrf_batched(dA, m=m)
    LU = dA.cpu().numpy()
    check(oracle, A, LU, ipiv.cpu().numpy(), info.cpu().numpy(), m, n)
    assert np.array_equal(LU[:, :, m:], A[:, :, m:])


@pytest.mark.parametrize("m,n", [(24, 40), (100, 260), (256, 300)])
def test_getrf_wide_batch(mb, oracle, m, n):
    A = uniform_batch(np.random.default_rng(m + n), 8, m, cols=n)
    dA = dev(np.tile(A, (64, 1, 1)))                      # 512 systems: the rule's line
    ipiv, info = mb.dgetrf_batched(dA, m=m)
    check(oracle, A, dA[-8:].cpu().numpy(), ipiv[-8:].cpu().numpy(), info[-8:].cpu().numpy(), m, n)


@pytest.mark.parametrize("n,nrhs,ld", [(129, 1, 129), (160, 16, 160), (161, 15, 170), (256, 16, 256), (300, 3, 301),
                                       (512, 5, 512)])
def test_gesv_edges(mb, oracle, n, nrhs, ld):
    rng = np.random.default_rng(n + nrhs)
    A, B = uniform_batch(rng, 3, n, ld=ld), uniform_batch(rng, 3, n, ld=ld, cols=nrhs)
    dA, dB = dev(A), dev(B)
    ipiv, info = mb.dgesv_batched(dA, dB)
    check(oracle, A, dA.cpu().numpy(), ipiv.cpu().numpy(), info.cpu().numpy(), n, n)
    X = dB.cpu().numpy()
    assert (oracle.gesv_backward_error(A, X, B, n) < TESTER_TOL).all()
    assert np.array_equal(X[:, :, n:], B[:, :, n:])


@pytest.mark.parametrize("n,nrhs", [(65, 1), (96, 16), (127, 3), (128, 4)])
def test_gesv_many_small(mb, oracle, n, nrhs):
    """1,536 systems of up to 128 rows: the line from the register-tile kernel."""
    rng = np.random.default_rng(n)
    A, B = uniform_batch(rng, 4, n), uniform_batch(rng, 4, n, cols=nrhs)
    dA, dB = dev(np.tile(A, (384, 1, 1))), dev(np.tile(B, (384, 1, 1)))
    ipiv, info = mb.dgesv_batched(dA, dB)
    check(oracle, A, dA[-4:].cpu().numpy(), ipiv[-4:].cpu().numpy(), info[-4:].cpu().numpy(), n, n)
    assert (oracle.gesv_backward_error(A, dB[-4:].cpu().numpy(), B, n) < TESTER_TOL).all()


@pytest.mark.parametrize("n", [33, 64, 100, 129, 200, 300])
def test_getrf_f32(mb, oracle, n):
    A = uniform_batch(np.random.default_rng(n), 3, n).astype(np.float32)
    dA = dev(A)
    ipiv, info = mb.sgetrf_batched(dA)
    A64 = A.astype(np.float64)
    assert (info.cpu().numpy() == 0).all()
    res = oracle.lu_residual(A64, dA.cpu().numpy().astype(np.float64), ipiv.cpu().numpy(), n, n)
    assert (res < 30 * np.finfo(np.float32).eps).all()


@pytest.mark.parametrize("kind", ["ties", "zero_column", "not_finite"])
def test_same_as_blocked(mb, oracle, kind):
    """Ties, an exactly singular column and entries that are not finite: the
    pivots, info and where the factors are finite are those of the
    launch-per-step blocked LU."""
    rng = np.random.default_rng(5)
    ns = [130, 144, 200, 257, 300]
    mats = []
    for n in ns:
        M = rng.integers(-2, 3, (n, n)).astype(np.float64) if kind == "ties" else rng.uniform(-1, 1, (n, n))
        if kind == "zero_column":
            M[:, n // 3] = 0.0
        if kind == "not_finite":
            M[n // 2, n // 4] = np.inf
            M[3, n - 2] = np.nan
            M[0, 0] = np.nan
        mats.append(M)
    out = []
    for v in (VARIANT_WG, VARIANT_BLOCKED):
        A, B = mb.VBatch(ns, ns), mb.VBatch(ns, [1] * len(ns))
        for i, M in enumerate(mats):
            A.set(i, M)
        ipiv, info = mb.IpivV(ns), torch.zeros(len(ns), dtype=torch.int32, device="cuda")
        plan = mb.VbatchedPlan(ns, [1] * len(ns), {b: v for b in range(22)})
        assert all(b["variant"] == v for b in plan.buckets())
        plan.execute(A, B, ipiv, info)
        torch.cuda.synchronize()
        plan.close()
        out.append((A, ipiv, info.cpu().numpy()))
    (A1, p1, i1), (A2, p2, i2) = out
    assert np.array_equal(i1, i2)
    for i, n in enumerate(ns):
        X, Y = A1.get(i), A2.get(i)
        if kind == "ties":
            # the first columns are exact small integers over powers of two: ties decide their pivots
            assert p1.get(i, n)[0] == p2.get(i, n)[0]
            assert np.array_equal(p1.get(i, n)[:2], oracle.dgetrf(np.ascontiguousarray(mats[i].T)[None])[1][0][:2])
            continue
        assert np.array_equal(p1.get(i, n), p2.get(i, n))
        assert np.array_equal(np.isfinite(X), np.isfinite(Y))
        f = np.isfinite(X)
        if kind == "zero_column":
            assert np.abs(X[f] - Y[f]).max() <= LU_FWD_TOL * np.abs(Y[f]).max()


@pytest.mark.parametrize("n,nrhs,ld", [(1, 1, 1), (15, 4, 15), (16, 1, 20), (17, 3, 17), (32, 4, 32), (33, 2, 33),
                                       (47, 4, 50), (48, 1, 48)])
def test_wave_lu(mb, oracle, n, nrhs, ld):
    """2,048 systems of up to 48 rows: one wave per system, FP64 LU and LU + solve."""
    rng = np.random.default_rng(n * 7)
    A, B = uniform_batch(rng, 8, n, ld=ld), uniform_batch(rng, 8, n, ld=ld, cols=nrhs)
    A[1, :, :n] = rng.integers(-1, 2, (n, n))                # exact ties
    A[2, n // 2, :n] = 0.0                                   # a zero column
    A[1] += 3.0 * np.eye(n, ld)
    tA, tB = np.tile(A, (256, 1, 1)), np.tile(B, (256, 1, 1))
    dA, dB, dF = dev(tA), dev(tB), dev(tA)
    ipiv, info = mb.dgesv_batched(dA, dB)
    ipf, inf = mb.dgetrf_batched(dF, m=n)
    assert torch.equal(dA, dF) and torch.equal(ipiv, ipf) and torch.equal(info, inf)
    keep = [0, 1, 3, 4, 5, 6, 7]
    last = np.array(keep) + 2040
    LU, X = dA.cpu().numpy()[last], dB.cpu().numpy()[last]
    check(oracle, A[keep], LU, ipiv.cpu().numpy()[last], info.cpu().numpy()[last], n, n)
    assert int(info[2042]) == int(oracle.dgetrf(A[2:3], m=n)[2][0]) != 0
    ok = info.cpu().numpy()[last] == 0
    assert (oracle.gesv_backward_error(A[keep], X, B[keep], n)[ok] < TESTER_TOL).all()
    assert np.array_equal(LU[:, :, n:], A[keep][:, :, n:]) and np.array_equal(X[:, :, n:], B[keep][:, :, n:])


@pytest.mark.parametrize("n", [1, 5, 16, 31, 48, 49, 63, 64])
def test_wave_lu_f32(mb, oracle, n):
    """FP32 up to 64 rows against the FP64 oracle on small-integer systems
    whose factors are exact, and by residual."""
    rng = np.random.default_rng(n)
    A = uniform_batch(rng, 5, n).astype(np.float32)
    dA = dev(A)
    ipiv, info = mb.sgetrf_batched(dA)
    assert (info.cpu().numpy() == 0).all()
    res = oracle.lu_residual(A.astype(np.float64), dA.cpu().numpy().astype(np.float64), ipiv.cpu().numpy(), n, n)
    assert (res < 30 * np.finfo(np.float32).eps).all()
    U = np.triu(rng.integers(-4, 5, (n, n))).astype(np.float32)
    U[np.arange(n), np.arange(n)] = rng.integers(1, 10, n)
    perm = rng.permutation(n)
    P = np.empty_like(U)
    P[perm] = U                                              # one non-zero candidate per column
    dP = dev(np.ascontiguousarray(P.T)[None])
    ip, inf = mb.sgetrf_batched(dP)
    assert np.array_equal(dP.cpu().numpy()[0].T, U) and int(inf[0]) == 0
    assert np.array_equal(ip.cpu().numpy()[0], oracle.dgetrf(np.ascontiguousarray(P.T.astype(np.float64))[None])[1][0])
