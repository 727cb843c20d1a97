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
