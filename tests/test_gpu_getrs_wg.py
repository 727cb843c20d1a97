"""The blocked MFMA solve at the edges of its blocks (32 rows), strips (16
right-hand sides), workgroup sizes (64, 128, 512 rows) and of the right-hand
sides' place (LDS or global memory), both directions, FP64 and FP32."""
import numpy as np
import pytest

from conftest import TESTER_TOL, uniform_batch

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("trans", [111, 112])
@pytest.mark.parametrize("n,nrhs,pad", [(1, 1, 0), (31, 5, 0), (32, 16, 0), (33, 17, 3), (64, 33, 0), (65, 16, 1),
                                        (128, 5, 0), (129, 6, 0), (280, 16, 0), (300, 16, 5), (512, 5, 0),
                                        (545, 3, 0), (700, 40, 0)])
def test_getrs(oracle, trans, n, nrhs, pad):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from magma_amd import batched as mb
    rng = np.random.default_rng(n * 5 + nrhs)
    ld = n + pad
    A, B = uniform_batch(rng, 3, n, ld=ld), uniform_batch(rng, 3, n, ld=ld, cols=nrhs)
    if pad:
        B[:, :, n:] = 7.0
    LU, piv, _ = oracle.dgetrf(A, m=n)
    dB = torch.from_numpy(B).cuda()
    mb.dgetrs_batched(trans, torch.from_numpy(LU).cuda(), torch.from_numpy(piv).cuda(), dB)
    X = dB.cpu().numpy()
    Aop = A[:, :, :n] if trans == 111 else np.transpose(A[:, :, :n], (0, 2, 1))
    be = oracle.gesv_backward_error(np.ascontiguousarray(Aop), X[:, :, :n].copy(), B[:, :, :n].copy(), n)
    assert (be < TESTER_TOL).all(), be.max()
    assert np.array_equal(X[:, :, n:], B[:, :, n:])
    if pad:
        return
    # FP32: the same factors rounded; the residual is that of the rounded system
    LUs, dBs = torch.from_numpy(LU.astype(np.float32)).cuda(), torch.from_numpy(B.astype(np.float32)).cuda()
    mb.sgetrs_batched(trans, LUs, torch.from_numpy(piv).cuda(), dBs)
    L64 = LUs.cpu().numpy().astype(np.float64)
    eye = np.arange(n)
    for s in range(3):
        M = L64[s].T
        L, U = np.tril(M, -1), np.triu(M)
        L[eye, eye] = 1.0
        P = L @ U
        for j in reversed(range(n)):                       # undo the interchanges: A = P^T L U
            p = piv[s][j] - 1
            P[[j, p]] = P[[p, j]]
        Pop = P if trans == 111 else P.T
        Xs, Bs = dBs[s].cpu().numpy().astype(np.float64).T, B[s].astype(np.float32).astype(np.float64).T
        r = np.abs(Bs - Pop @ Xs).max() / (n * np.abs(L).sum(1).max() * np.abs(U).sum(1).max() * np.abs(Xs).max())
        assert r < 30 * np.finfo(np.float32).eps, r


@pytest.mark.parametrize("batch", [1024, 1025])
@pytest.mark.parametrize("n,nrhs", [(1, 1), (16, 4), (64, 1), (65, 3), (129, 4), (256, 2)])
def test_getrs_few_and_many(oracle, batch, n, nrhs):
    """Both sides of the line between one workgroup and one wave per system:
    three systems repeated through the batch, every copy with the same answer."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from magma_amd import batched as mb
    rng = np.random.default_rng(n * 7 + nrhs)
    A, B = uniform_batch(rng, 3, n, ld=n), uniform_batch(rng, 3, n, ld=n, cols=nrhs)
    LU, piv, _ = oracle.dgetrf(A, m=n)
    pick = torch.arange(batch) % 3
    dB = torch.from_numpy(B)[pick].cuda()
    mb.dgetrs_batched(111, torch.from_numpy(LU)[pick].cuda(), torch.from_numpy(piv)[pick].cuda(), dB)
    X = dB.cpu()
    assert torch.equal(X, X[:3][pick])
    be = oracle.gesv_backward_error(A, X[:3].numpy(), B, n)
    assert (be < TESTER_TOL).all(), be.max()
