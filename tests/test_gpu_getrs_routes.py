"""Batched solves on both sides of the lines between their kernels (order,
number of right-hand sides, number of systems, direction, precision): three
systems repeated through the batch, every copy with the same answer."""
import numpy as np
import pytest

from conftest import TESTER_TOL, uniform_batch

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

TRANS = 112
CASES = [(111, n, r, b) for n, r, b in ((1, 64, 3), (8, 8, 5000), (8, 9, 1706), (8, 9, 1707), (9, 5, 30), (4, 40, 30),
                                        (16, 17, 512), (16, 17, 513), (33, 40, 3), (64, 33, 30), (65, 33, 3))]
CASES += [(TRANS, n, r, b) for n, r, b in ((32, 2, 9), (33, 1, 768), (33, 2, 769), (128, 2, 30), (129, 2, 30), (64, 3, 30),
                                           (193, 2, 6), (192, 1, 6), (480, 3, 3), (481, 4, 3), (1536, 3, 3), (1537, 3, 3),
                                           (1537, 4, 3))]


@pytest.mark.parametrize("trans,n,nrhs,batch", CASES)
def test_getrs(oracle, trans, n, nrhs, batch):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from magma_amd import batched as mb
    rng = np.random.default_rng(n * 3 + nrhs)
    A, B = uniform_batch(rng, 3, n), uniform_batch(rng, 3, n, cols=nrhs)
    LU, piv, _ = oracle.dgetrf(A)
    pick = torch.arange(batch) % 3
    Aop = A if trans == 111 else np.ascontiguousarray(np.transpose(A, (0, 2, 1)))
    for dt, fn in ((torch.float64, mb.dgetrs_batched), (torch.float32, mb.sgetrs_batched)):
        F, R = torch.from_numpy(LU).to(dt), torch.from_numpy(B).to(dt)
        dB = R[pick].cuda()
        fn(trans, F[pick].cuda(), torch.from_numpy(piv)[pick].cuda(), dB)
        X = dB.cpu()
        assert torch.equal(X, X[:3][pick])
        if dt == torch.float64:
            be = oracle.gesv_backward_error(Aop, X[:3].numpy(), B, n)
            assert (be < TESTER_TOL).all(), be.max()
            continue
        for s in range(3):                       # the residual of the system that the rounded factors multiply out to
            M = F[s].double().numpy().T
            L, U = np.tril(M, -1) + np.eye(n), np.triu(M)
            P = L @ U
            for j in reversed(range(n)):
                p = piv[s][j] - 1
                P[[j, p]] = P[[p, j]]
            x, b = X[s].double().numpy().T, R[s].double().numpy().T
            r = np.abs(b - (P if trans == 111 else P.T) @ x).max()
            r /= n * np.abs(L).sum(1).max() * np.abs(U).sum(1).max() * np.abs(x).max()
            assert r < 30 * np.finfo(np.float32).eps, r
