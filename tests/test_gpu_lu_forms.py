"""Inputs on which the batched LU kernels must follow LAPACK step by step, at
batch sizes on both sides of the lines between the kernels, against the
oracle."""
import sys
from pathlib import Path

import numpy as np
import pytest

from conftest import EPS

torch = pytest.importorskip("torch")

sys.path.insert(0, str(Path(__file__).resolve().parent / "emu"))

import lu_inputs  # noqa: E402

pytestmark = pytest.mark.gpu

LU_FWD_TOL = 1e3 * EPS


@pytest.fixture(scope="module")
def mb():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from magma_amd import batched
    return batched


@pytest.mark.parametrize("n,batch,cols", [(32, 2047, [0]), (32, 2048, [0]), (48, 2048, [3, 20]), (80, 1535, [0]),
                                          (80, 1536, [0]), (130, 2, [5, 20, 40]), (300, 2, [0, 70])])
def test_zero_pivot_above_a_nan(mb, oracle, n, batch, cols):
    A = lu_inputs.zero_columns_with_nan(np.random.default_rng(n), n, cols)
    dA = torch.from_numpy(A).cuda().repeat(batch, 1, 1)
    ipiv, info = mb.dgetrf_batched(dA)
    LUo, ipo, info_o = oracle.dgetrf(A)
    assert (info.cpu().numpy() == info_o[0]).all()
    assert (ipiv.cpu().numpy() == ipo[0]).all()
    if batch >= 1536 or n > 128:          # the register tile spreads a NaN over its 16-row blocks
        assert np.array_equal(np.isfinite(dA[-1].cpu().numpy()), np.isfinite(LUo[0]))


@pytest.mark.parametrize("m,n,zeros", [(80, 80, [0]), (130, 130, [5, 20, 40]), (64, 20, [17])])
def test_zero_pivot_without_pivoting(mb, oracle, m, n, zeros):
    M = lu_inputs.dominant_with_zeros(np.random.default_rng(m), m, n, zeros)
    ref, info_ref = lu_inputs.getf2_nopiv(M)
    dA = torch.from_numpy(np.ascontiguousarray(M.T)[None]).cuda()
    info = mb.dgetrf_nopiv_batched(dA, m=m)
    assert int(info[0]) == info_ref
    assert oracle.lu_forward_error(ref.T[None], dA.cpu().numpy(), m)[0] < LU_FWD_TOL


@pytest.mark.parametrize("m,n", [(13, 14), (13, 48), (13, 49), (20, 24), (20, 48), (21, 30)])
def test_few_wide_rows(mb, oracle, m, n):
    """Wide systems on both sides of the line to the LDS kernel, 512 of them."""
    A = lu_inputs.uniform(np.random.default_rng(m * n), 4, m, n)
    dA = torch.from_numpy(A).cuda().repeat(128, 1, 1)
    ipiv, info = mb.dgetrf_batched(dA, m=m)
    LUo, ipo, info_o = oracle.dgetrf(A, m=m)
    clear = oracle.pivot_margin(A, m) > 1e-10
    assert (info.cpu().numpy() == 0).all() and (info_o == 0).all()
    assert np.array_equal(ipiv[-4:].cpu().numpy()[clear], ipo[clear])
    assert (oracle.lu_forward_error(LUo[clear], dA[-4:].cpu().numpy()[clear], m) < LU_FWD_TOL).all()
    assert torch.equal(dA, dA[-4:].repeat(128, 1, 1))


def test_dense_zero_pivot_above_a_nan(oracle):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from magma_amd import dense
    A = lu_inputs.zero_columns_with_nan(np.random.default_rng(12), 300, [0, 40, 130])
    LUo, ipo, info_o = oracle.dgetrf(A)
    ipiv, info = dense.getrf_gpu(torch.from_numpy(A[0].copy()).cuda())
    assert info == info_o[0] and np.array_equal(np.asarray(ipiv), ipo[0])


@pytest.mark.parametrize("n,batch", [(2, 2048), (33, 2048), (48, 2048), (48, 2047), (128, 1535), (127, 1536), (128, 1536),
                                     (256, 3), (301, 3), (512, 3)])
def test_tied_candidates(mb, oracle, n, batch):
    A = np.concatenate([lu_inputs.tied_pairs(np.random.default_rng(n + s), n, 2.0 ** -50) for s in range(3)])
    pick = torch.arange(batch) % 3
    ipiv, info = mb.dgetrf_batched(torch.from_numpy(A)[pick].cuda())
    assert (info == 0).all()
    assert torch.equal(ipiv.cpu(), torch.from_numpy(oracle.dgetrf(A)[1])[pick])


@pytest.mark.parametrize("n", [5, 32, 64, 100, 300])
def test_tied_candidates_f32(mb, oracle, n):
    A = np.concatenate([lu_inputs.tied_pairs(np.random.default_rng(n + s), n, 2.0 ** -20) for s in range(3)])
    ipiv, info = mb.sgetrf_batched(torch.from_numpy(A.astype(np.float32)).cuda())
    assert (info == 0).all() and np.array_equal(ipiv.cpu().numpy(), oracle.dgetrf(A)[1])
