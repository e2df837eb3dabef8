"""CSR products with a lane group per row: averages on both sides of the dispatch lines (8 and 128
entries per row), rows of 0, 1 and many entries, every width of the interleaved pass and its
remainder, with and without workspace, and the x . Ax partials that CG and Lanczos read."""
import numpy as np
import pytest
import scipy.sparse
import torch

import cola_amd as ca
from cola_amd import _native as N
from cola_amd._blocks import ld_of
from cola_amd.linalg import HipCG, inv

pytestmark = pytest.mark.gpu


def matrix(n, avg, seed):
    """Rows of uneven length around avg: empty ones, single entries and one row four times as long."""
    rs = np.random.RandomState(seed)
    lens = np.minimum(rs.poisson(avg, n), n)
    lens[::7] = np.minimum(lens[::7], 1)
    lens[n // 2] = min(n, 4 * avg)
    lens[0] = 0
    rows = np.repeat(np.arange(n), lens)
    cols = rs.randint(0, n, rows.size)  # a pair drawn twice becomes one entry
    vals = rs.randn(rows.size).astype(np.float32)
    return scipy.sparse.csr_matrix((vals, (rows, cols)), (n, n))


@pytest.mark.parametrize("n,avg", [(65, 14), (700, 5), (700, 12), (700, 40), (700, 90), (301, 230), (5000, 11)])
@pytest.mark.parametrize("nrhs", [1, 2, 3, 5, 8, 11])
@pytest.mark.parametrize("room", [True, False])
def test_csr_group_product(dev, n, avg, nrhs, room):
    M = matrix(n, avg, n + avg)
    A = ca.Sparse.from_csr(torch.from_numpy(M.indptr).to(dev), torch.from_numpy(M.indices).to(dev),
                           torch.from_numpy(M.data).to(dev), (n, n))
    X = np.random.RandomState(nrhs).randn(n, nrhs).astype(np.float32)
    ref = 0.5 * (M.astype(np.float64) @ X.astype(np.float64)) + 2.0 * X
    mag = 0.5 * (abs(M).astype(np.float64) @ np.abs(X).astype(np.float64)) + 2.0 * np.abs(X)
    op, keep = A.hip_op()
    op.scale, op.shift = 0.5, 2.0
    ld = ld_of(n)
    Xb = torch.full((nrhs, ld), float("nan"), device=dev)  # padding is never gathered
    Xb[:, :n] = torch.from_numpy(X.T.copy()).to(dev)
    Yb = torch.empty_like(Xb)
    wb = N.q("ck_op_workspace_bytes", op, nrhs)
    work = torch.empty(max(wb, 4) // 4, device=dev) if room else None
    N.call("ck_op_apply", op, nrhs, N.ptr(Xb), ld, N.ptr(Yb), ld, N.ptr(work), wb if room else 0, N.stream_ptr(dev))
    err = np.abs(Yb[:, :n].T.double().cpu().numpy() - ref)
    depth = np.diff(M.indptr)[:, None] + 8  # roundings of a row's sum
    assert (err <= 6e-8 * depth * mag + 1e-30).all()


def hubs(n, avg, length, seed):
    """Rows of about avg entries, three of them `length` long: first, last and in the middle of a wave's."""
    rs = np.random.RandomState(seed)
    lens = np.maximum(rs.poisson(avg, n), 1)
    lens[[0, n // 2 + 5, n - 1]] = length
    ptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    cols = rs.randint(0, n, ptr[-1]).astype(np.int32)  # several entries may share a column
    return scipy.sparse.csr_matrix((rs.randn(ptr[-1]).astype(np.float32), cols, ptr), (n, n)), ptr, cols


@pytest.mark.parametrize("n,avg,length", [(1001, 12, 127), (1001, 12, 129), (1001, 12, 257), (1001, 40, 300), (640, 12, 20001),
                                          (1001, 100, 1025)])
@pytest.mark.parametrize("nrhs", [1, 2, 4, 7])
def test_csr_hub_rows(dev, n, avg, length, nrhs):
    """Rows far longer than the average, with and without the x . Ax partials: right, and rounded like sums
    shared by a wave.  A lane adds length / 64 products, in pairs and batches; random signs let the errors
    of a sum grow like the root of its additions, so 2 sqrt(length / 64 + 8) units of sqrt(sum v^2 x^2)."""
    M, ptr, cols = hubs(n, avg, length, length)
    A = ca.Sparse.from_csr(*(torch.from_numpy(a).to(dev) for a in (ptr, cols, M.data)), (n, n))
    X = torch.from_numpy(np.random.RandomState(nrhs).randn(n, nrhs).astype(np.float32)).to(dev)
    X64 = X.double().cpu().numpy()
    M64 = M.astype(np.float64)
    err = (A @ X).double().cpu().numpy() - M64 @ X64
    size = np.sqrt(M64.multiply(M64) @ X64**2)
    for row in (0, n // 2 + 5, n - 1):
        assert (np.abs(err[row]) <= 6e-8 * 2 * np.sqrt(length / 64 + 8) * size[row]).all()
    assert (np.abs(err) <= 6e-8 * 12 * size).all() or length > 2000
    S = scipy.sparse.diags(np.asarray(abs(M64).sum(1)).ravel() + np.asarray(abs(M64).sum(0)).ravel() + 1.0) - (
        abs(M64) + abs(M64).T)
    S = S.tocsr().astype(np.float32)  # CG takes p . Ap from the product
    As = ca.Sparse.from_csr(*(torch.from_numpy(a).to(dev) for a in (S.indptr, S.indices, S.data)), (n, n))
    x = inv(ca.PSD(As), HipCG(tol=1e-6, max_iters=400)) @ X
    res = S.astype(np.float64) @ x.double().cpu().numpy() - X64
    assert (np.linalg.norm(res, axis=0) <= 4e-6 * np.linalg.norm(X64, axis=0)).all()


@pytest.mark.parametrize("avg,nrhs", [(40, 1), (90, 1), (120, 1), (120, 3), (120, 8)])
def test_csr_rounds_like_a_wave_a_row(dev, avg, nrhs):
    """The error of a whole product against that of 64 sums a row added as a tree (the mean over 20000 rows;
    its spread over matrices is below 1 %).  A lane's plain chain gives 1.03 to 1.45."""
    n, rs = 20000, np.random.RandomState(avg)
    M, ptr, cols = hubs(n, avg, avg, avg)
    A = ca.Sparse.from_csr(*(torch.from_numpy(a).to(dev) for a in (ptr, cols, M.data)), (n, n))
    X = rs.randn(n, nrhs).astype(np.float32)
    ref = M.astype(np.float64) @ X.astype(np.float64)
    err = lambda Y: np.linalg.norm(Y - ref)  # noqa: E731
    length = np.diff(ptr)
    k = np.arange(192)
    at = np.minimum(ptr[:-1, None] + k, ptr[1:, None] - 1)
    v = np.where(k < length[:, None], M.data[at], 0).astype(np.float64)
    assert length.max() <= 192
    ours = (A @ torch.from_numpy(X).to(dev)).double().cpu().numpy()
    wave = np.empty((n, nrhs))
    for b in range(nrhs):
        x = X[cols[at], b].astype(np.float64)
        s = np.zeros((n, 64), np.float32)
        for c in range(3):
            s = (s + v[:, 64 * c:64 * c + 64] * x[:, 64 * c:64 * c + 64]).astype(np.float32)
        while s.shape[1] > 1:
            s = s[:, ::2] + s[:, 1::2]
        wave[:, b] = s[:, 0]
    print(avg, nrhs, err(ours) / err(wave), flush=True)
    assert err(ours) < 1.025 * err(wave)


def test_csr_group_ignores_other_columns_nonfinite(dev):
    """Lanes past a row's end read its last entry again: an infinity there counts once, elsewhere not."""
    M = matrix(300, 12, 1)
    A = ca.Sparse.from_csr(torch.from_numpy(M.indptr).to(dev), torch.from_numpy(M.indices).to(dev),
                           torch.from_numpy(M.data).to(dev), (300, 300))
    x = torch.ones(300, 4)
    x[5] = float("inf")
    touches = torch.from_numpy((M[:, 5] != 0).toarray()[:, 0])
    y = (A @ x.to(dev)).cpu()
    assert bool(torch.isfinite(y[~touches]).all()) and bool(torch.isinf(y[touches]).all())


@pytest.mark.parametrize("n,avg,nrhs", [(2000, 12, 1), (2000, 12, 4), (1500, 200, 3), (140000, 12, 9)])
def test_cg_on_group_partials(dev, n, avg, nrhs):
    """CG's p . Ap from the product's epilogue: solutions against a 64-bit direct solve."""
    M = matrix(n, avg, 3)
    S = abs(M) + abs(M).T
    L = scipy.sparse.diags(np.asarray(S.sum(1)).ravel() + 1.0) - 0.5 * S
    L = L.tocsr().astype(np.float32)
    A = ca.Sparse.from_csr(torch.from_numpy(L.indptr).to(dev), torch.from_numpy(L.indices).to(dev),
                           torch.from_numpy(L.data).to(dev), (n, n))
    b = torch.from_numpy(np.random.RandomState(0).randn(n, nrhs).astype(np.float32)).to(dev)
    x = inv(ca.PSD(A), HipCG(tol=1e-6, max_iters=400)) @ b
    L64 = L.astype(np.float64)
    res = L64 @ x.cpu().double().numpy() - b.cpu().double().numpy()
    # tol * ||r0|| + tol on the recursive residual of a normalised column, plus rounding
    assert (np.linalg.norm(res, axis=0) <= 4e-6 * np.linalg.norm(b.cpu().double().numpy(), axis=0)).all()
