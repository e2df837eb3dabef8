"""Dense products at any order, leading dimension and 4-byte alignment: fp32 with 1 to 33 rhs at the
edges of the 4-column pieces, the 1024-column chunks and the 8/16/32-row blocks; the X . Y partials that
CG takes from the epilogue; and the FP64-accumulating product of the refinement residuals."""
import ctypes

import pytest
import torch

import cola_amd as ca
from cola_amd import _native as N
from cola_amd.linalg import HipCG, HipMixedCG, PivotedCholeskyPreconditioner, inv

pytestmark = pytest.mark.gpu


def problem(n, lda, off, nrhs, dev, dtype=torch.float32):
    """A (n, n) at element `off` of a buffer with leading dimension lda; what lies between rows is NaN."""
    g = torch.Generator().manual_seed(n * 7 + nrhs)
    A, X = torch.randn(n, n, generator=g), torch.randn(n, nrhs, generator=g)
    buf = torch.full((off + n * lda + 3, ), float("nan"))
    torch.as_strided(buf, (n, n), (lda, 1), off).copy_(A)
    buf = buf.to(dev)
    ldx = n + 3
    Xb = torch.full((nrhs, ldx), float("nan"), dtype=dtype)
    Xb[:, :n] = X.T.to(dtype)
    return A.double(), X.double(), buf, Xb.to(dev), ldx


@pytest.mark.parametrize("n,pad,off", [(1, 0, 0), (2, 1, 1), (3, 0, 3), (5, 2, 0), (31, 0, 1), (257, 0, 0), (1023, 1, 2),
                                       (1025, 0, 0), (1028, 0, 1), (2051, 0, 3), (4097, 3, 0), (4200, 0, 0), (8195, 0, 1)])
@pytest.mark.parametrize("nrhs", [1, 2, 3, 5, 9, 33])
def test_dense_any_alignment(dev, n, pad, off, nrhs):
    A, X, buf, Xb, ldx = problem(n, n + pad, off, nrhs, dev)
    Yb = torch.full((nrhs, ldx), -7.0, device=dev)
    op = N.CkOp()
    op.kind, op.n, op.scale, op.shift = N.CK_OP_DENSE_F32, n, 0.5, 2.0
    op.a, op.lda = buf.data_ptr() + 4 * off, n + pad
    N.call("ck_op_apply", op, nrhs, N.ptr(Xb), ldx, N.ptr(Yb), ldx, None, 0, N.stream_ptr(dev))
    ref = 0.5 * (A @ X) + 2.0 * X
    mag = 0.5 * (A.abs() @ X.abs()) + 2.0 * X.abs()
    err = (Yb[:, :n].T.double().cpu() - ref).abs()
    # a lane adds n / 64 products one after another, the wave's sums add 10 more roundings
    assert bool((err <= 6e-8 * (n / 64 + 16) * mag).all())
    assert bool((Yb[:, n:] == -7.0).all())


@pytest.mark.parametrize("n,pad,off", [(3, 1, 1), (511, 0, 1), (513, 0, 0), (1030, 3, 2)])
@pytest.mark.parametrize("nrhs", [1, 8, 11])
def test_dense_f64acc_any_alignment(dev, n, pad, off, nrhs):
    A, X, buf, Xb, ldx = problem(n, n + pad, off, nrhs, dev, torch.float64)
    Yb = torch.empty((nrhs, ldx), dtype=torch.float64, device=dev)
    N.call("ck_dense_apply_f64acc", n, ctypes.c_void_p(buf.data_ptr() + 4 * off), n + pad, 0.5, 2.0, nrhs, N.ptr(Xb),
           ldx, N.ptr(Yb), ldx, N.stream_ptr(dev))
    ref = 0.5 * (A @ X) + 2.0 * X
    assert float((Yb[:, :n].T.cpu() - ref).norm() / ref.norm()) < 1e-14


@pytest.mark.parametrize("n", [3, 131, 257, 513, 516, 1030])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_dense_products_infinite_entry(dev, n, dtype):
    """An infinite entry in any column of its row, everything else positive: that row is infinite (and no NaN),
    the others finite, at one and several rhs (lanes past a row's end may read its last entries again)."""
    for col in {0, n - 1, n // 2, max(n - 4, 0), n - n % 4 - 1}:
        A = torch.rand(n, n, device=dev) + 0.1
        A[n - 2, col] = float("inf")
        for nrhs in (1, 2, 5, 8):
            X = torch.rand(n, nrhs, device=dev, dtype=dtype) + 0.1
            if dtype == torch.float32:
                Y = ca.Dense(A) @ X
            else:
                Xb, Yb = X.T.contiguous(), torch.empty(nrhs, n, device=dev, dtype=dtype)
                N.call("ck_dense_apply_f64acc", n, N.ptr(A), n, 1.0, 0.0, nrhs, N.ptr(Xb), n, N.ptr(Yb), n,
                       N.stream_ptr(dev))
                Y = Yb.T
            hit = torch.zeros_like(Y, dtype=torch.bool)
            hit[n - 2] = True
            assert bool((torch.isposinf(Y) == hit).all()) and bool((torch.isfinite(Y) == ~hit).all()), (col, nrhs)


@pytest.mark.parametrize("n,nrhs", [(2047, 4), (2049, 3), (4099, 8), (8201, 5)])
def test_cg_on_odd_orders(dev, n, nrhs):
    """Chained CG with p . Ap from the dense epilogue, and the fused Woodbury step of a refined solve."""
    g = torch.Generator().manual_seed(n)
    P = torch.rand(n, 3, generator=g).to(dev)
    d2 = sum((P[:, c, None] - P[None, :, c])**2 for c in range(3))
    K = ca.Dense(torch.exp(-d2 / (2 * 0.3**2)))
    A = ca.PSD(K + 0.5 * ca.I_like(K))
    b = torch.randn(n, nrhs, generator=g).to(dev)
    A64 = K.A.double()
    A64.diagonal().add_(0.5)

    def res(x):
        return float(((A64 @ x.double() - b.double()).norm(dim=0) / b.double().norm(dim=0)).max())

    assert res(inv(A, HipCG(tol=1e-5, max_iters=400, fused=False)) @ b) < 1e-3  # kappa ~ n / 5 at tol 1e-5
    P64 = PivotedCholeskyPreconditioner(K, 64, 0.5)
    solver = inv(A, HipMixedCG(tol=1e-9, P=P64))
    assert res(solver @ b) < 2e-9
    assert max(solver.info["inner_iterations"]) < 100
