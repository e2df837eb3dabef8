"""The on-the-fly stationary kernel product (CK_OP_RBF_F32) at the edges of its tiles: 128 rows per
block, 256 columns per staged tile split over four waves, up to 8 rhs per pass, dimensions rounded
up to a template size, with the columns split over blocks (workspace) and not (none)."""
import math

import pytest
import torch

import cola_amd as ca
from cola_amd import _native as N
from cola_amd._blocks import ld_of

pytestmark = pytest.mark.gpu

FNS = ("rbf", "matern12", "matern32", "matern52")


def reference(fam, X, V, ell):
    d2 = ((X[:, None, :] - X[None, :, :])**2).sum(-1)
    r = d2.sqrt()
    if fam == 0:
        K = torch.exp(-d2 / (2 * ell * ell))
    elif fam == 1:
        K = torch.exp(-r / ell)
    else:
        a = (3.0 if fam == 2 else 5.0)**0.5 * r / ell
        K = ((1 + a) if fam == 2 else (1 + a + a * a / 3)) * torch.exp(-a)
    return K @ V, K.abs() @ V.abs()


@pytest.mark.parametrize("n,dim,nrhs", [(1, 1, 1), (63, 2, 2), (64, 3, 3), (127, 4, 4), (129, 5, 5), (255, 6, 7), (257, 7, 8),
                                        (513, 8, 9), (1025, 3, 17)])
@pytest.mark.parametrize("fam", [0, 1, 2, 3])
@pytest.mark.parametrize("split", [True, False])
def test_stationary_product_edges(dev, n, dim, nrhs, fam, split):
    g = torch.Generator().manual_seed(100 * fam + n)
    ldp, ell = dim + 3, 0.4
    pts = torch.randn(n, ldp, generator=g)
    V = torch.randn(n, nrhs, generator=g)
    ref, mag = reference(fam, pts[:, :dim].double(), V.double(), ell)
    ref = 1.5 * ref - 0.25 * V.double()
    Pd = pts.to(dev)
    ld = ld_of(n)
    Xb = torch.full((nrhs, ld), float("nan"), device=dev)  # padding is never read
    Xb[:, :n] = V.T.to(dev)
    Yb = torch.empty_like(Xb)
    op = N.CkOp()
    op.kind, op.n, op.scale, op.shift = N.CK_OP_RBF_F32, n, 1.5, -0.25
    op.a, op.lda, op.dim, op.aux_f, op.rank = Pd.data_ptr(), ldp, dim, ell, fam
    wb = N.q("ck_op_workspace_bytes", op, nrhs)
    assert (wb > 0) == (n > 256)
    work = torch.empty(max(wb, 4) // 4, device=dev) if split else None
    N.call("ck_op_apply", op, nrhs, N.ptr(Xb), ld, N.ptr(Yb), ld, N.ptr(work), wb if split else 0, N.stream_ptr(dev))
    err = (Yb[:, :n].T.double().cpu() - ref).abs()
    # an entry's relative error: 2u per squared difference and its sum, halved by the root, times the
    # exponent |t| < 12 at these distances (about 60 u); the sums add n u / 4 at most
    bound = 6e-8 * (60 + n / 4) * (1.5 * mag + 0.25 * V.double().abs()) + 1e-30
    assert bool((err <= bound).all())


def test_stationary_product_repeats_bitwise(dev):
    g = torch.Generator().manual_seed(1)
    X, V = torch.rand(3000, 3, generator=g).to(dev), torch.randn(3000, 4, generator=g).to(dev)
    A = ca.ops.Kernel(X, X, ca.ops.matern52(0.3), 1024, 1024)
    assert torch.equal(A @ V, A @ V)


@pytest.mark.parametrize("fam", [0, 1, 2, 3])
@pytest.mark.parametrize("dim,nrhs,n", [(1, 1, 203), (3, 4, 203), (3, 4, 600)])
def test_stationary_subnormal_entries(dev, fam, dim, nrhs, n):
    """Columns of K itself, from 2^-100 down to the last subnormal: the exponent t is rounded a few times at
    |t| <= 110 (1e-5 of an entry), a subnormal once or twice by 2^-149."""
    ell = 0.4
    t = torch.linspace(70.0, 108.0, n - 1, dtype=torch.float64)  # -log of the exponential
    t[:80] = 126 * math.log(2) * (1 + torch.linspace(-2e-6, 2e-6, 80, dtype=torch.float64))  # around the last normal one
    root = 3.0**0.5 if fam == 2 else 5.0**0.5 if fam == 3 else 1.0
    r = ell * ((2 * t).sqrt() if fam == 0 else t / root)
    pts = torch.zeros(n, dim)
    pts[1:, dim - 1] = r.float()
    V = torch.zeros(n, nrhs)
    V[0] = 1.0
    ref, _ = reference(fam, pts.double(), V.double(), float(torch.tensor(ell)))
    fn = (ca.ops.rbf, ca.ops.matern12, ca.ops.matern32, ca.ops.matern52)[fam](ell)
    Pd = pts.to(dev)
    out = (ca.ops.Kernel(Pd, Pd, fn, 1024, 1024) @ V.to(dev)).cpu().double()
    assert bool(((out - ref).abs() <= 2e-5 * ref + 3e-45).all())
    assert bool((out[1:81] > 0).all(dim=0)[0])
    assert float((out[1:, 0] > 0).double().mean()) > 0.9 * float((ref[1:, 0] > 1.5e-45).double().mean())


@pytest.mark.parametrize("fam", [1, 2, 3])
def test_stationary_subnormal_distances(dev, fam):
    """Squared distances around 1e-39, with a lengthscale to match."""
    g = torch.Generator().manual_seed(fam)
    pts, V, ell = torch.rand(300, 2, generator=g) * 6e-20, torch.randn(300, 2, generator=g), 3e-20
    ref, mag = reference(fam, pts.double(), V.double(), float(torch.tensor(ell)))
    fn = (None, ca.ops.matern12, ca.ops.matern32, ca.ops.matern52)[fam](ell)
    Pd = pts.to(dev)
    out = (ca.ops.Kernel(Pd, Pd, fn, 1024, 1024) @ V.to(dev)).cpu().double()
    assert bool(((out - ref).abs() <= 1e-3 * mag).all())
