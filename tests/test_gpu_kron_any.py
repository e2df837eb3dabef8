"""Kronecker products with factors of any order up to 64 (kron_any.hip): orders on both sides of the
16-wide tiles and below the 4-wide loads, planes of odd and single width, several slabs per block, and
the X . Y partials that CG and Lanczos take from the second pass."""
import pytest
import torch

import cola_amd as ca
from cola_amd import _native as N
from cola_amd._blocks import ld_of
from cola_amd.linalg import HipCG, HipLanczos, inv, log

pytestmark = pytest.mark.gpu


def factors(dims, g, spd=False):
    out = []
    for d in dims:
        A = torch.randn(d, d, generator=g)
        out.append((A @ A.T / d + 0.2 * torch.eye(d)) if spd else A)
    return out


def kron64(fs, X):
    V = X.double().reshape(*[f.shape[0] for f in fs], -1)
    for i, f in enumerate(fs):
        V = torch.movedim(torch.tensordot(f.double(), V, dims=([1], [i])), 0, i)
    return V.reshape(X.shape)


DIMS = [(1, 1, 1), (2, 3, 5), (3, 1, 1), (1, 4, 3), (5, 1, 7), (16, 16, 16), (17, 15, 33), (31, 48, 49), (63, 64, 62), (64, 17, 1),
        (48, 2, 64), (64, 64, 63), (3, 1), (1, 1), (16, 50), (63, 33), (64, 64)]


@pytest.mark.parametrize("dims", DIMS)
@pytest.mark.parametrize("nrhs", [1, 3])
def test_kron_any_product(dev, dims, nrhs):
    g = torch.Generator().manual_seed(sum(dims) + nrhs)
    fs = factors(dims, g)
    n = 1
    for d in dims:
        n *= d
    X = torch.randn(n, nrhs, generator=g)
    K = ca.Kronecker(*[ca.Dense(f.to(dev)) for f in fs])
    op, keep = K.hip_op()
    op.scale, op.shift = 0.5, 2.0
    ld = ld_of(n) + 64
    Xb = torch.full((nrhs, ld), float("nan"), device=dev)  # what lies past a vector is never used
    Xb[:, :n] = X.T.to(dev)
    Yb = torch.full_like(Xb, -7.0)
    wb = N.q("ck_op_workspace_bytes", op, nrhs)
    work = torch.full((max(wb, 4) // 4, ), float("nan"), device=dev)
    N.call("ck_op_apply", op, nrhs, N.ptr(Xb), ld, N.ptr(Yb), ld, N.ptr(work), wb, N.stream_ptr(dev))
    ref = 0.5 * kron64(fs, X) + 2.0 * X.double()
    mag = 0.5 * kron64([f.abs() for f in fs], X.abs()) + 2.0 * X.abs().double()
    err = (Yb[:, :n].T.double().cpu() - ref).abs()
    assert bool((err <= 6e-8 * (sum(dims) + 8) * mag + 1e-30).all())  # the sums' roundings
    assert bool((Yb[:, n:] == -7.0).all())


@pytest.mark.parametrize("dims,factor", [(d, f) for d in ((3, 20, 17), (20, 5, 4), (4, 3, 50), (33, 64, 20), (20, 7), (1, 60))
                                         for f in range(len(d))])
def test_kron_any_infinite_entry(dev, dims, factor):
    """One infinite entry of a factor, everything else positive: infinite where it enters, finite elsewhere
    (the padding to 16 is zeros times the other operand, whatever that holds)."""
    g = torch.Generator().manual_seed(sum(dims))
    fs = [torch.rand(d, d, generator=g) + 0.1 for d in dims]
    at = dims[factor] - 1
    fs[factor][at, 0] = float("inf")
    X = torch.rand(torch.Size(dims).numel(), 2, generator=g) + 0.1
    Y = (ca.Kronecker(*[ca.Dense(f.to(dev)) for f in fs]) @ X.to(dev)).cpu().reshape(*dims, 2)
    hit = torch.zeros(*dims, 2, dtype=torch.bool)
    hit.select(factor, at).fill_(True)
    assert bool((torch.isposinf(Y) == hit).all()) and bool((torch.isfinite(Y) == ~hit).all())


def test_kron_any_many_slabs(dev):
    """Enough slabs that a block walks several of them, the last block fewer."""
    dims, nrhs = (63, 18, 20), 53
    g = torch.Generator().manual_seed(0)
    fs = factors(dims, g)
    X = torch.randn(63 * 18 * 20, nrhs, generator=g)
    out = ca.Kronecker(*[ca.Dense(f.to(dev)) for f in fs]) @ X.to(dev)
    ref = kron64(fs, X)
    assert float((out.double().cpu() - ref).norm() / ref.norm()) < 1e-6


def test_kron_any_padding_reads_no_neighbour(dev):
    """The rows and columns that pad an operand to 16 are zeros, not what lies next to it in memory: an
    infinite vector leaves its neighbours on both sides finite."""
    dims = (3, 17, 18)
    g = torch.Generator().manual_seed(5)
    fs = factors(dims, g)
    X = torch.randn(3 * 17 * 18, 3, generator=g)
    X[:, 1] = float("inf")
    y = (ca.Kronecker(*[ca.Dense(f.to(dev)) for f in fs]) @ X.to(dev)).cpu()
    assert bool(torch.isfinite(y[:, [0, 2]]).all())


@pytest.mark.parametrize("dims,nrhs", [((20, 30, 25), 1), ((5, 33, 40), 4), ((48, 17, 31), 33), ((30, 40), 3)])
def test_cg_and_lanczos_on_any_orders(dev, dims, nrhs):
    g = torch.Generator().manual_seed(2)
    fs = factors(dims, g, spd=True)
    n = 1
    for d in dims:
        n *= d
    K = ca.Kronecker(*[ca.Dense(f.to(dev)) for f in fs])
    A = K + 1.0 * ca.I_like(K)
    b = torch.randn(n, nrhs, generator=g)
    x = inv(ca.PSD(A), HipCG(tol=1e-6, max_iters=500)) @ b.to(dev)
    xc = x.cpu().double()
    res = kron64(fs, xc) + xc - b.double()
    assert bool((res.norm(dim=0) <= 5e-6 * b.double().norm(dim=0)).all())
    w, Q = zip(*[torch.linalg.eigh(f.double()) for f in fs])
    lam = w[0]
    for v in w[1:]:
        lam = (lam[:, None] * v[None, :]).reshape(-1)
    ref = kron64(list(Q), torch.log(lam + 1.0)[:, None] * kron64([q.T for q in Q], b.double()))
    out = log(ca.SelfAdjoint(A), HipLanczos(max_iters=40, tol=1e-7)) @ b.to(dev)
    # 40 steps resolve log on these spectra to about 1e-5
    assert float((out.cpu().double() - ref).norm() / ref.norm()) < 1e-4
