"""The training kernels at the edges of their tiles: the network's forward and backward passes (16 and
64 points per block, 16-wide tiles of inputs and outputs, strided outputs), the small SPD inverse (two
pivots per step, orders odd and even, batches), the loss factors and the tall-skinny product."""
import numpy as np
import pytest
import torch

from cola_amd import _native as N
from cola_amd.linalg import PointMLP
from cola_amd.linalg import learned as L

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float((a.double().cpu() - b.double().cpu()).norm() / b.double().norm().clamp_min(1e-300))


@pytest.mark.parametrize("n", [1, 3, 15, 16, 17, 63, 65, 130, 4161])
@pytest.mark.parametrize("din,dout", [(1, 1), (3, 15), (4, 64), (5, 17), (7, 65), (8, 128), (4, 33)])
def test_mlp_edges(dev, n, din, dout):
    g = torch.Generator().manual_seed(n * 131 + dout)
    rs = np.random.RandomState(n + dout)
    net = PointMLP(din, dout, device=dev, params=(rs.randn(int(N.q("ck_mlp_param_count", din, dout))) * 0.3).astype(
        np.float32))
    X = torch.randn(n, din, generator=g)
    G, Z1, Z2 = net.forward(X.to(dev), save=True)
    dG = torch.full((dout, G.shape[1]), float("nan"))
    dG[:, :n] = torch.randn(dout, n, generator=g)  # what pads a column block is never read
    Z1[:, n:] = Z2[:, n:] = float("nan")
    grad = net.backward(X.to(dev), Z1, Z2, dG.to(dev), scale=0.5)
    sizes = [din * 128, 128, 128 * 128, 128, 128 * dout, dout]
    P = [p.double().cpu().requires_grad_(True) for p in torch.split(net.params, sizes)]
    act = torch.nn.functional.gelu
    z1 = X.double() @ P[0].view(din, 128) + P[1]
    z2 = act(z1) @ P[2].view(128, 128) + P[3]
    out = act(z2) @ P[4].view(128, dout) + P[5]
    ref = 0.5 * torch.cat([q.reshape(-1) for q in torch.autograd.grad((out * dG[:, :n].T.double()).sum(), P)])
    # sums of at most 128 products and a few roundings of the activations, 6e-8 each, on unit scales
    assert rel(Z1[:, :n].T, z1) < 1e-6 and rel(Z2[:, :n].T, z2) < 2e-6 and rel(G[:, :n].T, out) < 2e-6
    assert rel(grad, ref) < 3e-6


def _chain(acc, x, w):
    """acc[i, j] + sum_k x[i, k] w[k, j] in fp32, k ascending, one fma a term (a product of two fp32 numbers
    is exact in 64 bits)."""
    acc = np.broadcast_to(acc, (x.shape[0], w.shape[1])).astype(np.float32)
    for k in range(x.shape[1]):
        acc = (acc.astype(np.float64) + x[:, k:k + 1].astype(np.float64) * w[k:k + 1].astype(np.float64)).astype(
            np.float32)
    return acc


@pytest.mark.parametrize("n,din,dout", [(150, 5, 37), (64, 8, 64), (17, 1, 128)])
def test_mlp_sums_in_index_order(dev, n, din, dout):
    """Every sum starts from its bias and adds its terms in index order.  At arguments of 20 and more GELU is
    the identity and its derivative one to the bit, so the whole pass can be restated exactly."""
    rs = np.random.RandomState(n)
    f = lambda *s: rs.randn(*s).astype(np.float32)  # noqa: E731
    W1, W2, W3, b3 = 0.3 * f(din, 128), 0.05 * f(128, 128), f(128, dout), f(dout)
    b1, b2 = 30 + f(128), 300 + f(128)
    X, dG = rs.rand(n, din).astype(np.float32), f(n, dout)
    net = PointMLP(din, dout, device=dev, params=np.concatenate([a.reshape(-1) for a in (W1, b1, W2, b2, W3, b3)]))
    Xd = torch.from_numpy(X).to(dev)
    G, Z1, Z2 = net.forward(Xd, save=True)
    z1 = _chain(b1, X, W1)
    z2 = _chain(b2, z1, W2)
    assert z1.min() > 20 and z2.min() > 20
    for got, want in ((Z1, z1), (Z2, z2), (G, _chain(b3, z2, W3))):
        assert np.array_equal(got[:, :n].cpu().numpy().T, want)
    d = torch.zeros(dout, G.shape[1])
    d[:, :n] = torch.from_numpy(dG.T.copy())
    grad = net.backward(Xd, Z1, Z2, d.to(dev), scale=1.0)
    dz2 = _chain(np.float32(0), dG, W3.T)
    dz1 = _chain(np.float32(0), dz2, W2.T)
    total, zero, one = 0.0, np.float32(0), np.ones((1, n), np.float32)
    for p in range(0, n, 64):  # a chunk's sums in fp32, the chunks' in fp64
        c = slice(p, p + 64)
        parts = [(X.T[:, c], dz1[c]), (one[:, c], dz1[c]), (z1.T[:, c], dz2[c]), (one[:, c], dz2[c]),
                 (z2.T[:, c], dG[c]), (one[:, c], dG[c])]
        total = total + np.concatenate([_chain(zero, a, b).astype(np.float64).reshape(-1) for a, b in parts])
    assert np.array_equal(grad.cpu().numpy(), total.astype(np.float32))


def test_mlp_row_major_output(dev):
    """Outputs and their gradient by rows, no saved pre-activations: the same numbers."""
    n, din, dout = 100, 4, 40
    net = PointMLP(din, dout, device=dev, seed=3)
    X = torch.rand(n, din, generator=torch.Generator().manual_seed(1)).to(dev)
    G, Z1, Z2 = net.forward(X, save=True)
    R = torch.empty(n, dout + 3, device=dev)
    N.call("ck_mlp_forward", n, din, dout, N.ptr(X), din, N.ptr(net.params), N.ptr(R), dout + 3, 1, None, None, 0,
           N.stream_ptr(dev))
    assert torch.equal(R[:, :dout], G[:, :n].T)
    dR = torch.randn(n, dout, generator=torch.Generator().manual_seed(2)).to(dev)
    dC = torch.zeros_like(G)
    dC[:, :n] = dR.T
    wb = N.q("ck_mlp_grad_workspace_bytes", n, din, dout)
    work, grad = torch.empty(wb // 4, device=dev), torch.empty_like(net.params)
    N.call("ck_mlp_backward", n, din, dout, N.ptr(X), din, N.ptr(net.params), N.ptr(Z1), N.ptr(Z2), Z1.stride(0),
           N.ptr(dR), dout, 1, 1.0, N.ptr(grad), N.ptr(work), wb, N.stream_ptr(dev))
    assert torch.equal(grad, net.backward(X, Z1, Z2, dC))


@pytest.mark.parametrize("k", [1, 2, 3, 5, 16, 31, 32, 33, 47, 63, 64])
def test_spd_inverse_orders(dev, k):
    rs = np.random.RandomState(k)
    mats, batch = [], 3
    for _ in range(batch):
        Q = rs.randn(k, k)
        mats.append(Q @ Q.T / k + 0.1 * np.eye(k))
    lda = k + 2
    A = np.full((batch, k, lda), np.nan)
    A[:, :, :k] = np.stack([np.tril(M) + np.triu(np.full((k, k), np.nan), 1) for M in mats])  # the lower triangle is read
    Ad = torch.from_numpy(A).to(dev)
    f64 = lambda: torch.empty(batch, k, k, dtype=torch.float64, device=dev)  # noqa: E731
    linv, inv, st = f64(), f64(), torch.full((batch, ), 9, dtype=torch.int32, device=dev)
    inv32, lT = torch.empty(batch, k, k, device=dev), torch.empty(batch, k, k, device=dev)
    N.call("ck_spd_inverse_f64", batch, k, N.ptr(Ad), lda, k * lda, 0.01, 0.05, N.ptr(linv), N.ptr(inv), N.ptr(inv32),
           N.ptr(lT), N.ptr(st), N.stream_ptr(dev))
    assert st.tolist() == [0] * batch
    for b, M in enumerate(mats):
        S = M + (0.05 + 0.01 * np.trace(M) / k) * np.eye(k)
        Li = np.linalg.inv(np.linalg.cholesky(S))
        cond = np.linalg.cond(S)
        tol = 1e-15 * cond * (k + 4)  # backward stable: k roundings times the condition number
        assert np.linalg.norm(linv[b].cpu().numpy() - Li) <= tol * np.linalg.norm(Li)
        assert np.linalg.norm(inv[b].cpu().numpy() - np.linalg.inv(S)) <= tol * np.linalg.norm(np.linalg.inv(S))
        assert torch.equal(inv32[b], inv[b].float()) and torch.equal(lT[b], linv[b].T.float())


@pytest.mark.parametrize("scale,e", [(1.0, 100), (1e-291, 100), (1e291, 511)])
def test_spd_inverse_divides(dev, scale, e):
    """[[p, a], [a, 4^e]] with a^2 / p below half a unit of 4^e: the inverse factor's (1, 0) entry is -a / p
    scaled by 2^-e, rounded once."""
    rs, n = np.random.RandomState(5), 4096
    p, a = scale * (1 + rs.rand(n)), scale * rs.rand(n)
    A = np.zeros((n, 2, 2))
    A[:, 0, 0], A[:, 1, 0], A[:, 1, 1] = p, a, 4.0**e
    f64 = lambda: torch.empty(n, 2, 2, dtype=torch.float64, device=dev)  # noqa: E731
    Ad, linv, st = torch.from_numpy(A).to(dev), f64(), torch.empty(n, dtype=torch.int32, device=dev)
    N.call("ck_spd_inverse_f64", n, 2, N.ptr(Ad), 2, 4, 0.0, 0.0, N.ptr(linv), None, None, None, N.ptr(st),
           N.stream_ptr(dev))
    assert not st.any()
    assert np.array_equal(linv[:, 1, 0].cpu().numpy(), -(a / p) * 2.0**-e)


@pytest.mark.parametrize("k,bad", [(7, 0), (7, 3), (8, 7), (33, 32), (64, 41)])
def test_spd_inverse_reports_the_failing_pivot(dev, k, bad):
    A = np.eye(k)
    A[bad, bad] = -1.0
    with pytest.raises(np.linalg.LinAlgError, match=f"pivot {bad}"):
        L.spd_inverse(torch.from_numpy(A).to(dev))


@pytest.mark.parametrize("k,m", [(1, 1), (5, 64), (64, 3), (33, 47), (64, 64)])
def test_energy_factors(dev, k, m):
    rs = np.random.RandomState(k * 100 + m)
    Q, T, w = rs.randn(k, k), rs.randn(m, k), rs.rand(m)
    S = np.linalg.inv(Q @ Q.T / k + np.eye(k))
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    C1, C2 = torch.empty(m, k, device=dev), torch.empty(k, k, device=dev)
    loss = torch.empty(1, dtype=torch.float64, device=dev)
    Sd, Td, wd = t(S), t(T), t(w)
    N.call("ck_energy_loss_f64", k, m, N.ptr(Sd), N.ptr(Td), N.ptr(wd), N.ptr(C1), N.ptr(C2), N.ptr(loss),
           N.stream_ptr(dev))
    P, c = T @ S, 2 / w.sum()
    assert abs(float(loss) - (1 - (w[:, None] * P * T).sum() / w.sum())) < 1e-12 * (1 + np.abs(P * T).sum())
    # rounded once to 32 bits
    assert np.allclose(C1.cpu().numpy(), -c * w[:, None] * P, rtol=1e-6, atol=1e-9)
    assert np.allclose(C2.cpu().numpy(), c * P.T @ (w[:, None] * P), rtol=1e-6, atol=1e-6 * np.abs(P).max()**2)


@pytest.mark.parametrize("n,kin,kout", [(1, 1, 1), (63, 64, 33), (65, 65, 31), (1000, 128, 64), (130, 3, 70)])
@pytest.mark.parametrize("by_rows", [True, False])
def test_rows_gemm(dev, n, kin, kout, by_rows):
    g = torch.Generator().manual_seed(n + kin)
    X, W, Y = torch.randn(n, kin, generator=g), torch.randn(kin, kout, generator=g), torch.randn(n, kout, generator=g)
    Xd = X.to(dev) if by_rows else X.T.contiguous().to(dev)
    Yd = Y.to(dev) if by_rows else Y.T.contiguous().to(dev)
    xs, ys = ((kin, 1), (kout, 1)) if by_rows else ((1, n), (1, n))
    L.rows_gemm(Xd, *xs, W.to(dev), Yd, *ys, n, alpha=0.5, beta=2.0)
    out = Yd if by_rows else Yd.T
    ref = 0.5 * X.double() @ W.double() + 2.0 * Y.double()
    mag = 0.5 * X.abs().double() @ W.abs().double() + 2.0 * Y.abs().double()
    assert bool(((out.cpu().double() - ref).abs() <= 6e-8 * (kin + 3) * mag).all())
