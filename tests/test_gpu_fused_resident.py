"""The persistent CG over several workgroups (rows in registers up to 3584 unknowns, read in every step
above) at the edges of its chunks of 512 columns, 16 or 20 rows a workgroup and 1 / 4 / 8 columns,
against FP64 and the chained launches; and concurrent solves of several threads."""
import importlib
import threading

import pytest
import torch

import cola_amd as ca
from cola_amd.linalg import run_batched_cg
from cola_amd.linalg.cg import fused_solve

pytestmark = pytest.mark.gpu

EPS = 2.0**-24


def rel(a, b):
    return float((a.double() - b.double()).norm() / b.double().norm())


def system(dev, n, seed, pad=0):
    g = torch.Generator(device=dev).manual_seed(seed)
    k = max(n // 4, 2)
    X = torch.randn(n, k, generator=g, device=dev)
    A = torch.zeros(n, n + pad, device=dev)[:, :n] if pad else torch.empty(n, n, device=dev)
    A.copy_(X @ X.T / k)
    A.diagonal().add_(0.3)
    return A, g


@pytest.mark.parametrize("n,B,nblocks", [(7, 8, 0), (15, 5, 0), (16, 6, 2), (17, 1, 17), (321, 1, 0), (257, 2, 0), (511, 3, 0),
                                         (512, 8, 0), (513, 5, 0), (1023, 4, 256), (1024, 7, 0), (1537, 2, 0), (2048, 8, 0),
                                         (2049, 4, 0), (2561, 3, 0), (3072, 4, 0), (3073, 1, 0), (3584, 4, 0), (3585, 1, 0),
                                         (4100, 1, 0), (7168, 1, 0)])
def test_resident(dev, n, B, nblocks):
    """||A|| <= 9.4 and cond(A) <= 32: stopped at 1e-6 of the residual, with the recursive residual within
    n EPS ||A|| of the true one, the solution is within cond * (2e-6 + n EPS) of FP64's."""
    A, g = system(dev, n, n + B, pad=n % 3)
    b = torch.randn(B, n, generator=g, device=dev).T
    Ad = A.double()
    sol = torch.linalg.solve(Ad, b.double())
    bound = 32 * (2e-6 + n * EPS)
    x, r, k, info = fused_solve(ca.Dense(A), b, None, 300, 1e-6, None, nblocks=nblocks)
    xc, rc, kc, ic = run_batched_cg(ca.Dense(A), b, None, 300, 1e-6, None, fused=False)
    print(n, B, nblocks, k, kc, rel(x, sol), rel(xc, sol), flush=True)
    assert info["status"] == ic["status"] == "ok" and info["fused"] and not ic["fused"]
    assert abs(k - kc) <= 2 and rel(x, sol) < bound and rel(xc, sol) < bound
    assert float((b.double() - Ad @ x.double() - r.double()).norm() / b.double().norm()) < 20 * n * EPS
    d = torch.rand(n, generator=g, device=dev) + 0.5
    x0 = 0.1 * torch.randn(n, B, generator=g, device=dev) / n**0.5  # A x0 of the size of a normalised column
    op = ca.Dense(A) * 2.0 + 0.25 * ca.I_like(ca.Dense(A))
    x, r, k, info = fused_solve(op, b, x0, 300, 1e-6, ca.Diagonal(d), nblocks=nblocks)
    Aop = 2.0 * Ad + 0.25 * torch.eye(n, device=dev, dtype=torch.float64)
    sol = torch.linalg.solve(Aop, b.double())
    # ||Aop|| <= 19, cond <= 23: ||r0|| <= 3, so the recursive residual ends below 4e-6; the true one differs
    # by roundings of random sign, a few sqrt(n) EPS ||Aop|| over the steps
    print(n, B, nblocks, "pre", k, rel(x, sol), flush=True)
    assert info["status"] == "ok" and rel(x, sol) < 23 * (4e-6 + 4 * n**0.5 * EPS)
    assert float((b.double() - Aop @ x.double() - r.double()).norm() / b.double().norm()) < 40 * n**0.5 * EPS


def test_limits(dev):
    for n, B in ((3585, 2), (7169, 1), (2049, 5), (64, 9)):
        A = torch.eye(n, device=dev)
        assert fused_solve(ca.Dense(A), torch.ones(n, B, device=dev)) is None


def test_threads(dev):
    """Eight threads with a stream each: the workgroups of their solves never exceed the device."""
    n, out = 2500, {}
    A, g = system(dev, n, 5)
    bs = [torch.randn(n, 2, generator=g, device=dev) for _ in range(8)]
    sol = torch.linalg.solve(A.double(), torch.cat(bs, 1).double())
    importlib.import_module("cola_amd.linalg.cg")._WORKGROUPS.clear()  # all threads ask for the device's CUs at once
    torch.cuda.synchronize()

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(3):
                out[i] = run_batched_cg(ca.Dense(A), bs[i], None, 300, 1e-6, None)
            torch.cuda.current_stream().synchronize()

    ts = [threading.Thread(target=work, args=(i, )) for i in range(8)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    for i in range(8):
        x, _, _, info = out[i]
        assert info["fused"] and info["status"] == "ok"
        assert rel(x, sol[:, 2 * i:2 * i + 2]) < 32 * (2e-6 + n * EPS)


@pytest.mark.parametrize("n", [64, 600])
def test_threads_on_the_default_stream(dev, n):
    """Six threads on one stream, equal shapes, right-hand sides of 1 to 6 eigenvectors: each solve reports
    its own steps (exactly as many in a diagonal system with that many distinct eigenvalues)."""
    A = torch.diag(torch.linspace(1, 2, n, device=dev))
    bs = torch.zeros(6, n, 1, device=dev)
    for i in range(6):
        bs[i, torch.arange(i + 1) * (n // 7)] = 1.0
    torch.cuda.synchronize()
    want = [run_batched_cg(ca.Dense(A), b, None, 100, 1e-5, None)[2] for b in bs]
    assert want == sorted(set(want)) and want[0] == 1
    got = {}

    def work(i):
        for _ in range(20):
            x, _, k, info = run_batched_cg(ca.Dense(A), bs[i], None, 100, 1e-5, None)
            got.setdefault(i, []).append((k, info["status"], rel(x, bs[i] / A.diagonal()[:, None]) < 1e-4))

    ts = [threading.Thread(target=work, args=(i, )) for i in range(6)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert got == {i: [(want[i], "ok", True)] * 20 for i in range(6)}
