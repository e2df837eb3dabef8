"""The fused Gram-Schmidt update and projection that reads the basis once (up to 128 columns, four
register layouts) and the two-sweep kernel beyond: bases that cross every line of the dispatch, vectors
of whole and of partial 1024-row tiles, padding that is never a number."""
import numpy as np
import pytest
import torch

import cola_amd as ca
from cola_amd import _native as N
from cola_amd.linalg._engine import lower
from cola_amd.linalg.lanczos import LanczosRun

pytestmark = pytest.mark.gpu


def lanczos64(d, s, m):
    q, Q, al, be = s / np.linalg.norm(s), [], [], []
    for _ in range(m):
        Q.append(q)
        w = d * q
        al.append(w @ q)
        for _ in range(2):
            B = np.stack(Q)
            w = w - B.T @ (B @ w)
        be.append(np.linalg.norm(w))
        q = w / be[-1]
    return np.array(al), np.array(be)


@pytest.mark.parametrize("n", [1024, 2048 + 1, 3000 + 3, 5118])
@pytest.mark.parametrize("nb", [1, 3])
def test_basis_across_every_layout(dev, n, nb):
    m = 140  # 32, 64, 96 and 128 columns are crossed on the way
    g = torch.Generator().manual_seed(n + nb)
    d = torch.rand(n, generator=g) * 4 + 0.5
    S = torch.randn(nb, n, generator=g)
    run = LanczosRun(n, nb, m, dev)
    run.V.fill_(float("nan"))
    Sb = torch.full((nb, run.ld), float("nan"), device=dev)
    Sb[:, :n] = S.to(dev)
    aop = lower(ca.Diagonal(d.to(dev)))
    s = N.stream_ptr(dev)
    N.call("ck_lanczos_start", n, nb, N.ptr(Sb), run.ld, N.ptr(run.V), run.ld, run.ldb, N.ptr(run.diag),
           N.ptr(run.subdiag), N.ptr(run.state), m, N.ptr(run.scratch), s)
    N.call("ck_lanczos_iterate", aop[0], n, nb, m, N.ptr(run.V), run.ld, run.ldb, N.ptr(run.diag), N.ptr(run.subdiag),
           N.ptr(run.state), 1e-7, 0, m, N.ptr(run.scratch), None, 0, s)
    for b in range(nb):
        Q = run.V[b, 1:m + 1, :n].double()
        # CGS2 in 32 bits: orthogonal to the rounding of a dot product of n unit-norm terms
        assert float((Q @ Q.T - torch.eye(m, dtype=torch.float64, device=dev)).abs().max()) < 2e-6
        al, be = lanczos64(d.double().numpy(), S[b].double().numpy(), m)
        T = run.diag[b].double().cpu().numpy(), run.subdiag[b, 1:m].double().cpu().numpy()
        ev = np.linalg.eigvalsh(np.diag(T[0]) + np.diag(T[1], 1) + np.diag(T[1], -1))
        ref = np.linalg.eigvalsh(np.diag(al) + np.diag(be[:-1], 1) + np.diag(be[:-1], -1))
        assert np.abs(ev - ref).max() < 2e-5 * ref.max()
        assert bool(torch.isnan(run.V[b, 2:m + 2, n:]).all())  # what pads a column is not written
