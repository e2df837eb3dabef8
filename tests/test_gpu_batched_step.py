"""The one-launch step of the batched CG (systems of up to 4096 unknowns) against the five-launch one and FP64."""
import numpy as np
import pytest
import torch

from cola_amd.linalg.batched import BatchedCG, BatchedSystems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [[1], [1, 2, 63, 64, 65], [1023, 1024, 1025], [2048, 7, 2049, 300], [4095, 4096, 1]])
@pytest.mark.parametrize("rows,graph", [(4, False), (16, True)])
def test_step(dev, sizes, rows, graph):
    """Both paths take the sums of a system in 32-bit rows and FP64 (the general one adds a tile's r.r in
    32 bits, 4 EPS apart): counts within one step, solutions within cond(A) <= 10 times the tolerance."""
    g = torch.Generator(device=dev).manual_seed(sum(sizes))
    mats, sols = [], []
    for n in sizes:
        X = torch.randn(n, max(n // 2, 1), generator=g, device=dev) / max(n // 2, 1)**0.5
        mats.append(X @ X.T + torch.eye(n, device=dev))
    sy = BatchedSystems.dense(mats, 0.25, dev)
    bs = [torch.randn(n, generator=g, device=dev) for n in sizes]
    b = sy.concat(bs)
    outs = []
    for general in (False, True):
        cg = BatchedCG(sy, rows, 200)
        assert 1 <= cg.plan.max_vtiles <= 4
        if general:
            cg.plan.max_vtiles = 0
        x, ks = cg.solve(b, 1e-6, use_graph=graph)
        torch.cuda.synchronize()
        outs.append(([v.clone() for v in sy.split(x)], ks, cg.gamma.clone(), cg.beta.clone()))
    for s, n in enumerate(sizes):
        sol = torch.linalg.solve(mats[s].double() + 0.25 * torch.eye(n, device=dev, dtype=torch.float64), bs[s].double())
        for xs, ks, _, _ in outs:
            assert float((xs[s].double() - sol).norm() / sol.norm()) < 10 * 1.5e-6 + 8 * n * 2.0**-24
        assert abs(int(outs[0][1][s]) - int(outs[1][1][s])) <= 1
    # a capped solve stops after the same number of steps on both, with every scalar close
    for general in (False, True):
        cg = BatchedCG(sy, rows, 3)
        cg.plan.max_vtiles = 0 if general else cg.plan.max_vtiles
        x, ks = cg.solve(b, 0.0, use_graph=graph)
        outs.append((x.clone(), ks, cg.gamma.clone(), cg.alpha.clone()))
    (x0, k0, g0, a0), (x1, k1, g1, a1) = outs[2:]
    big = torch.tensor([n > 8 for n in sizes], device=dev)
    assert np.all(k0 == 3) and np.all(k1 == 3)
    assert float((x0 - x1).norm() / x1.norm()) < 1e-5
    assert torch.allclose(g0[big], g1[big], rtol=1e-3) and torch.allclose(a0[big], a1[big], rtol=1e-4)
