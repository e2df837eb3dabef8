"""The core of the fused Woodbury step at the edges of its tiles of 128 rows (sixteen waves, eight tiles
each at once) and its 4-column pieces of C^-1, against the unfused step on the same columns."""
import pytest
import torch

import cola_amd as ca
from cola_amd.linalg.cg import run_batched_cg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k", [(100, 1), (128, 3), (129, 4), (1920, 5), (2048, 33), (2049, 63), (4000, 64),
                                 (16384, 7), (16385, 64)])
def test_core(dev, n, k):
    """A = 2 I + F F^T with the preconditioner's F and its shift of 1, so that the preconditioned spectrum lies
    in [1, 2]: ten steps leave 0.17^10, and both runs differ by 32-bit rounding of n-term sums, 8 EPS sqrt(n),
    carried over ten steps."""
    g = torch.Generator(device=dev).manual_seed(n + k)
    F = torch.randn(n, k, generator=g, device=dev) / n**0.5 * 3.0
    A = F @ F.T
    A.diagonal().add_(2.0)
    P = ca.WoodburyInverse(F, 1.0)
    op = ca.PSD(ca.Dense(A))
    b = torch.randn(n, 8, generator=g, device=dev)
    x, _, kf, info = run_batched_cg(op, b, None, 10, 0.0, P)
    sol = torch.linalg.solve(A.double(), b.double()) if n <= 4000 else None
    for j in (0, 6):
        xu, _, ku, _ = run_batched_cg(op, b[:, j:j + 2].contiguous(), None, 10, 0.0, P)
        d = float((x[:, j:j + 2] - xu).norm() / xu.norm())
        print(n, k, kf, ku, d, flush=True)
        assert kf == ku == 10 and d < 10 * 8 * n**0.5 * 2.0**-24
    if sol is not None:
        assert float((x.double() - sol).norm() / sol.norm()) < 10 * 8 * n**0.5 * 2.0**-24 + 0.18**10 * 4
