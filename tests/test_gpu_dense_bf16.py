"""Products of bf16-stored matrices at the edges of the kernels' tiles and of the rule that picks them."""
import pytest
import torch

import cola_amd as ca

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [8, 16, 504, 512, 520, 1016, 1024, 1032, 2048, 2056, 8192, 8200, 11584, 11592, 12296])
def test_dense_bf16(dev, n):
    """Products with the stored values in 32 bits: a lane adds at most n / 64 + 8 of them one after another
    and the wave six times more, so an entry errs by at most that many EPS of sum |a| |x|; and an infinity,
    a NaN and 1e-36 go through as in 32-bit arithmetic."""
    g = torch.Generator(device=dev).manual_seed(n)
    A = torch.randn(n, n, generator=g, device=dev).to(torch.bfloat16)
    op = 1.5 * ca.ops.DenseBF16(A) + 0.5 * ca.I_like(ca.ops.DenseBF16(A))
    X = torch.randn(n, 17, generator=g, device=dev)
    X[:, 1] *= 1e-36
    rows = torch.unique(torch.cat([torch.arange(min(n, 300), device=dev), torch.arange(max(n - 300, 0), n, device=dev)]))
    Ad = A[rows].double()
    ref = 1.5 * (Ad @ X.double()) + 0.5 * X[rows].double()
    mag = 1.5 * (Ad.abs() @ X.double().abs()) + 0.5 * X[rows].double().abs()
    for B in (1, 2, 3, 4, 5, 8, 9, 16, 17):
        Y = op @ X[:, :B].contiguous()
        assert Y.shape == (n, B)
        assert torch.all((Y[rows].double() - ref[:, :B]).abs() <= (n / 64 + 16) * 2.0**-24 * mag[:, :B] + 1e-44 * n)
    A2 = A.clone()
    A2[n // 2, n - 1] = float("inf")
    X2 = torch.ones(n, 4, device=dev)
    X2[0, 3] = float("nan")
    for B in (1, 2, 4):
        Y = ca.ops.DenseBF16(A2) @ X2[:, 4 - B:].contiguous()
        assert bool(torch.isnan(Y[:, -1]).all())
        if B > 1:
            assert float(Y[n // 2, 0]) == float("inf") and int(torch.isfinite(Y[:, 0]).sum()) == n - 1
