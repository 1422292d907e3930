"""Outputs of wide elements just below and just above the size from which the
scans store past the caches (128 MB a launch), with every gradient, against
the CPU kernels on the same inputs.

Tolerance: with |A[t]| <= 0.9 a step's rounding error dies out as 0.9^k, so
an output carries at most about 2 (1 - 0.9)^-1 = 20 roundings of 2^-53 of the
row's largest value per pass and operand; 1e-13 of the largest value allows
for 45 times that over two passes."""
import pytest

pytestmark = pytest.mark.gpu


def _both(f, args, gy):
    """f's outputs and gradients on the GPU and on the CPU."""
    import torch

    out = []
    for dev in ("cuda", "cpu"):
        ts = [v.to(dev).requires_grad_(True) for v in args]
        y = f(*ts)
        out.append([v.detach().cpu() for v in (y, *torch.autograd.grad(y, ts, gy.to(dev)))])
    for i, (a, b) in enumerate(zip(*out)):
        assert float((a - b).abs().max()) <= 1e-13 * float(b.abs().max()), i


@pytest.mark.parametrize("T", [4095, 4097])  # y: 128 MB at 4096
def test_scan(hip, T):
    import torch

    from philtorch_amd import lpv

    g = torch.Generator().manual_seed(T)
    B = 4096
    A = (torch.rand(B, T, generator=g, dtype=torch.float64) - 0.5) * 1.8
    x, gy = (torch.randn(B, T, generator=g, dtype=torch.float64) for _ in range(2))
    zi = torch.randn(B, generator=g, dtype=torch.float64)
    _both(lambda A, zi, x: lpv.linear_recurrence(A, zi, x), (A, zi, x), gy)


@pytest.mark.parametrize("T", [2730, 2731])  # states and y: 128 MB between the two
def test_state_space(hip, T):
    import torch

    from philtorch_amd import lpv

    g = torch.Generator().manual_seed(T)
    B = 2048
    A = (torch.rand(B, T, 2, 2, generator=g, dtype=torch.float64) - 0.5) * 0.9
    b, zi = torch.randn(B, T, 2, generator=g, dtype=torch.float64), torch.randn(B, 2, generator=g, dtype=torch.float64)
    x, gy = (torch.randn(B, T, generator=g, dtype=torch.float64) for _ in range(2))
    _both(lambda A, b, zi, x: lpv.state_space(A, x, B=b, zi=zi, unroll_factor=1, out_idx=0)[0], (A, b, zi, x), gy)
