"""philtorch::mimo_ss_states (phs_mimo_ss_hs): the multi-input multi-output
state space that keeps its states for the coefficient gradients."""
import numpy as np
import pytest

from tests import _data as D

pytestmark = pytest.mark.gpu


# one step, a lane's chunk, a wave's span and a tile (16 fp32 or 8 fp64 steps
# a lane, 64 lanes, 3 waves), each side of them
@pytest.mark.parametrize("T", [1, 15, 16, 17, 512, 1025, 3071, 3073, 12289])
@pytest.mark.parametrize("rev", [False, True])
@pytest.mark.parametrize("M,F,P", [(1, 1, 2), (2, 2, 1), (3, 3, 4), (4, 2, 2), (4, 4, 3)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_states(hip, dtype, M, F, P, rev, T):
    """y and zf mimo_ss's, hs the pass with C the identity, which the other
    tests hold to the oracle: bit for bit within one tile; over more a tile's
    entry state is summed from whichever predecessors have published, so
    calls agree to the rounding of those double sums (once rounded to fp32)."""
    import torch

    def same(a, b):
        if T <= 3 * 64 * (16 if dtype == np.float32 else 8):
            return torch.equal(a, b)
        eps = float(torch.finfo(a.dtype).eps)
        return float((a - b).abs().max()) <= 8 * eps * float(b.abs().max())

    g = D.rng(D.seed_of(np.dtype(dtype).name, M, F, P, rev, T))
    B = 3
    up = lambda *s: torch.from_numpy(g.standard_normal(s).astype(dtype)).cuda()  # noqa: E731
    Bm, C, Dm, zi, x = up(M, F), up(B, P, M), up(P, F), up(B, M), up(B, T, F)
    A = np.stack([np.linalg.qr(g.standard_normal((M, M)))[0] * 0.9 for _ in range(B)])
    A = torch.from_numpy(A.astype(dtype)).cuda()
    op = torch.ops.philtorch.mimo_ss
    y, zf = op(A, Bm, C, Dm, zi, x, rev)
    y1, zf1, hs = torch.ops.philtorch.mimo_ss_states(A, Bm, C, Dm, zi, x, rev)
    assert same(y, y1) and same(zf, zf1)
    assert same(hs, op(A, Bm, torch.eye(M, dtype=x.dtype, device="cuda"), None, zi, x, rev)[0])
    y0, zf0, hs0 = torch.ops.philtorch.mimo_ss_states(A, Bm, C[:, :0], None, zi, x, rev)  # the states alone
    assert y0.shape == (B, T, 0) and same(zf0, zf) and same(hs0, hs)


@pytest.mark.parametrize("M,F,P", [(1, 2, 2), (2, 4, 4), (3, 2, 2), (4, 2, 2), (4, 1, 3)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_gradients(hip, dtype, M, F, P):
    """state_space's gradients through the kept states, and the sums' whole-vector
    reads (F = P = 2 or 4), against the composed route's autograd in double."""
    import torch

    from philtorch_amd import lti
    from philtorch_amd.lti.ssm import _mimo_composite

    g = D.rng(D.seed_of("grad", np.dtype(dtype).name, M, F, P))
    B, T = 5, 2 * 16384 + 77  # more rows than outputs: a C of (rows, M) reads as one vector per row
    A = np.stack([np.linalg.qr(g.standard_normal((M, M)))[0] * 0.9 for _ in range(B)])
    vals = [A, g.standard_normal((M, F)), g.standard_normal((P, M)), g.standard_normal((P, F)),
            g.standard_normal((B, M)), g.standard_normal((B, T, F))]
    gy = g.standard_normal((B, T, P)).astype(dtype)
    ts = [torch.from_numpy(v.astype(dtype)).cuda().requires_grad_(True) for v in vals]
    A, Bm, C, Dm, zi, x = ts
    y, _ = lti.state_space(A, x, B=Bm, C=C, D=Dm, zi=zi, unroll_factor=1)
    got = torch.autograd.grad(y, ts, torch.from_numpy(gy).cuda())
    td = [t.detach().double().requires_grad_(True) for t in ts]
    yd, _ = _mimo_composite(*td)
    ref = torch.autograd.grad(yd, td, torch.from_numpy(gy).cuda().double())
    for name, a, b in zip("A B C D zi x".split(), got, ref):
        D.check(a.cpu().numpy(), b.cpu().numpy().astype(dtype), name)


def test_opcheck(hip):
    import torch

    t = lambda *s: torch.randn(*s, dtype=torch.float64, device="cuda")  # noqa: E731
    args = (t(2, 2, 2) * 0.4, t(2, 2), t(3, 2), t(3, 2), t(2, 2), t(2, 9, 2))
    torch.library.opcheck(torch.ops.philtorch.mimo_ss_states.default, args)
    for a in args:
        a.requires_grad_(True)
    f = lambda *a: torch.ops.philtorch.mimo_ss_states(*a)[:2]  # noqa: E731
    assert torch.autograd.gradcheck(f, args)
