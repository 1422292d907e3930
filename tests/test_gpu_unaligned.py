"""Rows and operands that start off a 16-byte boundary.

The kernels read and write rows as 16-byte vectors at element alignment, so
the same call on operands shifted by 1 to 3 elements, and on rows of odd
length (whose starts fall on every residue), must give the same bits as on
freshly allocated operands.  The aligned calls are held to the oracle by the
other GPU tests, at odd lengths too."""
import numpy as np
import pytest

from tests import _data as D

pytestmark = pytest.mark.gpu

# either side of a 16-byte vector, of one wave's round and of the kernels' tiles
LENGTHS = [1, 3, 1537, 6143, 8193, 30721]


def _operands(kind, B, T, dtype):
    g = D.rng(D.seed_of(B, T, kind))
    n = lambda *s: D.normal(g, s, dtype)  # noqa: E731
    if kind == "recur":
        return [D.coef(g, (B, T), dtype), n(B), n(B, T)], n(B, T)
    if kind == "lti_recur":
        return [D.coef(g, (B,), dtype), n(B), n(B, T)], n(B, T)
    M = int(kind[-1])
    A = (n(B, T, M, M) if kind.startswith("recurN") else n(B, M, M)) * np.dtype(dtype).type(0.9 / M)
    A = np.clip(A.real, -0.9 / M, 0.9 / M).astype(dtype)
    return [A, n(B, M), n(B, T, M)], n(B, T, M)


def _shifted(v, off):
    """v on the GPU, `off` elements past the start of an allocation."""
    import torch

    t = torch.from_numpy(np.ascontiguousarray(v)).cuda()
    buf = torch.empty(t.numel() + off, dtype=t.dtype, device="cuda")
    out = buf[off:].view(t.shape)
    out.copy_(t)
    return out


@pytest.mark.parametrize("T", LENGTHS)
@pytest.mark.parametrize("kind,dtype", [("recur", np.float32), ("recur", np.float64), ("lti_recur", np.float32),
                                        ("lti_recur", np.complex64), ("recurN2", np.float32), ("recurN3", np.float32),
                                        ("lti_recurN2", np.float32), ("lti_recurN2", np.float64)])
def test_scans(hip, kind, dtype, T):
    import torch

    base = kind.rstrip("23")
    fwd, bwd = getattr(torch.ops.philtorch, base), getattr(torch.ops.philtorch, base + "_backward")
    ins, gy = _operands(kind, 3, T, dtype)

    def run(off):
        A, zi, x = (_shifted(v, off) for v in ins)
        y = fwd(A, zi, x)
        return [y, *bwd(A, zi, _shifted(y.cpu().numpy(), off), _shifted(gy, off))]

    ref = run(0)
    for off in (1, 2, 3):
        for i, (a, b) in enumerate(zip(run(off), ref)):
            assert torch.equal(a, b), (off, i)


@pytest.mark.parametrize("T", LENGTHS)
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("order", [1, 2, 4])
def test_filters(hip, order, dtype, T):
    """lfilter, filtfilt, sosfilt (order 2) and the LPV state space, with every gradient."""
    import torch

    from philtorch_amd import lpv, lti

    B = 3
    g = D.rng(D.seed_of(B, T, order))
    a = (0.4 / order * g.uniform(-1, 1, (B, order))).astype(dtype)
    b = g.standard_normal((B, order + 1)).astype(dtype)
    x, gy = D.normal(g, (B, T), dtype), D.normal(g, (B, T), dtype)
    A = (g.uniform(-1, 1, (B, T, order, order)) * 0.9 / order).astype(dtype)
    bv, zi = g.standard_normal((B, T, order)).astype(dtype), D.normal(g, (B, order), dtype)
    sos = np.concatenate([b, np.ones((B, 1), dtype), a], 1)[:, None].astype(dtype) if order == 2 else None

    def run(off):
        up = lambda v: _shifted(v, off).requires_grad_(True)  # noqa: E731
        calls = [((b, a, x), lambda b, a, x: lti.lfilter(b, a, x, unroll_factor=1)),
                 ((A, bv, zi, x), lambda A, bv, zi, x: lpv.state_space(A, x, B=bv, zi=zi, unroll_factor=1, out_idx=0)[0])]
        if T > 3:
            calls.append(((b, a, x), lambda b, a, x: lti.filtfilt(b, a, x, padlen=3, unroll_factor=1)))
        if sos is not None:
            calls.append(((sos, x), lti.sosfilt))
        out = []
        for args, f in calls:
            ts = [up(v) for v in args]
            y = f(*ts)
            out += [y, *torch.autograd.grad(y, ts, _shifted(gy, off))]
        return out

    ref = run(0)
    for off in (1, 2, 3):
        for i, (p, q) in enumerate(zip(run(off), ref)):
            assert torch.equal(p, q), (off, i)
