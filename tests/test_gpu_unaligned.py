"""Rows and operands that start off a 16-byte boundary.

The kernels read and write rows as 16-byte vectors at element alignment, so
the same call on operands shifted by 1 to 3 elements, and on rows of odd
length (whose starts fall on every residue), must give the same bits as on
freshly allocated operands where a row is one tile.  Over several tiles a
tile's entry state is summed, in 64 bits, from whichever predecessors have
published, so two calls differ by the rounding of those sums.  The aligned
calls are held to the oracle by the other GPU tests, at odd lengths too."""
import numpy as np
import pytest

from tests import _data as D

pytestmark = pytest.mark.gpu

# either side of a 16-byte vector, of one wave's round and of the kernels' tiles
LENGTHS = [1, 3, 381, 1537, 6143, 8193, 30721]
ONE_TILE = 384  # the shortest tile among these kernels (orders 2 to 4, fp64, time-varying)


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


def _same(got, ref, what):
    """Bit for bit within a tile.  Beyond, an entry state may differ by a few
    roundings of the storage type; the models' memory is some tens of steps
    (|A| <= 0.99, drawn per step or row), which carries that to at most 64
    roundings of a row's largest value.  A gradient summed over the row takes
    that once per tile, of terms whose sum grows with the root of their
    number: the root of T covers it."""
    import torch

    for i, (a, b) in enumerate(zip(got, ref)):
        T = what[0]
        if T <= ONE_TILE:
            assert torch.equal(a, b), (what, i)
            continue
        per_step = a.dim() > 1 and a.size(1) == T
        tol = 64 * torch.finfo(a.dtype).eps * (1 if per_step else T ** 0.5)
        assert float((a - b).abs().max()) <= tol * float(b.abs().max()), (what, i)


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
        _same(run(off), ref, (T, off))


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
        _same(run(off), ref, (T, off))


@pytest.mark.parametrize("T", LENGTHS)
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("M,F,P", [(1, 2, 1), (2, 1, 2), (3, 3, 2), (4, 2, 2), (4, 4, 4)])
def test_multi_input(hip, M, F, P, dtype, T):
    """The multi-input state spaces, A per row and A per step, with every gradient."""
    import torch

    from philtorch_amd import lpv, lti

    B = 5  # a C of (rows, M) or (steps, M) reads as a vector per row or step: neither is P
    g = D.rng(D.seed_of(B, T, M, F, P))
    A = (g.uniform(-1, 1, (B, M, M)) * 0.9 / M).astype(dtype)
    At = (g.uniform(-1, 1, (B, T, M, M)) * 0.9 / M).astype(dtype)
    rest = [g.standard_normal(s).astype(dtype) for s in ((M, F), (P, M), (P, F), (B, M), (B, T, F))]
    gy = g.standard_normal((B, T, P)).astype(dtype)

    def run(off):
        out = []
        for a, f in ((A, lti.state_space), (At, lpv.state_space)):
            ts = [_shifted(v, off).requires_grad_(True) for v in (a, *rest)]
            y, zf = f(ts[0], ts[5], B=ts[1], C=ts[2], D=ts[3], zi=ts[4], unroll_factor=1)
            out += [y, zf, *torch.autograd.grad(y, ts, _shifted(gy, off).view(y.shape))]
        return out

    ref = run(0)
    for off in (1, 2, 3):
        _same(run(off), ref, (T, off))
