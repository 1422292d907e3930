"""Outputs of wide elements, with every gradient, against the CPU kernels on
the same inputs (sizes around 128 MB of outputs), and the launches that store
past the caches (from 1 GiB of outputs on, rows of whole 128-byte lines)
against the same rows in launches that do not.

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


# bytes a step and row of the backward's outputs, elements and steps of one
# row: from 1 GiB on with an even number of lines a row, below it, and with
# rows that start inside a line
@pytest.mark.parametrize("T,rows", [(8192, None), (8192, -1), (8200 + 5, None)])
@pytest.mark.parametrize("kind", ["recur f32", "recur f64", "recur c64", "lti_recur f64", "lti_recur c64", "recur2 f32",
                                  "recur2 f64"])
def test_past_the_caches(hip, kind, T, rows):
    """A launch that streams against two launches of half its rows, which do
    not: within a launch every row is computed for itself.  The entry states
    of a row's tiles are sums in compute precision (64 bits) of whichever
    predecessors have published, rounded once, so calls agree to a few
    roundings of the storage type, which die out as above."""
    import torch

    name, dt = kind.split()
    dt = {"f32": torch.float32, "f64": torch.float64, "c64": torch.complex64}[dt]
    es = torch.empty((), dtype=dt).element_size()
    per_step = {"recur": 2, "lti_recur": 1, "recur2": 6}[name] * es
    B = -(-(1 << 30) // (8192 * per_step)) + (rows or 0)
    B += B % 2 if rows is None else 0
    g = torch.Generator(device="cuda").manual_seed(B)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda", dtype=dt)  # noqa: E731
    if name == "recur2":
        A = (torch.rand(B, T, 2, 2, generator=g, device="cuda") - 0.5).to(dt) * 0.9
        zi, x, gy = r(B, 2), r(B, T, 2), r(B, T, 2)
    else:
        A = ((torch.rand(*((B, T) if name == "recur" else (B,)), generator=g, device="cuda") - 0.5) * 1.8).to(dt)
        zi, x, gy = r(B), r(B, T), r(B, T)
    fwd = getattr(torch.ops.philtorch, name)
    bwd = getattr(torch.ops.philtorch, "recurN_backward" if name == "recur2" else name + "_backward")

    def run(*ts):
        y = fwd(*ts[:3])
        return [y, *bwd(*ts[:2], y, ts[3])]

    whole = run(A, zi, x, gy)
    h = B // 2
    eps = torch.finfo(dt).eps
    for lo, hi in ((0, h), (h, B)):
        part = run(*(v[lo:hi].contiguous() for v in (A, zi, x, gy)))
        for i, (p, q) in enumerate(zip(whole, part)):
            # an LTI coefficient's gradient sums a whole row
            tol = 64 * eps if not (i == 1 and name == "lti_recur") else 64 * eps * T ** 0.5
            assert float((p[lo:hi] - q).abs().max()) <= tol * float(q.abs().max()), i


# 16 MiB of per-step gradients and grad_x, from which on the time-varying state
# space's gradients leave past the caches: just above, and halves below
@pytest.mark.parametrize("T", [4096, 4099])
@pytest.mark.parametrize("operands", ["every one", "shared A", "constant b"])
@pytest.mark.parametrize("M", [1, 2])
@pytest.mark.parametrize("dt", ["float32", "float64"])
def test_state_space_gradients(hip, dt, M, operands, T):
    """One launch that streams against two of half its rows that do not.  With
    A shared by the rows its gradient is a sum over them, of rows that each
    agree as above: the halves' sums add up to the whole's."""
    import torch

    from philtorch_amd import lpv

    dt = getattr(torch, dt)
    es = torch.empty((), dtype=dt).element_size()
    per_step = {"every one": M * M + M + 2, "shared A": M * M + M + 2, "constant b": M * M + 1}[operands] * es
    B = 2 * (-(-(1 << 24) // (T * per_step)) // 2 + 1)
    g = torch.Generator(device="cuda").manual_seed(B + T)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda", dtype=dt)  # noqa: E731
    A = ((torch.rand(*(() if operands == "shared A" else (B,)), T, M, M, generator=g, device="cuda") - 0.5) * 0.9).to(dt)
    b, d = (r(M), None) if operands == "constant b" else (r(B, T, M), r(B, T))
    zi, x, gy = r(B, M), r(B, T), r(B, T)

    def run(lo, hi):
        part = lambda t: t if t is None or t.size(0) != B else t[lo:hi].contiguous()  # noqa: E731
        ts = [None if t is None else part(t).detach().requires_grad_(True) for t in (A, b, d, zi, x)]
        y, zf = lpv.state_space(ts[0], ts[4], B=ts[1], D=ts[2], zi=ts[3], unroll_factor=1, out_idx=0)
        wanted = [t for t in ts if t is not None]
        return [y.detach(), zf.detach()] + list(torch.autograd.grad(y, wanted, gy[lo:hi].contiguous()))

    whole, first, second = run(0, B), run(0, B // 2), run(B // 2, B)
    eps = torch.finfo(dt).eps
    for i, (w, p, q) in enumerate(zip(whole, first, second)):
        if w.size(0) == B:
            want, tol = torch.cat([p, q]), 64 * eps
        else:  # summed over the rows
            want, tol = p + q, 64 * eps * B ** 0.5
        assert float((w - want).abs().max()) <= tol * float(want.abs().max()), i


@pytest.mark.parametrize("dt", ["float32", "float64"])
def test_3x3_backward_time(hip, dt):
    """The 3x3 scan's stores are a lane's own vectors, 36 to 144 bytes apart:
    past the caches they reach memory as partial lines, and the backward took
    six (fp32) to nine (fp64) times its forward.  It moves 27 elements a step
    where the forward moves 15; 1.6 times is measured."""
    import torch

    dt = getattr(torch, dt)
    B, T = 256, 16384
    A = (torch.rand(B, T, 3, 3, device="cuda") - 0.5).to(dt) * 0.6
    zi, x = torch.randn(B, 3, device="cuda", dtype=dt), torch.randn(B, T, 3, device="cuda", dtype=dt)
    y = torch.ops.philtorch.recurN(A, zi, x)

    def time(f):
        out = []
        for _ in range(7):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            f()
            a.record()
            f()
            b.record()
            b.synchronize()
            out.append(a.elapsed_time(b))
        return min(out)

    fwd = time(lambda: torch.ops.philtorch.recurN(A, zi, x))
    assert time(lambda: torch.ops.philtorch.recurN_backward(A, zi, y, x)) < 3.2 * fwd
