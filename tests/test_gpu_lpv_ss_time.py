"""The time-varying state space's forward against the plain 2x2 scan of the
same matrices."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("with_cd", [False, True])
def test_order2_forward_time(hip, with_cd):
    """Both are bound by memory: a step moves 24 bytes, 36 with b, c and d per
    step, and the scan's 32.  With four waves a SIMD the state space takes
    0.99 and 1.22 times the scan's time; with three it took 1.19 and 1.37.
    The limits lie between."""
    import torch

    from philtorch_amd import lpv

    B, T = 32, 1 << 20
    A = (torch.rand(B, T, 2, 2, device="cuda") - 0.5) * 0.9
    zi, xs, x = (torch.randn(*s, device="cuda") for s in ((B, 2), (B, T, 2), (B, T)))
    kw = dict(B=torch.randn(B, T, 2, device="cuda"), D=torch.randn(B, T, device="cuda")) if with_cd else dict(
        B=torch.randn(2, device="cuda"))
    buf = torch.empty(128 << 20, device="cuda")  # read between calls: 512 MB, no call finds its inputs cached

    def time(f):
        out = []
        for _ in range(9):
            buf.sum()
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            f()
            b.record()
            b.synchronize()
            out.append(a.elapsed_time(b))
        return sorted(out[2:])[3]

    with torch.no_grad():
        scan = time(lambda: torch.ops.philtorch.recur2(A, zi, xs))
        ss = time(lambda: lpv.state_space(A, x, zi=zi, unroll_factor=1, out_idx=0, **kw))
    assert ss < (1.30 if with_cd else 1.09) * scan, (ss, scan)
