"""Order 4 with 3 or 4 inputs: the widths whose lanes hold fewer steps (fp32
with 4 inputs) or have a form with fewer steps for few tiles (fp64)."""
import numpy as np
import pytest

from tests import _data as D

pytestmark = pytest.mark.gpu


def _case(B, T, F, P, dtype):
    g = D.rng(D.seed_of(B, T, F, P, np.dtype(dtype).name))
    A = np.stack([np.linalg.qr(g.standard_normal((4, 4)))[0] * 0.9 for _ in range(B)])
    vals = [A, g.standard_normal((4, F)), g.standard_normal((B, P, 4)), g.standard_normal((P, F)),
            g.standard_normal((B, 4)), g.standard_normal((B, T, F))]
    return [v.astype(dtype) for v in vals]


# one step; a lane's chunk (4 or 8 fp64 steps, 8 or 16 fp32), a wave's span and a tile of
# either form, each side of them; more tiles than one look-back window's part of a row
@pytest.mark.parametrize("B,T", [(3, 1), (3, 3), (3, 4), (3, 5), (3, 8), (3, 9), (2, 255), (2, 257), (2, 513),
                                 (3, 767), (3, 769), (2, 1535), (2, 1537), (2, 3073), (2, 24001),
                                 # fp64: the last launch of the short form and the first of the long one
                                 (511, 1536), (512, 1536), (255, 1537), (256, 1537)])
@pytest.mark.parametrize("F,P", [(3, 1), (3, 4), (4, 1), (4, 4)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_states_and_outputs(hip, dtype, F, P, B, T):
    """mimo_ss and mimo_ss_states, forward against the oracle in double on the
    same bits, and reversed against the forward of the reversed input."""
    import torch

    import oracle

    vals = _case(B, T, F, P, dtype)
    A, Bm, C, Dm, zi, x = vals
    ref, ref_zf = oracle.lti_state_space_mimo(*(v.astype(np.float64) for v in (A, x, Bm, C, Dm, zi)))
    up = lambda v: torch.from_numpy(np.ascontiguousarray(v)).cuda()  # noqa: E731
    ts = [up(v) for v in vals]
    y, zf = torch.ops.philtorch.mimo_ss(*ts, False)
    D.check(y.cpu().numpy(), ref.astype(dtype), "y")
    D.check(zf.cpu().numpy(), ref_zf.astype(dtype), "zf")
    ys, zfs, hs = torch.ops.philtorch.mimo_ss_states(*ts, False)
    D.check(ys.cpu().numpy(), ref.astype(dtype), "y with states")
    D.check(zfs.cpu().numpy(), ref_zf.astype(dtype), "zf with states")
    got = torch.einsum("bpm,btm->btp", ts[2].double().cpu(), hs.double().cpu()) + torch.einsum(
        "pf,btf->btp", ts[3].double().cpu(), ts[5].double().cpu())
    D.check(got.numpy().astype(dtype), ref.astype(dtype), "C hs + D x")
    yr, zfr = torch.ops.philtorch.mimo_ss(*ts[:5], ts[5].flip(1).contiguous(), True)
    D.check(yr.flip(1).cpu().numpy(), ref.astype(dtype), "reversed y")
    D.check(zfr.cpu().numpy(), ref_zf.astype(dtype), "reversed zf")


@pytest.mark.parametrize("forced", ["fallback", "aggregates"])
@pytest.mark.parametrize("F", [3, 4])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_look_back_routes(hip, dtype, F, forced):
    """The bounded wait's fallback (which folds the row again) and rows of aggregates alone."""
    import torch

    import oracle
    from tests import capi

    lib = capi.load()
    A, Bm, C, Dm, zi, x = _case(4, 24001, F, 2, dtype)
    ref, _ = oracle.lti_state_space_mimo(*(v.astype(np.float64) for v in (A, x, Bm, C, Dm, zi)))
    ts = [torch.from_numpy(np.ascontiguousarray(v)).cuda() for v in (A, Bm, C, Dm, zi, x)]
    try:
        if forced == "fallback":
            lib.phs_debug_set_spin_limit(1)
        else:
            lib.phs_debug_set_aggregates_only(1)
        y, _ = torch.ops.philtorch.mimo_ss(*ts, False)
        torch.cuda.synchronize()
    finally:
        lib.phs_debug_set_spin_limit(0)
        lib.phs_debug_set_aggregates_only(0)
    D.check(y.cpu().numpy(), ref.astype(dtype), forced)
