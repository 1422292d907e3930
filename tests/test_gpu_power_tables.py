"""The LTI state spaces' power tables at orders 3 and 4 (4 x 4 fp64 matrix
instructions, order 3 padded): models whose powers stay near one for a whole
row, so that every entry, up to the look-back's powers of the tile matrix,
carries weight in the result."""
import numpy as np
import pytest

from tests import _data as D

pytestmark = pytest.mark.gpu


def _model(M, B, F, P, seed):
    g = D.rng(seed)
    A = np.stack([np.linalg.qr(g.standard_normal((M, M)))[0] * 0.99999 for _ in range(B)])
    return g, A, g.standard_normal((B, M, F)), g.standard_normal((B, P, M))


@pytest.mark.parametrize("T", [8 * 64, 3 * 8 * 64 + 1, 70 * 6144 + 3])
@pytest.mark.parametrize("M", [3, 4])
def test_slow_models(hip, M, T):
    import torch

    import oracle
    from philtorch_amd import lti

    B, F, P = 2, 2, 3
    g, A, Bm, C = _model(M, B, F, P, D.seed_of(M, T))
    x, zi = g.standard_normal((B, T, F)), g.standard_normal((B, M))
    up = lambda v: torch.from_numpy(np.ascontiguousarray(v)).cuda()  # noqa: E731
    y, zf = lti.state_space(up(A), up(x), B=up(Bm), C=up(C), zi=up(zi), unroll_factor=1)
    y_ref, zf_ref = oracle.lti_state_space_mimo(A, x, Bm, C, None, zi)
    D.check(y.cpu().numpy(), y_ref, "mimo y")
    D.check(zf.cpu().numpy(), zf_ref, "mimo zf")
    for dt in (np.float64, np.float32):
        a, u, b, c, z = (v.astype(dt) for v in (A, x[..., 0], Bm[..., 0], C[:, 0], zi))
        y, zf = lti.state_space(up(a), up(u), B=up(b), C=up(c), zi=up(z), unroll_factor=1)
        # the reference in double on the same bits
        y_ref, zf_ref = oracle.lti_state_space(*(v.astype(np.float64) for v in (a, u, b, c)), None,
                                               z.astype(np.float64))
        D.check(y.cpu().numpy(), y_ref.astype(dt), "ss y")
        D.check(zf.cpu().numpy(), zf_ref.astype(dt), "ss zf")
