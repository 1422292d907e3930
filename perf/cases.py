"""The work the linear-recurrence framework is timed on, through its public API.

A case is a dict of plain values; `listed` gives the named ones, `draw` more
of the same ranges.  `prepare` makes what a program has in hand before the
call (on the GPU, from the seed alone), `run` is one call of the framework,
with its gradients where a training step takes them, and `exact` is the same
computation in 64 bits in plain torch.

Kinds of cases, each with what stands behind it:
  lfilter   lti.lfilter: an IIR filter from b and a.  A chain of biquads from
            coefficient tables, trained or applied; a single filter of order
            1 to 4; a stream's blocks with the state carried (zi).
  sos       lti.sosfilt: a cascade of second-order sections at once.
  filtfilt  lti.filtfilt: zero-phase filtering.
  lpv       lpv.linear_recurrence: the first-order scan whose coefficient
            varies in time (one-pole smoothers, gated recurrences).
  diag      lti.LTIRecurrence: per-channel complex poles, the scan of a
            diagonal state-space model.
  lpvm      lpv.state_space_recursion: M x M matrices that vary in time.
  lpvss     lpv.state_space of a time-varying filter, one input and output.
  mimo      lti.state_space with several inputs and outputs per step.
"""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from philtorch_amd import lpv, lti

_DTYPES = {"f32": torch.float32, "f64": torch.float64, "c64": torch.complex64}
_BYTES = {"f32": 4, "f64": 8, "c64": 8}


def listed():
    return [
        # a real-time stereo stream: one biquad, one block, the state carried over
        dict(name="stream_block", kind="lfilter", B=2, T=512, order=2, chain=1, dtype="f32", grad="none", zi=True),
        # an equaliser's eight biquads per signal, trained: one lfilter per column of the coefficient tables
        dict(name="biquad_chain_train", kind="lfilter", B=16, T=480000, order=2, chain=8, dtype="f32", grad="coef",
             zi=False),
        # five-second clips at 44.1 kHz (an odd number of samples) through a fourth-order filter
        dict(name="lfilter4_clip", kind="lfilter", B=8, T=220501, order=4, chain=1, dtype="f32", grad="none",
             zi=False),
        # the same equaliser as one cascade, trained
        dict(name="sos_train", kind="sos", B=16, T=480000, sections=8, dtype="f32", grad="coef"),
        # zero-phase filtering of a batch of ten-second signals
        dict(name="filtfilt", kind="filtfilt", B=16, T=480000, order=2, dtype="f32", grad="none"),
        # the headline workload: the first-order time-varying scan, forward and backward
        dict(name="lpv_scan_train", kind="lpv", B=64, T=65536, dtype="f32", grad="coef"),
        # the same on a training batch of one-second clips, odd length
        dict(name="lpv_scan_clip_train", kind="lpv", B=16, T=24001, dtype="f32", grad="coef"),
        # a few very long rows in double precision
        dict(name="lpv_scan_long_f64", kind="lpv", B=8, T=1 << 24, dtype="f64", grad="coef"),
        # a diagonal state-space layer: 1024 channels of complex poles, forward and backward
        dict(name="diag_train", kind="diag", B=1024, T=262144, dtype="c64", grad="coef"),
        # 2 x 2 matrices per sample (time-varying biquad denominators), forward and backward
        dict(name="lpv_matrix_train", kind="lpvm", B=32, T=1 << 20, M=2, dtype="f32", grad="coef"),
        # a time-varying biquad with its zeros, every coefficient trained
        dict(name="lpv_filter_train", kind="lpvss", B=16, T=441000, M=2, dtype="f32", grad="coef"),
        # a fourth-order model with two inputs and two outputs, every matrix trained
        dict(name="mimo_train", kind="mimo", B=16, T=480000, M=4, F=2, P=2, dtype="f32", grad="coef"),
    ]


def _log_int(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["lfilter", "lfilter", "sos", "filtfilt", "lpv", "lpv", "diag", "lpvm", "lpvss", "mimo"])
    # (rows, steps, rows * steps) at most, as in the listed case of the kind
    rows, steps, most = {
        "lfilter": (64, 1 << 20, 16 * 480000), "sos": (64, 1 << 20, 16 * 480000),
        "filtfilt": (64, 1 << 20, 16 * 480000), "lpv": (64, 1 << 24, 8 << 24), "diag": (1024, 262144, 1 << 28),
        "lpvm": (64, 1 << 20, 32 << 20), "lpvss": (64, 1 << 20, 8 << 20), "mimo": (64, 1 << 20, 16 * 480000),
    }[kind]
    B = _log_int(rng, 1, rows)
    T = min(_log_int(rng, 256, steps), most // B)
    dtype = "c64" if kind == "diag" else rng.choice(["f32", "f32", "f32", "f64"])
    if dtype == "f64":  # the bytes of the largest listed case of the kind bound the drawn ones
        T = T if kind == "lpv" else max(256, T // 2)
    case = dict(kind=kind, B=B, T=T, dtype=dtype, grad=rng.choice(["none", "x", "coef", "coef"]))
    if kind == "lfilter":
        case.update(order=rng.choice([1, 2, 2, 3, 4]), chain=rng.choice([1, 1, 4, 8]), zi=False)
        case["zi"] = case["chain"] == 1 and rng.random() < 0.5
    elif kind == "sos":
        case.update(sections=rng.randint(1, 8))
    elif kind == "filtfilt":
        case.update(order=rng.randint(1, 4))
    elif kind in ("lpvm", "lpvss"):
        case.update(M=rng.choice([2, 2, 3]))
        case["T"] = max(256, case["T"] * 4 // case["M"] ** 2)
    elif kind == "mimo":
        # more rows than outputs: a C of (rows, M) would be read as one vector per row
        case.update(M=rng.randint(2, 4), F=rng.randint(1, 3), P=rng.randint(1, 3), B=max(4, case["B"]))
        case["T"] = min(case["T"], most // case["B"])
    return case


# ---------------------------------------------------------------- inputs
def _poly(roots_r, roots_th, real_r):
    """Denominators after the leading 1 of pole pairs (r, theta) [..., n] and real poles [..., m]."""
    p = torch.ones(roots_r.shape[:-1] + (1,), dtype=roots_r.dtype, device=roots_r.device)
    for i in range(roots_r.size(-1)):
        r, th = roots_r[..., i], roots_th[..., i]
        p = _mul(p, torch.stack([torch.ones_like(r), -2 * r * torch.cos(th), r * r], -1))
    for i in range(real_r.size(-1)):
        p = _mul(p, torch.stack([torch.ones_like(real_r[..., i]), -real_r[..., i]], -1))
    return p


def _mul(p, q):
    out = p.new_zeros(p.shape[:-1] + (p.size(-1) + q.size(-1) - 1,))
    for i in range(q.size(-1)):
        out[..., i:i + p.size(-1)] += p * q[..., i:i + 1]
    return out


class _Draws:
    """Seeded random tensors on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def uniform(self, low, high, *shape, dtype=torch.float64):
        return torch.rand(*shape, generator=self.g, device="cuda", dtype=dtype) * (high - low) + low

    def normal(self, *shape, dtype=torch.float64):
        return torch.randn(*shape, generator=self.g, device="cuda", dtype=dtype)

    def filters(self, order, *shape):
        """(b, a) of stable filters: poles of radius 0.5 to 0.98, zeros within 1.2."""
        n, m = order // 2, order % 2
        a = _poly(self.uniform(0.5, 0.98, *shape, n), self.uniform(0, math.pi, *shape, n),
                  self.uniform(0.5, 0.98, *shape, m))
        b = _poly(self.uniform(0, 1.2, *shape, n), self.uniform(0, math.pi, *shape, n),
                  self.uniform(0, 1.2, *shape, m))
        return b, a[..., 1:]

    def curve(self, low, high, B, T):
        """A parameter per step: one uniform value every 64 steps, interpolated."""
        frames = self.uniform(low, high, B, 1, T // 64 + 2)
        return F.interpolate(frames, size=T, mode="linear", align_corners=True).squeeze(1)


def _inputs(case, seed):
    """The call's tensors by name, in the case's type; "gy" is the upstream gradient."""
    r, kind, B, T = _Draws(seed), case["kind"], case["B"], case["T"]
    dt = _DTYPES[case["dtype"]]
    real = torch.float64 if dt == torch.float64 else torch.float32
    t = {}
    if kind == "lfilter":
        t["b"], t["a"] = r.filters(case["order"], B, case["chain"])
        if case["zi"]:
            t["zi"] = r.normal(B, case["order"])
        t["x"] = r.normal(B, T, dtype=real)
    elif kind == "sos":
        b, a = r.filters(2, B, case["sections"])
        t["sos"] = torch.cat([b, torch.ones_like(a[..., :1]), a], -1)
        t["x"] = r.normal(B, T, dtype=real)
    elif kind == "filtfilt":
        t["b"], t["a"] = r.filters(case["order"], B)
        t["x"] = r.normal(B, T, dtype=real)
    elif kind == "lpv":
        t["a"] = r.uniform(-0.99, 0.99, B, T, dtype=real)
        t["zi"] = r.normal(B)
        t["x"] = r.normal(B, T, dtype=real)
    elif kind == "diag":
        t["a"] = torch.polar(r.uniform(0.9, 0.999, B), r.uniform(0, math.pi, B))
        t["zi"] = torch.complex(r.normal(B), r.normal(B))
        t["x"] = torch.complex(r.normal(B, T, dtype=real), r.normal(B, T, dtype=real))
    elif kind in ("lpvm", "lpvss"):
        M = case["M"]
        a = _poly(torch.stack([r.curve(0.5, 0.98, B, T)] * (M // 2), -1),
                  torch.stack([r.curve(0, math.pi, B, T)] * (M // 2), -1),
                  torch.stack([r.curve(0.5, 0.9, B, T)] * (M % 2), -1) if M % 2
                  else torch.zeros(B, T, 0, device="cuda", dtype=torch.float64))[..., 1:]
        t["A"] = torch.zeros(B, T, M, M, device="cuda", dtype=torch.float64)
        t["A"][..., 0] = -a
        for i in range(M - 1):
            t["A"][..., i, i + 1] = 1
        t["zi"] = r.normal(B, M)
        if kind == "lpvm":
            t["x"] = r.normal(B, T, M, dtype=real)
        else:
            bn = torch.stack([r.curve(-1, 1, B, T) for _ in range(M + 1)], -1)
            t["b"], t["d"] = bn[..., 1:] - bn[..., :1] * a, bn[..., 0]
            t["x"] = r.normal(B, T, dtype=real)
    elif kind == "mimo":
        M, Fn, P = case["M"], case["F"], case["P"]
        # rotations and decays in an orthogonal basis per row
        q = torch.linalg.qr(r.normal(B, M, M).cpu())[0].cuda()
        d = torch.zeros(B, M, M, device="cuda", dtype=torch.float64)
        for i in range(0, M - 1, 2):
            rad, th = r.uniform(0.5, 0.98, B), r.uniform(0, math.pi, B)
            d[:, i, i] = d[:, i + 1, i + 1] = rad * torch.cos(th)
            d[:, i, i + 1], d[:, i + 1, i] = -rad * torch.sin(th), rad * torch.sin(th)
        if M % 2:
            d[:, M - 1, M - 1] = r.uniform(0.5, 0.98, B)
        t["A"] = _matmul(_matmul(q, d), q.mT)
        t["B"], t["C"], t["D"] = r.normal(M, Fn), r.normal(P, M), r.normal(P, Fn)
        t["zi"] = r.normal(B, M)
        t["x"] = r.normal(B, T, Fn, dtype=real)
    shape = {"lpvm": (B, T, case.get("M")), "mimo": (B, T, case.get("P"))}.get(kind, (B, T))
    if case["grad"] != "none":
        gy = r.normal(*shape, dtype=real)
        t["gy"] = torch.complex(gy, r.normal(*shape, dtype=real)) if kind == "diag" else gy
    return {k: v.to(dt).contiguous() for k, v in t.items()}


def _wanted(case):
    """The names of the tensors whose gradients the pass returns."""
    if case["grad"] == "none":
        return ()
    coefs = {"lfilter": ("b", "a"), "sos": ("sos",), "filtfilt": ("b", "a"), "lpv": ("a", "zi"), "diag": ("a", "zi"),
             "lpvm": ("A", "zi"), "lpvss": ("A", "b", "d", "zi"), "mimo": ("A", "B", "C", "D", "zi")}[case["kind"]]
    return ("x",) + (coefs if case["grad"] == "coef" else ())


def prepare(case, seed):
    t = _inputs(case, seed)
    for k in _wanted(case):
        t[k].requires_grad_(True)
    return case, t


# ---------------------------------------------------------------- the pass
def _call(case, t):
    """(outputs that the call returns): y, and the final state where the call gives one."""
    kind = case["kind"]
    if kind == "lfilter":
        if case["zi"]:
            return lti.lfilter(t["b"][:, 0], t["a"][:, 0], t["x"], zi=t["zi"], unroll_factor=1)
        y = t["x"]
        for s in range(case["chain"]):
            y = lti.lfilter(t["b"][:, s], t["a"][:, s], y, form="tdf2", unroll_factor=1)
        return (y,)
    if kind == "sos":
        return (lti.sosfilt(t["sos"], t["x"]),)
    if kind == "filtfilt":
        return (lti.filtfilt(t["b"], t["a"], t["x"], unroll_factor=1),)
    if kind == "lpv":
        return (lpv.linear_recurrence(t["a"], t["zi"], t["x"], unroll_factor=1),)
    if kind == "diag":
        return (lti.LTIRecurrence.apply(t["a"], t["zi"], t["x"]),)
    if kind == "lpvm":
        return (lpv.state_space_recursion(t["A"], t["zi"], t["x"], unroll_factor=1),)
    if kind == "lpvss":
        return lpv.state_space(t["A"], t["x"], B=t["b"], D=t["d"], zi=t["zi"], unroll_factor=1, out_idx=0)
    return lti.state_space(t["A"], t["x"], B=t["B"], C=t["C"], D=t["D"], zi=t["zi"], unroll_factor=1)


def run(state):
    case, t = state
    wanted = _wanted(case)
    if not wanted:
        with torch.no_grad():
            return list(_call(case, t))
    out = _call(case, t)
    grads = torch.autograd.grad(out[0], [t[k] for k in wanted], t["gy"])
    return [v.detach() for v in out] + list(grads)


def work(case):
    """Bytes: every input read once and every output written once.  Operations: the recurrence, its adjoint and
    the coefficient gradients as a sequential program does them."""
    kind, B, T = case["kind"], case["B"], case["T"]
    es, n = _BYTES[case["dtype"]], B * T
    back, coef = case["grad"] != "none", case["grad"] == "coef"
    if kind in ("lfilter", "sos", "filtfilt"):
        order = 2 if kind == "sos" else case["order"]
        stages = case["sections"] if kind == "sos" else 2 if kind == "filtfilt" else case["chain"]
        sig, par, per = 1, 0, stages * (4 * order + 2)
        per_grad = per * back + stages * (4 * order + 2) * coef
    elif kind in ("lpv", "diag"):
        sig, par = 1, (1 if kind == "lpv" else 0)
        cx = 4 if kind == "diag" else 1
        per, per_grad = 2 * cx, 2 * cx * back + 2 * cx * coef
    elif kind == "lpvm":
        M = case["M"]
        sig, par, per, per_grad = M, M * M, 2 * M * M, 2 * M * M * back + M * M * coef
    elif kind == "lpvss":
        M = case["M"]
        sig, par, per = 1, M * M + M + 1, 2 * (M * M + 2 * M + 1)
        per_grad = per * back + (M * M + M + 1) * coef
    else:
        M, Fn, P = case["M"], case["F"], case["P"]
        sig, par, per = Fn, 0, 2 * (M + P) * (M + Fn)
        per_grad = per * back + 2 * (M + P) * (M + Fn) * coef
    out = case["P"] if kind == "mimo" else sig
    # x, the per-step coefficients and gy in; y, grad x and the per-step coefficients' gradients out
    moved = sig + par + out + (out + sig) * back + par * coef
    return {"bytes": n * es * moved, "flops": n * (per + per_grad)}


# About four times the largest relative error of a pass against `exact` in 32 bits that draws showed, scaled to the
# type's rounding (in 64 bits `exact` rounds as the pass does, and ill-conditioned filters show it).  Chains of filters and orders above two amplify a sample's rounding by their gain (poles that
# nearly coincide, up to radius 0.98), as poles that vary in time do; scans of poles within 0.99 round once.
_REL = {"lpv": 3e-7, "diag": 4e-5, "lpvm": 1e-4, "lpvss": 1.5e-4, "mimo": 1e-6}


def tolerance(case):
    simple = case.get("order", case.get("sections", 0) + 1) <= 2 and case.get("chain", 1) == 1
    rel = _REL.get(case["kind"], 1e-5 if simple else 2e-4)
    return {"rel": rel * (2.0 ** -22 if case["dtype"] == "f64" else 1.0)}


# ---------------------------------------------------------------- in 64 bits
def _matmul(p, q):
    """p q of (batches of) small matrices, term by term."""
    return sum(p[..., :, k:k + 1] * q[..., k:k + 1, :] for k in range(p.size(-1)))


def _matvec(p, v):
    return sum(p[..., :, k] * v[..., k:k + 1] for k in range(p.size(-1)))


def _prefix(A, x):
    """h[t] = A[t] h[t-1] + x[t], h[-1] = 0, by doubling.  x [B, T, M]; A [B, T, M, M] or one per row [B, 1, M, M]."""
    h, T, fixed, d = x, x.size(1), A.size(1) == 1, 1
    while d < T:
        h = torch.cat([h[:, :d], h[:, d:] + _matvec(A if fixed else A[:, d:], h[:, :-d])], 1)
        if fixed:
            A = _matmul(A, A)
        elif 2 * d < T:
            A = torch.cat([A[:, :d], _matmul(A[:, d:], A[:, :-d])], 1)
        d *= 2
    return h


class _Scan(torch.autograd.Function):
    """_prefix with its adjoint, l[t] = g[t] + A[t+1]^H l[t+1]."""

    @staticmethod
    def forward(ctx, A, x):
        h = _prefix(A, x)
        ctx.save_for_backward(A, h)
        return h

    @staticmethod
    def backward(ctx, g):
        A, h = ctx.saved_tensors
        AH = A.mT.conj()
        if A.size(1) > 1:
            AH = torch.roll(AH, -1, 1).flip(1)
        lam = _prefix(AH, g.flip(1)).flip(1)
        prev = torch.cat([torch.zeros_like(h[:, :1]), h[:, :-1]], 1).conj()
        if A.size(1) > 1:
            return lam.unsqueeze(-1) * prev.unsqueeze(-2), lam
        M = h.size(-1)
        gA = [(lam[..., i] * prev[..., j]).sum(1) for i in range(M) for j in range(M)]
        return torch.stack(gA, -1).reshape(-1, 1, M, M), lam


def _states(A, zi, u):
    """(states before every step, state after the last) of h[t+1] = A[t] h[t] + u[t], h[0] = zi."""
    first = u[:, :1] + _matvec(A[:, :1], zi.unsqueeze(1))
    h = _Scan.apply(A, torch.cat([first, u[:, 1:]], 1))
    return torch.cat([zi.unsqueeze(1), h[:, :-1]], 1), h[:, -1]


def _filter(b, a, x, zi):
    """(y, zf) of b / a (a after its leading 1) per row, transposed direct form II."""
    M = a.size(-1)
    cols = [torch.zeros_like(a).unsqueeze(-1)] * (M - 1)
    A = torch.cat([-a.unsqueeze(-1)] + cols, -1) + torch.diag_embed(a.new_ones(M - 1), 1)
    g = b[..., 1:] - b[..., :1] * a
    h, zf = _states(A.unsqueeze(1), zi, x.unsqueeze(-1) * g.unsqueeze(1))
    return h[..., 0] + b[..., :1] * x, zf


def _reference(case, t):
    kind = case["kind"]
    if kind == "lfilter":
        y = t["x"]
        zi = t["zi"] if case["zi"] else y.new_zeros(case["B"], case["order"])
        for s in range(case["chain"]):
            y, zf = _filter(t["b"][:, s], t["a"][:, s], y, zi)
        return (y, zf) if case["zi"] else (y,)
    if kind == "sos":
        y = t["x"]
        for s in range(case["sections"]):
            q = t["sos"][:, s] / t["sos"][:, s, 3:4]
            y, _ = _filter(q[:, :3], q[:, 4:], y, y.new_zeros(case["B"], 2))
        return (y,)
    if kind == "filtfilt":
        b, a, x = t["b"], t["a"], t["x"]
        e = 3 * b.size(-1)
        # the state of a settled filter at a unit input, z = A z + g
        g = b[..., 1:] - b[..., :1] * a
        z = [b.sum(-1) / (1 + a.sum(-1)) - b[..., 0]]
        for i in range(a.size(-1) - 1):
            z.append(z[-1] + a[..., i] * z[0] - g[..., i])
        z = torch.stack(z, -1)
        y = F.pad(x, (e, e), mode="replicate")
        for _ in range(2):
            y = _filter(b, a, y, z * y[:, :1])[0].flip(-1)
        return (y[:, e:-e],)
    if kind in ("lpv", "diag"):
        A = t["a"].reshape(case["B"], -1, 1, 1)
        first = t["x"][:, :1] + A[:, 0, 0] * t["zi"].unsqueeze(1)
        return (_Scan.apply(A, torch.cat([first, t["x"][:, 1:]], 1).unsqueeze(-1)).squeeze(-1),)
    if kind == "lpvm":
        h, zf = _states(t["A"], t["zi"], t["x"])
        return (torch.cat([h[:, 1:], zf.unsqueeze(1)], 1),)
    if kind == "lpvss":
        h, zf = _states(t["A"], t["zi"], t["x"].unsqueeze(-1) * t["b"])
        return h[..., 0] + t["d"] * t["x"], zf
    h, zf = _states(t["A"].unsqueeze(1), t["zi"], _matvec(t["B"], t["x"]))
    return _matvec(t["C"], h) + _matvec(t["D"], t["x"]), zf


def exact(case, seed):
    t = {k: v.to(torch.complex128 if v.is_complex() else torch.float64) for k, v in _inputs(case, seed).items()}
    wanted = _wanted(case)
    for k in wanted:
        t[k].requires_grad_(True)
    out = _reference(case, t)
    grads = torch.autograd.grad(out[0], [t[k] for k in wanted], t["gy"]) if wanted else ()
    return [v.detach() for v in out] + list(grads)
