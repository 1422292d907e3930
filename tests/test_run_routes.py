"""philtorch_amd._run and _run_scan: the short route of plain eager calls against the op's
registered autograd, over the calls that must keep finding the op."""
import pytest
import torch

import philtorch_amd as pa
from philtorch_amd import lpv, lti

if not pa.EXTENSION_LOADED:  # pragma: no cover
    pytest.skip("extension not built", allow_module_level=True)


def _scan_case(name, dtype=torch.float64):
    g = torch.Generator().manual_seed(7)
    r = lambda *s: torch.rand(*s, generator=g, dtype=torch.float64).to(dtype) - 0.5  # noqa: E731
    B, T, M = 3, 7, 2
    return {"recur": (r(B, T), r(B), r(B, T)), "lti_recur": (r(B), r(B), r(B, T)),
            "recur2": (r(B, T, M, M), r(B, M), r(B, T, M)), "recurN": (r(T, 3, 3), r(B, 3), r(B, T, 3)),
            "lti_recur2": (r(B, M, M), r(B, M), r(B, T, M)), "lti_recurN": (r(3, 3), r(B, 3), r(B, T, 3))}[name]


SCANS = ["recur", "lti_recur", "recur2", "recurN", "lti_recur2", "lti_recurN"]


@pytest.mark.parametrize("name", SCANS)
@pytest.mark.parametrize("needs", [(0,), (1,), (2,), (0, 1, 2)])
def test_same_gradients_as_the_op(name, needs):
    op = getattr(torch.ops.philtorch, name)

    def grads(call):
        ts = [t.clone().requires_grad_(i in needs) for i, t in enumerate(_scan_case(name))]
        y = call(*ts)
        g = torch.linspace(-1, 1, y.numel(), dtype=y.dtype).reshape(y.shape)
        first = torch.autograd.grad(y, [ts[i] for i in needs], g, create_graph=True)
        again = torch.autograd.grad(call(*ts), [ts[i] for i in needs], g)
        # second order, where the first gradient depends on the inputs
        s = sum((f * f).sum() for f in first)
        second = torch.autograd.grad(s, [ts[i] for i in needs], allow_unused=True) if s.requires_grad else ()
        return [y, *first, *again, *second]

    for a, b in zip(grads(lambda *t: pa._run_scan(name, *t)), grads(op)):
        assert (a is None) == (b is None)
        assert a is None or torch.allclose(a, b, rtol=1e-12, atol=1e-12)


@pytest.mark.parametrize("name", SCANS)
def test_no_gradient_recorded(name):
    ts = _scan_case(name)
    want = getattr(torch.ops.philtorch, name)(*ts)
    y = pa._run_scan(name, *ts)
    assert not y.requires_grad and torch.equal(y, want)
    with torch.no_grad():
        y = pa._run_scan(name, *[t.clone().requires_grad_(True) for t in ts])
    assert not y.requires_grad and torch.equal(y, want)


def test_saved_tensor_hooks_see_the_saved_tensors():
    seen = []
    ts = [t.clone().requires_grad_(True) for t in _scan_case("recur")]
    with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(t.shape) or t, lambda t: t):
        y = lpv.linear_recurrence(ts[0], ts[1], ts[2], unroll_factor=1)
    assert len(seen) >= 3
    y.sum().backward()
    assert all(t.grad is not None for t in ts)


def test_forward_mode_keeps_its_route():
    """The Functions with a jvp keep it; the ops without one refuse as before."""
    import torch.autograd.forward_ad as fw

    A, zi, x = _scan_case("recur2")
    with fw.dual_level():
        xd = fw.make_dual(x, torch.ones_like(x))
        assert not pa._plain((A, zi, xd))
        t = fw.unpack_dual(lpv.state_space_recursion(A, zi, xd, unroll_factor=1)).tangent
        assert t is not None and torch.allclose(t, lpv.state_space_recursion(A, 0 * zi, torch.ones_like(x)))
        a, z, u = _scan_case("lti_recur")
        ud = fw.make_dual(u, torch.ones_like(u))
        t = fw.unpack_dual(lti.LTIRecurrence.apply(a, z, ud)).tangent
        assert torch.allclose(t, lti.LTIRecurrence.apply(a, 0 * z, torch.ones_like(u)))
        a, z, u = _scan_case("recur")
        out = []
        for call in (lambda v: pa._run_scan("recur", a, z, v), lambda v: torch.ops.philtorch.recur(a, z, v)):
            try:
                out.append(fw.unpack_dual(call(fw.make_dual(u, torch.ones_like(u)))).tangent is None)
            except (RuntimeError, NotImplementedError) as e:
                out.append(type(e))
        assert out[0] == out[1]


def test_functorch_grad_and_modes_reach_the_op():
    from torch.utils._python_dispatch import TorchDispatchMode

    a, z, u = _scan_case("recur")
    with pytest.raises(RuntimeError):  # torch.library's autograd has no functorch rule: refused by op and API alike
        torch.func.grad(lambda v: lpv.linear_recurrence(a, z, v, unroll_factor=1).sum())(u)
    b, zb, ub = _scan_case("lti_recur")  # the Function with a setup_context has one
    got = torch.func.grad(lambda v: (lti.LTIRecurrence.apply(b, zb, v) ** 2).sum())(ub)
    v = ub.clone().requires_grad_(True)
    (lti.LTIRecurrence.apply(b, zb, v) ** 2).sum().backward()
    assert torch.allclose(got, v.grad)
    v = u.clone().requires_grad_(True)

    calls = []

    class Log(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            calls.append(str(func))
            return func(*args, **(kwargs or {}))

    with Log():
        lpv.linear_recurrence(a, z, u, unroll_factor=1)
    assert any("philtorch.recur" in c for c in calls)

    class Sub(torch.Tensor):
        pass

    assert not pa._plain((a.as_subclass(Sub),))
    assert pa._plain((a, torch.nn.Parameter(z)))
    y = torch.compile(lambda v: lpv.linear_recurrence(a, z, v, unroll_factor=1), backend="aot_eager")(v)
    assert torch.allclose(y, lpv.linear_recurrence(a, z, u, unroll_factor=1))


def _whole_graph_cases():
    """name -> (call, arguments, the op the captured graph has to hold).  The matrix scans and
    LTIRecurrence have a jvp of their own, which dynamo refuses where a gradient is recorded."""
    g = torch.Generator().manual_seed(3)
    r = lambda *s: torch.rand(*s, generator=g) - 0.5  # noqa: E731
    B, T, M = 3, 9, 2
    return {
        "lpv.linear_recurrence": (lambda a, z, x: lpv.linear_recurrence(a, z, x, unroll_factor=1),
                                  (r(B, T), r(B), r(B, T)), "recur"),
        "LTIRecurrence": (lti.LTIRecurrence.apply, (r(B), r(B), r(B, T)), "lti_recur"),
        "lpv.state_space_recursion": (lambda A, z, x: lpv.state_space_recursion(A, z, x, unroll_factor=1),
                                      (r(B, T, M, M), r(B, M), r(B, T, M)), "recur2"),
        "lti.state_space_recursion": (lambda A, z, x: lti.state_space_recursion(A, z, x, unroll_factor=1),
                                      (r(B, 3, 3), r(B, 3), r(B, T, 3)), "lti_recurN"),
        "lti.lfilter": (lambda b, a, x: lti.lfilter(b, a, x, unroll_factor=1), (r(B, 3), r(B, 2), r(B, T)),
                        "lti_recur2"),
        "lti.filtfilt": (lambda b, a, x: lti.filtfilt(b, a, x, padlen=3, unroll_factor=1),
                         (r(B, 3), r(B, 2), r(B, T)), "lti_recur2"),
    }


@pytest.mark.parametrize("grad,name", [(False, n) for n in _whole_graph_cases()] + [(True, "lpv.linear_recurrence")])
def test_compiles_whole(grad, name):
    f, args, op = _whole_graph_cases()[name]
    args = [t.clone().requires_grad_(grad) for t in args]
    seen = []

    def backend(gm, example):
        seen.extend(str(n.target) for n in gm.graph.nodes)
        return gm.forward

    torch._dynamo.reset()
    y = torch.compile(lambda *t: f(*t), fullgraph=True, backend=backend)(*args)
    assert any(f"philtorch.{op}" in s for s in seen)
    want = f(*args)
    assert torch.allclose(y, want, rtol=1e-5, atol=1e-6)  # the same kernel on the same inputs
    if grad:
        for p, q in zip(torch.autograd.grad(y.sum(), args), torch.autograd.grad(want.sum(), args)):
            assert torch.allclose(p, q, rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("name", ["_fused_lfilter", "_fused_biquad", "_fused_filtfilt", "_sosfilt_fused"])
def test_fused_routes_are_captured_whole(name):
    """The routes of HIP tensors, where a gradient is recorded: what dynamo hands its backend (their
    kernels take no CPU tensors, so the graph is looked at and not run)."""
    from philtorch_amd.lti import filtering

    g = torch.Generator().manual_seed(3)
    r = lambda *s: (torch.rand(*s, generator=g) - 0.5).requires_grad_(True)  # noqa: E731
    b, a, x = r(3, 3), r(3, 2), r(3, 9)
    sos = torch.cat([torch.rand(3, 2, 3), torch.ones(3, 2, 1), torch.rand(3, 2, 2) / 4], -1).requires_grad_(True)
    f, args, op = {
        "_fused_lfilter": (lambda b, a, x: filtering._fused_lfilter(b, a, x, None, "tdf2"), (b, a, x),
                           "lfilter_ss_states"),
        "_fused_biquad": (lambda b, a, x: filtering._fused_biquad(b, a, x, None), (b, a, x), "biquad"),
        "_fused_filtfilt": (lambda b, a, x: filtering._fused_filtfilt(b, a, x, None, 0), (b, a, x),
                            "filtfilt_states"),
        "_sosfilt_fused": (lambda s, x: filtering._sosfilt_fused(s, x, None)[0], (sos, x), "sosfilt"),
    }[name]
    seen = []

    def backend(gm, example):
        seen.extend(str(n.target) for n in gm.graph.nodes)
        raise RuntimeError("seen")

    torch._dynamo.reset()
    with pytest.raises(Exception, match="seen"):
        torch.compile(f, fullgraph=True, backend=backend)(*args)
    assert any(f"philtorch.{op}" in s for s in seen)


@pytest.mark.parametrize("name", list(_whole_graph_cases()))
def test_exports_strictly(name):
    f, args, op = _whole_graph_cases()[name]

    class Mod(torch.nn.Module):
        def forward(self, *t):
            return f(*t)

    ep = torch.export.export(Mod(), args, strict=True)
    assert any(f"philtorch.{op}" in str(n.target) for n in ep.graph.nodes)
    assert torch.allclose(ep.module()(*args), f(*args), rtol=1e-5, atol=1e-6)
