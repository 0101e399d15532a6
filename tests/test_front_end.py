"""The layer's front-end kernel (``ttc_lqr_front_end`` / ``_backward``) against the same formulas as torch
operators in 64 bits, and the layer's route through it."""
import ctypes

import pytest
import torch

from ttc.layers.front_end import front_end, front_end_torch

# (tokens, heads, d, du, b_rank, q_rank): one wave's width and its neighbours, ranks beyond it, no rank
SHAPES = [(1, 1, 1, 1, 1, 1), (3, 2, 16, 16, 16, 16), (5, 3, 63, 20, 65, 7), (2, 8, 64, 64, 32, 64), (4, 1, 65, 3, 0, 130),
          (33, 5, 24, 20, 8, 33), (3, 2, 7, 0, 4, 4), (2, 1, 0, 5, 1, 0)]


def _proj(N, H, d, du, rb, rq, dtype, device):
    g = torch.Generator().manual_seed(N + d)
    x = torch.randn(N, (3 * d + 2 * du + rq + 1) * H + rb + rq, generator=g) * 4.0
    x[0, ::7] = 25.0   # softplus is the identity above 20
    x[-1, ::5] = -40.0  # and underflows; R is clamped at 1e-6
    if N > 2:
        x[1] = 0.0
    return x.to(device=device, dtype=dtype)


def _reference64(proj, bias, dims):
    """The front-end in the dtype of its arguments throughout (``front_end_torch`` normalises in fp32), and per
    normalised output the factor s = 1 / sqrt(|v|^2 + 1e-6) of its rows."""
    H, d, du, rb, rq = dims
    head = [d, d, du, rq, 1 + du + d]
    heads, cB, cQ = torch.split(proj, [sum(head) * H, rb, rq], dim=-1)
    h0, A, R, cQf, lg = torch.split(heads.reshape(-1, H, sum(head)), head, dim=-1)
    F = torch.nn.functional
    vs = [A, cB, F.softplus(cQ), F.softplus(R), F.softplus(cQf)]
    ss = [torch.rsqrt((v * v).sum(-1, keepdim=True) + 1e-6) for v in vs]
    A, cB, cQ, R, cQf = (v * s for v, s in zip(vs, ss))
    lg = -F.softplus(lg) - (0 if bias is None else F.relu(-bias))
    lgA, lgB, lgQ = torch.split(lg, [1, du, d], dim=-1)
    return (A, cB, cQ, torch.clamp(R, min=1e-6), cQf, lgA.squeeze(-1), lgB, lgQ, h0), ss


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("with_bias", [False, True])
def test_front_end_kernel(shape, with_bias):
    """Values and gradients against 64 bits, to first order in u = 2^-24.  A softplus (expf, log1pf) is 6 u off; a sum
    of n products in a wave adds n / 64 + 6 roundings; so s = rsqrt(sum + 1e-6) is (n / 128 + 12) u off
    and a value (n / 128 + 20) u of itself.  The gradient s g_i - v_i (v . g) s^3 has terms of at most
    s |g_i| and s |g|, off by (n / 128 + 20) u and (5 n / 128 + 65) u with the softplus's derivative."""
    N, H, d, du, rb, rq = shape
    dims = (H, d, du, rb, rq)
    n, u = max(d, du, rb, rq), 2.0 ** -24
    a = _proj(*shape, torch.float32, "cuda").requires_grad_(True)
    b = a.detach().double().cpu().requires_grad_(True)
    bias = torch.linspace(-2, 1, 1 + du + d) if with_bias else None
    ba = None if bias is None else bias.cuda().requires_grad_(True)
    bb = None if bias is None else bias.double().requires_grad_(True)
    ya, (yb, ss) = front_end(a, ba, dims), _reference64(b, bb, dims)
    g = torch.Generator().manual_seed(9)
    # (R's clamp is a step in its gradient: entries within rounding of it are left out)
    ws = [torch.randn(y.shape, generator=g).double() for y in yb]
    ws[3] = ws[3] * ((yb[3].detach() - 1e-6).abs() > 1e-9)
    ins_a, ins_b = [a] + ([ba] if with_bias else []), [b] + ([bb] if with_bias else [])
    ga = torch.autograd.grad([(y * w.float().cuda()).sum() for y, w in zip(ya, ws)], ins_a)
    gb = torch.autograd.grad([(y * w).sum() for y, w in zip(yb, ws)], ins_b)
    for x, y in list(zip(ya, yb)) + list(zip(ga, gb)):
        assert x.is_contiguous() and x.shape == y.shape
    for x, y in zip(ya, yb):
        assert bool(((x.detach().double().cpu() - y.detach()).abs() <= (n / 128 + 20) * u * y.detach().abs()).all())
    size = [s.detach() * (w.abs() + w.norm(dim=-1, keepdim=True)) for s, w in zip(ss, ws)]
    lg = torch.cat([ws[5].unsqueeze(-1), ws[6], ws[7]], dim=-1)
    heads = torch.cat([ws[8], size[0], size[3], size[4], lg], dim=-1)
    size = torch.cat([heads.reshape(N, -1), size[1], size[2]], dim=-1).abs()
    assert bool(((ga[0].double().cpu() - gb[0]).abs() <= (n / 25 + 65) * u * size).all())
    if with_bias:
        assert bool(((ga[1].double().cpu() - gb[1]).abs() <= (N * H + 1) * u * lg.abs().sum((0, 1))).all())


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(9, 2, 6, 5, 3, 4), (7, 3, 65, 3, 2, 70)])
def test_front_end_keeps_nan_and_infinity(shape):
    """NaN and infinities in the projection, the bias and the gradients come out where the operators have them,
    forward and backward, and leave the other segments alone; finite values agree to fp32 rounding."""
    N, H, d, du, rb, rq = shape
    dims, nan, inf = shape[1:], float("nan"), float("inf")
    x = _proj(*shape, torch.float32, "cuda")
    head = 3 * d + 2 * du + rq + 1
    at = [0, d, 2 * d, 2 * d + du, 2 * d + du + rq, 2 * d + du + rq + 1, head - 1]  # h0, A, R, coeff_Qf, lgA, lgB, lgQ
    for n, v in ((2, nan), (3, inf), (4, -inf)):
        for k, c in enumerate(at):  # alternating heads
            x[n, (k % H) * head + c] = v
        x[n, H * head] = x[n, H * head + rb] = v
    bias = torch.linspace(-2, 1, 1 + du + d, device="cuda")
    bias[[2, 1, 3, 1 + du]] = torch.tensor([nan, inf, -inf, nan], device="cuda")
    g = torch.Generator().manual_seed(5)
    ws = None
    got = []
    for f in (front_end, front_end_torch):
        a, b = x.clone().requires_grad_(True), bias.clone().requires_grad_(True)
        ys = f(a, b, dims)
        if ws is None:
            ws = [torch.randn(y.shape, generator=g).cuda() for y in ys]
            ws[6][-1, 0, 0] = inf  # reaches the bias whose relu is off
        got.append([y.detach() for y in ys] + list(torch.autograd.grad(ys, [a, b], ws)))
    for p, q in zip(*got):
        assert torch.equal(p.isnan(), q.isnan()) and torch.equal(p.isinf(), q.isinf())
        assert torch.equal(p[q.isinf()], q[q.isinf()])
        ok = q.isfinite()
        scale = max(float(q[ok].abs().max()), 1.0)
        assert float((p - q)[ok].abs().max()) <= (max(dims) / 2 + 10) * 2.0 ** -24 * 8 * scale


@pytest.mark.gpu
@pytest.mark.parametrize("factored", [True, False])
def test_layer_raises_on_a_nan_bias(factored):
    """A NaN in ``bias_gamma`` reaches the solver, whose status word raises."""
    from ttc import TTCLayer
    torch.manual_seed(0)
    layer = TTCLayer(32, 32, 16, 2, 8, 8, gamma_bias=True, factored=factored).cuda()
    x = torch.randn(5, 32, device="cuda")
    layer(x, T=4)
    with torch.no_grad():
        layer.bias_gamma[3] = float("nan")
    with pytest.raises(RuntimeError):
        layer(x, T=4)


@pytest.mark.gpu
def test_front_end_beyond_one_launch():
    """2^26 + 6 (token, head) units, more than the 2^32 - 1 threads of one launch hold: both ends of the
    tokens, and the seam of the two launches, get the operators' values, forward and backward.  The
    norms' gradients are differences of two terms of at most s = 1 / |v| <= 5 here (inputs of magnitude
    1/2 to 3/2, softplus at least 0.2), with about four roundings each: 8 * 2^-24 * 5 apart at most."""
    N, dims = (1 << 25) + 3, (1, 1, 1, 0, 0)
    proj = torch.rand(N, 6, device="cuda", generator=torch.Generator(device="cuda").manual_seed(3)) * 2 - 1
    proj = (proj + proj.sign() * 0.5).requires_grad_(True)
    ys = front_end(proj, None, dims)
    ws = [torch.ones_like(y) for y in ys]
    (g,) = torch.autograd.grad(ys, proj, ws)
    for part in (slice(0, 64), slice(N // 2, N // 2 + 64), slice(N - 128, N)):
        p = proj.detach()[part].clone().requires_grad_(True)
        want = front_end_torch(p, None, dims)
        (gw,) = torch.autograd.grad(want, p, [w[part] for w in ws])
        for a, b in zip([y[part] for y in ys] + [g[part]], list(want) + [gw]):
            assert torch.allclose(a, b, rtol=1e-5, atol=3e-6)


@pytest.mark.gpu
def test_front_end_second_derivative_and_partial_gradients():
    """Under create_graph the backward is differentiable, as the operators' is; outputs without a
    gradient count as zero."""
    dims = (2, 6, 5, 3, 4)
    a = _proj(3, *dims, torch.float32, "cuda").requires_grad_(True)
    b = a.detach().clone().requires_grad_(True)
    for t, f in ((a, front_end), (b, front_end_torch)):
        y = f(t, None, dims)
        (g,) = torch.autograd.grad((y[3] ** 2).sum() + (y[0] * 3).sum(), t, create_graph=True)
        t.first = g.detach()
        (t.second,) = torch.autograd.grad((g ** 2).sum(), t)
    assert torch.allclose(a.first, b.first, rtol=1e-4, atol=1e-6)
    assert torch.allclose(a.second, b.second, rtol=1e-3, atol=1e-6)
    (p,) = torch.autograd.grad(front_end(a, None, dims)[8].sum(), a)
    assert float(p.sum()) == 3 * 2 * 6


@pytest.mark.gpu
def test_other_sizes_broadcast_or_raise():
    """A projection of another width raises and a bias of another size broadcasts or raises, as in the operators:
    the kernel, which would read beyond either, is not launched."""
    dims = (2, 6, 5, 3, 4)
    x = _proj(3, *dims, torch.float32, "cuda")
    for wrong in (x[:, :-1], torch.cat([x, x], dim=1), x[:, :40]):
        with pytest.raises(RuntimeError):
            front_end(wrong, None, dims)
    for bias in (torch.full((1,), -0.5, device="cuda"), torch.full((), -0.5, device="cuda")[None]):
        for p, q in zip(front_end(x, bias, dims), front_end_torch(x, bias, dims)):
            assert torch.equal(p, q)
    for n in (11, 13, 24):
        with pytest.raises(RuntimeError):
            front_end(x, torch.zeros(n, device="cuda"), dims)


def test_front_end_argument_validation():
    from ttc.solvers._lib import lib
    p = ctypes.c_void_p(16)
    assert lib.ttc_lqr_front_end(p, None, 0, 1, 4, 4, 2, 2, *[p] * 9, None) == 0      # nothing to do
    assert lib.ttc_lqr_front_end(None, None, 1, 1, 4, 4, 2, 2, *[p] * 9, None) == 1
    assert lib.ttc_lqr_front_end(p, None, 1, 0, 4, 4, 2, 2, *[p] * 9, None) == 1
    assert lib.ttc_lqr_front_end(p, None, 1, 1, 4, -1, 2, 2, *[p] * 9, None) == 1
    assert lib.ttc_lqr_front_end(p, None, 1, 1, 4, 4, 2, 2, *[p] * 8, None, None) == 1
    assert lib.ttc_lqr_front_end_backward(p, 1, 1, 4, 4, 2, 2, *[p] * 9, None, None) == 1
    assert lib.ttc_lqr_front_end_backward(p, 0, 1, 4, 4, 2, 2, *[None] * 9, None, None) == 0


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_front_end_compiles_as_one_graph(device):
    """``torch.compile(fullgraph=True)`` of the layer's front-end traces the operators, forward and backward."""
    from ttc import TTCLayer
    torch.manual_seed(0)
    layer = TTCLayer(8, 8, 4, 2, 3, 3, gamma_bias=True, solver_impl="riccati" if device == "cpu" else "hip").to(device)
    x = torch.randn(5, 8, device=device)
    for f in (layer.solver_inputs, layer.factored_inputs):
        torch._dynamo.reset()
        got, want = torch.compile(f, backend="aot_eager", fullgraph=True)(x), f(x)
        assert all(torch.allclose(p, q, rtol=1e-5, atol=1e-7) for p, q in zip(got, want))
        ws = list(layer.parameters())
        gs = [torch.autograd.grad(sum((y * y).sum() for y in ys), ws, allow_unused=True) for ys in (got, want)]
        assert all(p is None or torch.allclose(p, q, rtol=1e-4, atol=1e-6) for p, q in zip(*gs))
    torch._dynamo.reset()


def test_cpu_and_other_dtypes_use_the_operators():
    dims = (2, 6, 5, 3, 4)
    for dt in (torch.float32, torch.bfloat16):
        x = _proj(2, *dims, dt, "cpu")
        for u, v in zip(front_end(x, None, dims), front_end_torch(x, None, dims)):
            assert u.dtype == dt and torch.equal(u, v)


@pytest.mark.gpu
def test_transforms_and_tracing_see_the_operators():
    """vmap, forward-mode AD (both interfaces), tracing and fake tensors, which see nothing of an autograd
    Function, get the operators' results (the same formulas, so the same bits)."""
    import torch.autograd.forward_ad as fwAD
    dims = (2, 6, 5, 3, 4)
    x = _proj(3, *dims, torch.float32, "cuda")
    v = torch.linspace(-1, 1, x.numel(), device="cuda").reshape(x.shape)
    for k in (0, 2, 3, 8):
        want = torch.func.jvp(lambda t: front_end_torch(t, None, dims)[k], (x,), (v,))
        got = torch.func.jvp(lambda t: front_end(t, None, dims)[k], (x,), (v,))
        assert all(torch.equal(p, q) for p, q in zip(got, want))
        with fwAD.dual_level():
            y = fwAD.unpack_dual(front_end(fwAD.make_dual(x, v), None, dims)[k])
            assert torch.equal(y.tangent, want[1])
    xs = torch.stack([x, 2 * x])
    want = torch.func.vmap(lambda t: front_end_torch(t, None, dims)[3])(xs)
    assert torch.equal(torch.func.vmap(lambda t: front_end(t, None, dims)[3])(xs), want)
    traced = torch.jit.trace(lambda t: front_end(t, None, dims)[3], x)
    assert torch.allclose(traced(2 * x), want[1], rtol=1e-5, atol=0)
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode() as mode:
        assert front_end(mode.from_tensor(x), None, dims)[3].shape == (3, 2, 5)


@pytest.mark.gpu
def test_dispatch_modes_and_batched_gradients_see_the_operators():
    """Dispatch modes over plain tensors (make_fx on real tensors, a mode that counts) record the operators, not
    empty outputs that a kernel fills unseen; batched gradients pass the backward; all with the operators'
    values, forward and backward."""
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.utils._python_dispatch import TorchDispatchMode
    dims = (2, 6, 5, 3, 4)
    x = _proj(3, *dims, torch.float32, "cuda")
    bias = torch.linspace(-2, 1, 12, device="cuda")

    def step(f):
        def run(t, b):
            t, b = t.detach().requires_grad_(), b.detach().requires_grad_()
            ys = f(t, b, dims)
            return [*ys, *torch.autograd.grad(sum((y * y).sum() for y in ys), (t, b))]
        return run

    traced = make_fx(step(front_end))(x, bias)
    for p, q in zip(traced(2 * x, 0.5 * bias), step(front_end_torch)(2 * x, 0.5 * bias)):
        assert torch.equal(p, q)

    class Names(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.seen = getattr(self, "seen", set()) | {func.overloadpacket}
            return func(*args, **(kwargs or {}))

    with Names() as mode:
        front_end(x, bias, dims)
    assert torch.ops.aten.softplus in mode.seen
    t = x.clone().requires_grad_()
    b = bias.clone().requires_grad_()
    ys = front_end(t, b, dims)
    with Names() as mode:
        torch.autograd.grad(ys, (t, b), [torch.ones_like(y) for y in ys], retain_graph=True)
    assert torch.ops.aten.softplus_backward in mode.seen

    def jacobian(f):
        t, b = x.clone().requires_grad_(), bias.clone().requires_grad_()
        y = f(t, b, dims)[3]
        seeds = torch.eye(y.numel(), device="cuda").reshape(-1, *y.shape)
        return torch.autograd.grad(y, (t, b), seeds, is_grads_batched=True, allow_unused=True)
    for p, q in zip(jacobian(front_end), jacobian(front_end_torch)):
        assert (p is None and q is None) or torch.equal(p, q)


@pytest.mark.gpu
def test_no_grad_forward_writes_no_stash(monkeypatch):
    """Under no_grad a layer whose parameters require gradients runs the forward without a stash (nothing
    asks whether one fits), with the same bits as a recorded forward."""
    from ttc import TTCLayer
    from ttc.solvers import hip_lqr as hl
    torch.manual_seed(0)
    x = torch.randn(64, 32, device="cuda")
    asked = []
    fits = hl._stash_fits
    monkeypatch.setattr(hl, "_stash_fits", lambda *a: asked.append(a) or fits(*a))
    for factored in (True, False):
        layer = TTCLayer(32, 32, 16, 8, 16, 16, factored=factored).cuda()
        y = layer(x, T=8)
        assert asked
        asked.clear()
        with torch.no_grad():
            assert torch.equal(y, layer(x, T=8))
        assert not asked
