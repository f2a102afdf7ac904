"""The torch flavour's native calls against the general way through the checks of the Python layer, and what autograd
offers around a node: a second backward, saved-tensor hooks, inference mode, other streams; transforms stay refused."""
import types
from fractions import Fraction

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DTYPES = (torch.bfloat16, torch.float16, torch.float32)


@pytest.fixture(scope="module")
def op():
    import rwkv_kernel
    return rwkv_kernel.RWKVKernelOperator(64, 1024)


def _inputs(B, T, H, dtype, grad=False, seed=3):
    g = torch.Generator().manual_seed(seed)
    C = H * 64
    r, k, v = (torch.randn(B, T, C, generator=g) for _ in range(3))
    w = torch.rand(B, T, C, generator=g) * 7.0 - 6.0
    u = torch.randn(H, 64, generator=g) * 0.5
    return [x.to(dtype).cuda().requires_grad_(grad) for x in (r, k, v, w, u)]


def _same(a, b):
    for x, y in zip(a, b):
        assert (x is None) == (y is None)
        assert x is None or (x.dtype == y.dtype and x.shape == y.shape and torch.equal(x, y))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("B,T,H", [(1, 1, 1), (3, 33, 2), (2, 100, 3)])
def test_plain_and_general_calls_agree(op, B, T, H, dtype):
    ins = _inputs(B, T, H, dtype)
    boxed = ins[:4] + [types.SimpleNamespace(value=ins[4])]   # a parameter in its wrapper: only the Python layer takes it
    _same(op(*ins), op(*boxed))
    _same(op(*ins, return_state=True), op(*boxed, return_state=True))
    for sdt in {torch.float32, torch.float32 if dtype == torch.float16 else dtype}:
        s0 = torch.randn(B, H, 64, 64, device="cuda").to(sdt)
        want = op(*ins, return_state=True, init_state=s0)
        assert want[1].dtype == sdt
        _same(want, op(*ins, return_state=True, init_state=s0, state_map=list(range(B))))
        spread = torch.empty(B, H, 64, 128, device="cuda", dtype=sdt)[..., ::2].copy_(s0)
        _same(want, op(*ins, return_state=True, init_state=spread))
        _same(op(*ins, return_state=True, init_state=s0[:1]), op(*ins, return_state=True, init_state=s0[0]))
    leaves = [x.requires_grad_(True) for x in ins]
    y = op(*leaves)[0]
    yb = op(*leaves[:4], types.SimpleNamespace(value=leaves[4]))[0]
    gy = torch.randn_like(y)
    _same(torch.autograd.grad(y, leaves, gy), torch.autograd.grad(yb, leaves, gy))


def test_fused_calls_agree(op):
    B, T, H = 2, 70, 2
    ins = _inputs(B, T, H, torch.bfloat16)
    boxed = ins[:4] + [types.SimpleNamespace(value=ins[4])]
    gate = torch.randn(B, T, H * 64, device="cuda", dtype=torch.bfloat16)
    sc, of = torch.randn(H, 64, device="cuda"), torch.randn(H * 64, device="cuda", dtype=torch.bfloat16)
    s0 = torch.randn(B, H, 64, 64, device="cuda")
    for kw in ({}, {"return_state": True}, {"return_state": True, "init_state": s0}, {"init_state": s0}):
        _same(op.forward_gn_gate(*ins, gate, sc, of, **kw), op.forward_gn_gate(*boxed, gate, sc.cpu(), of, **kw))
    leaves = [x.requires_grad_(True) for x in ins + [gate, sc, of]]
    out = op.forward_gn_gate(*leaves)[0]
    outb = op.forward_gn_gate(*leaves[:4], types.SimpleNamespace(value=leaves[4]), *leaves[5:])[0]
    g = torch.randn_like(out)
    # scale and offset are summed by additions whose order is not fixed; the others come out the same
    a, b = torch.autograd.grad(out, leaves, g), torch.autograd.grad(outb, leaves, g)
    _same(a[:6], b[:6])
    for x, y, leaf in zip(a, b, leaves):
        assert x.shape == leaf.shape and x.dtype == leaf.dtype
        torch.testing.assert_close(x, y, rtol=1e-2, atol=1e-4 * float(y.abs().max()))


@pytest.mark.parametrize("dtype,T", [(torch.bfloat16, 96), (torch.float32, 96), (torch.float32, 40)])
def test_autograd_around_the_node(op, dtype, T):
    leaves = _inputs(2, T, 2, dtype, grad=True)
    gy = torch.randn(2, T, 128, device="cuda", dtype=dtype)
    y = op(*leaves)[0]
    want = torch.autograd.grad(y, leaves, gy, retain_graph=True)
    again = torch.autograd.grad(y, leaves, gy)           # the saved states are gone: the plain backward
    with pytest.raises(RuntimeError):
        torch.autograd.grad(y, leaves, gy)               # ... and now the graph is
    for a, b in zip(want, again):
        torch.testing.assert_close(a, b, rtol=0, atol=(2e-2 if dtype == torch.bfloat16 else 1e-4) * float(a.abs().max()))
    with torch.autograd.graph.save_on_cpu():
        hooked = op(*leaves)[0]
    _same(torch.autograd.grad(hooked, leaves, gy), want)
    with pytest.raises(RuntimeError):                    # a saved input changed in place
        y = op(*leaves)[0]
        with torch.no_grad():
            leaves[0].mul_(1)
        torch.autograd.grad(y, leaves, gy)
    part = [x.detach() for x in leaves]
    part[2].requires_grad_(True)
    (gv,) = torch.autograd.grad(op(*part)[0], part[2:3], gy.expand_as(gy))
    _same([gv], want[2:3])
    with torch.inference_mode():
        z = op(*leaves)[0]
    assert z.is_inference() and torch.equal(z, y)
    with torch.no_grad():
        assert not op(*leaves)[0].requires_grad
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = torch.autograd.grad(op(*leaves)[0], leaves, gy)
    torch.cuda.current_stream().wait_stream(side)
    _same(got, want)


def test_transforms_stay_refused(op):
    ins = _inputs(2, 96, 2, torch.float32)
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda r: op(r, *ins[1:])[0].sum())(ins[0])
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda r: op(r, *ins[1:])[0])(ins[0][None])
    with pytest.raises((RuntimeError, NotImplementedError)):
        torch.func.jvp(lambda r: op(r, *ins[1:])[0], (ins[0],), (ins[0],))


@pytest.mark.parametrize("again", [False, True])
def test_parameters_gradients_hold_nothing_else(op, again):
    """torch takes a parameter's gradient over as it is: its storage is the parameter's own size, to the allocator's
    rounding at most, and not a block that also holds gradients of the size of the activations."""
    B, T, H, R = 4, 96, 4, 32
    C = H * 64
    mk = lambda *s: (torch.randn(*s, device="cuda") * 0.2).requires_grad_(True)

    def check(params, out, g):
        for i in range(2 if again else 1):           # (a second backward over one graph goes another way)
            for q in params:
                q.grad = None
            out.backward(g, retain_graph=again)
        for q in params:
            assert q.grad.shape == q.shape and q.grad.dtype == q.dtype
            assert q.grad.untyped_storage().nbytes() <= q.numel() * q.element_size() + 512

    for dtype in DTYPES:
        ins = _inputs(B, T, H, dtype, grad=True)
        y = op(*ins)[0]
        check(ins[4:], y, torch.randn_like(y))
    ins = _inputs(B, T, H, torch.bfloat16, grad=True)
    gate, sc, of = mk(B, T, C).bfloat16(), mk(H, 64), mk(C)
    out = op.forward_gn_gate(*ins, gate, sc, of)[0]
    check([ins[4], sc, of], out, torch.randn_like(out))
    ps = [mk(C), mk(5 * R, C), mk(5, C, R), mk(5, C)]
    outs = torch.stack(op.shift_mix(mk(B, T, C).bfloat16(), *ps))
    check(ps, outs, torch.randn_like(outs))


def test_flags_and_numbers_of_any_type(op):
    """return_state is anything with a truth, epsilon anything with a value, as in a Python signature."""
    ins = _inputs(2, 33, 2, torch.bfloat16)
    gate, p = ins[0], torch.ones(128, device="cuda")
    want = {s: op(*ins, return_state=s) for s in (False, True)}
    fused = {s: op.forward_gn_gate(*ins, gate, p, p, 0.25, return_state=s) for s in (False, True)}
    for flag in (0, 1, None, [], [0], "", "yes", torch.tensor(True), torch.zeros(1).cuda(), np.bool_(True), object()):
        _same(op(*ins, return_state=flag), want[bool(flag)])
        _same(op.forward_gn_gate(*ins, gate, p, p, 0.25, return_state=flag), fused[bool(flag)])
    for eps in (np.float32(0.25), torch.tensor(0.25), Fraction(1, 4), "0.25"):
        _same(op.forward_gn_gate(*ins, gate, p, p, eps, return_state=True), fused[True])
    with pytest.raises(Exception):
        op(*ins, return_state=torch.zeros(2))


@pytest.mark.parametrize("dtype", DTYPES)
def test_tensors_without_elements_are_refused(op, dtype):
    for B, T, C in ((2, 3, 0), (0, 3, 64), (2, 0, 64)):
        z, u = torch.zeros(B, T, C, dtype=dtype, device="cuda"), torch.zeros(C // 64, 64, dtype=dtype, device="cuda")
        sc = torch.zeros(C, device="cuda")
        for kw in ({}, {"return_state": True}):
            with pytest.raises(Exception):
                op(z, z, z, z, u, **kw)
            with pytest.raises(Exception):
                op.forward_gn_gate(z, z, z, z, u, z, sc, sc, **kw)


def test_input_side_gradients_of_some_outputs(op):
    B, T, C, R = 2, 40, 128, 32
    mk = lambda *s: torch.randn(*s, device="cuda") * 0.2
    x = mk(B, T, C).bfloat16().requires_grad_(True)
    ps = [p.requires_grad_(True) for p in (mk(C), mk(5 * R, C), mk(5, C, R), mk(5, C))]
    g = mk(B, T, C).bfloat16()
    outs = op.shift_mix(x, *ps)
    got = torch.autograd.grad(outs[3], [x, *ps], g)
    outs = op.shift_mix(x, *ps)
    want = torch.autograd.grad(outs, [x, *ps], [g if i == 3 else torch.zeros_like(g) for i in range(5)])
    for a, b, leaf in zip(got, want, [x, *ps]):
        assert a.shape == leaf.shape and a.dtype == leaf.dtype
        torch.testing.assert_close(a, b, rtol=0, atol=1e-5 * float(b.abs().max()) + 1e-30)
