"""Forward and backward of a training call captured in graphs of their own."""
import pytest
import torch

pytestmark = pytest.mark.gpu

N = 64
NAMES = "gr gk gv gw gu ggate gscale goffset".split()
SHAPES = [(1, 70, 3),       # tile form
          (5, 150, 32),     # block form
          (9, 150, 32),     # block form, two pairs to a workgroup
          (1, 1100, 2),     # segments in tile form
          (2, 1100, 8)]     # segments in block form


def _leaves(B, T, H, fused, dtype=torch.bfloat16):
    g = torch.Generator(device="cuda").manual_seed(B * T + H)

    def normal(*shape, dt=dtype):
        return torch.randn(*shape, generator=g, device="cuda").to(dt)

    r, k, v, gate, gout = (normal(B, T, H * N) for _ in range(5))
    w = (torch.rand(B, T, H * N, generator=g, device="cuda") * 7 - 6).to(dtype)
    leaves = [r, k, v, w, normal(H, N)]
    if fused:
        leaves += [gate, normal(H, N, dt=torch.float32), normal(H, N, dt=torch.float32)]
    return [x.requires_grad_(True) for x in leaves], gout if dtype != torch.float16 else gout.float()


def _forward(leaves, fused):
    import rwkv_kernel

    op = rwkv_kernel.RWKVKernelOperator(N, 16384)
    return (op.forward_gn_gate if fused else op)(*leaves)[0]


def _agree(got, want, B, T):
    for name, a, b in zip(NAMES, got, want):
        if name in ("gscale", "goffset"):
            # fp32 sums of the same B T terms in another order: each addition rounds by 2^-24 of a partial sum, some sqrt(B T) of which
            # matter where terms of either sign cancel
            assert (a - b).norm() <= 2.0 ** -24 * (B * T) ** 0.5 * b.norm() + 1e-5, name
        else:
            assert torch.equal(a, b), name


CASES = [(s, True, torch.bfloat16) for s in SHAPES] + [((2, 1100, 8), False, torch.bfloat16), ((5, 150, 32), False, torch.bfloat16),
                                                       ((2, 100, 3), False, torch.float32), ((1, 400, 8), False, torch.float16)]


@pytest.mark.parametrize("shape,fused,dtype", CASES)
def test_replays_of_a_backward_over_one_forward(shape, fused, dtype):
    B, T, H = shape
    leaves, gout = _leaves(B, T, H, fused, dtype)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        want = [x.clone() for x in torch.autograd.grad(_forward(leaves, fused), leaves, gout)]
        out = _forward(leaves, fused)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        got = torch.autograd.grad(out, leaves, gout, retain_graph=True)   # (what it reads stays allocated)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        _agree(got, want, B, T)
        torch.full((1 << 20,), float("nan"), device="cuda")   # (the program's own work between replays)


@pytest.mark.parametrize("shape,fused,dtype", CASES)
def test_gradients_outlive_replays_of_the_forward(shape, fused, dtype):
    B, T, H = shape
    leaves, gout = _leaves(B, T, H, fused, dtype)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        want = [x.clone() for x in torch.autograd.grad(_forward(leaves, fused), leaves, gout)]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        out = _forward(leaves, fused)
    graph.replay()
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        kept = torch.autograd.grad(out, leaves, gout)
    torch.cuda.synchronize()
    _agree(kept, want, B, T)
    graph.replay()
    torch.cuda.synchronize()
    _agree(kept, want, B, T)


@pytest.mark.parametrize("shape", SHAPES)
def test_make_graphed_callables(shape):
    # forward and backward in graphs of their own, two backward passes over one forward
    B, T, H = shape
    leaves, gout = _leaves(B, T, H, True)
    want = torch.autograd.grad(_forward(leaves, True), leaves, gout)
    call = torch.cuda.make_graphed_callables(lambda *x: _forward(x, True), tuple(x.detach().clone().requires_grad_(True) for x in leaves))
    for _ in range(2):
        out = call(*leaves)
        for _ in range(2):
            got = [x.clone() for x in torch.autograd.grad(out, leaves, gout, retain_graph=True)]
            _agree(got, want, B, T)
