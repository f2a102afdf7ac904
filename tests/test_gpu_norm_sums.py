"""Gradients of the norm's scale and offset: sums that the forward clears for the first backward over a graph."""
import pytest
import torch

pytestmark = pytest.mark.gpu

N = 64


SHAPES = [(1, 70, 3),        # tile form, a pair to a workgroup
          (3, 64, 100),      # tile form, several pairs to a workgroup
          (5, 150, 32),      # block form
          (9, 150, 32),      # block form, two pairs to a workgroup
          (1, 1100, 2),      # segments in tile form
          (2, 1100, 8),      # segments in block form
          (9, 800, 32)]     # inputs read past the caches


@pytest.mark.parametrize("B,T,H", SHAPES)
def test_the_forward_clears_the_sums(B, T, H):
    from rwkv_kernel import _native

    lib, C = _native.load(), H * N
    g = torch.Generator(device="cuda").manual_seed(T)
    r, k, v, gate = (torch.randn(B, T, C, generator=g, device="cuda").bfloat16() for _ in range(4))
    w = (torch.rand(B, T, C, generator=g, device="cuda") * 7 - 6).bfloat16()
    u, scale, offset = torch.randn(H, N, device="cuda").bfloat16(), torch.randn(H, N, device="cuda"), torch.randn(H, N, device="cuda")
    n = int(lib.wkv6_saved_bytes(_native.BF16, _native.ALGO_CHUNK, B, T, C, H))
    out, y, stats, saved = torch.empty_like(r), torch.empty_like(r), torch.empty(B, T, H, 2, device="cuda"), torch.empty(n, dtype=torch.uint8, device="cuda")
    sums = torch.full((4, H, N), float("nan"), device="cuda")
    P = lambda t: t.data_ptr()
    _native.check(lib.wkv6_forward_gn_gate_save_sums(torch.cuda.current_stream().cuda_stream, _native.BF16, B, T, C, H, P(r), P(k), P(v), P(w), P(u),
                                                     P(gate), P(scale), P(offset), 64e-5, P(out), P(y), P(stats), P(saved), n, P(sums[1]), P(sums[2])))
    torch.cuda.synchronize()
    assert (sums[1:3] == 0).all() and torch.isnan(sums[0]).all() and torch.isnan(sums[3]).all()


@pytest.mark.parametrize("B,T,H", SHAPES)
def test_first_and_second_backward_give_the_same_sums(B, T, H):
    import rwkv_kernel

    op = rwkv_kernel.RWKVKernelOperator(N, 16384)
    g = torch.Generator(device="cuda").manual_seed(T)

    def normal(*shape, dtype=torch.bfloat16):
        return torch.randn(*shape, generator=g, device="cuda").to(dtype)

    r, k, v, gate, gout = (normal(B, T, H * N) for _ in range(5))
    w = (torch.rand(B, T, H * N, generator=g, device="cuda") * 7 - 6).bfloat16()
    u, scale, offset = normal(H, N), normal(H, N, dtype=torch.float32), normal(H, N, dtype=torch.float32)
    scale.requires_grad_(True)
    offset.requires_grad_(True)
    for _ in range(2):
        poison = [torch.full((H, N), float("nan"), device="cuda") for _ in range(8)]   # (what the allocator hands out next for a sum is not zero)
        del poison
        out, _ = op.forward_gn_gate(r, k, v, w, u, gate, scale, offset)
        first = torch.autograd.grad(out, [scale, offset], gout, retain_graph=True)
        second = torch.autograd.grad(out, [scale, offset], gout)
        for a, b in zip(first, second):
            # fp32 sums of the same B T terms in another order: each addition rounds by 2^-24 of a partial sum, some sqrt(B T) of which
            # matter where terms of either sign cancel
            assert a.data_ptr() != b.data_ptr() and torch.isfinite(a).all()
            assert (a - b).norm() <= 2.0 ** -24 * (B * T) ** 0.5 * b.norm() + 1e-5
        # and of outputs that are no leaves' only use: the offset's gradient is the sum of gout * gate over the tokens
        want = (gout.double() * gate.double()).sum((0, 1)).view(H, N)
        assert (first[1].double() - want).norm() <= 1e-5 * want.norm()
