"""Large calls without a backward read their inputs past the caches, the largest write their output past them: the same bits as smaller calls."""
import pytest
import torch

pytestmark = pytest.mark.gpu

N = 64
MIB = 2 ** 20


@pytest.fixture(scope="module")
def op():
    assert torch.cuda.is_available(), "these tests need the GPU"
    import rwkv_kernel

    return rwkv_kernel.RWKVKernelOperator(N, 16384)


# A pair's result does not depend on the pairs around it, so the first `few` rows by themselves, a call that stays below the limits
# (28 MiB a tensor for what is read, 320 MiB for what is written), have to be what they are among all rows.
@pytest.mark.parametrize("B,few,T,H,sdt", [(9, 8, 800, 32, torch.float32),      # read past the caches, 28.1 MiB; several pairs to a workgroup
                                           (8, 7, 897, 32, torch.bfloat16),     # one pair to a workgroup and a chunk of one token, 28.0 MiB
                                           (20, 8, 820, 32, torch.float32),     # 64.1 MiB, a ragged end
                                           (65, 16, 320, 24, torch.float32),    # 60.9 MiB, heads that do not divide the chip
                                           (37, 8, 448, 32, None)])             # 64.75 MiB, without a state
@pytest.mark.parametrize("fused", [False, True])
def test_large_calls_give_the_bits_of_small_ones(op, B, few, T, H, sdt, fused):
    assert few * T * H * N * 2 < 28 * MIB <= B * T * H * N * 2
    g = torch.Generator(device="cuda").manual_seed(B)

    def normal(*shape, dtype=torch.bfloat16):
        return torch.randn(*shape, generator=g, device="cuda").to(dtype)

    C = H * N
    r, k, v = (normal(B, T, C) for _ in range(3))
    w = (torch.rand(B, T, C, generator=g, device="cuda") * 7 - 6).bfloat16()
    w[2, T // 2:, :N] = 6.0    # a pair that is redone one timestep at a time
    u = normal(H, N)
    s0 = None if sdt is None else normal(B, H, N, N, dtype=sdt)
    gate, scale, offset = normal(B, T, C), normal(H, N, dtype=torch.float32), normal(H, N, dtype=torch.float32)

    def call(n):
        ins = [x[:n].contiguous() for x in (r, k, v, w)]
        state = None if s0 is None else s0[:n].contiguous()
        if fused:
            return op.forward_gn_gate(*ins, u, gate[:n].contiguous(), scale, offset, return_state=True, init_state=state)
        return op(*ins, u, return_state=True, init_state=state)

    y, s = call(B)
    y_few, s_few = call(few)
    assert torch.equal(y[:few], y_few) and torch.equal(s[:few], s_few)


@pytest.mark.parametrize("fused", [False, True])
def test_outputs_larger_than_the_caches(op, fused):
    # 323 MiB a tensor, a ragged end: y or the fused output is written past the caches, too
    test_large_calls_give_the_bits_of_small_ones(op, 81, 6, 1023, 32, torch.float32, fused)


# (several pairs to a workgroup in both calls: the backward of one pair to a workgroup is another kernel, whose gw rounds differently)
@pytest.mark.parametrize("B,few,T,H", [(15, 10, 500, 32),     # 29.3 MiB, a ragged end
                                       (43, 12, 401, 32),     # 67.4 MiB
                                       (33, 11, 512, 32)])    # 66 MiB, whole chunks
def test_large_training_calls_with_the_output_stage(op, B, few, T, H):
    # the saving forward reads past the caches: the output and every row's gradients as in a call below the limit
    assert few * T * H * N * 2 < 28 * MIB <= B * T * H * N * 2
    g = torch.Generator(device="cuda").manual_seed(B)

    def normal(*shape, dtype=torch.bfloat16):
        return torch.randn(*shape, generator=g, device="cuda").to(dtype)

    C = H * N
    r, k, v, gate, gout = (normal(B, T, C) for _ in range(5))
    w = (torch.rand(B, T, C, generator=g, device="cuda") * 7 - 6).bfloat16()
    w[2, T // 2:, :N] = 6.0    # a pair that is redone one timestep at a time
    u, scale, offset = normal(H, N), normal(H, N, dtype=torch.float32), normal(H, N, dtype=torch.float32)

    def call(n):
        rows = [x[:n].clone().requires_grad_(True) for x in (r, k, v, w, gate)]
        out, _ = op.forward_gn_gate(*rows[:4], u, rows[4], scale, offset)
        return [out, *torch.autograd.grad(out, rows, gout[:n].contiguous())]

    for name, a, b in zip("out gr gk gv gw ggate".split(), call(B), call(few)):
        assert torch.equal(a[:few], b), name


@pytest.mark.parametrize("B,T,H", [(9, 800, 32), (3, 100, 4)])   # past the caches, and a call of which no form asks
@pytest.mark.parametrize("sdt", [torch.float32, torch.bfloat16])
def test_inference_is_the_stateful_call(B, T, H, sdt):
    from rwkv_kernel import _native

    lib, C = _native.load(), H * N
    g = torch.Generator(device="cuda").manual_seed(T)
    r, k, v = (torch.randn(B, T, C, generator=g, device="cuda").bfloat16() for _ in range(3))
    w = (torch.rand(B, T, C, generator=g, device="cuda") * 7 - 6).bfloat16()
    u, s = torch.randn(H, N, generator=g, device="cuda").bfloat16(), torch.randn(B, H, N, N, generator=g, device="cuda").to(sdt)
    code = {torch.float32: _native.F32, torch.bfloat16: _native.BF16}[sdt]
    P = lambda t: None if t is None else t.data_ptr()

    def call(entry, has, y, ys):
        return entry(torch.cuda.current_stream().cuda_stream, _native.BF16, code, _native.ALGO_AUTO, B, T, C, H, has, None, P(r), P(k), P(v), P(w),
                     P(u), P(s) if has else None, P(y), P(ys), None, 0)

    entries = (lib.wkv6_forward_inference, lib.wkv6_forward_with_state_ex, lib.wkv6_forward_with_state_for_backward)
    for has in (0, 1):
        got = []
        for entry in entries:
            y, ys = torch.full_like(r, float("nan")), torch.full_like(s, float("nan"))
            _native.check(call(entry, has, y, ys))
            y2 = torch.full_like(r, float("nan"))
            _native.check(call(entry, has, y2, None))        # (the final state is not wanted)
            assert torch.equal(y, y2)
            got.append((y, ys))
        for y, ys in got[1:]:
            assert torch.equal(y, got[0][0]) and torch.equal(ys, got[0][1])
    for entry in entries:   # refused alike
        assert call(entry, 1, None, s) == call(entries[1], 1, None, s) != 0
