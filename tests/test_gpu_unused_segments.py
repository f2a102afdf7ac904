"""Training pair in time segments: nothing of what the last segment would leave alone (backward in time: the first) is read."""
import pytest
import torch

pytestmark = pytest.mark.gpu

N = 64


@pytest.mark.parametrize("B,T,H", [(2, 1400, 48),      # two segments
                                   (3, 1000, 28),      # three, the last of one token less than whole chunks
                                   (1, 8192, 32),      # eight
                                   (1, 1025, 4),       # sixteen and one token
                                   (1, 1300, 1)])      # tile form
def test_whatever_the_block_held_before(oracle, B, T, H):
    from rwkv_kernel import _native

    lib, C = _native.load(), H * N
    ins = oracle.make_inputs(B, T, H, N, 33)
    r, k, v, w, u, gy = (x.bfloat16().cuda().contiguous() for x in ins[:6])
    n = int(lib.wkv6_saved_bytes(_native.BF16, 0, B, T, C, H))
    st = torch.cuda.current_stream().cuda_stream
    P = lambda t: t.data_ptr()

    def run(fill):
        saved = torch.full((n,), fill, dtype=torch.uint8, device="cuda")   # (255: NaN wherever the kernels do not write)
        y, gr, gk, gv, gw = (torch.full_like(r, float("nan")) for _ in range(5))
        gu, gu_sum = torch.full((B, C), float("nan"), dtype=torch.bfloat16, device="cuda"), torch.full_like(u, float("nan"))
        _native.check(lib.wkv6_forward_save(st, _native.BF16, 0, B, T, C, H, P(r), P(k), P(v), P(w), P(u), P(y), P(saved), n))
        _native.check(lib.wkv6_backward_saved_sum(st, _native.BF16, 0, B, T, C, H, P(r), P(k), P(v), P(w), P(u), P(gy), P(gr), P(gk), P(gv),
                                                  P(gw), P(gu), P(gu_sum), P(saved), n))
        torch.cuda.synchronize()
        return y, gr, gk, gv, gw, gu, gu_sum

    for a, b in zip(run(255), run(0)):
        assert torch.isfinite(a).all() and torch.equal(a, b)
