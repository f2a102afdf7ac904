"""Full-precision forward: y and the saved states leave through waves of their own."""
import pytest
import torch

from _util import cast_inputs, check_close

pytestmark = pytest.mark.gpu

N = 64


@pytest.mark.parametrize("dt", [torch.float32, torch.float16])
@pytest.mark.parametrize("B,T,H", [(2, 64, 3),       # two whole chunks
                                   (3, 65, 2),       # a chunk of one token, the first of its wave's rows
                                   (1, 79, 5),       # the last row of the first half of a chunk
                                   (2, 127, 4),      # all rows but one
                                   (9, 96, 32)])     # more pairs than compute units
def test_saving_and_plain_forward_store_the_same(oracle, B, T, H, dt):
    import rwkv_kernel

    op = rwkv_kernel.RWKVKernelOperator(N, 16384)
    dev, ref = cast_inputs(oracle.make_inputs(B, T, H, N, 40 + T)[:5], dt)
    y_plain, _ = op(*dev)                                    # no states kept
    y_state, sT = op(*dev, return_state=True)                # a final state
    leaves = [x.clone().requires_grad_(True) for x in dev]
    y_saved, _ = op(*leaves)                                 # chunk states kept
    assert torch.equal(y_plain, y_saved) and torch.equal(y_plain, y_state)
    y_ref, sT_ref = oracle.forward_c(*ref, N)
    check_close("y", y_saved, y_ref, torch.float32)
    check_close("sT", sT, sT_ref, torch.float32)
    gy = torch.randn_like(y_saved)
    grads = torch.autograd.grad(y_saved, leaves, gy)         # from the saved states
    want = oracle.backward_c(*ref, gy.double().cpu().numpy(), N)
    for name, g, g_ref in zip("gr gk gv gw gu".split(), grads, want):
        # (fp16 tensors: the gradients are rounded to fp16 once, 2^-11 of a value)
        check_close(name, g.reshape(g_ref.shape), g_ref, torch.float32 if dt == torch.float32 else torch.float16, is_grad=True)
