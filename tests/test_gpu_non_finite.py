"""Infinities and NaN in the inputs."""
import pytest
import torch

from _util import cast_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("B,T,H,fused", [(5, 128, 32, False), (3, 127, 48, True), (2, 1024, 16, False)])
def test_v_out_of_range_reaches_no_token_of_an_earlier_group(oracle, B, T, H, fused, bad):
    # block form, in one piece, ragged and with the output stage, and in time segments: tokens in front of the 16 that hold an
    # infinity or a NaN keep their values, bit for bit, whether those 16 open a block of 32 or close it
    from rwkv_kernel import RWKVKernelOperator

    op = RWKVKernelOperator(64, T)
    dev, _ = cast_inputs(oracle.make_inputs(B, T, H, 64, 74)[:5], torch.bfloat16)
    gate, one, zero = torch.ones_like(dev[0]), torch.ones(H, 64, device="cuda"), torch.zeros(H, 64, device="cuda")
    call = lambda v: op.forward_gn_gate(dev[0], dev[1], v, dev[3], dev[4], gate, one, zero)[0] if fused else op(dev[0], dev[1], v, dev[3], dev[4], return_state=True)[0]
    want = call(dev[2])
    for t in (16, 27, 32, 47, 64 + 21):
        v = dev[2].clone()
        v[B - 1, t] = bad
        got = call(v)
        first = t // 16 * 16
        assert torch.equal(got[:, :first], want[:, :first]) and torch.equal(got[:B - 1], want[:B - 1]), t
        assert torch.isfinite(got[:, :first]).all() and not torch.isfinite(got[B - 1, t]).all()
