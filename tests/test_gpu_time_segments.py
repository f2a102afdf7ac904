"""Time segments of bf16 sequences: what a segment hands to the next one."""
import ctypes

import numpy as np
import pytest
import torch

from _util import cast_inputs, rel_l2, to_np

pytestmark = pytest.mark.gpu

N = 64


@pytest.fixture(scope="module")
def op():
    assert torch.cuda.is_available(), "these tests need the GPU"
    import rwkv_kernel

    return rwkv_kernel.RWKVKernelOperator(N, 16384)


def _inputs(oracle, B, T, H, seed, strong=False, slow=False):
    ins = oracle.make_inputs(B, T, H, N, seed, with_state=True)
    if slow:
        ins[3] -= 3.0
    if strong:   # in every 32 tokens one whose decay leaves the reach of the scaled operands, in six channels of each head
        ins[3].view(B, T, H, N)[:, 5::32, :, 3:9] = 6.0
        ins[3].view(B, T, H, N)[:, -1, :, 3:9] = 6.0   # (the last segment may be of one token)
    dev, ref = cast_inputs(ins[:5], torch.bfloat16)
    s_dev, s_ref = cast_inputs([ins[6][:B]], torch.float32)
    return dev, ref, s_dev[0], s_ref[0]


def _state_of_scaled_tiles(ref, s0):
    """The final state in float64 with the tile form's one rounding: k decayed to the end of its 16 tokens, as bf16."""
    k, v, w = (torch.tensor(x) for x in ref[1:4])
    B, T, C = k.shape
    S = torch.tensor(s0)
    for t0 in range(0, T, 16):
        x = torch.exp(w[:, t0:t0 + 16].reshape(B, -1, C // N, N))
        c = x.cumsum(1)
        kk = (k[:, t0:t0 + 16].reshape(x.shape) * torch.exp(c - c[:, -1:])).float().bfloat16().double()
        vv = v[:, t0:t0 + 16].reshape(x.shape)
        S = S * torch.exp(-c[:, -1]).unsqueeze(-1) + torch.matmul(kk.permute(0, 2, 3, 1), vv.permute(0, 2, 1, 3))
    return S.numpy()


@pytest.mark.parametrize("B,T,H", [(1, 449, 16), (1, 1337, 32), (2, 512, 8), (1, 2049, 5), (1, 2880, 17)])
def test_segments_round_k_once_to_the_end_of_its_sixteen_tokens(op, oracle, B, T, H):
    # 1 to 3 chunks to a segment, whole and ragged; decays slow enough for a state to be made of many tiles.  fp32 leaves e^c an error
    # of some 2^-24 |c log2 e| a tile, |c| <= 2.2: about 4e-7 with the roundings around it, so one element in 5000 rounds the other
    # way, by 2^-8 of itself: 2^-8 / sqrt(5000) = 6e-5 of the state.  (Rounded anywhere else the two states are as far apart as each
    # is from float64, some 1e-3.)
    dev, ref, s_dev, s_ref = _inputs(oracle, B, T, H, 71, slow=True)
    _, sT = op(*dev, return_state=True, init_state=s_dev)
    assert rel_l2(to_np(sT), _state_of_scaled_tiles(ref, s_ref)) <= 6e-5


@pytest.mark.parametrize("B,T,H", [(1, 449, 16), (1, 1337, 32), (2, 512, 8), (1, 1025, 43), (2, 4096, 8)])
def test_state_of_strong_decays_stays_fp32_across_segments(op, oracle, B, T, H):
    # Rows out of the scaled operands' reach are redone one timestep at a time in fp32; the decays here forget what is older than
    # some hundred tokens, so a state carries the rounding of few steps: 5.5e-8 measured, 2^-20 (sixteen times 2^-24) allowed.
    dev, ref, s_dev, s_ref = _inputs(oracle, B, T, H, 72, strong=True)
    gate = torch.ones_like(dev[0])
    one, zero = torch.ones(H, N, device="cuda"), torch.zeros(H, N, device="cuda")
    want = oracle.forward_c(*ref, N, s_ref)[1]
    _, sT = op(*dev, return_state=True, init_state=s_dev)
    _, oT = op.forward_gn_gate(*dev, gate, one, zero, return_state=True, init_state=s_dev)
    assert rel_l2(to_np(sT), want) <= 2.0 ** -20 and rel_l2(to_np(oT), want) <= 2.0 ** -20


@pytest.mark.parametrize("B,T,H", [(1, 1100, 8), (2, 2048, 8), (1, 4095, 24)])
def test_gradient_of_the_state_behind_strong_decays_stays_fp32(op, oracle, B, T, H):
    # the same backwards in time: dL/dS_0 is chained from what every segment sends back, read back to front
    dev, ref, s_dev, s_ref = _inputs(oracle, B, T, H, 73, strong=True)
    gy_dev, gy_ref = cast_inputs([torch.randn(B, T, H * N, generator=torch.Generator().manual_seed(1))], torch.bfloat16)
    gs = torch.randn(B, H, N, N, generator=torch.Generator().manual_seed(2))
    leaves = [x.clone().requires_grad_(True) for x in dev + [s_dev]]
    y, sT = op(*leaves[:5], return_state=True, init_state=leaves[5])
    got = torch.autograd.grad((y, sT), leaves, (gy_dev[0], gs.cuda()))[5]
    want = oracle.backward_state_c(*ref, gy_ref[0], N, s_ref, to_np(gs))[5]
    assert rel_l2(to_np(got), want) <= 2.0 ** -20
    assert np.isfinite(to_np(sT)).all()


@pytest.mark.parametrize("B,T,H,launches", [(1, 1023, 8, 2), (2, 1000, 24, 2), (1, 1024, 8, 7), (2, 2047, 64, 2), (2, 2048, 64, 7)])
def test_backward_through_the_state_in_segments_where_its_launches_pay(oracle, B, T, H, launches):
    from rwkv_kernel import _native

    lib, C = _native.load(), H * N
    r, k, v, w, u, gy = (x.bfloat16().cuda().contiguous() for x in oracle.make_inputs(B, T, H, N, 76))
    s0, gs = (torch.randn(B, H, N, N, device="cuda") for _ in range(2))
    outs, gu, gs0 = [torch.empty_like(r) for _ in range(4)], torch.empty(B, C, dtype=torch.bfloat16, device="cuda"), torch.empty_like(s0)
    n = lib.wkv6_backward_with_state_workspace_bytes(_native.BF16, 0, B, T, C, H)
    ws = torch.empty(int(n), dtype=torch.uint8, device="cuda")
    P = lambda t: t.data_ptr()

    def call():
        _native.check(lib.wkv6_backward_with_state(torch.cuda.current_stream().cuda_stream, _native.BF16, 0, B, T, C, H, *map(P, (r, k, v, w, u, s0, gy, gs)),
                                                   *map(P, outs), P(gu), P(gs0), P(ws), n))

    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        call()
    nodes = ctypes.c_size_t()
    hip = ctypes.CDLL(next(x.split()[-1] for x in open("/proc/self/maps") if "libamdhip64" in x))   # the one that torch runs on
    assert hip.hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(nodes)) == 0
    assert nodes.value == launches
