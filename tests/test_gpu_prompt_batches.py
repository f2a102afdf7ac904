"""Batches of prompts of any length in time segments (wkv6_forward_workspace_bytes_any_length)."""
import numpy as np
import pytest
import torch

from _util import cast_inputs, check_close, check_composite, rel_l2, to_np

pytestmark = pytest.mark.gpu

N = 64
CHUNK = 2


# fit: segments of each sequence, counted by the workspace: two states and a decay a segment and pair
@pytest.mark.parametrize("B,T,H,segments", [(2, 1000, 8, 16),     # whole chunks, the last of 40 tokens
                                            (3, 705, 16, 4),      # the last segment of one chunk, of one token
                                            (7, 577, 12, 3),      # 84 pairs, three segments
                                            (2, 1030, 1, 6),      # tile form, segments of three chunks
                                            (4, 200, 16, 4), (3, 260, 28, 3), (2, 330, 64, 2),   # the shortest (the last two with the output stage alone)
                                            (2, 4161, 5, 14),     # the last one of a single token
                                            (4, 2100, 32, 2)])    # two segments
@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("sdt", [torch.float32, torch.bfloat16])
def test_any_length(oracle, B, T, H, segments, fused, sdt):
    from rwkv_kernel import _native

    lib, C = _native.load(), H * N
    code = {torch.bfloat16: _native.BF16, torch.float32: _native.F32}
    n = int(lib.wkv6_forward_workspace_bytes_any_length(_native.BF16, CHUNK, B, T, C, H))
    assert n == B * segments * H * (2 * N * N + N) * 4
    assert int(lib.wkv6_forward_workspace_bytes(_native.BF16, CHUNK, B, T, C, H)) == 0   # (none of these lengths divides evenly)
    ins = oracle.make_inputs(B, T, H, N, 90 + B, with_state=True)
    ins[3].view(B, T, H, N)[B - 1, T // 2, 0, 3:9] = 6.0    # a segment that is redone one timestep at a time
    dev, ref = cast_inputs(ins[:5], torch.bfloat16)
    kinds = min(2, B)
    s_dev, s_ref = cast_inputs([ins[6][:kinds]], sdt)
    smap = torch.tensor([(b + 1) % kinds for b in range(B)], device="cuda")
    g = torch.Generator(device="cuda").manual_seed(B)
    gate = torch.randn(B, T, C, generator=g, device="cuda").bfloat16()
    scale, offset = (torch.randn(H, N, generator=g, device="cuda") for _ in range(2))
    ws = torch.empty(n + 64, dtype=torch.uint8, device="cuda")
    P = lambda t: None if t is None else t.data_ptr()

    def run(s_in, s_out, index, size):
        y = torch.full((B, T, C), float("nan"), dtype=torch.bfloat16, device="cuda")
        ws.fill_(255)   # (NaN in every state it holds)
        st = torch.cuda.current_stream().cuda_stream
        if fused:
            _native.check(lib.wkv6_forward_gn_gate_ex(st, _native.BF16, code[sdt], B, T, C, H, 1, P(index), *map(P, dev), P(s_in),
                                                      P(gate), P(scale), P(offset), 64e-5, P(y), P(s_out), P(ws), size))
        else:
            _native.check(lib.wkv6_forward_with_state_ex(st, _native.BF16, code[sdt], CHUNK, B, T, C, H, 1, P(index), *map(P, dev), P(s_in),
                                                         P(y), P(s_out), P(ws), size))
        torch.cuda.synchronize()
        assert (ws[size:] == 255).all()
        return y, s_out

    y, sT = run(s_dev[0], torch.empty(B, H, N, N, dtype=sdt, device="cuda"), smap, n)
    y_ref, sT_ref = oracle.forward_c(*ref, N, s_ref[0], smap.tolist())
    if fused:
        f64 = lambda t: torch.tensor(to_np(t))
        z = torch.nn.functional.layer_norm(torch.tensor(y_ref).view(B, T, H, N), (N,), eps=64e-5)
        check_composite("out", y, ((z * f64(scale) + f64(offset)).view(B, T, C) * f64(gate)).numpy())
    else:
        check_close("y", y, y_ref, torch.bfloat16)
    check_close("sT", sT, sT_ref, torch.bfloat16)
    # in one piece with less than the workspace of the segments, and close to it
    y1, sT1 = run(s_dev[0], torch.empty_like(sT), smap, n - 16)
    assert rel_l2(to_np(sT1), to_np(sT)) <= 1e-2 and np.isfinite(to_np(y1)).all()
    # the final states where the initial ones lie
    s_all = s_dev[0][smap].contiguous()
    y2, sT2 = run(s_all, torch.empty_like(sT), None, n)
    assert torch.equal(y, y2) and torch.equal(sT, sT2)
    y3, sT3 = run(s_all, s_all, None, n)
    assert torch.equal(y, y3) and torch.equal(sT, sT3)


@pytest.mark.parametrize("B,T,H", [(2, 330, 16), (2, 1000, 8), (3, 705, 16), (7, 577, 12), (1, 1337, 32), (2, 1300, 64)])
def test_segments_are_no_less_exact_than_one_piece(oracle, B, T, H):
    # segments run the block form, one piece of so few pairs the tile form.  y of many thousands of values: the 2-norm of its error
    # differs by 0.2 % from seed to seed, the two forms' on the same inputs by less than that around their own difference
    from rwkv_kernel import _native

    lib, C = _native.load(), H * N
    dev, ref = cast_inputs(oracle.make_inputs(B, T, H, N, 60 + B)[:5], torch.bfloat16)
    n = int(lib.wkv6_forward_workspace_bytes_any_length(_native.BF16, CHUNK, B, T, C, H))
    ws = torch.empty(n, dtype=torch.uint8, device="cuda")
    P = lambda t: t.data_ptr()

    def run(size):
        y, sT = torch.empty_like(dev[0]), torch.empty(B, H, N, N, device="cuda")
        _native.check(lib.wkv6_forward_with_state_ex(torch.cuda.current_stream().cuda_stream, _native.BF16, _native.F32, CHUNK, B, T, C, H, 0, None,
                                                     *map(P, dev), None, P(y), P(sT), P(ws), size))
        return to_np(y), to_np(sT)

    y_ref, s_ref = oracle.forward_c(*ref, N)
    (y, s), (y1, s1) = run(n), run(0)
    assert n > 0 and not np.array_equal(y, y1)
    assert rel_l2(y, y_ref) <= rel_l2(y1, y_ref)
    assert rel_l2(s, s_ref) <= 1.001 * rel_l2(s1, s_ref)   # (the same roundings in another order of additions)
