"""The final states written where the initial ones lie (ys = s, which the interface allows without a state_map or with the
identity): the same bits as with buffers apart."""
import pytest
import torch

pytestmark = pytest.mark.gpu

N = 64
AUTO, CHUNK = 0, 2
BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


def _compare(oracle, dt, sdt, B, T, H, fused=False, identity=False, strong=False, algo=AUTO, twice=3):
    from rwkv_kernel import _native

    lib, C = _native.load(), H * N
    code = {BF16: _native.BF16, F16: _native.F16, F32: _native.F32}
    ins = oracle.make_inputs(B, T, H, N, 75, with_state=True)
    if strong:   # pairs that are redone one timestep at a time: one decay out of reach in the middle, one at the end of a sequence
        ins[3].view(B, T, H, N)[:, T // 2, ::2, 3:9] = 6.0
        ins[3].view(B, T, H, N)[B - 1, T - 1, :, 20:24] = 6.0
    r, k, v, w, u = (x.to(dt).cuda().contiguous() for x in ins[:5])
    s = ins[6].to(sdt).cuda().contiguous()
    gate, one, zero = torch.ones_like(r), torch.ones(H, N, device="cuda"), torch.zeros(H, N, device="cuda")
    smap = torch.arange(B, device="cuda") if identity else None
    n = lib.wkv6_forward_workspace_bytes(code[dt], CHUNK if fused else algo, B, T, C, H)
    ws = torch.empty(max(int(n), 16), dtype=torch.uint8, device="cuda")
    P = lambda t: None if t is None else t.data_ptr()

    def run(s_in, s_out):
        y = torch.full((B, T, C), float("nan"), dtype=torch.float32 if dt == F16 else dt, device="cuda")
        st = torch.cuda.current_stream().cuda_stream
        if fused:
            _native.check(lib.wkv6_forward_gn_gate_ex(st, code[dt], code[sdt], B, T, C, H, 1, P(smap), P(r), P(k), P(v), P(w), P(u), P(s_in),
                                                      P(gate), P(one), P(zero), 64e-5, P(y), P(s_out), P(ws), n))
        else:
            _native.check(lib.wkv6_forward_with_state_ex(st, code[dt], code[sdt], algo, B, T, C, H, 1, P(smap), P(r), P(k), P(v), P(w), P(u),
                                                         P(s_in), P(y), P(s_out), P(ws), n))
        torch.cuda.synchronize()
        return y, s_out

    y, sT = run(s, torch.full_like(s, float("nan")))
    assert torch.isfinite(y).all() and torch.isfinite(sT).all()
    for _ in range(twice):
        s_io = s.clone()
        y2, _ = run(s_io, s_io)
        assert torch.equal(y, y2) and torch.equal(sT, s_io)
    return n


@pytest.mark.parametrize("identity", [False, True])
@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("sdt", [F32, BF16])
@pytest.mark.parametrize("B,T,H,strong", [(1, 449, 16, False), (1, 1337, 32, True), (2, 4096, 8, False), (1, 1025, 43, False), (4, 512, 16, True)])
def test_time_segments(oracle, B, T, H, strong, sdt, fused, identity):
    # 8, 7, 16, 5 and 4 segments in block form: the last one of a sequence ends while others may still start
    assert _compare(oracle, BF16, sdt, B, T, H, fused, identity, strong, CHUNK) > 0


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("sdt", [F32, BF16])
@pytest.mark.parametrize("B,T,H", [(5, 64, 32), (9, 150, 32), (70, 70, 4)])
def test_pairs_redone_per_timestep_in_block_form(oracle, B, T, H, sdt, fused):
    # one pair to a workgroup, two of them, ragged; every other head holds a decay out of reach
    _compare(oracle, BF16, sdt, B, T, H, fused, strong=True, algo=CHUNK)


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("sdt", [F32, BF16])
@pytest.mark.parametrize("B,T,H", [(4, 150, 32), (3, 100, 32), (2, 320, 5), (1, 50, 2), (3, 64, 100)])
def test_pairs_redone_per_timestep_in_tile_form(oracle, B, T, H, sdt, fused):
    # a pair shared by two workgroups, by four (whole chunks, and shorter than one; with the output stage always one), and several pairs to
    # a workgroup
    _compare(oracle, BF16, sdt, B, T, H, fused, strong=True, algo=CHUNK)


@pytest.mark.parametrize("dt", [F32, F16])
@pytest.mark.parametrize("B,T,H", [(2, 64, 3), (3, 203, 32), (2, 1100, 4)])
def test_pairs_redone_per_timestep_in_full_precision(oracle, B, T, H, dt):
    _compare(oracle, dt, F32, B, T, H, strong=True)


@pytest.mark.parametrize("dt,sdt", [(F32, F32), (F16, F32), (BF16, F32), (BF16, BF16)])
@pytest.mark.parametrize("B,T,H", [(9, 1, 5), (3, 20, 4), (8, 128, 32)])
def test_calls_in_one_piece(oracle, B, T, H, dt, sdt):
    # a single timestep, the per-timestep kernels and the chunk forms, no pair redone
    _compare(oracle, dt, sdt, B, T, H)
