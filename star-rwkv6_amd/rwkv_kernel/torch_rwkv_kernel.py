"""torch flavour of the WKV6 operator: autograd nodes over libwkv6_gfx950.so.

Mirrors rwkv_kernel/torch_rwkv_kernel.py of the reference (constructor, call signature, argument
checks, 2-tuple return, dtype rules) but launches on torch's CURRENT stream.  Calls in their plain form
(contiguous tensors of one shape, one initial state per row or none) go straight to csrc/torch_binding.cpp, built
ahead of time; what that declines is checked, or brought into that form, here.

Where the reference's torch flavour is broken as committed, the behaviour of its working
flavours is implemented: the default state_map for a single shared state has length batch
(ops_rwkv_kernal.py:54, against torch_rwkv_kernel.py:155), the stateful call actually runs
(torch_rwkv_kernel.py:93 names a binding that does not exist), and state_map is moved to the
device before the kernel reads it.
"""
import torch

from . import _native

_DTYPE_CODE = {torch.bfloat16: _native.BF16, torch.float16: _native.F16, torch.float32: _native.F32}


def _out_dtype(dt):
    # rwkv_kernel/torch_rwkv_kernel.py:35 -- float16 inputs produce float32 outputs
    return torch.float32 if dt == torch.float16 else dt


def _stream():
    return torch.cuda.current_stream().cuda_stream


_STAGGER = 256   # bytes


def _staggered(count, shape, dtype, device, first=1):
    """`count` tensors of one shape out of ONE allocation, the k-th starting (first + k) * 256 bytes
    past where a tensor of its own would start.  A workgroup of the kernels walks all (B,T,C) tensors
    of a call row by row in step; torch's allocator hands out large blocks on 2 MiB boundaries, and
    tensors whose bases agree modulo 4 KiB keep sending those streams to the same memory channel at
    the same moment (about 5 % of the training pair at B8 T1024 C2048).  The tensors are views of
    the common block, which lives as long as any of them."""
    n = 1
    for d in shape:
        n *= d
    es = torch.empty((), dtype=dtype).element_size()
    step = (n * es + _STAGGER - 1) // _STAGGER * _STAGGER + _STAGGER
    block = torch.empty(count * step + first * _STAGGER, dtype=torch.uint8, device=device)
    return [block[first * _STAGGER + i * step: first * _STAGGER + i * step + n * es].view(dtype).view(shape) for i in range(count)]


def _ptr(t):
    return None if t is None else t.data_ptr()


class _WKV6:
    """Stateless operator with gradients (rwkv_kernel/torch_rwkv_kernel.py:14-75)."""

    @staticmethod
    def apply(B, T, C, H, r, k, v, w, u, algo):
        assert r.dtype == k.dtype == v.dtype == w.dtype == u.dtype
        assert r.dtype in _DTYPE_CODE
        for x in (r, k, v, w, u):
            assert x.is_contiguous()
        return _native.load_torch().wkv6(r, k, v, w, u, H, algo)


class _ShiftMixX(torch.autograd.Function):
    """x + (previous token - x) * mix with gradients, bf16 (wkv6_shift_mix_x and its backward): the fixed
    token-shift mix of rwkv6_model.py:136 (time mix) and :57-60 (channel mix)."""

    @staticmethod
    def forward(ctx, x, mix):
        lib = _native.load()
        with torch.no_grad():
            B, T, C = x.shape
            mx = mix.detach().to(torch.float32).contiguous()
            out = torch.empty_like(x)
            with torch.cuda.device(x.device):
                _native.check(lib.wkv6_shift_mix_x(_stream(), _DTYPE_CODE[x.dtype], B, T, C, _ptr(x), _ptr(mx), _ptr(out)))
            ctx.save_for_backward(x, mx)
            ctx.mix_dtype = mix.dtype
            return out

    @staticmethod
    def backward(ctx, gout):
        lib = _native.load()
        with torch.no_grad():
            x, mx = ctx.saved_tensors
            B, T, C = x.shape
            gout = gout.to(x.dtype).contiguous()
            gx = torch.empty_like(x)
            gmx = torch.empty(C, device=x.device, dtype=torch.float32)
            with torch.cuda.device(x.device):
                _native.check(lib.wkv6_shift_mix_x_backward(_stream(), _DTYPE_CODE[x.dtype], B, T, C, _ptr(x), _ptr(mx), None, None,
                                                            _ptr(gout), _ptr(gx), _ptr(gmx)))
            return gx, gmx.to(ctx.mix_dtype)


def _forward_with_state(B, T, C, H, state_map, r, k, v, w, u, init_state, algo=_native.ALGO_AUTO, state_dtype=None, backward_follows=False):
    """Stateful forward, no gradient (rwkv_kernel/torch_rwkv_kernel.py:76-95)."""
    # state_map None with an init_state means the identity map (row b starts from init_state[b])
    assert init_state is not None or state_map is None, "state_map needs init_state"
    assert state_map is None or state_map.dtype == torch.int64
    sdt = init_state.dtype if init_state is not None else (state_dtype or _out_dtype(r.dtype))
    return _native.load_torch().forward_with_state(H, state_map, r, k, v, w, u, init_state, algo, _DTYPE_CODE[sdt], backward_follows)


class _WKV6State(torch.autograd.Function):
    """Stateful operator WITH gradients through the state: y, S_T = f(r, k, v, w, u, S_0), states fp32
    (B,H,N,N), one per batch row.  Not part of the reference, whose stateful call carries no gradient
    (rwkv_kernel/torch_rwkv_kernel.py:145-168); it makes back-propagation over a sequence cut into
    pieces possible (the state's gradient is handed from one piece to the one before)."""

    @staticmethod
    def forward(ctx, B, T, C, H, r, k, v, w, u, s0, algo):
        ctx.dims = (B, T, C, H)
        ctx.algo = algo
        ctx.has_s0 = s0 is not None
        ctx.set_materialize_grads(False)   # an unused output arrives as None, not as a tensor of zeros
        y, sT = _forward_with_state(B, T, C, H, None, r, k, v, w, u, s0, algo, state_dtype=torch.float32, backward_follows=True)
        ctx.save_for_backward(r, k, v, w, u, *((s0,) if s0 is not None else ()))
        return y, sT

    @staticmethod
    def backward(ctx, gy, gsT):
        B, T, C, H = ctx.dims
        r, k, v, w, u = ctx.saved_tensors[:5]
        s0 = ctx.saved_tensors[5] if ctx.has_s0 else None
        with torch.no_grad():
            odt = _out_dtype(r.dtype)
            gy = torch.zeros((B, T, C), device=r.device, dtype=odt) if gy is None else gy.to(odt).contiguous()
            gsT = None if gsT is None else gsT.float().contiguous()
            gr, gk, gv, gw, gu, gs0 = _backward_with_state(B, T, C, H, r, k, v, w, u, s0, gy, gsT, ctx.algo, ctx.has_s0)
            gu = torch.sum(gu, 0).reshape(u.shape)
        return (None, None, None, None, gr.to(r.dtype), gk.to(r.dtype), gv.to(r.dtype), gw.to(r.dtype), gu.to(u.dtype), gs0, None)


def _backward_with_state(B, T, C, H, r, k, v, w, u, s0, gy, gsT, algo, want_gs0):
    """gr, gk, gv, gw, per-row gu (B, C), dL/dS_0 or None, through wkv6_backward_with_state."""
    lib = _native.load()
    odt = _out_dtype(r.dtype)
    gr, gk, gv, gw = _staggered(4, (B, T, C), odt, r.device, first=7)
    gu = torch.empty((B, C), device=r.device, dtype=odt)
    gs0 = torch.empty((B, H, C // H, C // H), device=r.device, dtype=torch.float32) if want_gs0 else None
    code = _DTYPE_CODE[r.dtype]
    with torch.cuda.device(r.device):
        n = lib.wkv6_backward_with_state_workspace_bytes(code, algo, B, T, C, H)
        ws = torch.empty(max(int(n), 16), device=r.device, dtype=torch.uint8)
        _native.check(lib.wkv6_backward_with_state(
            _stream(), code, algo, B, T, C, H, _ptr(r), _ptr(k), _ptr(v), _ptr(w), _ptr(u), _ptr(s0),
            _ptr(gy), _ptr(gsT), _ptr(gr), _ptr(gk), _ptr(gv), _ptr(gw), _ptr(gu), _ptr(gs0), _ptr(ws), n))
    return gr, gk, gv, gw, gu, gs0


class RWKVKernelOperator:
    def __init__(self, head_size, max_sequence_length):
        lib = _native.load()
        self._torch = _native.load_torch()
        assert isinstance(head_size, int) and isinstance(max_sequence_length, int)
        assert head_size > 0 and max_sequence_length > 0
        assert head_size % 4 == 0, "head_size must be a multiple of 4"
        if not lib.wkv6_supports_head_size(head_size):
            raise _native.WKV6Error("libwkv6_gfx950 is built for head sizes 64 (all paths) and the other multiples of 4 up to 128 (plain calls), got %d" % head_size)
        self.head_size = head_size
        # the reference bakes this into a per-thread array bound (-D_T_); nothing here is sized by
        # it, so longer sequences simply work
        self.max_sequence_length = max_sequence_length
        self.algo = _native.ALGO_AUTO
        self._zero_maps = {}
        self.normal_kernenl = _WKV6
        self.kernel_with_state = _forward_with_state

    def __getstate__(self):
        """Copies and pickles leave the native module out (a module can be neither) and find it again."""
        return {k: v for k, v in self.__dict__.items() if k != "_torch"}

    def __setstate__(self, state):
        self.__dict__.update(state)
        self._torch = _native.load_torch()

    def _check(self, r, k, v, w, u, init_state, state_map):
        """Argument checks shared by every entry; returns (B, T, C, H, N, u, init_state, state_map)."""
        B, T, C = r.shape
        N = self.head_size
        assert C % N == 0
        H = C // N
        if not isinstance(u, torch.Tensor):
            u = u.value

        for x in (r, k, v, w, u):
            assert x.is_cuda
        assert r.device == k.device == v.device == w.device == u.device
        assert r.dtype == k.dtype == v.dtype == w.dtype == u.dtype
        assert r.shape == k.shape == v.shape == w.shape
        assert u.numel() == C, "u must hold one value per channel"

        if init_state is not None:
            assert init_state.dim() in (3, 4), \
                "init_state must be (state_kinds <= batch, H, N, N) or (H, N, N)"
            if init_state.dim() == 3:
                init_state = init_state[None, :]
            assert tuple(init_state.shape[1:]) == (H, N, N) and init_state.shape[0] <= B, \
                "init_state must be (state_kinds <= batch, H, N, N) or (H, N, N)"
            s_dtype = _out_dtype(r.dtype)
            assert init_state.dtype in (s_dtype, torch.float32), "init_state dtype must be %s" % s_dtype
            assert init_state.device == r.device

        if state_map is not None:
            if isinstance(state_map, (list, tuple)):
                state_map = torch.tensor(state_map, dtype=torch.int64)
            elif isinstance(state_map, torch.Tensor):
                assert state_map.dtype in (torch.int32, torch.int64), "state_map must be int32/int64 of shape (batch,)"
                state_map = state_map.to(torch.int64)
            assert tuple(state_map.shape) == (B,), "state_map must have shape (batch,)"
        return B, T, C, H, N, u, init_state, state_map

    def _resolve_state(self, B, r, init_state, state_map):
        """Default / validated state_map on the device (None = identity), contiguous init_state."""
        if init_state is None:
            assert state_map is None, "state_map needs init_state"
            return None, None
        n_state = init_state.shape[0]
        if state_map is None:
            assert n_state == 1 or n_state == B, "cannot infer state_map; pass it explicitly"
            if n_state == 1 and B > 1:
                key = (B, r.device)
                if key not in self._zero_maps:
                    self._zero_maps[key] = torch.zeros(B, dtype=torch.int64, device=r.device)
                state_map = self._zero_maps[key]
            # n_state == B: identity, expressed as "no map" so that a decode loop pays
            # neither a host-to-device copy nor a range check per step
        else:
            assert bool((state_map >= 0).all()) and bool((state_map < n_state).all()), \
                "state_map values must lie in [0, %d)" % n_state
            state_map = state_map.to(r.device).contiguous()
        return init_state.contiguous(), state_map

    def __call__(self, r, k, v, w, u, return_state=False, init_state=None, state_map=None):
        if state_map is None:
            res = self._torch.try_call(self.head_size, self.algo, r, k, v, w, u, return_state, init_state)
            if res is not None:
                return res
        B, T, C, H, N, u, init_state, state_map = self._check(r, k, v, w, u, init_state, state_map)
        if return_state:
            init_state, state_map = self._resolve_state(B, r, init_state, state_map)
            for x in (r, k, v, w, u):
                assert x.is_contiguous()
            leaves = (r, k, v, w, u) + ((init_state,) if init_state is not None else ())
            if torch.is_grad_enabled() and any(x.requires_grad for x in leaves):
                # gradients through the state (not in the reference): one fp32 state per batch row
                assert state_map is None and (init_state is None or init_state.shape[0] == B), \
                    "gradients through the state need one init_state row per batch row and no state_map"
                assert init_state is None or init_state.dtype == torch.float32, \
                    "gradients through the state need an fp32 init_state"
                return _WKV6State.apply(B, T, C, H, r, k, v, w, u, init_state, self.algo)
            return _forward_with_state(B, T, C, H, state_map, r, k, v, w, u, init_state, self.algo)
        o = _WKV6.apply(B, T, C, H, r, k, v, w, u, self.algo)
        return o, None

    def shift_mix_supported(self, x, decomposer_size):
        """Whether ``shift_mix`` takes this tensor (bf16 on the GPU, rank 32 or 64)."""
        if not (x.is_cuda and x.dtype == torch.bfloat16 and x.dim() == 3):
            return False
        return bool(_native.load().wkv6_shift_mix_supported(_DTYPE_CODE[x.dtype], x.shape[2], decomposer_size))

    def shift_mix_x(self, x, mix):
        """``x + (previous token - x) * mix`` (zero before a sequence's first token), differentiable in both
        arguments: the fixed token-shift mix of rwkv6_model.py:136 and of the channel-mix layer
        (:57-60).  bf16 tensors on the GPU, ``mix`` one value per channel.  Not part of the reference's operator."""
        assert x.is_contiguous() and x.dim() == 3 and mix.numel() == x.shape[2]
        assert mix.device == x.device, "x and mix must be on one device"
        assert self.shift_mix_supported(x, 32), "shift_mix_x takes bf16 tensors on the GPU, channels a multiple of 64"
        return _ShiftMixX.apply(x, mix.reshape(x.shape[2]))

    def shift_mix(self, x, mix_x, a, w2t, bias):
        """The layer's input side, rwkv6_model.py:134-146: from the layer input ``x`` (B,T,C) to the
        inputs ``(xr, xk, xv, xw, xg)`` of the projections that produce r, k, v, w and the gate:
        ``x_s = x + xx * (tanh((x + xx * mix_x) a_s^T) w2t_s^T + bias_s)`` with ``xx`` the previous token
        minus the token.  ``a`` (5R, C): the five mixers' first weights stacked in the order r, k, v, w, g;
        ``w2t`` (5, C, R) and ``bias`` (5, C): their second weights and biases.  Differentiable in all
        five arguments.  Not part of the reference's operator."""
        B, T, C = x.shape
        assert x.is_contiguous() and mix_x.numel() == C
        R = w2t.shape[2]
        assert a.shape == (5 * R, C) and w2t.shape == (5, C, R) and bias.shape == (5, C)
        assert self.shift_mix_supported(x, R), "shift_mix takes bf16 tensors on the GPU with rank 32 or 64"
        return self._torch.shift_mix(x, mix_x.reshape(C), a, w2t, bias)

    def forward_gn_gate(self, r, k, v, w, u, gate, gn_scale, gn_offset, epsilon=64e-5,
                        return_state=False, init_state=None, state_map=None):
        """Forward with the layer's next two steps fused into the kernel's output stage: returns
        ``(group_norm(y) * gate, state)`` where group_norm is the per-head layer norm with scale and
        offset of rwkv6_model.py:94-99 and ``* gate`` is rwkv6_model.py:158-160.  bf16 tensors;
        gn_scale / gn_offset hold one value per channel.  Without gradients (inference) y itself is
        never written and the stateful arguments work as in ``__call__``.  With gradients enabled and
        required (training; no state arguments) the call is differentiable in r, k, v, w, u, gate,
        gn_scale and gn_offset.  Not part of the reference's operator."""
        if state_map is None:
            res = self._torch.try_gn_gate(self.head_size, r, k, v, w, u, gate, gn_scale, gn_offset, epsilon, return_state, init_state)
            if res is not None:
                return res
        B, T, C, H, N, u, init_state, state_map = self._check(r, k, v, w, u, init_state, state_map)
        assert r.dtype == torch.bfloat16, "the fused output stage takes bf16 tensors"
        assert gate.shape == r.shape and gate.dtype == r.dtype and gate.device == r.device
        assert gn_scale.numel() == C and gn_offset.numel() == C
        if torch.is_grad_enabled() and any(x.requires_grad for x in (r, k, v, w, u, gate, gn_scale, gn_offset)):
            assert not return_state and init_state is None and state_map is None, \
                "the differentiable fused call takes no state arguments"
            for x in (r, k, v, w, u, gate):
                assert x.is_contiguous()
            lib = _native.load()
            if lib.wkv6_forward_gn_gate_save_supported(_DTYPE_CODE[r.dtype], B, T, C, H):
                return self._torch.wkv6_gn_gate(r, k, v, w, u, gate, gn_scale.to(r.device), gn_offset.to(r.device), H, float(epsilon)), None
            # (a shape the fused training kernels do not take, e.g. a sequence too long for the chunk form: unfused calls)
            y, _ = self(r, k, v, w, u)
            z = torch.nn.functional.layer_norm(y.float().view(B, T, H, N), (N,), eps=epsilon).view(B, T, C)
            out = (z * gn_scale.reshape(1, 1, C).float() + gn_offset.reshape(1, 1, C).float()) * gate.float()
            return out.to(r.dtype), None
        init_state, state_map = self._resolve_state(B, r, init_state, state_map)
        for x in (r, k, v, w, u, gate):
            assert x.is_contiguous()
        return self._torch.forward_gn_gate(H, state_map, r, k, v, w, u, init_state, gate, gn_scale, gn_offset, float(epsilon), bool(return_state))
