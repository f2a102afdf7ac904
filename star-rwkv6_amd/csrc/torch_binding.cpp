// torch's side of the operator in native code: argument checks, allocation, the autograd nodes of the operator, of the
// operator with group norm and gate and of the layer's input side, and the calls into libwkv6_gfx950.
//
// Why not Python: a training step is one or two kernel pairs of 40 to 110 us, and the same nodes written as
// torch.autograd.Function with ctypes calls took 185 us of host time per step at any size (265 with group norm and gate,
// 250 for the input side, 26 for one decoded token): every training shape up to about 2^25 elements ran at the speed of
// the interpreter, and the backward, which torch runs in a thread of its own, had to be handed the interpreter first.
//
// Rules of this file:
//  * every call holds no state between calls; tensors that outlive a forward are torch's saved variables (hooks and
//    version checks apply) or live in the node, as the saved chunk states do until the first backward takes them;
//  * `try_*` take a call only in its plain form and return None for anything else, and the Python layer then says what
//    is wrong with it or brings it into that form; what a call is refused for is decided there alone;
//  * kernels go to the current stream of the tensors' device; the interpreter's lock is not held meanwhile.
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>

#include <initializer_list>
#include <optional>
#include <vector>

#include "wkv6.h"

namespace {

namespace py = pybind11;
using at::ScalarType;
using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

constexpr int kChunk = WKV6_ALGO_CHUNK;

int code_of(ScalarType t) {
  switch (t) {
    case at::kBFloat16: return WKV6_BF16;
    case at::kHalf: return WKV6_F16;
    case at::kFloat: return WKV6_F32;
    default: return -1;
  }
}

// rwkv_kernel/torch_rwkv_kernel.py:35 of the reference: float16 inputs produce float32 outputs
ScalarType out_type(ScalarType t) { return t == at::kHalf ? at::kFloat : t; }

// The package's own exception for a failed library call, also out of a backward's thread.
void check(int status) {
  if (status == 0) return;
  py::gil_scoped_acquire gil;
  try {
    py::module_::import("rwkv_kernel._native").attr("check")(status);
  } catch (py::error_already_set &e) {
    e.restore();
    python_error err;
    err.persist();
    throw err;
  }
}

void *stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
// whether what goes to the current stream of the current device is recorded into a graph, to run any number of times
bool is_captured() { return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None; }

const void *in(const Tensor &t) { return t.defined() ? t.const_data_ptr() : nullptr; }
void *out(const Tensor &t) { return t.defined() ? t.mutable_data_ptr() : nullptr; }
const float *in_f(const Tensor &t) { return static_cast<const float *>(in(t)); }
float *out_f(const Tensor &t) { return static_cast<float *>(out(t)); }

Tensor bytes(const Tensor &like, size_t n) {
  return n ? at::empty({static_cast<int64_t>(n)}, at::TensorOptions().dtype(at::kByte).device(like.device())) : Tensor();
}

// Tensors of different shapes and types out of ONE allocation, each `slot` * 256 bytes past a 4 KiB boundary of it.  A
// workgroup of the kernels walks all (B,T,C) tensors of a call row by row in step; torch's allocator hands out large
// blocks on 2 MiB boundaries, and tensors whose bases agree modulo 4 KiB keep sending those streams to the same memory
// channel at the same moment (about 5 % of the training pair at B8 T1024 C2048).  The block lives as long as any of them.
struct Piece {
  at::DimVector shape;
  ScalarType type;
  int64_t slot;
};

std::vector<Tensor> carve(const Tensor &like, std::initializer_list<Piece> pieces) {
  std::vector<int64_t> offset;
  int64_t total = 0;
  for (const Piece &p : pieces) {
    const int64_t n = c10::multiply_integers(p.shape) * static_cast<int64_t>(c10::elementSize(p.type));
    offset.push_back(total + p.slot * 256);
    total += (p.slot * 256 + n + 4095) / 4096 * 4096;
  }
  const Tensor block = bytes(like, total ? total : 4096);
  std::vector<Tensor> res;
  size_t i = 0;
  for (const Piece &p : pieces) {
    auto impl = c10::make_intrusive<c10::TensorImpl>(c10::Storage(block.storage()), block.key_set(), c10::scalarTypeToTypeMeta(p.type));
    impl->set_storage_offset(offset[i++] / static_cast<int64_t>(c10::elementSize(p.type)));
    impl->set_sizes_contiguous(p.shape);
    res.emplace_back(std::move(impl));
  }
  return res;
}

// The gradient of a parameter gets an allocation of its own: torch takes it over as the parameter's .grad as it is, where it
// stays for as long as the caller keeps gradients, and with it whatever shares its block.
Tensor parameter_gradient(const Tensor &like, at::IntArrayRef shape, ScalarType type) {
  return at::empty(shape, at::TensorOptions().dtype(type).device(like.device()));
}

bool any_requires_grad(std::initializer_list<const Tensor *> ts) {
  for (const Tensor *t : ts)
    if (t->defined() && t->requires_grad()) return true;
  return false;
}

struct Dims {
  int64_t B, T, C, H;
};

Dims dims_of(const Tensor &r, int64_t H) { return {r.size(0), r.size(1), r.size(2), H}; }

// The operator's backward from the arriving gradient: through the saved block when there is one, which it uses up.
// Gradients of r, k, v, w and u, in that order.
std::vector<Tensor> wkv6_grads(const Dims &d, int algo, const Tensor &r, const Tensor &k, const Tensor &v, const Tensor &w,
                               const Tensor &u, const Tensor &gy, const Tensor &saved) {
  const auto [B, T, C, H] = d;
  const int code = code_of(r.scalar_type());
  const ScalarType ot = out_type(r.scalar_type());
  const at::DimVector big{B, T, C};
  // torch hands the gradient of an fp16 tensor on as fp16 whatever a node returns, in a kernel per gradient: the library
  // rounds where it stores them, where its kernels can
  const ScalarType gt = saved.defined() && algo != kChunk ? r.scalar_type() : ot;
  std::vector<Tensor> g = carve(r, {{big, gt, 7}, {big, gt, 8}, {big, gt, 9}, {big, gt, 10}, {{B, C}, ot, 0}});
  const Tensor gu_rows = std::move(g[4]);
  if (saved.defined()) {
    g[4] = parameter_gradient(r, u.sizes(), gt);
    // the batch sum of u's gradient (rwkv_kernel/torch_rwkv_kernel.py:73 of the reference) comes out of the same launch
    check(wkv6_backward_saved_sum_ex(stream_of(r), code, code_of(gt), algo, B, T, C, H, in(r), in(k), in(v), in(w), in(u), in(gy),
                                     out(g[0]), out(g[1]), out(g[2]), out(g[3]), out(gu_rows), out(g[4]), out(saved), saved.numel()));
    return g;
  }
  const size_t n = wkv6_backward_workspace_bytes_ex(code, algo, B, T, C, H);
  const Tensor ws = bytes(r, n);
  check(wkv6_backward_ex(stream_of(r), code, algo, B, T, C, H, in(r), in(k), in(v), in(w), in(u), in(gy), out(g[0]), out(g[1]),
                         out(g[2]), out(g[3]), out(gu_rows), out(ws), n));
  g[4] = at::sum(gu_rows, 0).reshape(u.sizes());
  return g;
}

// The saved chunk states, handed from the forward to the first backward, which gives their memory back.  A second backward over
// the same graph (retain_graph) finds none and runs the plain backward.  (torch holds the node's lock while a backward runs.  One
// that is captured leaves the states as they were for its replays: each of them reads them and arms their counters again.)
// The same goes for sums that the forward cleared, which only one run of a backward can add to: see Wkv6GnGate.
void keep(AutogradContext *ctx, const Tensor &saved, const char *name = "states") {
  if (saved.defined()) ctx->saved_data[name] = saved;
}

Tensor take(AutogradContext *ctx, const char *name = "states") {
  auto it = ctx->saved_data.find(name);
  if (it == ctx->saved_data.end()) return Tensor();
  Tensor t = it->second.toTensor();
  ctx->saved_data.erase(it);
  return t;
}

// Stateless operator with gradients (rwkv_kernel/torch_rwkv_kernel.py:14-75 of the reference).  When a gradient will be
// needed and the library has something worth keeping for it (the chunked kernels' per-chunk states), the forward runs as
// wkv6_forward_save and the backward as wkv6_backward_saved_sum; otherwise the plain pair.
struct Wkv6 : torch::autograd::Function<Wkv6> {
  static Tensor forward(AutogradContext *ctx, const Tensor &r, const Tensor &k, const Tensor &v, const Tensor &w, const Tensor &u,
                        int64_t H, int64_t algo) {
    const c10::DeviceGuard guard(r.device());
    const auto [B, T, C, H_] = dims_of(r, H);
    const int code = code_of(r.scalar_type());
    const size_t nsave = any_requires_grad({&r, &k, &v, &w, &u}) ? wkv6_saved_bytes(code, algo, B, T, C, H) : 0;
    const Piece yp{{B, T, C}, out_type(r.scalar_type()), 5};
    Tensor y;
    if (nsave) {
      const auto t = carve(r, {yp, {{static_cast<int64_t>(nsave)}, at::kByte, 6}});
      y = t[0];
      check(wkv6_forward_save(stream_of(r), code, algo, B, T, C, H, in(r), in(k), in(v), in(w), in(u), out(y), out(t[1]), nsave));
      keep(ctx, t[1]);
    } else {
      y = carve(r, {yp})[0];
      // optional workspace: a long sequence of few (batch, head) pairs runs as time segments
      const size_t n = wkv6_forward_workspace_bytes_any_length(code, algo, B, T, C, H);
      const Tensor ws = bytes(r, n);
      // (no gradient is wanted, or the per-timestep kernels run, which read their inputs in one way only)
      check(wkv6_forward_inference(stream_of(r), code, code_of(out_type(r.scalar_type())), algo, B, T, C, H, 0, nullptr, in(r), in(k), in(v),
                                   in(w), in(u), nullptr, out(y), nullptr, out(ws), n));
    }
    ctx->saved_data["H"] = H;
    ctx->saved_data["algo"] = algo;
    ctx->save_for_backward({r, k, v, w, u});
    return y;
  }

  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const at::NoGradGuard no_grad;
    const auto s = ctx->get_saved_variables();
    const Tensor &r = s[0];
    const c10::DeviceGuard guard(r.device());
    TORCH_CHECK(grads[0].is_cuda() && grads[0].scalar_type() == out_type(r.scalar_type()), "wkv6: the gradient must have y's device and dtype");
    const Tensor gy = grads[0].contiguous();
    auto g = wkv6_grads(dims_of(r, ctx->saved_data["H"].toInt()), static_cast<int>(ctx->saved_data["algo"].toInt()), r, s[1], s[2],
                        s[3], s[4], gy, take(ctx));
    return {g[0], g[1], g[2], g[3], g[4], Tensor(), Tensor()};
  }
};

// out = (group_norm_head(wkv6(r, k, v, w, u)) * scale + offset) * gate, bf16, zero initial state: the operator and what the
// layer does with its output next (rwkv6_model.py:94-99,158-160 of the reference) in one forward kernel, the norm's and
// the gate's backward in one elementwise kernel, then the operator's backward from the saved chunk states.
struct Wkv6GnGate : torch::autograd::Function<Wkv6GnGate> {
  static Tensor forward(AutogradContext *ctx, const Tensor &r, const Tensor &k, const Tensor &v, const Tensor &w, const Tensor &u,
                        const Tensor &gate, const Tensor &scale, const Tensor &offset, int64_t H, double eps) {
    const c10::DeviceGuard guard(r.device());
    const auto [B, T, C, H_] = dims_of(r, H);
    const int code = code_of(r.scalar_type());
    const Tensor sc = scale.to(at::kFloat).contiguous(), of = offset.to(at::kFloat).contiguous();
    const int64_t nsave = wkv6_saved_bytes(code, kChunk, B, T, C, H);
    // out and what stays for the backward lie in blocks of their own: an output that a caller keeps holds nothing else
    const Tensor res = carve(r, {{{B, T, C}, r.scalar_type(), 5}})[0];
    const auto t = carve(r, {{{B, T, C}, r.scalar_type(), 6}, {{nsave}, at::kByte, 7}, {{B, T, H, 2}, at::kFloat, 0}});
    if (is_captured()) {   // (each replay would clear the sums again, and with them the gradients a backward gave out)
      check(wkv6_forward_gn_gate_save(stream_of(r), code, B, T, C, H, in(r), in(k), in(v), in(w), in(u), in(gate), in_f(sc), in_f(of),
                                      static_cast<float>(eps), out(res), out(t[0]), out_f(t[2]), out(t[1]), nsave));
    } else {
      // the norm's gradients, which this forward clears for the first backward to add to
      const Tensor gscale = parameter_gradient(r, sc.sizes(), at::kFloat), goffset = parameter_gradient(r, of.sizes(), at::kFloat);
      check(wkv6_forward_gn_gate_save_sums(stream_of(r), code, B, T, C, H, in(r), in(k), in(v), in(w), in(u), in(gate), in_f(sc), in_f(of),
                                           static_cast<float>(eps), out(res), out(t[0]), out_f(t[2]), out(t[1]), nsave, out_f(gscale),
                                           out_f(goffset)));
      keep(ctx, gscale, "gscale");
      keep(ctx, goffset, "goffset");
    }
    keep(ctx, t[1]);
    ctx->saved_data["H"] = H;
    ctx->saved_data["scale_type"] = static_cast<int64_t>(scale.scalar_type());
    ctx->saved_data["offset_type"] = static_cast<int64_t>(offset.scalar_type());
    ctx->save_for_backward({r, k, v, w, u, gate, sc, of, t[0], t[2]});
    return res;
  }

  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const at::NoGradGuard no_grad;
    const auto s = ctx->get_saved_variables();
    const Tensor &r = s[0];
    const c10::DeviceGuard guard(r.device());
    const Dims d = dims_of(r, ctx->saved_data["H"].toInt());
    const auto [B, T, C, H] = d;
    TORCH_CHECK(grads[0].scalar_type() == r.scalar_type(), "wkv6: the gradient must have the output's dtype");
    const Tensor gout = grads[0].contiguous();
    const ScalarType t = r.scalar_type();
    const Tensor gy = carve(r, {{{B, T, C}, t, 5}})[0];
    const Tensor ggate = carve(r, {{{B, T, C}, t, 6}})[0];
    // (captured: the forward cleared its sums once, while the replays of this backward, however many follow one forward, each have to
    // start from zero, in memory of the graph's own)
    Tensor gscale, goffset;
    if (!is_captured()) { gscale = take(ctx, "gscale"); goffset = take(ctx, "goffset"); }
    const auto norm_backward = gscale.defined() ? wkv6_gn_gate_backward_sums : wkv6_gn_gate_backward;
    if (!gscale.defined()) {   // (also a second backward over the same graph, and one whose forward was captured)
      gscale = parameter_gradient(r, s[6].sizes(), at::kFloat);
      goffset = parameter_gradient(r, s[7].sizes(), at::kFloat);
    }
    check(norm_backward(stream_of(r), code_of(t), B, T, C, H, in(gout), in(s[8]), in_f(s[9]), in(s[5]), in_f(s[6]), in_f(s[7]), out(gy),
                        out(ggate), out_f(gscale), out_f(goffset)));
    auto w = wkv6_grads(d, kChunk, r, s[1], s[2], s[3], s[4], gy, take(ctx));
    return {w[0], w[1], w[2], w[3], w[4], ggate,
            gscale.to(static_cast<ScalarType>(ctx->saved_data["scale_type"].toInt())),
            goffset.to(static_cast<ScalarType>(ctx->saved_data["offset_type"].toInt())), Tensor(), Tensor()};
  }
};

// A parameter as the kernels read it: of this type, contiguous and on a 16-byte boundary.  (One that already has the type and
// is contiguous may be a view into a flat buffer of parameters, anywhere in it.)
Tensor laid_out(const Tensor &t, ScalarType type) {
  const Tensor c = t.to(type).contiguous();
  return reinterpret_cast<uintptr_t>(c.const_data_ptr()) % 16 == 0 ? c : c.clone();
}

// The layer's input side (rwkv6_model.py:134-146 of the reference) with gradients, bf16: x -> (xr, xk, xv, xw, xg).
struct ShiftMix : torch::autograd::Function<ShiftMix> {
  static variable_list forward(AutogradContext *ctx, const Tensor &x, const Tensor &mix_x, const Tensor &a, const Tensor &w2t,
                               const Tensor &bias) {
    const c10::DeviceGuard guard(x.device());
    const int64_t B = x.size(0), T = x.size(1), C = x.size(2), R = w2t.size(2);
    const int code = code_of(x.scalar_type());
    const Tensor mx = mix_x.to(at::kFloat).contiguous(), b32 = bias.to(at::kFloat).contiguous();
    const ScalarType wt = a.scalar_type() == w2t.scalar_type() && a.scalar_type() == at::kBFloat16 ? at::kBFloat16 : at::kFloat;
    // (bf16 second weights are handed through, and refused off a 16-byte boundary, like x and the biases)
    const Tensor aw = laid_out(a, wt), ww = w2t.scalar_type() == at::kBFloat16 ? w2t.to(wt).contiguous() : laid_out(w2t, wt);
    const int64_t nw = wkv6_shift_mix_weights_bytes(C, R);
    const ScalarType t = x.scalar_type();
    const at::DimVector big{B, T, C};
    auto o = carve(x, {{big, t, 1}, {big, t, 2}, {big, t, 3}, {big, t, 4}, {big, t, 5}});
    // (not out of the outputs' block: a caller may change an output in place)
    const auto kept = carve(x, {{{B, T, 5 * R}, t, 6}, {{nw}, at::kByte, 0}});
    check(wkv6_shift_mix_forward(stream_of(x), code, code_of(wt), B, T, C, R, in(x), in_f(mx), in(aw), in(ww), in_f(b32), out(kept[1]),
                                 nw, out(kept[0]), out(o[0]), out(o[1]), out(o[2]), out(o[3]), out(o[4])));
    ctx->saved_data["weight_type"] = static_cast<int64_t>(wt);
    ctx->saved_data["types"] = std::vector<int64_t>{static_cast<int64_t>(mix_x.scalar_type()), static_cast<int64_t>(a.scalar_type()),
                                                    static_cast<int64_t>(w2t.scalar_type()), static_cast<int64_t>(bias.scalar_type())};
    ctx->save_for_backward({x, kept[0], kept[1], mx, b32});
    return o;
  }

  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const at::NoGradGuard no_grad;
    const auto s = ctx->get_saved_variables();
    const Tensor &x = s[0], &h = s[1], &weights = s[2], &mx = s[3], &b32 = s[4];
    const c10::DeviceGuard guard(x.device());
    const int64_t B = x.size(0), T = x.size(1), C = x.size(2), R = h.size(2) / 5;
    const ScalarType t = x.scalar_type(), wt = static_cast<ScalarType>(ctx->saved_data["weight_type"].toInt());
    const int code = code_of(t);
    for (Tensor &g : grads) g = g.to(t).contiguous();
    const Tensor gx = carve(x, {{{B, T, C}, t, 6}})[0];
    const Tensor gmix = parameter_gradient(x, {C}, at::kFloat), ga = parameter_gradient(x, {5 * R, C}, wt),
                 gw2t = parameter_gradient(x, {5, C, R}, wt), gbias = parameter_gradient(x, {5, C}, at::kFloat);
    const size_t n = wkv6_shift_mix_backward_workspace_bytes(code, B, T, C, R);
    const Tensor ws = bytes(x, n);
    check(wkv6_shift_mix_backward(stream_of(x), code, code_of(wt), B, T, C, R, in(x), in_f(mx), in_f(b32), in(weights), in(h),
                                  in(grads[0]), in(grads[1]), in(grads[2]), in(grads[3]), in(grads[4]), out(gx), out_f(gmix),
                                  out(ga), out(gw2t), out_f(gbias), out(ws), n));
    const auto types = ctx->saved_data["types"].toIntVector();
    const auto as = [&](const Tensor &v, int i) { return v.to(static_cast<ScalarType>(types[i])); };
    return {gx, as(gmix, 0), as(ga, 1), as(gw2t, 2), as(gbias, 3)};
  }
};

// (B, H, N, N)
at::DimVector state_shape(const Dims &d) {
  TORCH_CHECK(d.H > 0, "wkv6: tensors without channels have no state");   // (the size per head below divides by it)
  return {d.B, d.H, d.C / d.H, d.C / d.H};
}

// Stateful forward without a gradient (rwkv_kernel/torch_rwkv_kernel.py:76-95 of the reference): y and the final state.
// An undefined map with an initial state means row b starts from s0[b].
std::pair<Tensor, Tensor> forward_with_state(int64_t H, const Tensor &map, const Tensor &r, const Tensor &k, const Tensor &v,
                                             const Tensor &w, const Tensor &u, const Tensor &s0, int64_t algo, ScalarType st,
                                             bool backward_follows = false) {
  const at::NoGradGuard no_grad;
  const c10::DeviceGuard guard(r.device());
  const Dims d = dims_of(r, H);
  const auto [B, T, C, H_] = d;
  const int code = code_of(r.scalar_type());
  const Tensor y = carve(r, {{{B, T, C}, out_type(r.scalar_type()), 5}})[0];
  const Tensor ys = at::empty(state_shape(d), r.options().dtype(st));
  // optional workspace: a long sequence of few (batch, head) pairs runs as time segments
  const size_t n = wkv6_forward_workspace_bytes_any_length(code, algo, B, T, C, H);
  const Tensor ws = bytes(r, n);
  const auto forward = backward_follows ? wkv6_forward_with_state_ex : wkv6_forward_inference;
  check(forward(stream_of(r), code, code_of(st), algo, B, T, C, H, s0.defined(), static_cast<const int64_t *>(in(map)), in(r), in(k),
                in(v), in(w), in(u), in(s0), out(y), out(ys), out(ws), n));
  return {y, ys};
}

// The same with group norm and gate in the output stage; the final state only on request.
std::pair<Tensor, Tensor> forward_gn_gate(int64_t H, const Tensor &map, const Tensor &r, const Tensor &k, const Tensor &v,
                                          const Tensor &w, const Tensor &u, const Tensor &s0, const Tensor &gate, const Tensor &scale,
                                          const Tensor &offset, double eps, bool want_state) {
  const at::NoGradGuard no_grad;
  const c10::DeviceGuard guard(r.device());
  const Dims d = dims_of(r, H);
  const auto [B, T, C, H_] = d;
  const int code = code_of(r.scalar_type());
  const Tensor sc = scale.to(r.device(), at::kFloat).contiguous(), of = offset.to(r.device(), at::kFloat).contiguous();
  const ScalarType st = s0.defined() ? s0.scalar_type() : at::kFloat;
  const Tensor res = carve(r, {{{B, T, C}, r.scalar_type(), 5}})[0];
  const Tensor ys = want_state ? at::empty(state_shape(d), r.options().dtype(st)) : Tensor();
  const size_t n = wkv6_forward_workspace_bytes_any_length(code, kChunk, B, T, C, H);
  const Tensor ws = bytes(r, n);
  check(wkv6_forward_gn_gate_ex(stream_of(r), code, code_of(st), B, T, C, H, s0.defined(), static_cast<const int64_t *>(in(map)), in(r),
                                in(k), in(v), in(w), in(u), in(s0), in(gate), in_f(sc), in_f(of), static_cast<float>(eps), out(res),
                                out(ys), out(ws), n));
  return {res, ys};
}

// ---- what the Python layer calls ----

// r, k, v, w and u as the kernels take them, with nothing left for the Python layer to check or to change.
bool plain(int64_t N, const Tensor &r, const Tensor &k, const Tensor &v, const Tensor &w, const Tensor &u) {
  if (r.dim() != 3 || !r.is_cuda() || code_of(r.scalar_type()) < 0 || r.size(2) == 0 || r.size(2) % N != 0 || u.numel() != r.size(2))
    return false;
  for (const Tensor *t : {&r, &k, &v, &w, &u})
    if (t->device() != r.device() || t->scalar_type() != r.scalar_type() || !t->is_contiguous()) return false;
  return k.sizes() == r.sizes() && v.sizes() == r.sizes() && w.sizes() == r.sizes();
}

// An initial state as the kernels take it, one per batch row.
bool plain_state(int64_t N, const Tensor &r, const Tensor &s) {
  return s.dim() == 4 && s.size(0) == r.size(0) && s.size(1) == r.size(2) / N && s.size(2) == N && s.size(3) == N &&
         s.device() == r.device() && s.is_contiguous() && (s.scalar_type() == at::kFloat || s.scalar_type() == out_type(r.scalar_type()));
}

const Tensor *tensor(const py::object &o) { return THPVariable_Check(o.ptr()) ? &THPVariable_Unpack(o.ptr()) : nullptr; }

py::object wrap(const Tensor &t) { return t.defined() ? py::reinterpret_steal<py::object>(THPVariable_Wrap(t)) : py::none(); }

// Whatever Python takes for true or false (pybind11's bool refuses lists, texts and other objects with a length).
bool truth(const py::object &o) {
  const int t = PyObject_IsTrue(o.ptr());
  if (t < 0) throw py::error_already_set();
  return t != 0;
}

py::tuple wrap(const std::pair<Tensor, Tensor> &p) { return py::make_tuple(wrap(p.first), wrap(p.second)); }

// Runs f without the interpreter's lock.  A Python error that torch has put into a C++ exception is restored as it was.
template <typename F> auto unlocked(F &&f) {
  try {
    py::gil_scoped_release nogil;
    return f();
  } catch (python_error &e) {
    py::gil_scoped_acquire gil;
    e.restore();
    throw py::error_already_set();
  }
}

py::object try_call(int64_t N, int64_t algo, const py::object &r_, const py::object &k_, const py::object &v_, const py::object &w_,
                    const py::object &u_, const py::object &return_state_, const py::object &s0_) {
  const Tensor *r = tensor(r_), *k = tensor(k_), *v = tensor(v_), *w = tensor(w_), *u = tensor(u_), *s0 = tensor(s0_);
  if (!r || !k || !v || !w || !u || !plain(N, *r, *k, *v, *w, *u)) return py::none();
  const int64_t H = r->size(2) / N;
  if (!truth(return_state_)) {
    if (!s0_.is_none()) return py::none();
    return py::make_tuple(wrap(unlocked([&] { return Wkv6::apply(*r, *k, *v, *w, *u, H, algo); })), py::none());
  }
  const Tensor state = s0 ? *s0 : Tensor();
  if (s0 ? !plain_state(N, *r, state) : !s0_.is_none()) return py::none();
  if (at::GradMode::is_enabled() && any_requires_grad({r, k, v, w, u, &state})) return py::none();
  const ScalarType st = s0 ? state.scalar_type() : out_type(r->scalar_type());
  return wrap(unlocked([&] { return forward_with_state(H, Tensor(), *r, *k, *v, *w, *u, state, algo, st); }));
}

py::object try_gn_gate(int64_t N, const py::object &r_, const py::object &k_, const py::object &v_, const py::object &w_,
                       const py::object &u_, const py::object &gate_, const py::object &scale_, const py::object &offset_,
                       const py::object &eps_, const py::object &return_state_, const py::object &s0_) {
  const Tensor *r = tensor(r_), *k = tensor(k_), *v = tensor(v_), *w = tensor(w_), *u = tensor(u_), *s0 = tensor(s0_);
  const Tensor *gate = tensor(gate_), *scale = tensor(scale_), *offset = tensor(offset_);
  if (!r || !k || !v || !w || !u || !gate || !scale || !offset || !plain(N, *r, *k, *v, *w, *u)) return py::none();
  const int64_t B = r->size(0), T = r->size(1), C = r->size(2), H = C / N;
  if (r->scalar_type() != at::kBFloat16 || gate->sizes() != r->sizes() || gate->scalar_type() != r->scalar_type() ||
      gate->device() != r->device() || !gate->is_contiguous() || scale->numel() != C || offset->numel() != C ||
      scale->device() != r->device() || offset->device() != r->device())
    return py::none();
  const Tensor state = s0 ? *s0 : Tensor();
  if (s0 ? !plain_state(N, *r, state) : !s0_.is_none()) return py::none();
  const bool return_state = truth(return_state_);
  const double eps = py::float_(eps_);
  if (at::GradMode::is_enabled() && any_requires_grad({r, k, v, w, u, gate, scale, offset})) {
    if (return_state || s0 || !wkv6_forward_gn_gate_save_supported(code_of(r->scalar_type()), B, T, C, H)) return py::none();
    return py::make_tuple(wrap(unlocked([&] { return Wkv6GnGate::apply(*r, *k, *v, *w, *u, *gate, *scale, *offset, H, eps); })), py::none());
  }
  return wrap(unlocked([&] {
    return forward_gn_gate(H, Tensor(), *r, *k, *v, *w, *u, state, *gate, *scale, *offset, eps, return_state);
  }));
}

Tensor given(const std::optional<Tensor> &t) { return t.has_value() ? *t : Tensor(); }

}  // namespace

PYBIND11_MODULE(_wkv6_torch, m) {
  m.def("try_call", &try_call);
  m.def("try_gn_gate", &try_gn_gate);
  m.def("wkv6", [](const Tensor &r, const Tensor &k, const Tensor &v, const Tensor &w, const Tensor &u, int64_t H, int64_t algo) {
    return unlocked([&] { return Wkv6::apply(r, k, v, w, u, H, algo); });
  });
  m.def("wkv6_gn_gate", [](const Tensor &r, const Tensor &k, const Tensor &v, const Tensor &w, const Tensor &u, const Tensor &gate,
                           const Tensor &scale, const Tensor &offset, int64_t H, double eps) {
    return unlocked([&] { return Wkv6GnGate::apply(r, k, v, w, u, gate, scale, offset, H, eps); });
  });
  m.def("shift_mix", [](const Tensor &x, const Tensor &mix_x, const Tensor &a, const Tensor &w2t, const Tensor &bias) {
    for (const Tensor *t : {&mix_x, &a, &w2t, &bias})
      TORCH_CHECK(t->device() == x.device(), "wkv6: x and the mixers' parameters must be on one device");   // (the kernels take addresses)
    const variable_list o = unlocked([&] { return ShiftMix::apply(x, mix_x, a, w2t, bias); });
    return py::make_tuple(wrap(o[0]), wrap(o[1]), wrap(o[2]), wrap(o[3]), wrap(o[4]));
  });
  m.def("forward_with_state", [](int64_t H, const std::optional<Tensor> &map, const Tensor &r, const Tensor &k, const Tensor &v,
                                 const Tensor &w, const Tensor &u, const std::optional<Tensor> &s0, int64_t algo, int state_code,
                                 bool backward_follows) {
    const ScalarType st = state_code == WKV6_F32 ? at::kFloat : state_code == WKV6_F16 ? at::kHalf : at::kBFloat16;
    return wrap(unlocked([&] { return forward_with_state(H, given(map), r, k, v, w, u, given(s0), algo, st, backward_follows); }));
  }, py::arg(), py::arg(), py::arg(), py::arg(), py::arg(), py::arg(), py::arg(), py::arg(), py::arg(), py::arg(), py::arg("backward_follows") = false);
  m.def("forward_gn_gate", [](int64_t H, const std::optional<Tensor> &map, const Tensor &r, const Tensor &k, const Tensor &v, const Tensor &w,
                              const Tensor &u, const std::optional<Tensor> &s0, const Tensor &gate, const Tensor &scale,
                              const Tensor &offset, double eps, bool want_state) {
    return wrap(unlocked([&] {
      return forward_gn_gate(H, given(map), r, k, v, w, u, given(s0), gate, scale, offset, eps, want_state);
    }));
  });
}
