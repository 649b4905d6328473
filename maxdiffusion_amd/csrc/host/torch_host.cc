// The torch-side host path in C++: what ops.py and attention_op.py do around a C-ABI call (checks, strides, allocation,
// the stream, the autograd node), for the inputs that need nothing unusual.  Every function returns None for any other
// input -- another dtype, a CPU tensor, a shape the kernels refuse -- and the Python path beside the call takes over and
// raises or converts as it always did; nothing is computed here that the kernels do not compute.  A backward call that a kernel
// refuses (a gradient at an unaligned address) raises the MdattnError that the Python nodes raise.
//
// Why native: a call of the smallest size is host time (4 heads x 126 tokens: 10 us of kernels).  The Python path took
// 36.7 us for prologue + attention (ctypes' conversion of twenty arguments, four stride structs, the checks), this one
// 16.5; a training step's backward runs in autograd's own thread without the interpreter: 255-465 us of host time per
// step become 91-108.
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <pybind11/stl.h>
#include <torch/csrc/utils/pybind.h>

#include <array>
#include <cmath>
#include <optional>

#include "mdattn.h"
#include "mdattn_host.h"

namespace {

namespace py = pybind11;
using at::Tensor;
using OptTensor = std::optional<Tensor>;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

void* stream() { return c10::hip::getCurrentHIPStream().stream(); }
const void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
void* mut(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
float* f32(const Tensor& t) { return t.defined() ? t.data_ptr<float>() : nullptr; }

Tensor value(const OptTensor& t) { return t.has_value() ? *t : Tensor(); }
// autograd's apply() takes an argument that may be missing as an optional, never as an undefined tensor
OptTensor opt(const Tensor& t) { return t.defined() ? OptTensor(t) : std::nullopt; }
bool bf16_on(const Tensor& t, const Tensor& ref) {
  return t.is_cuda() && t.scalar_type() == at::kBFloat16 && t.get_device() == ref.get_device() && !t.is_neg();
}
bool wants_grad(std::initializer_list<const Tensor*> ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t->defined() && t->requires_grad()) return true;
  return false;
}
// what a saved-tensor hook hands back is read with the form that the forward checked, or refused
void unpacked(bool ok) { TORCH_CHECK_VALUE(ok, "a tensor saved for the backward pass came back from its hook with another dtype, shape or layout"); }
// a backward call: _lib.check(rc, where), whose MdattnError autograd's engine carries back to the thread that waits for it
void must(int rc, const char* where) {
  if (rc == MDATTN_OK) return;
  py::gil_scoped_acquire gil;
  try {
    py::module_::import("maxdiffusion_amd._lib").attr("check")(rc, where);
  } catch (py::error_already_set& e) {
    e.restore();
  }
  python_error err;
  err.persist();
  throw err;
}
// thrown by a node's forward when a kernel refuses the request, before anything was saved: the Python path takes the call
struct Refused {};
template <class F>
auto unless_refused(F&& apply) -> std::optional<decltype(apply())> {
  try {
    return apply();
  } catch (const Refused&) {
    return std::nullopt;
  }
}

// [B,S,H,D] as the kernels walk it, over a rank-3 [B,S,H*D] or a rank-4 [B,H,S,D] tensor (attention_op._as_bshd)
struct View {
  int64_t b = 0, s = 0, h = 0, d = 0;
  mdattn_strides st{0, 0, 0};
};
std::optional<View> as_view(const Tensor& t, int64_t heads) {
  View v;
  if (t.dim() == 3) {
    const int64_t n = t.size(2);
    if (t.stride(2) != 1 || heads <= 0 || n % heads) return std::nullopt;
    v.b = t.size(0); v.s = t.size(1); v.h = heads; v.d = n / heads;
    v.st = {t.stride(0), t.stride(1), v.d};
  } else if (t.dim() == 4) {
    if (t.stride(3) != 1) return std::nullopt;
    v.b = t.size(0); v.h = t.size(1); v.s = t.size(2); v.d = t.size(3);
    v.st = {t.stride(0), t.stride(2), t.stride(1)};
  } else {
    return std::nullopt;
  }
  return v;
}
bool aligned(const Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; }
// Whether the kernels read this place and these strides (their own checks refuse the others): the padding of a head dim makes
// a copy, and with it takes views at any address, so head dims walked unpadded have to fall back to it before a node exists.
bool walkable(const Tensor& t, const View& v) {
  const int64_t m = v.st.batch | v.st.seq | v.st.head;
  return aligned(t) && m % 8 == 0 && v.st.seq >= v.d && v.st.seq < (1 << 23) && v.st.head > 0;
}
// a logical [B,S,H,D] tensor
mdattn_strides strides4(const Tensor& t) { return {t.stride(0), t.stride(1), t.stride(2)}; }

Tensor alloc_bshd(const Tensor& like, int64_t b, int64_t s, int64_t h, int64_t d, bool bhsd) {
  return bhsd ? at::empty({b, h, s, d}, like.options().dtype(at::kBFloat16)).permute({0, 2, 1, 3})
              : at::empty({b, s, h, d}, like.options().dtype(at::kBFloat16));
}
// A gradient as the kernels read it: bf16, last axis contiguous, with the strides of `like` when given.
Tensor grad_like(const Tensor& g, const Tensor& like) {
  Tensor x = g.scalar_type() == at::kBFloat16 ? g : g.to(at::kBFloat16);
  if (like.defined()) return x.strides() == like.strides() ? x : at::empty_strided(like.sizes(), like.strides(), x.options()).copy_(x);
  return x.stride(-1) == 1 ? x : x.contiguous();
}
// The gradients of a prologue's outputs, all with the strides of the first: the kernels walk them with one set.  A first one
// that is expanded (stride 0, as the sum over an axis hands it back) is read in place only when the others are too: nothing
// can be copied into its layout.
bool repeats(const Tensor& t) {
  for (int64_t i = 0; i < t.dim(); ++i)
    if (t.size(i) > 1 && t.stride(i) == 0) return true;
  return false;
}
void grads_alike(std::initializer_list<Tensor*> gs) {
  Tensor& first = **gs.begin();
  first = grad_like(first, Tensor());
  if (repeats(first))
    for (const Tensor* g : gs)
      if (g->defined() && (g->strides() != first.strides() || !aligned(*g) || g->scalar_type() != at::kBFloat16)) {
        first = first.contiguous();
        break;
      }
  for (Tensor* g : gs)
    if (g->defined() && g != &first) *g = grad_like(*g, first);
}

// ------------------------------------------------------------------------------------------------ attention
// A key mask as the kernels take it, in one buffer: the additive bias f32 [B, ceil32(Skv)], then the tile lists
struct Mask {
  float* bias = nullptr;
  int* tiles = nullptr;
  int64_t stride = 0;
  static int64_t cols(int64_t skv) { return (skv + 31) / 32 * 32; }
  static int64_t floats(const View& vk) { return vk.b * cols(vk.s) + mdattn_host_key_tiles_ints((int)vk.b, (int)vk.s); }
  Mask(const Tensor& m, const View& vk) {
    if (!m.defined()) return;
    stride = cols(vk.s);
    bias = m.data_ptr<float>();
    tiles = reinterpret_cast<int*>(bias + vk.b * stride);
  }
};

int fwd(const Tensor& q, const Tensor& k, const Tensor& v, const View& vq, const View& vk, const View& vv, const Tensor& out, const Tensor& lse,
        const Tensor& mask, double scale) {
  const Mask m(mask, vk);
  const mdattn_strides so{out.stride(0), out.stride(1), vq.d};
  const int64_t nws = m.bias ? 0 : mdattn_host_fwd_workspace_floats((int)vq.b, (int)vq.h, (int)vq.s, (int)vk.s, (int)vq.d);
  const Tensor ws = nws ? at::empty({nws}, q.options().dtype(at::kFloat)) : Tensor();
  return mdattn_host_fwd_bf16(stream(), ptr(q), ptr(k), ptr(v), mut(out), f32(lse), (int)vq.b, (int)vq.h, (int)vq.s, (int)vk.s, (int)vq.d, &vq.st, &vk.st,
                              &vv.st, &so, (float)scale, m.bias, m.stride, m.tiles, f32(ws), nws);
}

bool operands(const Tensor& q, const Tensor& k, const Tensor& v, int64_t heads, View& vq, View& vk, View& vv) {
  if (!q.is_cuda() || !bf16_on(q, q) || !bf16_on(k, q) || !bf16_on(v, q)) return false;
  const auto a = as_view(q, heads), b = as_view(k, heads), c = as_view(v, heads);
  if (!a || !b || !c || a->b != b->b || a->b != c->b || a->h != b->h || a->h != c->h || a->d != b->d || a->d != c->d || b->s != c->s) return false;
  vq = *a; vk = *b; vv = *c;
  return true;
}

// q, k, v in the caller's own rank; out [B,Sq,H*D]
struct FlashFn : torch::autograd::Function<FlashFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const OptTensor& mask_, int64_t heads, double scale) {
    const Tensor mask = value(mask_);
    const View vq = *as_view(q, heads), vk = *as_view(k, heads), vv = *as_view(v, heads);
    Tensor out = at::empty({vq.b, vq.s, vq.h * vq.d}, q.options());
    Tensor lse = at::empty({vq.b, vq.h, vq.s}, q.options().dtype(at::kFloat));
    if (fwd(q, k, v, vq, vk, vv, out, lse, mask, scale) != MDATTN_OK) throw Refused{};
    ctx->save_for_backward({q, k, v, out, lse});
    ctx->saved_data["mask"] = mask;  // not for hooks: its tile lists are indices
    ctx->saved_data["heads"] = heads;
    ctx->saved_data["scale"] = scale;
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &q = saved[0], &k = saved[1], &v = saved[2], &out = saved[3], &lse = saved[4];
    const Tensor mask = ctx->saved_data["mask"].toTensor();
    const int64_t heads = ctx->saved_data["heads"].toInt();
    const double scale = ctx->saved_data["scale"].toDouble();
    View vq, vk, vv;
    unpacked(operands(q, k, v, heads, vq, vk, vv) && q.is_non_overlapping_and_dense() && k.is_non_overlapping_and_dense() &&
             v.is_non_overlapping_and_dense() && bf16_on(out, q) && out.is_contiguous() && out.sizes() == grads[0].sizes() && out.dim() == 3 &&
             out.size(0) == vq.b && out.size(1) == vq.s && out.size(2) == vq.h * vq.d && lse.is_cuda() && lse.scalar_type() == at::kFloat &&
             lse.is_contiguous() && lse.numel() == vq.b * vq.h * vq.s && (!mask.defined() || mask.numel() == Mask::floats(vk)));
    const Mask m(mask, vk);
    Tensor dout = grad_like(grads[0], out);
    if (vq.d != 64 && vq.d != 128 && !aligned(dout)) dout = dout.clone();  // (a padded call's backward copies it as well)
    Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
    const int B = (int)vq.b, H = (int)vq.h, Sq = (int)vq.s, Skv = (int)vk.s, D = (int)vq.d;
    mdattn_host_bwd_plan plan;
    const int64_t nws = mdattn_host_bwd_plan_floats(B, H, Sq, Skv, D, m.bias != nullptr, -1, &plan);
    Tensor ws = at::empty({nws}, lse.options());
    const mdattn_strides so{out.stride(0), out.stride(1), vq.d};
    const int rc = mdattn_host_bwd_bf16(stream(), ptr(q), ptr(k), ptr(v), ptr(out), ptr(dout), f32(lse), mut(dq), mut(dk), mut(dv), f32(ws), nws, B, H, Sq,
                                        Skv, D, &vq.st, &vk.st, &vv.st, &so, (float)scale, m.bias, m.stride, m.tiles, &plan);
    must(rc, "mdattn_bwd_bf16");
    return {dq, dk, dv, Tensor(), Tensor(), Tensor()};
  }
};

// [B,Skv] keep-mask (bool or uint8) -> Mask, or undefined when it needs the Python path
Tensor make_mask(const Tensor& keep, const View& vk, const Tensor& ref) {
  if (!keep.is_cuda() || keep.get_device() != ref.get_device() || (keep.scalar_type() != at::kBool && keep.scalar_type() != at::kByte) ||
      keep.dim() != 2 || keep.size(0) != vk.b || keep.size(1) != vk.s || !keep.is_contiguous())
    return Tensor();
  const int B = (int)vk.b, S = (int)vk.s;
  Tensor m = at::empty({Mask::floats(vk)}, keep.options().dtype(at::kFloat));
  const Mask v(m, vk);
  return mdattn_host_key_tiles(stream(), ptr(keep), v.bias, v.tiles, B, S, v.stride) == MDATTN_OK ? m : Tensor();
}

// The registry entry's operands, checked: false when the Python path has to take over
bool flash_args(const Tensor& q, const Tensor& k, const Tensor& v, int64_t heads, double scale, const OptTensor& keep, View& vq, View& vk, View& vv,
                Tensor& mask) {
  if (!operands(q, k, v, heads, vq, vk, vv) || !(scale > 0)) return false;
  if (!mdattn_host_head_dim((int)vq.d)) return false;  // padded first
  if (q.numel() == 0 || k.numel() == 0 || std::max(vq.s, vk.s) >= ((int64_t)1 << 31)) return false;
  return !keep.has_value() || (mask = make_mask(*keep, vk, q)).defined();
}

// The registry entry `hip_flash`: [B,S,H*D] or [B,H,S,D] operands -> [B,Sq,H*D]; q_mul is rounded into q first.
OptTensor flash(const Tensor& q, const Tensor& k, const Tensor& v, int64_t heads, double scale, const OptTensor& keep, double q_mul) {
  View vq, vk, vv;
  Tensor mask;
  if (!flash_args(q, k, v, heads, scale, keep, vq, vk, vv, mask)) return std::nullopt;
  at::NoGradGuard guard;
  Tensor qf = q;
  if (q_mul != 1.0) {
    qf = q.mul(q_mul);
    const auto w = as_view(qf, heads);
    if (!w) return std::nullopt;
    vq = *w;
  }
  Tensor out = at::empty({vq.b, vq.s, vq.h * vq.d}, q.options());
  if (fwd(qf, k, v, vq, vk, vv, out, Tensor(), mask, scale) != MDATTN_OK) return std::nullopt;
  return out;
}

OptTensor flash_autograd(const Tensor& q, const Tensor& k, const Tensor& v, int64_t heads, double scale, const OptTensor& keep) {
  View vq, vk, vv;
  Tensor mask;
  for (const Tensor* t : {&q, &k, &v})
    if (!t->is_non_overlapping_and_dense()) return std::nullopt;  // their gradients take the same strides
  if (!operands(q, k, v, heads, vq, vk, vv) || !walkable(q, vq) || !walkable(k, vk) || !walkable(v, vv)) return std::nullopt;
  if (!flash_args(q, k, v, heads, scale, keep, vq, vk, vv, mask)) return std::nullopt;
  return unless_refused([&] { return FlashFn::apply(q, k, v, opt(mask), heads, scale); });
}

// The registry entry `hip_flash_fp8`: dense bf16 operands of either rank -> [B,Sq,H*D]
OptTensor flash_fp8(const Tensor& q, const Tensor& k, const Tensor& v, int64_t heads, double scale, const OptTensor& keep) {
  View vq, vk, vv;
  Tensor mask;
  for (const Tensor* t : {&q, &k, &v})  // the quantised copies are dense [B,S,H,D]
    if (t->dim() == 4 ? !t->permute({0, 2, 1, 3}).is_contiguous() : !t->is_contiguous()) return std::nullopt;
  if (!flash_args(q, k, v, heads, scale, keep, vq, vk, vv, mask) || (vq.d != 64 && vq.d != 128)) return std::nullopt;
  at::NoGradGuard guard;
  const auto bytes = q.options().dtype(at::kByte);
  Tensor q8 = at::empty({q.numel()}, bytes), k8 = at::empty({k.numel()}, bytes), v8 = at::empty({v.numel()}, bytes);
  Tensor ws = at::empty({mdattn_host_quant3_floats()}, q.options().dtype(at::kFloat));
  if (mdattn_host_quant3_e4m3(stream(), ptr(q), ptr(k), ptr(v), mut(q8), mut(k8), mut(v8), f32(ws), q.numel(), k.numel(),
                              (float)(scale * 1.4426950408889634)) != MDATTN_OK)
    return std::nullopt;
  Tensor out = at::empty({vq.b, vq.s, vq.h * vq.d}, q.options());
  auto dense = [](const View& x) { return mdattn_strides{x.s * x.h * x.d, x.h * x.d, x.d}; };
  const mdattn_strides sq = dense(vq), skv = dense(vk);
  const float *s = f32(ws), scale8 = (float)0.6931471805599453;  // q's quantisation carries scale * log2(e)
  const int B = (int)vq.b, H = (int)vq.h, Sq = (int)vq.s, Skv = (int)vk.s, D = (int)vq.d;
  const Mask m(mask, vk);
  const int rc = m.bias ? mdattn_fwd_fp8_bias(stream(), ptr(q8), ptr(k8), ptr(v8), mut(out), nullptr, B, H, Sq, Skv, D, &sq, &skv, &skv, &sq, scale8, s,
                                              s + 2, s + 4, m.bias, m.stride)
                        : mdattn_fwd_fp8(stream(), ptr(q8), ptr(k8), ptr(v8), mut(out), nullptr, B, H, Sq, Skv, D, &sq, &skv, &skv, &sq, scale8, s, s + 2,
                                         s + 4, MDATTN_FP8_SOFTMAX_BYTE_GRID);
  if (rc != MDATTN_OK) return std::nullopt;
  return out;
}

// One ring step (ops.flash_attention_merge) on logical [B,S,H,D] views; false: the Python path takes it
bool flash_merge(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o_run, const Tensor& lse_run, double scale) {
  if (!q.is_cuda() || !bf16_on(q, q) || !bf16_on(k, q) || !bf16_on(v, q) || q.dim() != 4 || k.dim() != 4 || v.dim() != 4 || o_run.dim() != 4)
    return false;
  if (q.stride(3) != 1 || k.stride(3) != 1 || v.stride(3) != 1 || o_run.stride(3) != 1 || k.sizes() != v.sizes() || k.size(0) != q.size(0) ||
      k.size(2) != q.size(2) || k.size(3) != q.size(3) || o_run.sizes() != q.sizes() || o_run.scalar_type() != at::kFloat || !o_run.is_cuda() ||
      lse_run.scalar_type() != at::kFloat || !lse_run.is_cuda() || !lse_run.is_contiguous() || lse_run.dim() != 3 || lse_run.size(0) != q.size(0) ||
      lse_run.size(1) != q.size(2) || lse_run.size(2) != q.size(1))
    return false;
  const mdattn_strides sq = strides4(q), sk = strides4(k), sv = strides4(v), so = strides4(o_run);
  return mdattn_fwd_bf16_merge(stream(), ptr(q), ptr(k), ptr(v), f32(o_run), f32(lse_run), (int)q.size(0), (int)q.size(2), (int)q.size(1),
                               (int)k.size(1), (int)q.size(3), &sq, &sk, &sv, &so, (float)scale) == MDATTN_OK;
}

// ------------------------------------------------------------------------------------------------ prologues
// A rotary table in one of the layouts that the kernels read in place (attention_op._rope_table)
struct Table {
  Tensor cos, sin;
  int64_t kind = MDATTN_TABLE_PLANES;
};
bool in_place(const Tensor& t, at::ScalarType dtype, int64_t numel, const Tensor& ref) {
  return t.is_cuda() && t.get_device() == ref.get_device() && t.scalar_type() == dtype && t.is_contiguous() && t.numel() == numel &&
         !t.is_conj() && !t.is_neg() && (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0;
}
std::optional<Table> as_table(const OptTensor& a, const OptTensor& b, int64_t s, int64_t d, bool per_head, const Tensor& ref) {
  Table t;
  if (!a.has_value()) return t;
  if (b.has_value()) {  // a (cos, sin) tuple
    if (per_head && in_place(*a, at::kFloat, s * d, ref) && in_place(*b, at::kFloat, s * d, ref)) t.kind = MDATTN_TABLE_REPEATED;
    else if (in_place(*a, at::kFloat, s * d / 2, ref) && in_place(*b, at::kFloat, s * d / 2, ref)) t.kind = MDATTN_TABLE_PLANES;
    else return std::nullopt;
    t.sin = *b;
  } else if (in_place(*a, at::kComplexFloat, s * d / 2, ref)) {
    t.kind = MDATTN_TABLE_COMPLEX;
  } else if (per_head && in_place(*a, at::kFloat, s * d * 2, ref)) {
    t.kind = MDATTN_TABLE_MATRIX;
  } else {
    return std::nullopt;
  }
  t.cos = *a;
  return t;
}
// Replaces a tensor that in_place has accepted, or two of one size (b may be undefined), by copies, in one launch.  False, and nothing
// replaced, for a size that is no multiple of 16 bytes: no kernel takes such rows either.
bool own(Tensor& a, Tensor& b) {
  const Tensor x = at::empty(a.sizes(), a.options()), y = b.defined() ? at::empty(b.sizes(), b.options()) : Tensor();
  if (mdattn_host_copy(stream(), ptr(a), mut(x), ptr(b), mut(y), (int64_t)a.nbytes()) != MDATTN_OK) return false;
  a = x;
  b = y;
  return true;
}
// The table as a node keeps it.  One that is read in place belongs to the caller, who may have made it in inference mode (autograd
// refuses to save such a tensor) or may rewrite it before the backward: a dense copy of it, one launch.  Half planes [S, D/2] were
// always saved as they are.
bool own_table(Table& t) { return !t.cos.defined() || t.kind == MDATTN_TABLE_PLANES || own(t.cos, t.sin); }
const float* table_ptr(const Tensor& t) { return t.defined() ? static_cast<const float*>(t.data_ptr()) : nullptr; }
bool weight_ok(const Tensor& w, int64_t n, const Tensor& ref) { return bf16_on(w, ref) && w.is_contiguous() && w.numel() == n; }

// a saved q (or fused q|k|v), the k beside it, their weights and table in the form that the forward took
bool rows_back(const Tensor& q, const Tensor& k, int64_t dim, bool dense) {
  return bf16_on(q, q) && q.dim() == dim && q.stride(-1) == 1 && (!dense || q.is_non_overlapping_and_dense()) &&
         (!k.defined() || (bf16_on(k, q) && k.sizes() == q.sizes() && k.strides() == q.strides()));
}
bool weights_back(std::initializer_list<const Tensor*> ws, int64_t n, const Tensor& ref) {
  for (const Tensor* w : ws)
    if (w->defined() && !weight_ok(*w, n, ref)) return false;
  return true;
}
bool table_back(const Tensor& cos, const Tensor& sin, int64_t kind, int64_t s, int64_t d, const Tensor& ref) {
  if (!cos.defined()) return true;
  if (kind == MDATTN_TABLE_COMPLEX) return in_place(cos, at::kComplexFloat, s * d / 2, ref);
  if (kind == MDATTN_TABLE_MATRIX) return in_place(cos, at::kFloat, s * d * 2, ref);
  const int64_t n = kind == MDATTN_TABLE_REPEATED ? s * d : s * d / 2;
  return in_place(cos, at::kFloat, n, ref) && in_place(sin, at::kFloat, n, ref);
}

struct Prologue {
  int64_t heads, kind, n_txt = 0;
  double eps, q_mul;
  bool bhsd;
  void save(AutogradContext* ctx) const {
    ctx->saved_data["i"] = c10::List<int64_t>({heads, kind, n_txt});
    ctx->saved_data["f"] = c10::List<double>({eps, q_mul});
  }
  static Prologue saved(AutogradContext* ctx) {
    const auto i = ctx->saved_data["i"].toIntVector();
    const auto f = ctx->saved_data["f"].toDoubleVector();
    return {i[0], i[1], i[2], f[0], f[1], false};
  }
};

// Wan: q, k [B,S,H*D] (k may be undefined) -> {q_out(, k_out)} or empty when a kernel refuses the request
variable_list fullrow_run(const Tensor& q, const Tensor& k, const Tensor& wq, const Tensor& wk, const Tensor& cos, const Tensor& sin, const Prologue& p) {
  const int64_t b = q.size(0), s = q.size(1), d = q.size(2) / p.heads;
  Tensor qo = alloc_bshd(q, b, s, p.heads, d, p.bhsd), ko = k.defined() ? alloc_bshd(q, b, s, p.heads, d, p.bhsd) : Tensor();
  const mdattn_strides so = strides4(qo);
  const int rc = mdattn_host_norm_rope_fullrow(stream(), ptr(q), ptr(k), mut(qo), mut(ko), ptr(wq), ptr(wk), table_ptr(cos), table_ptr(sin), (int)p.kind,
                                               (int)b, (int)s, (int)p.heads, (int)d, (float)p.eps, (float)p.q_mul, q.stride(0), q.stride(1), &so);
  if (rc != MDATTN_OK) return {};
  return k.defined() ? variable_list{qo, ko} : variable_list{qo};
}
struct FullrowFn : torch::autograd::Function<FullrowFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const OptTensor& k_, const Tensor& wq, const OptTensor& wk_,
                               const OptTensor& cos_, const OptTensor& sin_, const Prologue& p) {
    const Tensor k = value(k_), wk = value(wk_), cos = value(cos_), sin = value(sin_);
    variable_list out = fullrow_run(q, k, wq, wk, cos, sin, p);
    if (out.empty()) throw Refused{};
    ctx->save_for_backward({q, k, wq, wk, cos, sin});
    p.save(ctx);
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto sv = ctx->get_saved_variables();
    const Tensor &q = sv[0], &k = sv[1], &wq = sv[2], &wk = sv[3];
    const Prologue p = Prologue::saved(ctx);
    unpacked(rows_back(q, k, 3, true) && q.numel() == g[0].numel());
    const int64_t b = q.size(0), s = q.size(1), n = q.size(2), d = n / p.heads;
    unpacked(weights_back({&wq, &wk}, n, q) && table_back(sv[4], sv[5], p.kind, s, d, q) && g[0].sizes() == at::IntArrayRef({b, s, p.heads, d}));
    const bool has_k = k.defined();
    Tensor gq = g[0], gk = has_k ? g[1] : Tensor();
    grads_alike({&gq, &gk});
    Tensor dq = at::empty_strided(q.sizes(), q.strides(), q.options()), dk = has_k ? at::empty_strided(q.sizes(), q.strides(), q.options()) : Tensor();
    Tensor dwq = at::empty({n}, q.options()), dwk = has_k ? at::empty({n}, q.options()) : Tensor();
    const int64_t nws = mdattn_norm_rope_bwd_workspace_floats(b * s, (has_k ? 2 : 1) * n);
    Tensor ws = at::empty({nws}, q.options().dtype(at::kFloat));
    const mdattn_strides sg = strides4(gq);
    must(mdattn_host_norm_rope_fullrow_bwd(stream(), ptr(q), ptr(k), nullptr, ptr(gq), ptr(gk), mut(dq), mut(dk), ptr(wq), ptr(wk), mut(dwq), mut(dwk),
                                           nullptr, 1, nullptr, nullptr, table_ptr(sv[4]), table_ptr(sv[5]), (int)p.kind, (int)b, (int)s, (int)p.heads, (int)d, (float)p.eps,
                                           (float)p.q_mul, q.stride(0), q.stride(1), dq.stride(0), dq.stride(1), &sg, f32(ws), nws),
         "mdattn_norm_rope_fullrow_bwd");
    return {dq, dk, dwq, dwk, Tensor(), Tensor(), Tensor()};
  }
};

std::optional<variable_list> norm_rope(const Tensor& q, const OptTensor& k_, const Tensor& wq, const OptTensor& wk_, const OptTensor& fa, const OptTensor& fb,
                                       int64_t heads, double eps, double q_mul, bool bhsd) {
  const Tensor k = value(k_), wk = value(wk_);
  if (!q.is_cuda() || !bf16_on(q, q) || q.dim() != 3 || q.numel() == 0 || q.stride(2) != 1 || heads <= 0 || q.size(2) % heads) return std::nullopt;
  const int64_t n = q.size(2);
  if (!weight_ok(wq, n, q)) return std::nullopt;
  if (k.defined() && (!bf16_on(k, q) || k.sizes() != q.sizes() || k.strides() != q.strides() || !wk.defined() || !weight_ok(wk, n, q))) return std::nullopt;
  auto t = as_table(fa, fb, q.size(1), n / heads, false, q);
  if (!t) return std::nullopt;
  const Prologue p{heads, t->kind, 0, eps, q_mul, bhsd};
  if (wants_grad({&q, &k, &wq, &wk})) {
    if (!q.is_non_overlapping_and_dense()) return std::nullopt;
    if (!own_table(*t)) return std::nullopt;
    return unless_refused([&] { return FullrowFn::apply(q, opt(k), wq, k.defined() ? opt(wk) : std::nullopt, opt(t->cos), opt(t->sin), p); });
  }
  variable_list out = fullrow_run(q, k, wq, wk, t->cos, t->sin, p);
  if (out.empty()) return std::nullopt;
  return out;
}

// Flux: q, k logical [B,S,H,D]
variable_list perhead_run(const Tensor& q, const Tensor& k, const Tensor& wq, const Tensor& wk, const Tensor& wqt, const Tensor& wkt, const Tensor& cos,
                          const Tensor& sin, const Prologue& p) {
  const int64_t b = q.size(0), s = q.size(1), h = q.size(2), d = q.size(3);
  Tensor qo = alloc_bshd(q, b, s, h, d, p.bhsd), ko = k.defined() ? alloc_bshd(q, b, s, h, d, p.bhsd) : Tensor();
  const mdattn_strides si = strides4(q), so = strides4(qo);
  const int rc = mdattn_host_norm_rope_perhead(stream(), ptr(q), ptr(k), mut(qo), mut(ko), ptr(wq), ptr(wk), ptr(wqt), ptr(wkt), (int)p.n_txt,
                                               table_ptr(cos), table_ptr(sin), (int)p.kind, (int)b, (int)s, (int)h, (int)d, (float)p.eps, (float)p.q_mul,
                                               &si, &so);
  if (rc != MDATTN_OK) return {};
  return k.defined() ? variable_list{qo, ko} : variable_list{qo};
}
struct PerheadFn : torch::autograd::Function<PerheadFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const OptTensor& k_, const Tensor& wq, const OptTensor& wk_, const OptTensor& wqt_,
                               const OptTensor& wkt_, const OptTensor& cos_, const OptTensor& sin_, const Prologue& p) {
    const Tensor k = value(k_), wk = value(wk_), wqt = value(wqt_), wkt = value(wkt_), cos = value(cos_), sin = value(sin_);
    variable_list out = perhead_run(q, k, wq, wk, wqt, wkt, cos, sin, p);
    if (out.empty()) throw Refused{};
    ctx->save_for_backward({q, k, wq, wk, wqt, wkt, cos, sin});
    p.save(ctx);
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto sv = ctx->get_saved_variables();
    const Tensor &q = sv[0], &k = sv[1], &wq = sv[2], &wk = sv[3], &wqt = sv[4], &wkt = sv[5];
    const Prologue p = Prologue::saved(ctx);
    unpacked(rows_back(q, k, 4, true) && q.sizes() == g[0].sizes());
    const int64_t b = q.size(0), s = q.size(1), h = q.size(2), d = q.size(3);
    unpacked(weights_back({&wq, &wk, &wqt, &wkt}, d, q) && table_back(sv[6], sv[7], p.kind, s, d, q));
    const bool has_k = k.defined();
    Tensor gq = g[0], gk = has_k ? g[1] : Tensor();
    grads_alike({&gq, &gk});
    Tensor dq = at::empty_strided(q.sizes(), q.strides(), q.options()), dk = has_k ? at::empty_strided(q.sizes(), q.strides(), q.options()) : Tensor();
    auto dw = [&](bool want) { return want ? at::empty({d}, q.options()) : Tensor(); };
    Tensor dwq = dw(true), dwk = dw(has_k), dwqt = dw(wqt.defined()), dwkt = dw(wkt.defined() && has_k);
    const int64_t nws = mdattn_norm_rope_bwd_workspace_floats(b * s * h, 4 * d);
    Tensor ws = at::empty({nws}, q.options().dtype(at::kFloat));
    const mdattn_strides si = strides4(q), sd = strides4(dq), sg = strides4(gq);
    must(mdattn_host_norm_rope_perhead_bwd(stream(), ptr(q), ptr(k), ptr(gq), ptr(gk), mut(dq), mut(dk), ptr(wq), ptr(wk), ptr(wqt),
                                           has_k ? ptr(wkt) : nullptr, (int)p.n_txt, mut(dwq), mut(dwk), mut(dwqt), mut(dwkt), 1, table_ptr(sv[6]),
                                           table_ptr(sv[7]), (int)p.kind, (int)b, (int)s, (int)h, (int)d, (float)p.eps, (float)p.q_mul, &si, &sd, &sg,
                                           f32(ws), nws),
         "mdattn_norm_rope_perhead_bwd");
    return {dq, dk, dwq, dwk, dwqt, dwkt, Tensor(), Tensor(), Tensor()};
  }
};

std::optional<variable_list> norm_rope_perhead(const Tensor& q, const OptTensor& k_, const Tensor& wq, const OptTensor& wk_, const OptTensor& wqt_,
                                               const OptTensor& wkt_, int64_t n_txt, const OptTensor& fa, const OptTensor& fb, double eps, double q_mul,
                                               bool bhsd) {
  const Tensor k = value(k_), wk = value(wk_), wqt = value(wqt_), wkt = value(wkt_);
  if (!q.is_cuda() || !bf16_on(q, q) || q.dim() != 4 || q.numel() == 0 || q.stride(3) != 1) return std::nullopt;
  const int64_t d = q.size(3);
  if (!weight_ok(wq, d, q) || (wqt.defined() && !weight_ok(wqt, d, q)) || (wkt.defined() && !weight_ok(wkt, d, q))) return std::nullopt;
  if (k.defined() ? (!bf16_on(k, q) || k.sizes() != q.sizes() || k.strides() != q.strides() || !wk.defined() || !weight_ok(wk, d, q)) : wkt.defined())
    return std::nullopt;
  auto t = as_table(fa, fb, q.size(1), d, true, q);
  if (!t) return std::nullopt;
  const Prologue p{q.size(2), t->kind, n_txt, eps, q_mul, bhsd};
  if (wants_grad({&q, &k, &wq, &wk, &wqt, &wkt})) {
    if (!q.is_non_overlapping_and_dense()) return std::nullopt;
    if (!own_table(*t)) return std::nullopt;
    return unless_refused([&] { return PerheadFn::apply(q, opt(k), wq, k.defined() ? opt(wk) : std::nullopt, opt(wqt), opt(wkt), opt(t->cos), opt(t->sin), p); });
  }
  variable_list out = perhead_run(q, k, wq, wk, wqt, wkt, t->cos, t->sin, p);
  if (out.empty()) return std::nullopt;
  return out;
}

// Wan over one fused q|k|v projection output with its biases
variable_list qkv_run(const Tensor& x, const Tensor& bias, const Tensor& wq, const Tensor& wk, const Tensor& cos, const Tensor& sin, const Prologue& p) {
  const int64_t b = x.size(0), s = x.size(1), d = x.size(2) / 3 / p.heads;
  Tensor o[3];
  for (Tensor& t : o) t = alloc_bshd(x, b, s, p.heads, d, p.bhsd);
  const mdattn_strides so = strides4(o[0]);
  const int rc = mdattn_host_norm_rope_qkv(stream(), ptr(x), ptr(bias), mut(o[0]), mut(o[1]), mut(o[2]), ptr(wq), ptr(wk), table_ptr(cos), table_ptr(sin),
                                           (int)p.kind, (int)b, (int)s, (int)p.heads, (int)d, (float)p.eps, (float)p.q_mul, x.stride(0), x.stride(1), &so);
  if (rc != MDATTN_OK) return {};
  return {o[0], o[1], o[2]};
}
struct QkvFn : torch::autograd::Function<QkvFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& bias, const Tensor& wq, const Tensor& wk, const OptTensor& cos_,
                               const OptTensor& sin_, const Prologue& p) {
    const Tensor cos = value(cos_), sin = value(sin_);
    variable_list out = qkv_run(x, bias, wq, wk, cos, sin, p);
    if (out.empty()) throw Refused{};
    ctx->save_for_backward({x, bias, wq, wk, cos, sin});
    p.save(ctx);
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto sv = ctx->get_saved_variables();
    const Tensor &x = sv[0], &bias = sv[1], &wq = sv[2], &wk = sv[3];
    const Prologue p = Prologue::saved(ctx);
    unpacked(rows_back(x, Tensor(), 3, false));
    const int64_t b = x.size(0), s = x.size(1), n = x.size(2) / 3, d = n / p.heads;
    unpacked(weights_back({&wq, &wk}, n, x) && weight_ok(bias, 3 * n, x) && table_back(sv[4], sv[5], p.kind, s, d, x) &&
             g[0].sizes() == at::IntArrayRef({b, s, p.heads, d}));
    Tensor gq = g[0], gk = g[1], gv = g[2];
    grads_alike({&gq, &gk, &gv});
    // the value block took a view at any address; the copy has gq's strides also where these leave gaps (a clone would close them)
    if (!aligned(gv)) gv = at::empty_strided(gq.sizes(), gq.strides(), gq.options()).copy_(gv);
    Tensor dx = at::empty({b, s, 3 * n}, x.options());
    Tensor dwq = at::empty({n}, x.options()), dwk = at::empty({n}, x.options()), db = at::empty({3 * n}, x.options());
    const int64_t nws = mdattn_norm_rope_bwd_workspace_floats(b * s, 5 * n);
    Tensor ws = at::empty({nws}, x.options().dtype(at::kFloat));
    const mdattn_strides sg = strides4(gq);
    const char* xp = static_cast<const char*>(ptr(x));
    char* dp = static_cast<char*>(mut(dx));
    must(mdattn_host_norm_rope_fullrow_bwd(stream(), xp, xp + 2 * n, ptr(bias), ptr(gq), ptr(gk), dp, dp + 2 * n, ptr(wq), ptr(wk), mut(dwq), mut(dwk),
                                           mut(db), 1, ptr(gv), dp + 4 * n, table_ptr(sv[4]), table_ptr(sv[5]), (int)p.kind, (int)b, (int)s, (int)p.heads, (int)d, (float)p.eps,
                                           (float)p.q_mul, x.stride(0), x.stride(1), dx.stride(0), dx.stride(1), &sg, f32(ws), nws),
         "mdattn_norm_rope_fullrow_bwd");
    return {dx, db, dwq, dwk, Tensor(), Tensor(), Tensor()};
  }
};

std::optional<variable_list> norm_rope_qkv(const Tensor& x, const Tensor& bias, const Tensor& wq, const Tensor& wk, const OptTensor& fa, const OptTensor& fb,
                                           int64_t heads, double eps, double q_mul, bool bhsd) {
  if (!x.is_cuda() || !bf16_on(x, x) || x.dim() != 3 || x.numel() == 0 || x.stride(2) != 1 || heads <= 0 || x.size(2) % (3 * heads)) return std::nullopt;
  const int64_t n = x.size(2) / 3;
  if (!weight_ok(wq, n, x) || !weight_ok(wk, n, x) || !weight_ok(bias, 3 * n, x)) return std::nullopt;
  auto t = as_table(fa, fb, x.size(1), n / heads, false, x);
  if (!t) return std::nullopt;
  const Prologue p{heads, t->kind, 0, eps, q_mul, bhsd};
  if (wants_grad({&x, &bias, &wq, &wk})) {
    if (!own_table(*t)) return std::nullopt;
    return unless_refused([&] { return QkvFn::apply(x, bias, wq, wk, opt(t->cos), opt(t->sin), p); });
  }
  variable_list out = qkv_run(x, bias, wq, wk, t->cos, t->sin, p);
  if (out.empty()) return std::nullopt;
  return out;
}

// LTX-2: q, or q and k with one table; f32 weights; tables of the tensors' own size (mode 1) or [B,H,S,D/2] (mode 2)
struct Rows {
  int64_t heads, mode;
  double eps, w_mul;
};
variable_list rows_run(const Tensor& q, const Tensor& k, const Tensor& wq, const Tensor& wk, const Tensor& cos, const Tensor& sin, const Rows& p) {
  const int64_t b = q.size(0), s = q.size(1), d = q.size(2) / p.heads;
  Tensor qo = alloc_bshd(q, b, s, p.heads, d, false), ko = k.defined() ? alloc_bshd(q, b, s, p.heads, d, false) : Tensor();
  const mdattn_strides so = strides4(qo);
  const int rc = mdattn_host_norm_rope_rows(stream(), ptr(q), ptr(k), q.scalar_type() == at::kFloat, mut(qo), mut(ko), f32(wq), f32(wk), f32(cos), f32(sin),
                                            (int)p.mode, (int)b, (int)s, (int)p.heads, (int)d, (float)p.eps, (float)p.w_mul, q.stride(0), q.stride(1), &so);
  if (rc != MDATTN_OK) return {};
  return k.defined() ? variable_list{qo, ko} : variable_list{qo};
}
struct RowsFn : torch::autograd::Function<RowsFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const OptTensor& k_, const Tensor& wq, const OptTensor& wk_, const OptTensor& cos_,
                               const OptTensor& sin_, const Rows& p) {
    const Tensor k = value(k_), wk = value(wk_), cos = value(cos_), sin = value(sin_);
    variable_list out = rows_run(q, k, wq, wk, cos, sin, p);
    if (out.empty()) throw Refused{};
    // a weight with a factor is saved as a copy, as its product with the factor was: the caller's may be an inference tensor, or
    // be updated before the backward
    Tensor kept_wq = wq, none;
    if (p.w_mul != 1.0 && !own(kept_wq, none)) throw Refused{};
    ctx->save_for_backward({q, k, kept_wq, wk, cos, sin});
    ctx->saved_data["i"] = c10::List<int64_t>({p.heads, p.mode, (int64_t)q.scalar_type()});
    ctx->saved_data["f"] = c10::List<double>({p.eps, p.w_mul});
    ctx->set_materialize_grads(false);  // an output that the loss does not reach: no gradient for its input and weight
    return out;
  }
  // A backward through one output frees what both have saved; the other output's is kept beside, with its versions, so that a
  // second backward through that one runs as it would through a node of its own.
  static void leave(AutogradContext* ctx, const variable_list& sv, int64_t which) {
    variable_list left(6);
    for (const int64_t i : {which, 2 + which, (int64_t)4, (int64_t)5}) left[i] = sv[i];
    c10::List<int64_t> versions;
    for (const Tensor& t : left) versions.push_back(!t.defined() || t.is_inference() ? 0 : t._version());
    ctx->saved_data["left"] = left;
    ctx->saved_data["versions"] = versions;
  }
  static variable_list saved(AutogradContext* ctx, int64_t one, bool pair) {
    try {
      return ctx->get_saved_variables();
    } catch (const c10::Error&) {
      const auto at = ctx->saved_data.find("left");
      if (pair || at == ctx->saved_data.end()) throw;
      const variable_list left = at->second.toTensorVector();
      const auto versions = ctx->saved_data["versions"].toIntVector();
      if (!left[one].defined()) throw;
      for (size_t i = 0; i < left.size(); ++i)
        TORCH_CHECK(!left[i].defined() || left[i].is_inference() || left[i]._version() == versions[i],
                    "one of the variables needed for gradient computation has been modified by an inplace operation");
      ctx->saved_data.erase(at);
      return left;
    }
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const bool has[2] = {grads[0].defined(), grads.size() > 1 && grads[1].defined()};
    if (!has[0] && !has[1]) return variable_list(7);
    const bool pair = has[0] && has[1];
    const int one = has[0] ? 0 : 1;  // the tensor of a backward of one
    const variable_list sv = saved(ctx, one, pair);
    if (!pair && sv[1 - one].defined()) leave(ctx, sv, 1 - one);
    const Tensor q = sv[one], k = pair ? sv[1] : Tensor(), wq = sv[2 + one], wk = pair ? sv[3] : Tensor();
    const auto iv = ctx->saved_data["i"].toIntVector();
    const auto fv = ctx->saved_data["f"].toDoubleVector();
    const int64_t heads = iv[0], mode = iv[1];
    unpacked(q.is_cuda() && (int64_t)q.scalar_type() == iv[2] && q.dim() == 3 && q.stride(2) == 1 && q.is_non_overlapping_and_dense() &&
             (!pair || (k.get_device() == q.get_device() && k.scalar_type() == q.scalar_type() && k.sizes() == q.sizes() && k.strides() == q.strides())));
    const int64_t b = q.size(0), s = q.size(1), n = q.size(2);
    unpacked(grads[one].sizes() == at::IntArrayRef({b, s, heads, n / heads}) && in_place(wq, at::kFloat, n, q) && (!pair || in_place(wk, at::kFloat, n, q)));
    for (const Tensor& t : {sv[4], sv[5]}) unpacked(!mode || in_place(t, at::kFloat, mode == 1 ? q.numel() : q.numel() / 2, q));
    Tensor gq = grads[one], gk = pair ? grads[1] : Tensor();
    grads_alike({&gq, &gk});
    Tensor dq = at::empty_strided(q.sizes(), q.strides(), q.options()), dk = pair ? at::empty_strided(q.sizes(), q.strides(), q.options()) : Tensor();
    Tensor dwq = at::empty({n}, wq.options()), dwk = pair ? at::empty({n}, wq.options()) : Tensor();
    const int64_t nws = mdattn_norm_rope_bwd_workspace_floats(b * s, (pair ? 2 : 1) * n);
    Tensor ws = at::empty({nws}, wq.options());
    const mdattn_strides sg = strides4(gq);
    must(mdattn_host_norm_rope_rows_bwd(stream(), ptr(q), ptr(k), q.scalar_type() == at::kFloat, ptr(gq), ptr(gk), mut(dq), mut(dk), f32(wq), f32(wk),
                                        f32(dwq), f32(dwk), f32(sv[4]), f32(sv[5]), (int)mode, (int)b, (int)s, (int)heads, (int)(n / heads), (float)fv[0],
                                        one ? 1.0f : (float)fv[1], q.stride(0), q.stride(1), dq.stride(0), dq.stride(1), &sg, f32(ws), nws),
         "mdattn_norm_rope_rows_bwd");
    if (one) return {Tensor(), dq, Tensor(), dwq, Tensor(), Tensor(), Tensor()};
    return {dq, dk, dwq, dwk, Tensor(), Tensor(), Tensor()};
  }
};

std::optional<variable_list> norm_rope_rows(const Tensor& q, const OptTensor& k_, const Tensor& wq, const OptTensor& wk_, const OptTensor& cos_,
                                            const OptTensor& sin_, int64_t heads, int64_t mode, double eps, double w_mul) {
  const Tensor k = value(k_), wk = value(wk_), cos = value(cos_), sin = value(sin_);
  if (!q.is_cuda() || (q.scalar_type() != at::kFloat && q.scalar_type() != at::kBFloat16) || q.is_neg() || q.dim() != 3 || q.numel() == 0 ||
      q.stride(2) != 1 || heads <= 0 || q.size(2) % heads)
    return std::nullopt;
  const int64_t b = q.size(0), s = q.size(1), n = q.size(2);
  if (!in_place(wq, at::kFloat, n, q)) return std::nullopt;
  if (k.defined() && (n > 4096 || k.scalar_type() != q.scalar_type() || !k.is_cuda() || k.get_device() != q.get_device() || k.is_neg() ||
                      k.sizes() != q.sizes() || k.strides() != q.strides() || !wk.defined() || !in_place(wk, at::kFloat, n, q)))
    return std::nullopt;
  if (mode) {
    const std::array<int64_t, 3> full{b, s, n};
    const std::array<int64_t, 4> half{b, heads, s, n / heads / 2};
    const at::IntArrayRef want = mode == 1 ? at::IntArrayRef(full) : at::IntArrayRef(half);
    for (const Tensor* t : {&cos, &sin})
      if (!t->defined() || t->sizes() != want || !in_place(*t, at::kFloat, t->numel(), q)) return std::nullopt;
  }
  const Rows p{heads, mode, eps, w_mul};
  const Tensor c = mode ? cos : Tensor(), sn = mode ? sin : Tensor();
  const bool grad_q = wants_grad({&q, &wq}), grad_k = k.defined() ? wants_grad({&k, &wk}) : grad_q;
  if (grad_q != grad_k) return std::nullopt;  // one call each: the other output needs no gradient
  if (grad_q) {
    if (!q.is_non_overlapping_and_dense()) return std::nullopt;
    return unless_refused([&] { return RowsFn::apply(q, opt(k), wq, k.defined() ? opt(wk) : std::nullopt, opt(c), opt(sn), p); });
  }
  variable_list out = rows_run(q, k, wq, wk, c, sn, p);
  if (out.empty()) return std::nullopt;
  return out;
}

// the id of the sources, behind the marker that build.py finds in the file (as in libmdattn.so)
const char kBuildIdRecord[] = "mdattn-build-id:" MDATTN_BUILD_ID;

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("build_id", [] { return std::string(kBuildIdRecord + 16); });
  // Other Python threads run meanwhile, as they do during a call through ctypes: a launch may wait for room in its queue, an
  // allocation for memory.
  using Unlocked = py::call_guard<py::gil_scoped_release>;
  m.def("flash", &flash, Unlocked());
  m.def("flash_autograd", &flash_autograd, Unlocked());
  m.def("flash_fp8", &flash_fp8, Unlocked());
  m.def("flash_merge", &flash_merge, Unlocked());
  m.def("norm_rope", &norm_rope, Unlocked());
  m.def("norm_rope_perhead", &norm_rope_perhead, Unlocked());
  m.def("norm_rope_qkv", &norm_rope_qkv, Unlocked());
  m.def("norm_rope_rows", &norm_rope_rows, Unlocked());
}
