// Autograd nodes of flash_attn / flash_attn_gqa and apply_rotary_qk in C++
// (Python module flash_attn_volta._fa_torch), a client of the C ABI in
// fa_mi355x.h.
//
// The reference's autograd.Function (flash_attn_volta/autograd.py:19-59)
// is Python, and so is this package's (autograd.py).  A Python backward
// node makes torch's autograd engine thread take the GIL while the thread
// that called backward() waits for it, a hand-off that costs about as much
// host time as the whole fwd+bwd launch work of a small config.  This node
// runs its backward in C++ without the GIL.  Python keeps the argument
// checks and the per-signature launch plan (forward.py); a plan handed
// here (make_plan) holds the sizes, strides, scale and workspace sizes the
// two C calls need, and attn() runs the forward and records the node.
#include <torch/extension.h>

#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <optional>
#include <tuple>
#include <unordered_set>
#include <vector>

#include "fa_mi355x.h"

// Weak, so that the module still loads beside a library of another ABI
// version without them, as far as the version check below.
extern "C" {
__attribute__((weak)) decltype(fa_rope_qk_fwd) fa_rope_qk_fwd;
__attribute__((weak)) decltype(fa_rope_qk_bwd) fa_rope_qk_bwd;
__attribute__((weak)) decltype(fa_rope_qk_workspace_bytes) fa_rope_qk_workspace_bytes;
}

namespace {

using torch::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// Launch arguments of one call signature.  Plans live until the process
// ends (deduplicated by content), so a node's plan pointer never dangles.
struct Plan {
  int B, Sq, Sk, H, Hk, D;
  int gqa, causal, dtype;
  float scale;
  int64_t q_st[4], k_st[4], v_st[4], o_st[4];   // kernel strides, 0 for size-1 dims
  int64_t dq_st[4], dk_st[4];                   // contiguous gradients
  size_t fwd_ws;                                // fa_fwd_ws workspace, 0: plain forward
  size_t ws_split, ws_plain;                    // backward workspace, split schedule or not
};

constexpr size_t kPlanInts = 9 + 24 + 3;

std::mutex g_mu;
std::map<std::vector<int64_t>, std::unique_ptr<Plan>> g_plans;
std::unordered_set<int64_t> g_handles;

int64_t make_plan(const std::vector<int64_t> &v, double scale) {
  TORCH_CHECK(v.size() == kPlanInts, "make_plan: expected ", kPlanInts, " integers, got ", v.size());
  std::vector<int64_t> key(v);
  const float s = static_cast<float>(scale);
  int32_t bits;
  std::memcpy(&bits, &s, sizeof bits);
  key.push_back(bits);
  std::lock_guard<std::mutex> lock(g_mu);
  auto it = g_plans.find(key);
  if (it != g_plans.end()) return reinterpret_cast<int64_t>(it->second.get());
  auto p = std::make_unique<Plan>();
  size_t i = 0;
  p->B = (int)v[i++]; p->Sq = (int)v[i++]; p->Sk = (int)v[i++];
  p->H = (int)v[i++]; p->Hk = (int)v[i++]; p->D = (int)v[i++];
  p->gqa = (int)v[i++]; p->causal = (int)v[i++]; p->dtype = (int)v[i++];
  for (int64_t *st : {p->q_st, p->k_st, p->v_st, p->o_st, p->dq_st, p->dk_st})
    for (int j = 0; j < 4; ++j) st[j] = v[i++];
  p->fwd_ws = (size_t)v[i++];
  p->ws_split = (size_t)v[i++];
  p->ws_plain = (size_t)v[i++];
  p->scale = s;
  const int64_t h = reinterpret_cast<int64_t>(p.get());
  g_handles.insert(h);
  g_plans.emplace(std::move(key), std::move(p));
  return h;
}

const Plan &plan_of(int64_t h) {
  std::lock_guard<std::mutex> lock(g_mu);
  TORCH_CHECK(g_handles.count(h), "flash_attn_volta._fa_torch: unknown plan handle");
  return *reinterpret_cast<const Plan *>(h);
}

void *stream_of(const Tensor &t) {
  return c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

bool aligned(const Tensor &t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; }

// The kernels' strides of a (B, S, H, D) tensor they can read in place (unit
// D stride, the others non-negative multiples of 8 elements, 128 rows of a
// head within 31-bit byte offsets; `half_cols`, the attention kernels at 16
// columns: a whole head), 0 for size-1 dims, as the plan's; false for any
// other layout.
bool kernel_strides(const Tensor &t, int64_t (&st)[4], bool half_cols = false) {
  const int64_t *size = t.sizes().data(), *stride = t.strides().data();
  if (stride[3] != 1) return false;
  for (int i = 0; i < 3; ++i) {
    st[i] = size[i] == 1 ? 0 : stride[i];
    if (st[i] < 0 || (st[i] & 7) != 0) return false;
  }
  st[3] = 1;
  if (half_cols && (double)(size[1] - 1) * st[1] * 2 + 64 > INT32_MAX) return false;
  return 127 * st[1] * 2 + 2 * size[3] <= INT32_MAX;
}

// `t` as the kernels read it, its strides in `st`: itself where the layout and
// alignment allow, else a contiguous copy.
Tensor kernel_ready(const Tensor &t, int64_t (&st)[4], bool half_cols = false) {
  if (kernel_strides(t, st, half_cols) && aligned(t)) return t;
  Tensor c = t.clone(at::MemoryFormat::Contiguous);
  kernel_strides(c, st);
  return c;
}

// What a node saved may come back changed: hooks on saved tensors
// (torch.autograd.graph) return a tensor of their own, save_on_cpu for one a
// contiguous copy of any view.  The strides that a backward passes are
// therefore the returned tensor's; one of another shape, type or device than
// was saved is refused, as the kernels would read past its end.
void check_saved(const Tensor &t, at::IntArrayRef sizes, at::ScalarType dtype, at::Device device) {
  TORCH_CHECK(t.defined() && t.sizes() == sizes && t.scalar_type() == dtype &&
                  t.device() == device,
              "flash_attn_volta: a saved tensor came back with another shape, dtype or device");
}

void check(int rc, const char *where) {
  TORCH_CHECK(rc == FA_OK, where, ": ", fa_strerror(rc), " (status ", rc, ")");
}

struct FlashAttnFn : public torch::autograd::Function<FlashAttnFn> {
  static Tensor forward(AutogradContext *ctx, const Tensor &q, const Tensor &k, const Tensor &v,
                        int64_t handle, bool split) {
    const Plan &p = *reinterpret_cast<const Plan *>(handle);
    const c10::DeviceGuard guard(q.device());
    // (head_dim 16 runs as half of p.D = 32)
    Tensor out = at::empty({p.B, p.Sq, p.H, q.size(3)}, q.options());
    Tensor lse = at::empty({p.B, p.H, p.Sq}, q.options().dtype(at::kFloat));
    void *stream = stream_of(q);
    if (p.fwd_ws) {
      Tensor ws = at::empty({(int64_t)p.fwd_ws}, q.options().dtype(at::kByte));
      check(fa_fwd_ws(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
                      lse.data_ptr<float>(), ws.data_ptr(), p.fwd_ws, p.B, p.Sq, p.Sk, p.H, p.Hk,
                      p.D, p.q_st, p.k_st, p.v_st, p.o_st, p.scale, p.causal, p.dtype, stream),
            "fa_fwd_ws");
    } else if (p.gqa) {
      check(fa_fwd_gqa(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
                       lse.data_ptr<float>(), p.B, p.Sq, p.Sk, p.H, p.Hk, p.D, p.q_st, p.k_st,
                       p.v_st, p.o_st, p.scale, p.causal, p.dtype, stream),
            "fa_fwd_gqa");
    } else {
      check(fa_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), lse.data_ptr<float>(),
                   p.B, p.Sq, p.H, p.D, p.q_st, p.k_st, p.v_st, p.o_st, p.scale, p.causal, stream),
            "fa_fwd");
    }
    ctx->save_for_backward({q, k, v, out, lse});
    ctx->saved_data["plan"] = handle;
    ctx->saved_data["split"] = split;
    return out;
  }

  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const Plan &p = *reinterpret_cast<const Plan *>(ctx->saved_data["plan"].toInt());
    const bool split = ctx->saved_data["split"].toBool();
    // the engine hands dO over in out's shape, on its device
    const at::Device device = grads[0].device();
    const auto dtype = (p.dtype & ~FA_HALF_COLS) == FA_DTYPE_BF16 ? at::kBFloat16 : at::kHalf;
    const int64_t cols = grads[0].size(3);
    const c10::DeviceGuard guard(device);
    for (int i : {0, 3}) check_saved(s[i], {p.B, p.Sq, p.H, cols}, dtype, device);
    for (int i : {1, 2}) check_saved(s[i], {p.B, p.Sk, p.Hk, cols}, dtype, device);
    check_saved(s[4], {p.B, p.H, p.Sq}, at::kFloat, device);
    int64_t q_st[4], k_st[4], v_st[4], o_st[4], do_st[4];
    const bool half = cols != p.D;
    const Tensor q = kernel_ready(s[0], q_st, half), k = kernel_ready(s[1], k_st, half),
                 v = kernel_ready(s[2], v_st, half), out = kernel_ready(s[3], o_st, half);
    const Tensor lse = s[4].is_contiguous() && aligned(s[4])
                           ? s[4] : s[4].clone(at::MemoryFormat::Contiguous);
    // dO as the kernels read it: the forward's dtype, in place when its
    // layout allows (a model's transposed (B, H, S, D) gradient does: making
    // it contiguous cost 11 us of 113 at (8,1024,12,64)), 16-byte aligned
    const Tensor dout = kernel_ready(
        grads[0].scalar_type() == dtype ? grads[0] : grads[0].to(dtype), do_st, half);
    Tensor dq = at::empty({p.B, p.Sq, p.H, cols}, q.options());
    // separate allocations, as the Python path's
    Tensor dk = at::empty({p.B, p.Sk, p.Hk, cols}, q.options());
    Tensor dv = at::empty({p.B, p.Sk, p.Hk, cols}, q.options());
    const size_t nb = split ? p.ws_split : p.ws_plain;
    Tensor ws = at::empty({(int64_t)nb}, q.options().dtype(at::kByte));
    void *stream = stream_of(q);
    if (p.gqa) {
      check(fa_bwd_gqa(dout.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
                       lse.data_ptr<float>(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(),
                       ws.data_ptr(), nb, p.B, p.Sq, p.Sk, p.H, p.Hk, p.D, do_st, q_st,
                       k_st, v_st, o_st, p.dq_st, p.dk_st, p.dk_st, p.scale, p.causal,
                       p.dtype, stream),
            "fa_bwd_gqa");
    } else {
      check(fa_bwd(dout.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
                   lse.data_ptr<float>(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(),
                   ws.data_ptr(), nb, p.B, p.Sq, p.H, p.D, do_st, q_st, k_st, v_st,
                   o_st, p.dq_st, p.dk_st, p.dk_st, p.scale, p.causal, stream),
            "fa_bwd");
    }
    return {dq, dk, dv, Tensor(), Tensor()};
  }
};

// The forward of plan `handle` on q, k, v (whose shapes, strides, dtype and
// device the caller matched to the plan), recording the backward node when
// any input requires grad.  None when a data pointer is not 16-byte
// aligned: the caller then takes its general path.
std::optional<Tensor> attn(int64_t handle, const Tensor &q, const Tensor &k, const Tensor &v,
                           bool split) {
  plan_of(handle);
  if (!aligned(q) || !aligned(k) || !aligned(v)) return std::nullopt;
  return FlashAttnFn::apply(q, k, v, handle, split);
}

// The QK-norm + rotary prologue (rope.py's apply_rotary_qk) on tensors the
// kernels read in place.  A step of it is three kernels of some 45 us at
// (1, 4096, 32 / 8 heads, 128); a Python node around them took 178 us of host
// time a step.
using OptTensor = std::optional<Tensor>;

int dtype_of(const Tensor &t) {
  return t.scalar_type() == at::kHalf ? FA_DTYPE_F16 : FA_DTYPE_BF16;
}

const void *ptr_or_null(const OptTensor &t) { return t && t->defined() ? t->data_ptr() : nullptr; }

// (b, s) strides of a (1 or B, S, D) or (S, D) table, 0 for size-1 dims.
void table_strides(const Tensor &t, int64_t (&st)[2]) {
  const int64_t d = t.dim();
  st[0] = d == 2 || t.size(0) == 1 ? 0 : t.stride(0);
  st[1] = t.size(d - 2) == 1 ? 0 : t.stride(d - 2);
}

// A table that the kernels read in place, its strides in `st`: unit D stride,
// the others non-negative multiples of 8 elements, 16-byte aligned.
bool table_ready(const Tensor &t, int64_t (&st)[2]) {
  table_strides(t, st);
  return t.stride(t.dim() - 1) == 1 && st[0] >= 0 && st[1] >= 0 && st[0] % 8 == 0 &&
         st[1] % 8 == 0 && aligned(t);
}

struct RopeFn : public torch::autograd::Function<RopeFn> {
  static variable_list forward(AutogradContext *ctx, const Tensor &q, const Tensor &k,
                               const Tensor &cos, const Tensor &sin, const OptTensor &wq,
                               const OptTensor &wk, double eps) {
    const c10::DeviceGuard guard(q.device());
    Tensor qo = at::empty(q.sizes(), q.options()), ko = at::empty(k.sizes(), k.options());
    int64_t q_st[4], k_st[4], qo_st[4], ko_st[4], cs[2];
    kernel_strides(q, q_st);
    kernel_strides(k, k_st);
    kernel_strides(qo, qo_st);
    kernel_strides(ko, ko_st);
    table_strides(cos, cs);
    check(fa_rope_qk_fwd(q.data_ptr(), k.data_ptr(), qo.data_ptr(), ko.data_ptr(), cos.data_ptr(),
                         sin.data_ptr(), ptr_or_null(wq), ptr_or_null(wk), (float)eps,
                         (int)q.size(0), (int)q.size(1), (int)q.size(2), (int)k.size(2),
                         (int)q.size(3), q_st, k_st, qo_st, ko_st, cs, dtype_of(q), stream_of(q)),
          "fa_rope_qk_fwd");
    // the forward's inputs are needed again only to recompute a norm
    ctx->save_for_backward({wq ? q : Tensor(), wk ? k : Tensor(), cos, sin, wq.value_or(Tensor()),
                            wk.value_or(Tensor())});
    ctx->saved_data["eps"] = eps;
    return {qo, ko};
  }

  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const double eps = ctx->saved_data["eps"].toDouble();
    // the engine hands the gradients over in the outputs' shapes and dtype
    const auto dtype = grads[0].scalar_type();
    const at::Device device = grads[0].device();
    const c10::DeviceGuard guard(device);
    const int B = (int)grads[0].size(0), S = (int)grads[0].size(1), H = (int)grads[0].size(2),
              Hk = (int)grads[1].size(2), D = (int)grads[0].size(3);
    const bool norm[2] = {s[4].defined(), s[5].defined()};
    Tensor cos = s[2], sin = s[3], w[2];
    const bool one = cos.dim() == 3 && cos.size(0) == 1;
    check_saved(cos, cos.dim() == 2 ? at::DimVector{S, D} : at::DimVector{one ? 1 : B, S, D}, dtype,
                device);
    check_saved(sin, cos.sizes(), dtype, device);
    int64_t g_st[2][4], x_st[2][4], d_st[2][4], cs[2], sn[2];
    if (!table_ready(cos, cs) || !table_ready(sin, sn) || cs[0] != sn[0] || cs[1] != sn[1]) {
      cos = cos.clone(at::MemoryFormat::Contiguous);
      sin = sin.clone(at::MemoryFormat::Contiguous);
      table_ready(cos, cs);
    }
    const auto opt = cos.options();
    Tensor g[2], x[2], d[2], dw[2];
    for (int i = 0; i < 2; ++i) {
      g[i] = kernel_ready(grads[i].scalar_type() == dtype ? grads[i] : grads[i].to(dtype),
                          g_st[i]);
      if (norm[i]) {
        check_saved(s[i], g[i].sizes(), dtype, device);
        check_saved(s[4 + i], {D}, dtype, device);
        x[i] = kernel_ready(s[i], x_st[i]);
        w[i] = s[4 + i].is_contiguous() && aligned(s[4 + i])
                   ? s[4 + i] : s[4 + i].clone(at::MemoryFormat::Contiguous);
        dw[i] = at::empty({D}, opt);   // the weight's dtype
      } else {
        x[i] = g[i];   // read for a normed side only
        std::copy(g_st[i], g_st[i] + 4, x_st[i]);
      }
      d[i] = at::empty(g[i].sizes(), opt);
      kernel_strides(d[i], d_st[i]);
    }
    Tensor ws;
    if (norm[0] || norm[1])
      ws = at::empty({(int64_t)fa_rope_qk_workspace_bytes(B, S, H, Hk, D)}, opt.dtype(at::kByte));
    auto ptr = [](const Tensor &t) -> void * { return t.defined() ? t.data_ptr() : nullptr; };
    check(fa_rope_qk_bwd(g[0].data_ptr(), g[1].data_ptr(), x[0].data_ptr(), x[1].data_ptr(),
                         cos.data_ptr(), sin.data_ptr(), ptr(w[0]), ptr(w[1]), (float)eps,
                         d[0].data_ptr(), d[1].data_ptr(), static_cast<float *>(ptr(dw[0])),   // FA_DW_16
                         static_cast<float *>(ptr(dw[1])), ptr(ws),
                         ws.defined() ? (size_t)ws.numel() : 0, B, S, H, Hk, D, g_st[0], g_st[1],
                         x_st[0], x_st[1], d_st[0], d_st[1], cs, dtype_of(cos) | FA_DW_16,
                         stream_of(cos)),
          "fa_rope_qk_bwd");
    return {d[0], d[1], Tensor(), Tensor(), dw[0], dw[1], Tensor()};
  }
};

// (q_out, k_out) with the node recorded, or None for anything the kernels do
// not take in place as it is (other dtypes, devices and layouts, empty or
// misaligned tensors, tables that need a cast or have unequal strides or
// gradients, invalid arguments): the caller's general path copies, casts or
// raises.
std::optional<std::tuple<Tensor, Tensor>> rope(const Tensor &q, const Tensor &k, const Tensor &cos,
                                               const Tensor &sin, const OptTensor &wq,
                                               const OptTensor &wk, double eps) {
  if (q.dim() != 4 || k.dim() != 4 || !q.is_cuda()) return std::nullopt;
  const auto dt = q.scalar_type();
  const int64_t B = q.size(0), S = q.size(1), H = q.size(2), D = q.size(3), Hk = k.size(2);
  if ((dt != at::kHalf && dt != at::kBFloat16) || q.numel() == 0 || k.numel() == 0 ||
      (D != 16 && D != 32 && D != 64 && D != 128) || k.size(0) != B || k.size(1) != S ||
      k.size(3) != D || B > INT32_MAX || S > INT32_MAX ||
      (double)B * S * (double)std::max(H, Hk) > 2147483647.0)
    return std::nullopt;
  auto same = [&](const Tensor &t) {
    return t.scalar_type() == dt && t.device() == q.device() && aligned(t);
  };
  int64_t st[4];
  if (!same(q) || !same(k) || !kernel_strides(q, st) || !kernel_strides(k, st))
    return std::nullopt;
  int64_t c_st[2], s_st[2];
  for (const Tensor *t : {&cos, &sin}) {
    const int64_t d = t->dim();
    if ((d != 2 && d != 3) || t->size(d - 1) != D || t->size(d - 2) != S ||
        (d == 3 && t->size(0) != 1 && t->size(0) != B) || !same(*t) || t->requires_grad() ||
        !table_ready(*t, t == &cos ? c_st : s_st))
      return std::nullopt;
  }
  if (cos.sizes() != sin.sizes() || c_st[0] != s_st[0] || c_st[1] != s_st[1]) return std::nullopt;
  for (const OptTensor *w : {&wq, &wk}) {
    if (!*w) continue;
    if ((*w)->dim() != 1 || (*w)->size(0) != D || !same(**w) || !(*w)->is_contiguous() ||
        !(std::isfinite(eps) && eps >= 0.0))
      return std::nullopt;
  }
  variable_list r = RopeFn::apply(q, k, cos, sin, wq, wk, eps);
  return std::make_tuple(r[0], r[1]);
}

}  // namespace

PYBIND11_MODULE(_fa_torch, m) {
  // This module calls the library's entry points with the argument lists of
  // the header it was compiled against; a library built from another ABI
  // version (the two .so files are built separately) would take them
  // without an error.  Refuse to load then: the Python autograd path, which
  // checks the version itself, takes over.
  if (fa_abi_version() != FA_ABI_VERSION) {
    PyErr_Format(PyExc_ImportError,
                 "_fa_torch was built for libfa_mi355x ABI %d, the loaded library has ABI %d: "
                 "rebuild both (flash_attn_volta.build)",
                 (int)FA_ABI_VERSION, (int)fa_abi_version());
    throw pybind11::error_already_set();
  }
  m.doc() = "C++ autograd nodes of flash_attn_volta's flash_attn / flash_attn_gqa / apply_rotary_qk";
  m.def("make_plan", &make_plan, "register a launch plan (ints, sm_scale) -> handle");
  m.def("rope", &rope, "QK-norm + rotary prologue, recording the C++ backward node, or None");
  m.def("attn", &attn, "forward of a plan, recording the C++ backward node");
  m.attr("PLAN_INTS") = (int64_t)kPlanInts;
}
