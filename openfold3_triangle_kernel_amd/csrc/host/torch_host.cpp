// Host path of the two operators for plain eager GPU tensors, in C++.
//
// The Python facades stay the definition of the operators: they validate,
// report and handle every form.  A small call is bound by what the host does
// around its launches (N = 128 attention, forward and backward: 45 us of
// kernels behind about 200 us of Python), so the common form is recognised and
// run here: the same checks, the same native calls with the same arguments,
// autograd through C++ nodes.  Everything else returns no value, before any
// launch, and the facade goes on in Python: other dtypes or devices, head
// dimensions that need padding, partially broadcast biases, misaligned
// storage, function transforms, forward-mode AD, dispatch modes.
#include <torch/extension.h>
#include <torch/version.h>

#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>

#include <atomic>
#include <cctype>
#include <cmath>
#include <cstdlib>
#include <optional>
#include <string>

#include "tpf_amd.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// Workspace budget of the attention backward (attention.set_sr_workspace_budget).
std::atomic<int64_t> g_budget{int64_t(8) << 30};

void check(int rc, const char* fn) {
  if (rc != TPF_OK)
    throw std::runtime_error(std::string(fn) + " failed (status " + std::to_string(rc) +
                             "): " + tpf_last_error());
}

void* stream() { return (void*)c10::hip::getCurrentHIPStream().stream(); }

// The policy variables as the facade reads them: the canonical name, then
// the older one, then "1"; surrounding blanks dropped.  Called with the GIL
// held: Python's os.environ assignments change the environment under it.
std::string env_flag(const char* canonical, const char* legacy) {
  const char* v = std::getenv(canonical);
  if (!v) v = std::getenv(legacy);
  std::string s = v ? v : "1";
  const char* ws = " \t\n\r\f\v";
  const size_t b = s.find_first_not_of(ws);
  if (b == std::string::npos) return "";
  return s.substr(b, s.find_last_not_of(ws) - b + 1);
}

bool transforms_active() {
  return c10::impl::tls_is_dispatch_key_included(at::DispatchKey::FuncTorchDynamicLayerFrontMode) ||
         c10::impl::dispatch_mode_enabled();
}

// An ordinary strided tensor on the current GPU.
bool plain(const Tensor& t, c10::DeviceIndex dev) {
  static const at::DispatchKeySet special{
      at::DispatchKey::FuncTorchBatched, at::DispatchKey::FuncTorchGradWrapper,
      at::DispatchKey::Functionalize,    at::DispatchKey::Python,
      at::DispatchKey::ZeroTensor,       at::DispatchKey::Conjugate,
      at::DispatchKey::Negative};
  return t.defined() && t.is_cuda() && t.device().index() == dev && t.layout() == at::kStrided &&
         !t.key_set().has_any(special) && !t._fw_grad(0).defined();
}

bool aligned16(const Tensor& t) { return (uintptr_t)t.const_data_ptr() % 16 == 0; }

// An upstream gradient as the kernels read it: bf16, contiguous, 16-byte aligned.
Tensor kernel_grad(const Tensor& g) {
  const Tensor t = g.to(at::kBFloat16).contiguous();
  return aligned16(t) ? t : t.clone();
}

at::TensorOptions like(const Tensor& t, at::ScalarType dtype) {
  return at::TensorOptions().device(t.device()).dtype(dtype);
}

// Whether `sizes`, aligned to the right of `prefix`, broadcasts to exactly it.
bool broadcasts(at::IntArrayRef sizes, at::IntArrayRef prefix) {
  if (sizes.size() > prefix.size()) return false;
  const size_t off = prefix.size() - sizes.size();
  for (size_t i = 0; i < sizes.size(); ++i)
    if (sizes[i] != 1 && sizes[i] != prefix[off + i]) return false;
  return true;
}

// ------------------------------------------------------------- attention

struct AttentionFn : torch::autograd::Function<AttentionFn> {
  // bias_k: the detached kernel bias; source_bias keeps the autograd edge.
  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v,
                        const Tensor& mask, const Tensor& bias_k, const Tensor& source_bias,
                        int64_t layout, int64_t bias_batches, bool shadow) {
    const int64_t B = q.size(0), O = q.size(1), H = q.size(2), N = q.size(3), D = q.size(4);
    const double scale = 1.0 / std::sqrt((double)D);
    Tensor out = at::empty({B, O, N, H, D}, like(q, at::kBFloat16));
    Tensor lse = at::empty({B, O, H, N}, like(q, at::kFloat));
    const int64_t ws_bytes = tpf_attn_forward_workspace_bytes(B, H, N, bias_batches);
    Tensor ws = at::empty({ws_bytes}, like(q, at::kByte)), res;
    if (shadow) {
      res = at::empty_like(out);
      check(tpf_attn_forward_shadow_bf16(
                q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(),
                (const float*)mask.const_data_ptr(), bias_k.const_data_ptr(), out.data_ptr(),
                (float*)lse.data_ptr(), res.data_ptr(), ws.data_ptr(), ws_bytes, B, O, H, N, D,
                (int)layout, bias_batches, scale, stream()),
            "tpf_attn_forward_shadow_bf16");
    } else {
      check(tpf_attn_forward_bf16(q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(),
                                  (const float*)mask.const_data_ptr(), bias_k.const_data_ptr(),
                                  out.data_ptr(), (float*)lse.data_ptr(), ws.data_ptr(), ws_bytes,
                                  B, O, H, N, D, (int)layout, bias_batches, scale, stream()),
            "tpf_attn_forward_bf16");
    }
    ctx->save_for_backward({q, k, v, mask, bias_k, out, lse, res});
    ctx->saved_data["layout"] = layout;
    ctx->saved_data["batches"] = bias_batches;
    ctx->saved_data["shape"] = source_bias.sizes().vec();
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const Tensor &q = s[0], &k = s[1], &v = s[2], &mask = s[3], &bias_k = s[4], &out = s[5],
                 &lse = s[6], &res = s[7];
    const int64_t layout = ctx->saved_data["layout"].toInt();
    const int64_t batches = ctx->saved_data["batches"].toInt();
    const int64_t B = q.size(0), O = q.size(1), H = q.size(2), N = q.size(3), D = q.size(4);
    const Tensor dout = kernel_grad(grads[0]);
    Tensor d[3];
    for (Tensor& t : d)
      t = layout & TPF_QKV_SEQ_MAJOR
              ? at::empty({B, O, N, H, D}, like(q, at::kBFloat16)).transpose(2, 3)
              : at::empty({B, O, H, N, D}, like(q, at::kBFloat16));
    // The fold writes the bf16 bias gradient in the bias's own storage order.
    Tensor dbias = at::empty({batches, H, N, N}, like(q, at::kBFloat16));
    const int64_t ws_bytes = tpf_attn_backward_workspace_bytes_budget(
        B, O, H, N, D, g_budget.load(std::memory_order_relaxed));
    Tensor ws = at::empty({ws_bytes}, like(q, at::kByte));
    check(tpf_attn_backward_fused_bf16(
              q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(), dout.const_data_ptr(),
              out.const_data_ptr(), res.defined() ? res.const_data_ptr() : nullptr,
              (const float*)lse.const_data_ptr(), (const float*)mask.const_data_ptr(),
              bias_k.const_data_ptr(), d[0].data_ptr(), d[1].data_ptr(), d[2].data_ptr(),
              dbias.data_ptr(), ws.data_ptr(), ws_bytes, B, O, H, N, D,
              (int)layout | TPF_DBIAS_BF16, batches, 1.0 / std::sqrt((double)D), stream()),
          "tpf_attn_backward_fused_bf16");
    if (layout & TPF_BIAS_TRANSPOSED) dbias = dbias.transpose(-1, -2);
    return {d[0], d[1], d[2], Tensor(), Tensor(),
            dbias.reshape(ctx->saved_data["shape"].toIntVector()), Tensor(), Tensor(), Tensor()};
  }
};

// backward, shadow: the policy variables (env_flag).
std::optional<Tensor> attention(const Tensor& q, const Tensor& k, const Tensor& v,
                                const Tensor& res_mask, const Tensor& pair_bias,
                                const std::string& backward, const std::string& sh) {
  if (transforms_active() || !q.is_cuda()) return std::nullopt;
  const c10::DeviceIndex dev = c10::hip::current_device();
  for (const Tensor* t : {&q, &k, &v, &res_mask, &pair_bias})
    if (!plain(*t, dev)) return std::nullopt;
  const int64_t nd = q.dim();
  if (nd < 5 || q.numel() == 0 || k.sizes() != q.sizes() || v.sizes() != q.sizes())
    return std::nullopt;
  for (const Tensor* t : {&q, &k, &v})
    if (t->scalar_type() != at::kBFloat16) return std::nullopt;
  const at::IntArrayRef prefix = q.sizes().slice(0, nd - 4);
  const int64_t O = q.size(-4), H = q.size(-3), N = q.size(-2), D = q.size(-1);
  const int64_t B = c10::multiply_integers(prefix);
  if (D % 8 || D > 64 || H > 65535 || B * O > 65535) return std::nullopt;
  const auto mt = res_mask.scalar_type();
  if ((mt != at::kFloat && mt != at::kBFloat16 && mt != at::kHalf) || res_mask.requires_grad() ||
      res_mask.dim() < 4 || res_mask.size(-4) != O || res_mask.size(-3) != 1 ||
      res_mask.size(-2) != 1 || res_mask.size(-1) != N ||
      !broadcasts(res_mask.sizes().slice(0, res_mask.dim() - 4), prefix))
    return std::nullopt;
  const auto bt = pair_bias.scalar_type();
  if ((bt != at::kFloat && bt != at::kBFloat16) || pair_bias.dim() < 4 || pair_bias.size(-4) != 1 ||
      pair_bias.size(-3) != H || pair_bias.size(-2) != N || pair_bias.size(-1) != N)
    return std::nullopt;
  const at::IntArrayRef bp = pair_bias.sizes().slice(0, pair_bias.dim() - 4);
  const bool shared = c10::multiply_integers(bp) == 1 && bp.size() <= prefix.size();
  if (!shared && bp != prefix) return std::nullopt;
  if (backward == "0" || (sh != "0" && sh != "1")) return std::nullopt;

  // One storage order for q, k and v: contiguous, or the transposed view of a
  // contiguous [*B, O, N, H, D] projection.
  auto order = [](const Tensor& t) {
    if (t.is_contiguous()) return 0;
    return t.transpose(-2, -3).is_contiguous() && aligned16(t) ? 1 : 2;
  };
  const int oq = order(q);
  if (oq == 2 || order(k) != oq || order(v) != oq || !aligned16(q) || !aligned16(k) ||
      !aligned16(v))
    return std::nullopt;
  int64_t layout = (oq ? TPF_QKV_SEQ_MAJOR : 0) | (N % 64 ? TPF_ANY_N : 0);
  auto flat = [&](const Tensor& t) { return nd == 5 ? t : t.reshape({B, O, H, N, D}); };

  Tensor mask = res_mask;
  if (res_mask.dim() != 5 || res_mask.size(0) != B || mt != at::kFloat || nd != 5 ||
      !res_mask.is_contiguous()) {
    std::vector<int64_t> full = prefix.vec();
    full.insert(full.end(), {O, 1, 1, N});
    mask = res_mask.expand(full).reshape({B, O, N}).to(at::kFloat).contiguous();
  }
  const Tensor bias = bt == at::kFloat ? pair_bias.to(at::kBFloat16) : pair_bias;
  Tensor bias_k = bias.detach();
  if (!bias_k.is_contiguous()) {
    if (bias_k.transpose(-1, -2).is_contiguous()) layout |= TPF_BIAS_TRANSPOSED;
    else bias_k = bias_k.contiguous();
  }
  if (!aligned16(mask) || !aligned16(bias_k)) return std::nullopt;
  const bool grad = at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() ||
                                                   v.requires_grad() || bias.requires_grad());
  Tensor out = AttentionFn::apply(flat(q), flat(k), flat(v), mask, bias_k, bias, layout,
                                  shared ? 1 : B, sh == "1" && grad);
  if (nd == 5) return out;
  std::vector<int64_t> shape = prefix.vec();
  shape.insert(shape.end(), {O, N, H, D});
  return out.reshape(shape);
}

// ---------------------------------------------------------------- TriMul

int64_t a256(int64_t v) { return (v + 255) / 256 * 256; }

// The forward's state in one allocation: z_ln, gate, a, b, x (bf16), LN_in's
// statistics (f32) and, for a backward, xln (bf16) and LN_out's (f32).
struct TrimulState {
  char* p[10] = {};
  int64_t bytes;
  TrimulState(int64_t B, int64_t N, int64_t C, bool save, char* base) {
    const int64_t rows = a256(B * N * N * C * 2);
    const int64_t planes = a256(B * C * N * tpf_trimul_plane_pitch(N) * 2);
    const int64_t stat = a256(B * N * N * 4);
    const int64_t sizes[10] = {rows, rows, planes, planes, planes, stat, stat, rows, stat, stat};
    bytes = 0;
    for (int i = 0; i < (save ? 10 : 7); ++i) {
      p[i] = base + bytes;
      bytes += sizes[i];
    }
  }
};

// params: p_in [2C, C], g_in [2C, C], g_out [C, C], p_out [C, C], then the
// weight and bias of LN_in and LN_out.
Tensor trimul_forward(const Tensor& z, const Tensor& mask, const variable_list& w, bool outgoing,
                      const TrimulState& st) {
  const int64_t B = z.size(0), N = z.size(1), C = z.size(3), cc = C * C;
  Tensor out = at::empty({B, N, N, C}, like(z, at::kBFloat16));
  const int64_t ws_bytes = tpf_trimul_forward_workspace_bytes(C);
  Tensor ws = at::empty({ws_bytes}, like(z, at::kByte));
  auto f = [&](int i) { return (const float*)w[i].const_data_ptr(); };
  check(tpf_trimul_forward_bf16(
            z.const_data_ptr(), (const float*)mask.const_data_ptr(), f(0), f(1), f(0) + cc,
            f(1) + cc, f(2), f(3), f(4), f(5), f(6), f(7), outgoing ? 1 : 0, B, N, C,
            out.data_ptr(), st.p[0], st.p[1], st.p[2], st.p[3], st.p[4], st.p[7], (float*)st.p[5],
            (float*)st.p[6], (float*)st.p[8], (float*)st.p[9], ws.data_ptr(), ws_bytes, stream()),
        "tpf_trimul_forward_bf16");
  return out;
}

struct TrimulFn : torch::autograd::Function<TrimulFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& z, const Tensor& mask,
                        const Tensor& p_in, const Tensor& g_in, const Tensor& g_out,
                        const Tensor& p_out, const Tensor& n_in_w, const Tensor& n_in_b,
                        const Tensor& n_out_w, const Tensor& n_out_b, bool outgoing) {
    const int64_t B = z.size(0), N = z.size(1), C = z.size(3);
    Tensor state = at::empty({TrimulState(B, N, C, true, nullptr).bytes}, like(z, at::kByte));
    Tensor out = trimul_forward(z, mask, {p_in, g_in, g_out, p_out, n_in_w, n_in_b, n_out_w, n_out_b},
                                outgoing, TrimulState(B, N, C, true, (char*)state.data_ptr()));
    ctx->save_for_backward({z, mask, state, p_in, g_in, g_out, p_out, n_in_w, n_out_w});
    ctx->saved_data["outgoing"] = outgoing;
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const Tensor &z = s[0], &mask = s[1], &state = s[2];
    const int64_t B = z.size(0), N = z.size(1), C = z.size(3), cc = C * C;
    const TrimulState st(B, N, C, true, (char*)state.data_ptr());
    const Tensor g = kernel_grad(grads[0]);
    const auto f32 = like(z, at::kFloat);
    Tensor dz = at::empty({B, N, N, C}, like(z, at::kBFloat16));
    Tensor dp = at::empty({2 * C, C}, f32), dg = at::empty({2 * C, C}, f32);
    Tensor dgo = at::empty({C, C}, f32), dpo = at::empty({C, C}, f32);
    Tensor dn[4];
    for (Tensor& t : dn) t = at::empty({C}, f32);
    const int64_t ws_bytes = tpf_trimul_backward_workspace_bytes(B, N, C);
    Tensor ws = at::empty({ws_bytes}, like(z, at::kByte));
    auto f = [&](int i) { return (const float*)s[i].const_data_ptr(); };
    auto o = [](const Tensor& t) { return (float*)t.data_ptr(); };
    check(tpf_trimul_backward_named_bf16(
              g.const_data_ptr(), z.const_data_ptr(), (const float*)mask.const_data_ptr(), f(3),
              f(4), f(3) + cc, f(4) + cc, f(5), f(6), f(7), f(8), st.p[0], st.p[1], st.p[2],
              st.p[3], st.p[4], st.p[7], (const float*)st.p[5], (const float*)st.p[6],
              (const float*)st.p[8], (const float*)st.p[9],
              ctx->saved_data["outgoing"].toBool() ? 1 : 0, B, N, C, dz.data_ptr(), o(dp), o(dg),
              o(dgo), o(dpo), o(dn[0]), o(dn[1]), o(dn[2]), o(dn[3]), ws.data_ptr(), ws_bytes,
              stream()),
          "tpf_trimul_backward_named_bf16");
    return {dz, Tensor(), dp, dg, dgo, dpo, dn[0], dn[1], dn[2], dn[3], Tensor()};
  }
};

std::optional<Tensor> trimul(const Tensor& z, const std::optional<Tensor>& mask_in,
                             const variable_list& w, bool outgoing) {
  if (transforms_active() || !z.is_cuda()) return std::nullopt;
  const c10::DeviceIndex dev = c10::hip::current_device();
  if (!plain(z, dev) || z.dim() < 3 || z.scalar_type() != at::kBFloat16 || z.numel() == 0 ||
      !z.is_contiguous() || !aligned16(z))
    return std::nullopt;
  const int64_t C = z.size(-1), N = z.size(-2);
  if (z.size(-3) != N) return std::nullopt;
  const int64_t B = z.numel() / (N * N * C);
  if (!tpf_trimul_shape_supported(B, N, C, 0)) return std::nullopt;
  for (size_t i = 0; i < w.size(); ++i) {
    const Tensor& t = w[i];
    if (!plain(t, dev) || t.scalar_type() != at::kFloat || !t.is_contiguous() || !aligned16(t))
      return std::nullopt;
    if (i < 4 ? (t.dim() != 2 || t.size(0) != (i < 2 ? 2 * C : C) || t.size(1) != C)
              : (t.dim() != 1 || t.size(0) != C))
      return std::nullopt;
  }
  Tensor mask;
  if (!mask_in.has_value()) {
    mask = at::ones({B, N, N}, like(z, at::kFloat));
  } else {
    mask = *mask_in;
    if (!plain(mask, dev) || mask.sizes() != z.sizes().slice(0, z.dim() - 1) ||
        !mask.is_contiguous() || mask.requires_grad())
      return std::nullopt;
    if (mask.scalar_type() != at::kFloat) mask = mask.to(at::kFloat);
  }
  bool grad = z.requires_grad();
  for (const Tensor& t : w) grad = grad || t.requires_grad();
  grad = grad && at::GradMode::is_enabled();
  if (grad && !tpf_trimul_shape_supported(B, N, C, 1)) return std::nullopt;
  const Tensor z4 = z.dim() == 4 ? z : z.view({B, N, N, C});
  Tensor out;
  if (grad) {
    out = TrimulFn::apply(z4, mask, w[0], w[1], w[2], w[3], w[4], w[5], w[6], w[7], outgoing);
  } else {
    Tensor scratch = at::empty({TrimulState(B, N, C, false, nullptr).bytes}, like(z, at::kByte));
    out = trimul_forward(z4, mask, w, outgoing, TrimulState(B, N, C, false, (char*)scratch.data_ptr()));
  }
  return z.dim() == 4 ? out : out.view(z.sizes());
}

}  // namespace

// Refuses the import beside another torch or C-ABI library than it was built
// with: both are called through their headers of that time.
void check_versions() {
  const auto torch = pybind11::module_::import("torch").attr("__version__").cast<std::string>();
  const std::string built = TORCH_VERSION;
  if (torch.compare(0, built.size(), built) != 0 ||
      (torch.size() > built.size() && std::isdigit((unsigned char)torch[built.size()])))
    throw pybind11::import_error("built for torch " + built + ", found " + torch);
  if (tpf_abi_version() != TPF_ABI_VERSION)
    throw pybind11::import_error("built for library ABI " + std::to_string(TPF_ABI_VERSION) +
                                 ", found " + std::to_string(tpf_abi_version()));
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  check_versions();
  m.def("attention", [](const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& res_mask,
                        const Tensor& pair_bias) {
    const std::string backward = env_flag("TURBOPAIRFORMER_SR_BACKWARD", "OPENFOLD3_SR_BACKWARD");
    const std::string shadow = env_flag("TURBOPAIRFORMER_SR_SHADOW", "OPENFOLD3_SR_SHADOW");
    pybind11::gil_scoped_release nogil;
    return attention(q, k, v, res_mask, pair_bias, backward, shadow);
  });
  m.def("trimul", &trimul, pybind11::call_guard<pybind11::gil_scoped_release>());
  m.def("set_workspace_budget", [](int64_t bytes) { g_budget.store(bytes); });
}
