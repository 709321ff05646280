// Allocation and launch of one operator pass per call, for the Python layer:
// each function allocates outputs and workspace with torch's allocator, takes
// the current stream of the operands' device and calls one entry point of
// libvafa.so (include/vafa.h).  Autograd, argument checks and the plan cache
// stay in Python.  With tensor factories, ctypes conversions and stream lookups
// there too, host time held every small call: us a call with cu_seqlens seen before
// (the plan cached), before -> now, 4 short sequences forward 31 -> 17 (host
// cu_seqlens), forward + backward 150 -> 93; 16 absorb samples forward 34 -> 25,
// forward + backward 220 -> 171.  With new lengths in every call planning adds 15 to
// 50 us: 4 sequences 73 -> 62, 16 absorb samples 84 -> 85.
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <dlfcn.h>
#include <torch/extension.h>

#include <initializer_list>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/vafa.h"

namespace {

using at::Tensor;

// Entry points of the library the Python layer loaded.
struct Api {
#define VAFA_FN(name) decltype(&::vafa_##name) name = nullptr;
#define VAFA_FNS(X)                                                                       \
  X(last_error) X(varlen_fwd_workspace) X(varlen_fwd) X(varlen_bwd_workspace)             \
  X(varlen_bwd) X(absorb_fwd_workspace) X(absorb_fwd) X(absorb_bwd_workspace)             \
  X(absorb_bwd) X(absorb_fwd_full_workspace) X(absorb_fwd_full) X(absorb_bwd_full)        \
  X(absorb_bwd_full_workspace)                                                            \
  X(absorb_project_workspace) X(absorb_project_fwd) X(absorb_project_bwd)                 \
  X(absorb_project_f32_workspace) X(absorb_project_f32_fwd) X(absorb_project_f32_bwd)
  VAFA_FNS(VAFA_FN)
#undef VAFA_FN
} api;

void bind_library(const std::string &path) {
  void *h = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
  TORCH_CHECK(h != nullptr, "cannot load ", path, ": ", dlerror());
#define VAFA_SYM(name)                                                                    \
  api.name = reinterpret_cast<decltype(api.name)>(dlsym(h, "vafa_" #name));               \
  TORCH_CHECK(api.name != nullptr, path, " lacks vafa_" #name);
  VAFA_FNS(VAFA_SYM)
#undef VAFA_SYM
}

struct AssertionFailed : std::runtime_error {
  using std::runtime_error::runtime_error;
};

void check(int rc) {
  if (rc == VAFA_OK) return;
  const std::string msg = api.last_error();
  if (rc == VAFA_ERR_VALUE) throw py::value_error(msg);
  if (rc == VAFA_ERR_ASSERT) throw AssertionFailed(msg);
  throw std::runtime_error("vafa error " + std::to_string(rc) + ": " + msg);
}

// A device plan: its items and info struct.
struct Plan {
  Tensor items;
  vafa_plan_info info;
  Plan(Tensor t, const std::string &bytes) : items(std::move(t)) {
    TORCH_CHECK(bytes.size() == sizeof(info), "plan info of ", bytes.size(), " bytes");
    std::memcpy(&info, bytes.data(), sizeof(info));
  }
  const int32_t *dev() const { return items.data_ptr<int32_t>(); }
};

int32_t dtype_of(const Tensor &t) {
  switch (t.scalar_type()) {
    case at::kFloat: return VAFA_F32;
    case at::kHalf: return VAFA_F16;
    case at::kBFloat16: return VAFA_BF16;
    default: throw AssertionFailed("dtype not supported (float32, float16, bfloat16)");
  }
}

// One call's device, stream and workspace.
struct Call {
  c10::DeviceGuard guard;
  at::TensorOptions opt;
  void *stream;
  Tensor ws;
  explicit Call(const Tensor &t)
      : guard(t.device()), opt(t.options()),
        stream(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream()) {}
  Tensor empty(at::IntArrayRef shape) const { return at::empty(shape, opt); }
  Tensor empty_f32(at::IntArrayRef shape) const { return at::empty(shape, opt.dtype(at::kFloat)); }
  Tensor like(const Tensor &t) const { return at::empty(t.sizes(), opt); }
  // a workspace of n bytes (none for 0); a negative size is the query's error
  void *workspace(int64_t n) {
    if (n < 0) check(VAFA_ERR_VALUE);
    if (n == 0) return nullptr;
    ws = at::empty({n}, opt.dtype(at::kByte));
    return ws.data_ptr();
  }
  int64_t ws_bytes() const { return ws.defined() ? ws.numel() : 0; }
};

void *ptr(const Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; }
const float *f32(const Tensor &t) { return static_cast<const float *>(ptr(t)); }
float *f32w(const Tensor &t) { return static_cast<float *>(ptr(t)); }

// An upstream gradient as the kernels read it: the operands' dtype,
// contiguous, 16-byte aligned.
Tensor grad_in(Tensor g, const Tensor &like) {
  g = g.contiguous();
  if (g.scalar_type() != like.scalar_type()) g = g.to(like.scalar_type());
  if (reinterpret_cast<uintptr_t>(g.data_ptr()) % 16 != 0) g = g.clone();
  return g;
}

std::tuple<Tensor, Tensor> varlen_fwd(const Tensor &q, const Tensor &k, const Tensor &v,
                                      const Plan &p, double scale) {
  Call c(q);
  const int64_t D = q.size(2);
  Tensor o = c.like(q), lse = c.empty_f32({q.size(0), q.size(1)});
  void *ws = c.workspace(api.varlen_fwd_workspace(&p.info, D));
  check(api.varlen_fwd(ptr(q), ptr(k), ptr(v), ptr(o), f32w(lse), p.dev(), &p.info, D, dtype_of(q),
                       (float)scale, ws, c.ws_bytes(), c.stream));
  return {o, lse};
}

std::tuple<Tensor, Tensor, Tensor> varlen_bwd(const Tensor &q, const Tensor &k, const Tensor &v,
                                              const Tensor &o, const Tensor &lse, const Tensor &g,
                                              const Plan &p, double scale) {
  Call c(q);
  const int64_t D = q.size(2);
  const Tensor dout = grad_in(g, q);
  Tensor dq = c.like(q), dk = c.like(k), dv = c.like(v);
  void *ws = c.workspace(api.varlen_bwd_workspace(&p.info, D));
  check(api.varlen_bwd(ptr(q), ptr(k), ptr(v), ptr(o), ptr(dout), f32(lse), ptr(dq), ptr(dk),
                       ptr(dv), p.dev(), &p.info, D, dtype_of(q), (float)scale, ws, c.ws_bytes(),
                       c.stream));
  return {dq, dk, dv};
}

std::tuple<Tensor, Tensor> absorb_fwd(const Tensor &u, const Tensor &X, const Tensor &W_V,
                                      const Plan &p, double scale) {
  Call c(u);
  const int64_t T_q = u.size(0), H = u.size(1), F = u.size(2), DH = W_V.size(2);
  Tensor O = c.empty({T_q, H, DH}), lse = c.empty_f32({T_q, H});
  void *ws = c.workspace(api.absorb_fwd_workspace(&p.info, F, DH));
  check(api.absorb_fwd(ptr(u), ptr(X), ptr(W_V), ptr(O), f32w(lse), p.dev(), &p.info, F, DH,
                       dtype_of(u), (float)scale, ws, c.ws_bytes(), c.stream));
  return {O, lse};
}

std::tuple<Tensor, Tensor, Tensor> absorb_bwd(const Tensor &u, const Tensor &X, const Tensor &W_V,
                                              const Tensor &O, const Tensor &lse, const Tensor &g,
                                              const Plan &p, double scale) {
  Call c(u);
  const int64_t F = u.size(2), DH = W_V.size(2);
  const Tensor dO = grad_in(g, u);
  Tensor du = c.like(u), dX = c.like(X), dW = c.like(W_V);
  void *ws = c.workspace(api.absorb_bwd_workspace(&p.info, F, DH));
  check(api.absorb_bwd(ptr(u), ptr(X), ptr(W_V), ptr(O), ptr(dO), f32(lse), ptr(du), ptr(dX),
                       ptr(dW), p.dev(), &p.info, F, DH, dtype_of(u), (float)scale, ws,
                       c.ws_bytes(), c.stream));
  return {du, dX, dW};
}

// The whole 16-bit forward: (q_proj, O, lse).
std::tuple<Tensor, Tensor, Tensor> absorb_full_fwd(const Tensor &q_raw, const Tensor &X,
                                                   const Tensor &W_Q, const Tensor &W_K,
                                                   const Tensor &W_V, const Plan &p,
                                                   double scale) {
  Call c(q_raw);
  const int64_t T_q = q_raw.size(0), DQ = q_raw.size(1), F = X.size(1), H = W_Q.size(1),
                DH = W_Q.size(2);
  Tensor q_proj = c.empty({T_q, H * DH}), O = c.empty({T_q, H, DH}), lse = c.empty_f32({T_q, H});
  void *ws = c.workspace(api.absorb_fwd_full_workspace(&p.info, DQ, F, DH));
  check(api.absorb_fwd_full(ptr(q_raw), ptr(X), ptr(W_Q), ptr(W_K), ptr(W_V), ptr(q_proj), ptr(O),
                            f32w(lse), T_q, p.dev(), &p.info, DQ, F, DH, dtype_of(q_raw),
                            (float)scale, ws, c.ws_bytes(), c.stream));
  return {q_proj, O, lse};
}

// Projections in 16 bits or fp32: (q_proj, u).
std::tuple<Tensor, Tensor> project_fwd(const Tensor &q_raw, const Tensor &W_Q, const Tensor &W_K) {
  Call c(q_raw);
  const int64_t T_q = q_raw.size(0), DQ = q_raw.size(1), H = W_Q.size(1), DH = W_Q.size(2),
                F = W_K.size(0);
  Tensor q_proj = c.empty({T_q, H * DH}), u = c.empty({T_q, H, F});
  if (q_raw.scalar_type() == at::kFloat) {
    check(api.absorb_project_f32_fwd(f32(q_raw), f32(W_Q), f32(W_K), f32w(q_proj), f32w(u), T_q, H,
                                     DQ, F, DH, c.stream));
  } else {
    void *ws = c.workspace(api.absorb_project_workspace(T_q, H, DQ, F, DH, 0));
    check(api.absorb_project_fwd(ptr(q_raw), ptr(W_Q), ptr(W_K), ptr(q_proj), ptr(u), T_q, H, DQ,
                                 F, DH, dtype_of(q_raw), ws, c.ws_bytes(), c.stream));
  }
  return {q_proj, u};
}

// (dq_raw, dW_Q, dW_K), None where not asked for.
using Grads3 = std::tuple<std::optional<Tensor>, std::optional<Tensor>, std::optional<Tensor>>;
Grads3 project_bwd(const Tensor &q_raw, const Tensor &W_Q, const Tensor &W_K, const Tensor &q_proj,
                   const Tensor &g, bool need_q, bool need_wq, bool need_wk) {
  Call c(q_raw);
  const int64_t T_q = q_raw.size(0), DQ = q_raw.size(1), H = W_Q.size(1), DH = W_Q.size(2),
                F = W_K.size(0);
  const Tensor du = grad_in(g, q_raw);
  Tensor dq, dwq, dwk;
  if (need_q) dq = c.like(q_raw);
  if (need_wq) dwq = c.like(W_Q);
  if (need_wk) dwk = c.like(W_K);
  if (q_raw.scalar_type() == at::kFloat) {
    void *ws = c.workspace(api.absorb_project_f32_workspace(T_q, H, DQ, F, DH));
    check(api.absorb_project_f32_bwd(f32(q_raw), f32(W_Q), f32(W_K), f32(q_proj), f32(du),
                                     f32w(dq), f32w(dwq), f32w(dwk), T_q, H, DQ, F, DH, ws,
                                     c.ws_bytes(), c.stream));
  } else {
    void *ws = c.workspace(api.absorb_project_workspace(T_q, H, DQ, F, DH, 1));
    check(api.absorb_project_bwd(ptr(q_raw), ptr(W_Q), ptr(W_K), ptr(q_proj), ptr(du), ptr(dq),
                                 ptr(dwq), ptr(dwk), T_q, H, DQ, F, DH, dtype_of(q_raw), ws,
                                 c.ws_bytes(), c.stream));
  }
  auto opt = [](const Tensor &t) { return t.defined() ? std::optional<Tensor>(t) : std::nullopt; };
  return {opt(dq), opt(dwq), opt(dwk)};
}

// Backward of the whole 16-bit op: (dq_raw, dX, dW_Q, dW_K, dW_V).
std::tuple<std::optional<Tensor>, Tensor, std::optional<Tensor>, std::optional<Tensor>, Tensor>
absorb_full_bwd(const Tensor &q_raw, const Tensor &W_Q, const Tensor &W_K, const Tensor &q_proj,
                const Tensor &X, const Tensor &W_V, const Tensor &O, const Tensor &lse,
                const Tensor &g, const Plan &p, double scale, bool need_q, bool need_wq,
                bool need_wk) {
  Call c(q_raw);
  const int64_t T_q = q_raw.size(0), DQ = q_raw.size(1), F = X.size(1), DH = W_Q.size(2);
  const Tensor dO = grad_in(g, q_raw);
  Tensor dX = c.like(X), dW_V = c.like(W_V), dq, dwq, dwk;
  if (need_q) dq = c.like(q_raw);
  if (need_wq) dwq = c.like(W_Q);
  if (need_wk) dwk = c.like(W_K);
  void *ws = c.workspace(api.absorb_bwd_full_workspace(&p.info, T_q, DQ, F, DH));
  check(api.absorb_bwd_full(ptr(q_raw), ptr(X), ptr(W_Q), ptr(W_K), ptr(W_V), ptr(q_proj), ptr(O),
                            ptr(dO), f32(lse), ptr(dq), ptr(dX), ptr(dwq), ptr(dwk), ptr(dW_V),
                            T_q, p.dev(), &p.info, DQ, F, DH, dtype_of(q_raw), (float)scale, ws,
                            c.ws_bytes(), c.stream));
  auto opt = [](const Tensor &t) { return t.defined() ? std::optional<Tensor>(t) : std::nullopt; };
  return {opt(dq), dX, opt(dwq), opt(dwk), dW_V};
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  py::register_exception_translator([](std::exception_ptr e) {
    try {
      if (e) std::rethrow_exception(e);
    } catch (const AssertionFailed &x) {
      PyErr_SetString(PyExc_AssertionError, x.what());
    }
  });
  py::class_<Plan>(m, "Plan").def(py::init([](Tensor items, const py::bytes &info) {
    return Plan(std::move(items), std::string(info));
  }));
  // allocation and launch may wait (a full queue, an allocator retry): other
  // Python threads run meanwhile, as they do under a ctypes call
  py::call_guard<py::gil_scoped_release> no_gil;
  m.def("bind", &bind_library);
  m.def("varlen_fwd", &varlen_fwd, no_gil);
  m.def("varlen_bwd", &varlen_bwd, no_gil);
  m.def("absorb_fwd", &absorb_fwd, no_gil);
  m.def("absorb_bwd", &absorb_bwd, no_gil);
  m.def("absorb_full_fwd", &absorb_full_fwd, no_gil);
  m.def("absorb_full_bwd", &absorb_full_bwd, no_gil);
  m.def("project_fwd", &project_fwd, no_gil);
  m.def("project_bwd", &project_bwd, no_gil);
}
