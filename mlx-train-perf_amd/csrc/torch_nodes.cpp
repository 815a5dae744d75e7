// The autograd nodes of flash_attention and linear_cross_entropy on plain tensors: the forward and backward of
// attention/api.py's _KernelAttention and core/loss.py's _KernelLCE, planned and launched from C++.
// Autograd runs a backward on a thread of its own; a Python node there holds the interpreter lock for the
// whole of it and pulls the interpreter's state to that thread's core, and the next forward pulls it back.
// A node here takes the lock for a moment: once to count the backward, and in a loss also for the workspace
// budget and the cached transposed head. A pass of an attention layer (B = 4, S = 509, 16/8 heads, head_dim 64)
// takes 75 or 122 us with the Python node, 45 or 78 with this one, by where the thread lands; of a small mean
// loss (N = 128, D = 256, V = 3000) 165 us, and 65 or 110. The entry points of the C-ABI library come from the
// Python layer (bind), so both use the one it loaded.
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>

#include <string>

#include "../../include/mtp_hip.h"

namespace {

struct Entries {
  decltype(&mtp_attn_fwd) fwd = nullptr;
  decltype(&mtp_attn_bwd) bwd = nullptr;
  decltype(&mtp_attn_bwd_workspace_bytes) ws = nullptr;
  decltype(&mtp_attn_fwd_f32) fwd32 = nullptr;
  decltype(&mtp_attn_bwd_f32) bwd32 = nullptr;
  decltype(&mtp_attn_bwd_f32_workspace_bytes) ws32 = nullptr;
  decltype(&mtp_lce_fwd) lce_fwd = nullptr;
  decltype(&mtp_lce_fwd_workspace_bytes) lce_fwd_ws = nullptr;
  decltype(&mtp_lce_bwd) lce_bwd = nullptr;
  decltype(&mtp_lce_bwd_workspace_bytes) lce_bwd_ws = nullptr;
  decltype(&mtp_lce_bwd_stage_chunk) lce_stage_chunk = nullptr;
  decltype(&mtp_lce_bwd_row_block) lce_row_block = nullptr;
  decltype(&mtp_lce_bwd_chunk) lce_chunk = nullptr;
  decltype(&mtp_lce_fwd_f32) lce_fwd32 = nullptr;
  decltype(&mtp_lce_fwd_f32_workspace_bytes) lce_fwd_ws32 = nullptr;
  decltype(&mtp_lce_bwd_f32) lce_bwd32 = nullptr;
  decltype(&mtp_lce_bwd_f32_workspace_bytes) lce_bwd_ws32 = nullptr;
  decltype(&mtp_lce_bwd_f32_chunk) lce_chunk32 = nullptr;
  decltype(&mtp_lce_mean) lce_mean = nullptr;
  decltype(&mtp_lce_mean_bwd) lce_mean_bwd = nullptr;
};
Entries g_api;
// Python: the typed error of a return code (_native.check), the call counters of the attention and the
// loss (VJP_CALLS), the loss layer's cache of transposed heads (_transposed_head) and its workspace budget
// (plan.launch.lce_bwd_budget_bytes), os.environ.get. Held until the process ends.
PyObject* g_check = nullptr;
PyObject* g_attn_calls = nullptr;
PyObject* g_lce_calls = nullptr;
PyObject* g_transposed_head = nullptr;
PyObject* g_budget = nullptr;
PyObject* g_env = nullptr;

void* stream_of(const at::Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// f(), a call of Python code with the lock held; its exception keeps its type, also out of the autograd
// thread.
template <class F>
auto python(F&& f) {
  py::gil_scoped_acquire gil;
  try {
    return f();
  } catch (py::error_already_set& e) {
    e.restore();
  }
  python_error err;
  err.persist();
  throw std::move(err);
}

void check(int rc, const char* domain = "attention") {
  if (rc == MTP_OK) return;
  python([&] {
    const py::handle raise(g_check);
    raise(rc, py::arg("domain") = domain);
    return 0;
  });
}

void count_backward(PyObject* counters, std::initializer_list<const char*> names) {
  python([&] {
    auto calls = py::reinterpret_borrow<py::dict>(counters);
    for (const char* name : names) calls[name] = py::int_(calls.contains(name) ? calls[name].cast<long>() + 1 : 1L);
    return 0;
  });
}

const int32_t* ints(const at::Tensor& t) { return t.defined() ? t.const_data_ptr<int32_t>() : nullptr; }
template <class T = void>
T* ptr(const at::Tensor& t) { return static_cast<T*>(t.data_ptr()); }
template <class T = void>
T* opt_ptr(const at::Tensor& t) { return t.defined() ? ptr<T>(t) : nullptr; }
py::object opt_object(const at::Tensor& t) { return t.defined() ? py::cast(t) : py::none(); }

// Not inputs of the node: they have no gradients, and may be missing.
struct Segments {
  at::Tensor id, start;
};

struct KernelAttention : torch::autograd::Function<KernelAttention> {
  static at::Tensor forward(torch::autograd::AutogradContext* ctx, const at::Tensor& q, const at::Tensor& k,
                            const at::Tensor& v, const Segments& seg, double scale, bool causal) {
    const c10::DeviceGuard device(q.device());
    const int64_t b = q.size(0), hq = q.size(1), s = q.size(2), dh = q.size(3), hkv = k.size(1);
    const at::Tensor o = at::empty_like(q), lse = at::empty({b, hq, s}, q.options().dtype(at::kFloat));
    if (q.scalar_type() == at::kFloat)
      check(g_api.fwd32(ptr<float>(q), ptr<float>(k), ptr<float>(v), b, hq, hkv, s, dh, (float)scale, causal, ints(seg.id),
                        ints(seg.start), ptr<float>(o), ptr<float>(lse), stream_of(q)));
    else
      check(g_api.fwd(ptr(q), ptr(k), ptr(v), b, hq, hkv, s, dh, (float)scale, causal, ints(seg.id), ints(seg.start), ptr(o),
                      ptr<float>(lse), stream_of(q)));
    ctx->save_for_backward({q, k, v, o, lse, seg.id, seg.start});
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["causal"] = causal;
    ctx->set_materialize_grads(false);
    return o;
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    count_backward(g_attn_calls, {"flash_attention", "flash_attention_kernel_bwd"});
    const auto saved = ctx->get_saved_variables();
    const at::Tensor &q = saved[0], &k = saved[1], &v = saved[2], &o = saved[3], &lse = saved[4];
    const at::Tensor &seg_id = saved[5], &seg_start = saved[6];
    const float scale = (float)ctx->saved_data["scale"].toDouble();
    const bool causal = ctx->saved_data["causal"].toBool();
    const c10::DeviceGuard device(q.device());
    const at::Tensor d_o = grads[0].defined() ? grads[0].contiguous() : at::zeros_like(o);
    const int64_t b = q.size(0), hq = q.size(1), s = q.size(2), dh = q.size(3), hkv = k.size(1);
    const bool f32 = q.scalar_type() == at::kFloat;
    const at::Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
    const size_t bytes = (f32 ? g_api.ws32 : g_api.ws)(b, hq, hkv, s, dh);
    const at::Tensor ws = at::empty({(int64_t)bytes}, q.options().dtype(at::kByte));
    if (f32)
      check(g_api.bwd32(ptr<float>(q), ptr<float>(k), ptr<float>(v), ptr<float>(o), ptr<float>(lse), ptr<float>(d_o), b, hq,
                        hkv, s, dh, scale, causal, ints(seg_id), ints(seg_start), ptr<float>(dq), ptr<float>(dk),
                        ptr<float>(dv), ptr(ws), bytes, stream_of(q)));
    else
      check(g_api.bwd(ptr(q), ptr(k), ptr(v), ptr(o), ptr<float>(lse), ptr(d_o), b, hq, hkv, s, dh, scale, causal,
                      ints(seg_id), ints(seg_start), ptr(dq), ptr(dk), ptr(dv), ptr(ws), bytes, stream_of(q)));
    return {dq, dk, dv, at::Tensor(), at::Tensor(), at::Tensor()};
  }
};

// A call of the loss. Its inputs are those of _KernelLCE that may ask for a gradient (also where they get none,
// as a frozen weight does): hidden, w, scales, biases and the head's own weight, owner.
struct LossCall {
  at::Tensor targets, w, w_q, scales, biases, owner;
  int64_t head_kind, fwd_kind, fwd_ws_bytes, ignore_index, bwd_chunk;
  bool mean;
};

// A switch of the environment as Python sees it (C's getenv may not run beside another thread's setenv).
bool env_is(const char* name, const char* value) {
  return python([&] {
    const py::handle get(g_env);
    const py::object x = get(name);
    return !x.is_none() && x.cast<std::string>() == value;
  });
}

size_t budget_bytes() {
  return python([] {
    const py::handle f(g_budget);
    return f().cast<size_t>();
  });
}

struct KernelLoss : torch::autograd::Function<KernelLoss> {
  static at::Tensor forward(torch::autograd::AutogradContext* ctx, const at::Tensor& hidden,
                            const std::optional<at::Tensor>& w, const std::optional<at::Tensor>& /*scales*/,
                            const std::optional<at::Tensor>& /*biases*/, const at::Tensor& /*owner*/, const LossCall& c) {
    const c10::DeviceGuard device(hidden.device());
    const int64_t n = hidden.size(0), d = hidden.size(1), v = c.head_kind == MTP_HEAD_DENSE ? c.w.size(0) : c.w_q.size(0);
    const bool f32 = hidden.scalar_type() == at::kFloat;
    const auto opt = hidden.options().dtype(at::kFloat);
    at::Tensor nll = at::empty({n}, opt), count;
    const at::Tensor lse = at::empty({n}, opt), tgt = at::empty({n}, opt);
    const size_t bytes = c.fwd_ws_bytes > 0 ? (size_t)c.fwd_ws_bytes
                         : f32              ? g_api.lce_fwd_ws32(n, d, v, c.head_kind)
                                            : g_api.lce_fwd_ws(n, d, v, c.head_kind);
    const at::Tensor ws = at::empty({(int64_t)std::max<size_t>(bytes, 16)}, hidden.options().dtype(at::kByte));
    const auto* t = ptr<int64_t>(c.targets);
    if (f32)
      check(g_api.lce_fwd32(ptr<float>(hidden), opt_ptr<float>(c.w), opt_ptr<uint32_t>(c.w_q), opt_ptr<float>(c.scales),
                            opt_ptr<float>(c.biases), t, n, d, v, c.fwd_kind, c.ignore_index, ptr<float>(nll),
                            ptr<float>(lse), ptr<float>(tgt), ptr(ws), bytes, stream_of(hidden)),
            "loss");
    else
      check(g_api.lce_fwd(ptr(hidden), opt_ptr(c.w), opt_ptr<uint32_t>(c.w_q), opt_ptr(c.scales), opt_ptr(c.biases), t, n, d,
                          v, c.fwd_kind, c.ignore_index, ptr<float>(nll), ptr<float>(lse), ptr<float>(tgt), ptr(ws), bytes,
                          stream_of(hidden)),
            "loss");
    at::Tensor out = nll;
    if (c.mean) {
      out = at::empty({}, opt);
      count = at::empty({}, opt);
      check(g_api.lce_mean(ptr<float>(nll), t, n, c.ignore_index, ptr<float>(out), ptr<float>(count), stream_of(hidden)),
            "loss");
    }
    ctx->save_for_backward({hidden, c.targets, lse, count});
    // The head is kept as it is, not as a saved tensor: its packed words never change, and a dense
    // weight is read again by the backward whatever its version.
    auto& sd = ctx->saved_data;
    if (c.w.defined()) sd["w"] = c.w;
    if (c.w_q.defined()) {
      sd["w_q"] = c.w_q;
      sd["scales"] = c.scales;
      sd["biases"] = c.biases;
    }
    sd["owner"] = c.owner;
    sd["head_kind"] = c.head_kind;
    sd["ignore_index"] = c.ignore_index;
    sd["bwd_chunk"] = c.bwd_chunk;
    sd["d_w"] = w.has_value() && w->requires_grad();
    ctx->set_materialize_grads(false);
    return out;
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    count_backward(g_lce_calls, {"kernel"});
    const auto saved = ctx->get_saved_variables();
    const at::Tensor &hidden = saved[0], &targets = saved[1], &lse = saved[2], &count = saved[3];
    auto& sd = ctx->saved_data;
    auto tensor = [&](const char* name) { return sd.count(name) ? sd[name].toTensor() : at::Tensor(); };
    const at::Tensor w = tensor("w"), w_q = tensor("w_q"), scales = tensor("scales"), biases = tensor("biases");
    int64_t kind = sd["head_kind"].toInt();
    const int64_t ignore_index = sd["ignore_index"].toInt(), bwd_chunk = sd["bwd_chunk"].toInt();
    const c10::DeviceGuard device(hidden.device());
    const int64_t n = hidden.size(0), d = hidden.size(1), v = kind == MTP_HEAD_DENSE ? w.size(0) : w_q.size(0);
    at::Tensor d_nll;
    if (!grads[0].defined()) {
      d_nll = at::zeros_like(lse);
    } else if (count.defined()) {  // the gradient of the mean
      const at::Tensor d_mean = grads[0].to(at::kFloat);
      d_nll = at::empty_like(lse);
      check(g_api.lce_mean_bwd(ptr<float>(d_mean), ptr<float>(count), n, ptr<float>(d_nll), stream_of(hidden)), "loss");
    } else {
      d_nll = grads[0].to(at::kFloat).contiguous();
    }
    const bool want_dw = sd["d_w"].toBool();
    const at::Tensor d_w = want_dw ? at::empty_like(w) : at::Tensor(), d_hidden = at::empty_like(hidden);
    auto workspace = [&](size_t bytes) { return at::empty({(int64_t)bytes}, hidden.options().dtype(at::kByte)); };
    const auto* t = ptr<int64_t>(targets);
    if (hidden.scalar_type() == at::kFloat) {
      const int64_t vpad = (v + 127) / 128 * 128;
      const int64_t chunk = bwd_chunk ? std::min(std::max<int64_t>(128, (bwd_chunk + 127) / 128 * 128), vpad)
                                      : g_api.lce_chunk32(n, d, v, budget_bytes());
      const size_t bytes = g_api.lce_bwd_ws32(n, d, v, chunk);
      const at::Tensor ws = workspace(bytes);
      check(g_api.lce_bwd32(ptr<float>(hidden), opt_ptr<float>(w), opt_ptr<uint32_t>(w_q), opt_ptr<float>(scales),
                            opt_ptr<float>(biases), t, n, d, v, kind, ignore_index, ptr<float>(lse), ptr<float>(d_nll),
                            ptr<float>(d_hidden), opt_ptr<float>(d_w), chunk, ptr(ws), bytes, stream_of(hidden)),
            "loss");
      return {d_hidden, d_w, {}, {}, {}, {}};
    }
    // The head and workspace plan of _KernelLCE.backward; the cached transposed copies are the Python
    // layer's.
    at::Tensor w_t;
    if (!want_dw || env_is("MTP_LCE_TRANSPOSED_HEAD", "1"))
      w_t = python([&] {
        const py::handle f(g_transposed_head);
        const py::object r = f(tensor("owner"), opt_object(w), opt_object(w_q), opt_object(scales), opt_object(biases), kind, v, d);
        return r.is_none() ? at::Tensor() : r.cast<at::Tensor>();
      });
    const bool staged = !w_t.defined() && d % 64 == 0 && !env_is("MTP_LCE_STAGE_HEAD", "0");
    if (staged) kind = kind == MTP_HEAD_Q4 ? MTP_HEAD_Q4_STAGED : MTP_HEAD_DENSE_STAGED;
    const int64_t vpad = (v + 255) / 256 * 256;
    int64_t chunk, rows = n;
    if (bwd_chunk) {
      chunk = std::min(std::max<int64_t>(256, (bwd_chunk + 255) / 256 * 256), vpad);
    } else if (staged) {
      chunk = g_api.lce_stage_chunk(n, d, v, kind, budget_bytes());
    } else {
      const size_t budget = budget_bytes();
      if (!want_dw) rows = g_api.lce_row_block(n, d, v, budget);
      chunk = rows < n ? vpad : g_api.lce_chunk(n, d, v, budget);
    }
    const size_t bytes = g_api.lce_bwd_ws(n, d, v, kind, chunk, rows);
    const at::Tensor ws = workspace(bytes);
    check(g_api.lce_bwd(ptr(hidden), opt_ptr(w), opt_ptr(w_t), opt_ptr<uint32_t>(w_q), opt_ptr(scales), opt_ptr(biases), t, n, d,
                        v, kind, ignore_index, ptr<float>(lse), ptr<float>(d_nll), ptr(d_hidden), opt_ptr(d_w), chunk, rows,
                        ptr(ws), bytes, stream_of(hidden)),
          "loss");
    return {d_hidden, d_w, {}, {}, {}, {}};
  }
};

// The node's result for a Python caller: typed errors as they are.
template <class F>
at::Tensor apply_node(F&& f) {
  try {
    py::gil_scoped_release no_gil;
    return f();
  } catch (python_error& e) {
    e.restore();
    throw py::error_already_set();
  }
}

at::Tensor loss(const at::Tensor& hidden, const at::Tensor& targets, const std::optional<at::Tensor>& w,
                const std::optional<at::Tensor>& w_q, const std::optional<at::Tensor>& scales,
                const std::optional<at::Tensor>& biases, int64_t head_kind, int64_t ignore_index, int64_t bwd_chunk,
                const at::Tensor& owner, bool mean, int64_t fwd_kind, int64_t fwd_ws_bytes) {
  const at::Tensor none;
  const LossCall call{targets, w.value_or(none), w_q.value_or(none), scales.value_or(none), biases.value_or(none), owner,
                      head_kind, fwd_kind, fwd_ws_bytes, ignore_index, bwd_chunk, mean};
  return apply_node([&] {
    return KernelLoss::apply(hidden, w, scales, biases, owner, call);
  });
}

at::Tensor attention(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const std::optional<at::Tensor>& seg_id,
                     const std::optional<at::Tensor>& seg_start, double scale, bool causal) {
  return apply_node([&] {
    return KernelAttention::apply(q, k, v, Segments{seg_id.value_or(at::Tensor()), seg_start.value_or(at::Tensor())}, scale,
                                  causal);
  });
}

void bind(const py::dict& entries, py::object check_fn) {
  auto set = [&](auto& f, const char* name) {
    f = reinterpret_cast<std::remove_reference_t<decltype(f)>>(entries[name].cast<uintptr_t>());
  };
  set(g_api.fwd, "mtp_attn_fwd");
  set(g_api.bwd, "mtp_attn_bwd");
  set(g_api.ws, "mtp_attn_bwd_workspace_bytes");
  set(g_api.fwd32, "mtp_attn_fwd_f32");
  set(g_api.bwd32, "mtp_attn_bwd_f32");
  set(g_api.ws32, "mtp_attn_bwd_f32_workspace_bytes");
  set(g_api.lce_fwd, "mtp_lce_fwd");
  set(g_api.lce_fwd_ws, "mtp_lce_fwd_workspace_bytes");
  set(g_api.lce_bwd, "mtp_lce_bwd");
  set(g_api.lce_bwd_ws, "mtp_lce_bwd_workspace_bytes");
  set(g_api.lce_stage_chunk, "mtp_lce_bwd_stage_chunk");
  set(g_api.lce_row_block, "mtp_lce_bwd_row_block");
  set(g_api.lce_chunk, "mtp_lce_bwd_chunk");
  set(g_api.lce_fwd32, "mtp_lce_fwd_f32");
  set(g_api.lce_fwd_ws32, "mtp_lce_fwd_f32_workspace_bytes");
  set(g_api.lce_bwd32, "mtp_lce_bwd_f32");
  set(g_api.lce_bwd_ws32, "mtp_lce_bwd_f32_workspace_bytes");
  set(g_api.lce_chunk32, "mtp_lce_bwd_f32_chunk");
  set(g_api.lce_mean, "mtp_lce_mean");
  set(g_api.lce_mean_bwd, "mtp_lce_mean_bwd");
  g_check = check_fn.release().ptr();
}
void bind_attention(py::object calls) { g_attn_calls = calls.release().ptr(); }
void bind_loss(py::object calls, py::object transposed_head, py::object budget, py::object env) {
  g_lce_calls = calls.release().ptr();
  g_transposed_head = transposed_head.release().ptr();
  g_budget = budget.release().ptr();
  g_env = env.release().ptr();
}

}  // namespace

PYBIND11_MODULE(_mtp_torch, m) {
  m.def("bind", &bind);
  m.def("bind_attention", &bind_attention);
  m.def("bind_loss", &bind_loss);
  m.def("loss", &loss);
  m.def("attention", &attention);
}
