// The host path of the operators over torch tensors: argument checks, output allocation and the call of the C ABI
// (include/lancet_hip.h), in one native call per operator; and the gradient rules of the MoE operators
// (src/op/grad/moe.cc:30-93) as native autograd nodes, so that a backward pass neither takes the interpreter's lock nor
// changes threads for it.
//
// A small call costs what its host path costs.  A launch takes the host 2.4 us; around its launches an encode + decode of 64
// tokens spent 16 us in Python (torch.empty 1.5 us for each output, checks, conversion of twenty arguments), and a training
// step of 10007 ragged tokens 140 of its 185 us in a backward pass of interpreted functions, which the engine's thread runs
// under the interpreter's lock.  Time per pass, Python path / this one, us: encode + decode of 64 tokens 29.5 / 17.5 (then
// bound by its four kernels), 4096 x 768 fp32 top-1 26.4 / 19.4, training step of 10007 x 1003 bf16 top-2 188 / 104 and of
// 16384 x 1024 fp32 184 / 147, partitions of 512 short rows: chain 96 / 48, pipelined layer 410 / 209; a LANS step over 674
// tensors occupied the host for 951 us, now for 40.
//
// A wrong argument is a ValueError or TypeError before anything is launched, a failed launch a capi.LancetError.  Nothing is
// kept between calls but the three Python objects that bind() is given.  The interpreter's lock is released around allocation
// and launch.
#include <Python.h>

#include <ATen/core/LegacyTypeDispatch.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/zeros.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/DynamicTypes.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>
#include <torch/csrc/utils/pybind.h>

#include <mutex>
#include <optional>
#include <string>
#include <vector>

#include "../../include/lancet_hip.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

PyObject* g_lancet_error = nullptr;    // capi.LancetError
PyObject* g_scan_pool = nullptr;       // ops._scan_pool
PyObject* g_scan_workspace = nullptr;  // ops._scan_workspace

// ---- statuses -----------------------------------------------------------------------------------------------------
struct Status : std::runtime_error {
  int code;
  const char* what_failed;
  Status(int c, const char* w) : std::runtime_error(w), code(c), what_failed(w) {}
};
inline void check(int status, const char* what) {
  if (status != LANCET_OK) throw Status(status, what);
}
// with the lock held: the Python exception of a status
void set_lancet_error(const Status& s) {
  THPObjectPtr args(Py_BuildValue("(is)", s.code, s.what_failed));
  THPObjectPtr e(args ? PyObject_Call(g_lancet_error, args.get(), nullptr) : nullptr);
  if (e) PyErr_SetObject(g_lancet_error, e.get());
}
// Every entry point: C++ exceptions become Python ones.
#define LANCET_TRY try {
#define LANCET_CATCH              \
  }                               \
  catch (const Status& s) {       \
    set_lancet_error(s);          \
    return nullptr;               \
  }                               \
  catch (python_error& e) {       \
    e.restore();                  \
    return nullptr;               \
  }                               \
  catch (...) {                   \
    torch::translate_exception_to_python(std::current_exception()); \
    return nullptr;               \
  }

// ---- argument helpers ---------------------------------------------------------------------------------------------
const Tensor& tensor_arg(PyObject* o, const char* name) {
  TORCH_CHECK_TYPE(THPVariable_Check(o), name, " must be a torch.Tensor, got ", Py_TYPE(o)->tp_name);
  return THPVariable_Unpack(o);
}
Tensor optional_arg(PyObject* o, const char* name) { return o == Py_None ? Tensor() : tensor_arg(o, name); }
int64_t int_arg(PyObject* o) {
  const long long v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) throw python_error();
  return v;
}
double float_arg(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw python_error();
  return v;
}
void need_args(Py_ssize_t got, Py_ssize_t want, const char* name) {
  TORCH_CHECK_TYPE(got == want, name, " takes ", want, " arguments, got ", got);
}
int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return LANCET_F32;
    case at::kBFloat16: return LANCET_BF16;
    case at::kHalf: return LANCET_F16;
    default: return -1;
  }
}
int rows_dtype(const Tensor& t) {
  const int c = dtype_code(t.scalar_type());
  TORCH_CHECK_TYPE(c >= 0, "token rows must be float32, bfloat16 or float16, got ", t.scalar_type());
  return c;
}
int gate_dtype(const Tensor& t, const char* name = "gate") {
  const int c = dtype_code(t.scalar_type());
  TORCH_CHECK_TYPE(c >= 0, name, " must be float32, bfloat16 or float16, got ", t.scalar_type());
  return c;
}
#define NEED(cond, ...) TORCH_CHECK_VALUE(cond, __VA_ARGS__)
void on_device(const Tensor& t, const char* name) {
  NEED(t.is_cuda(), name, " must live on the GPU");
  NEED(t.is_contiguous(), name, " must be contiguous");
}
inline void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
inline void* current_stream() { return c10::hip::getCurrentHIPStream().stream(); }
Tensor new_tensor(at::IntArrayRef shape, at::ScalarType dtype, const Tensor& like) {
  return at::empty(shape, at::TensorOptions().dtype(dtype).device(like.device()));
}
bool is_mask(const Tensor& t) { return t.scalar_type() == at::kInt && t.dim() == 2 && t.size(0) == 2; }
int64_t mask_tokens(const Tensor& il, int64_t top_k) {
  on_device(il, "indices_locations");
  NEED(is_mask(il), "indices_locations must be int32 [2, k*S]");
  NEED((top_k == 1 || top_k == 2) && il.size(1) % top_k == 0, "top_k must be 1 or 2 and divide the mask length");
  return il.size(1) / top_k;
}
void check_rows_and_gate(const Tensor& data, const Tensor& gate) {
  on_device(data, "data"), on_device(gate, "gate");
  NEED(data.dim() == 2, "Expected input data to be 2D.");
  NEED(gate.dim() == 2, "Expected input gate to be 2D.");
  NEED(data.size(0) == gate.size(0), "Input data and gate should have matching shape in dim 0.");
  gate_dtype(gate);
  rows_dtype(data);
}
void check_noise(const Tensor& noise, const Tensor& gate, int64_t top_k) {
  if (!noise.defined()) return;
  on_device(noise, "gate2_noise");
  NEED(top_k == 2, "gate2_noise only exists for the second choice (top_k = 2)");
  NEED(noise.sizes() == gate.sizes() && noise.scalar_type() == gate.scalar_type(), "gate2_noise must have the gate's shape and dtype");
}
int64_t capacity_of(int64_t S, int64_t E, double factor) { return lancet_moe_capacity(S, E, static_cast<float>(factor)); }

// n tensors of a Python sequence
struct TensorSeq {
  THPObjectPtr fast;
  Py_ssize_t n;
  explicit TensorSeq(PyObject* o, const char* name) : fast(PySequence_Fast(o, name)), n(0) {
    if (!fast) throw python_error();
    n = PySequence_Fast_GET_SIZE(fast.get());
  }
  const Tensor& at(Py_ssize_t i, const char* name) const { return tensor_arg(PySequence_Fast_GET_ITEM(fast.get(), i), name); }
};

// The scan's workspace: the caller's, or the one kept for the data's device and its current stream.  ops._scan_workspace
// knows the rules; the common case (one that is kept already and large enough) is looked up here.
Tensor scan_workspace(size_t nbytes, const Tensor& data, PyObject* given) {
  THPObjectPtr ws;
  if (given == Py_None) {
    const int idx = data.device().index();
    THPObjectPtr key(Py_BuildValue("(iK)", idx, reinterpret_cast<unsigned long long>(c10::hip::getCurrentHIPStream(idx).stream())));
    if (!key) throw python_error();
    PyObject* kept = PyDict_GetItemWithError(g_scan_pool, key.get());
    if (!kept && PyErr_Occurred()) throw python_error();
    if (kept) {
      THPObjectPtr buf(PyObject_GetAttrString(kept, "buf"));
      if (!buf) throw python_error();
      const Tensor t = tensor_arg(buf.get(), "workspace");
      if (static_cast<size_t>(t.numel()) >= nbytes) return t;
    }
  }
  THPObjectPtr dev(THPDevice_New(data.device())), size(PyLong_FromSize_t(nbytes));
  ws = PyObject_CallFunctionObjArgs(g_scan_workspace, size.get(), dev.get(), given, nullptr);
  if (!ws) throw python_error();
  THPObjectPtr buf(PyObject_GetAttrString(ws.get(), "buf"));
  if (!buf) throw python_error();
  return tensor_arg(buf.get(), "workspace");
}
// A call is several launches that pass tables through its workspace, and the interpreter's lock is released around them: threads
// that share a stream share the workspace kept for it, so one enqueues all its launches before the next may (they then run
// one after the other on the stream).  Taken without the interpreter's lock, held over launches alone; a workspace given by
// the caller serves one call at a time by its contract.
std::unique_lock<std::mutex> launches_on(const Tensor& workspace, bool kept) {
  static std::mutex locks[64];  // by address, so that threads on streams of their own do not wait for one another
  if (!kept) return {};
  return std::unique_lock<std::mutex>(locks[(reinterpret_cast<uintptr_t>(workspace.data_ptr()) >> 12) % 64]);
}
// a plain scratch buffer: the caller's, or a new one
Tensor scratch(size_t nbytes, const Tensor& like, const Tensor& given) {
  if (given.defined()) {
    NEED(given.is_cuda() && given.scalar_type() == at::kByte && static_cast<size_t>(given.numel()) >= nbytes,
         "workspace must be a uint8 GPU tensor of at least ", nbytes, " bytes");
    return given;
  }
  return new_tensor({static_cast<int64_t>(std::max<size_t>(nbytes, 4))}, at::kByte, like);
}

// ---- the operators ------------------------------------------------------------------------------------------------
struct Encoded {
  Tensor gates_s, indloc, used, elems, disp;
};
struct EncodeArgs {
  double capacity_factor = 1.0;  // as the caller gave it
  std::optional<int64_t> capacity;
  int64_t top_k = 1;
  unsigned flags = 0;
  bool prioritized = false;  // batch-prioritised: the batch is cut into n_partitions, the call covers one
  int64_t n_partitions = 0, partition_id = 0;
  Tensor workspace;
  bool kept_workspace = false;  // scan_workspace's own, which other threads may find too
};

size_t encode_workspace_bytes(const Tensor& gate, const EncodeArgs& a) {
  return a.prioritized ? lancet_moe_encode_bpr_workspace_bytes(gate.size(0), gate.size(1), static_cast<int>(a.n_partitions))
                            : lancet_moe_encode_workspace_bytes(gate.size(0), gate.size(1), static_cast<int>(a.top_k));
}
// everything that is checked before the workspace is asked for
int64_t check_encode(const Tensor& data, const Tensor& gate, const Tensor& noise, const Tensor& used, const EncodeArgs& a) {
  check_rows_and_gate(data, gate);
  const int64_t S = data.size(0), E = gate.size(1);
  if (a.prioritized) {
    NEED(a.n_partitions > 0, "n_partitions should be greater than 0.");
    NEED(0 <= a.partition_id && a.partition_id < a.n_partitions, "partition_id should be less than n_partitions.");
    return capacity_of(S / a.n_partitions, E, a.capacity_factor);
  }
  NEED(a.top_k == 1 || a.top_k == 2, "top_k must be 1 or 2");
  check_noise(noise, gate, a.top_k);
  const int64_t cap = a.capacity ? *a.capacity : capacity_of(S, E, a.capacity_factor * (a.top_k == 2 ? 2.0 : 1.0));
  NEED(cap >= 0, "capacity must not be negative");
  if (used.defined()) {
    on_device(used, "used_capacity");
    NEED(used.dim() == 1 && used.numel() == E && used.scalar_type() == at::kInt, "Input used_capacity should be 1-D int32 of length E.");
  }
  return cap;
}
Encoded new_encoded(const Tensor& data, const Tensor& gate, int64_t cap, const EncodeArgs& a) {
  const int64_t S = a.prioritized ? data.size(0) / a.n_partitions : data.size(0), k = a.prioritized ? 1 : a.top_k, E = gate.size(1);
  return {new_tensor({k * S}, gate.scalar_type(), data), new_tensor({2, k * S}, at::kInt, data), new_tensor({E}, at::kInt, data),
          new_tensor({E}, at::kUInt64, data), new_tensor({E, cap, data.size(1)}, data.scalar_type(), data)};
}
void encode(const Tensor& data, const Tensor& gate, const Tensor& noise, const Tensor& used, int64_t cap, const EncodeArgs& a,
            const Encoded& o) {
  NEED(o.gates_s.scalar_type() == gate.scalar_type(), "gates_s takes the gate's dtype");
  const int dt = rows_dtype(data), gd = gate_dtype(gate);
  const auto elems = static_cast<uint64_t*>(ptr(o.elems));
  const auto il = static_cast<int32_t*>(ptr(o.indloc));
  const auto used_out = static_cast<int32_t*>(ptr(o.used));
  const auto lock = launches_on(a.workspace, a.kept_workspace);
  if (a.prioritized) {
    check(lancet_moe_encode_bpr(ptr(data), ptr(gate), data.size(0), data.size(1), gate.size(1), cap, static_cast<int>(a.n_partitions),
                                static_cast<int>(a.partition_id), dt, gd, a.flags, ptr(o.gates_s), il, used_out, elems,
                                ptr(o.disp), ptr(a.workspace), a.workspace.numel(), current_stream()),
          "lancet_moe_encode_bpr");
  } else {
    check(lancet_moe_encode(ptr(data), ptr(gate), ptr(noise), static_cast<const int32_t*>(ptr(used)), data.size(0), data.size(1),
                            gate.size(1), cap, static_cast<int>(a.top_k), dt, gd, a.flags, ptr(o.gates_s), il, used_out, elems,
                            ptr(o.disp), ptr(a.workspace), a.workspace.numel(), current_stream()),
          "lancet_moe_encode");
  }
}

Tensor decode(const Tensor& data, const Tensor& gate, const Tensor& il, int64_t top_k, Tensor out) {
  on_device(data, "data"), on_device(gate, "gate"), on_device(il, "indices_locations");
  NEED(data.dim() == 3, "Expected input data to be 3D.");
  NEED(gate.dim() == 1, "Expected input gate to be 1D.");
  const int gd = gate_dtype(gate);
  NEED(is_mask(il) && il.size(1) == gate.size(0), "indices_locations must be int32 [2, k*S]");
  const int dt = rows_dtype(data);
  NEED(top_k != 0 && gate.size(0) % top_k == 0, "gate length must be a multiple of top_k");
  const int64_t S = gate.size(0) / top_k, E = data.size(0), C = data.size(1), M = data.size(2);
  if (!out.defined()) out = new_tensor({S, M}, data.scalar_type(), data);
  check(lancet_moe_decode(ptr(data), ptr(gate), static_cast<const int32_t*>(ptr(il)), S, M, E, C, static_cast<int>(top_k), dt, gd,
                          ptr(out), current_stream()),
        "lancet_moe_decode");
  return out;
}

Tensor encode_dx(const Tensor& dy, const Tensor& il, int64_t top_k, Tensor out) {
  on_device(dy, "dy");
  NEED(dy.dim() == 3, "Input dy should be 3-D.");
  const int64_t S = mask_tokens(il, top_k), E = dy.size(0), C = dy.size(1), M = dy.size(2);
  if (!out.defined()) out = new_tensor({S, M}, dy.scalar_type(), dy);
  check(lancet_moe_encode_dx(ptr(dy), static_cast<const int32_t*>(ptr(il)), S, M, E, C, static_cast<int>(top_k), rows_dtype(dy),
                             ptr(out), current_stream()),
        "lancet_moe_encode_dx");
  return out;
}

Tensor encode_dg(const Tensor& dy, const Tensor& il, int64_t n_experts, int64_t top_k, Tensor out) {
  on_device(dy, "dy");
  NEED(dy.dim() == 1, "Input dy should be 1-D.");
  const int64_t S = mask_tokens(il, top_k);
  NEED(dy.size(0) == top_k * S, "dy and indices_locations disagree");
  if (!out.defined()) out = new_tensor({S, n_experts}, dy.scalar_type(), dy);
  NEED(out.scalar_type() == dy.scalar_type(), "the gate gradient takes dy's dtype");
  check(lancet_moe_encode_dg(ptr(dy), static_cast<const int32_t*>(ptr(il)), S, n_experts, static_cast<int>(top_k),
                             gate_dtype(dy, "dy"), ptr(out), current_stream()),
        "lancet_moe_encode_dg");
  return out;
}

Tensor encode_dgate(const Tensor& dy, const Tensor& gate, const Tensor& il, int64_t top_k, bool is_logits, Tensor out) {
  on_device(dy, "dy"), on_device(gate, "gate");
  NEED(dy.dim() == 1 && gate.dim() == 2, "dy must be 1-D and gate 2-D");
  const int64_t S = mask_tokens(il, top_k);
  NEED(dy.size(0) == top_k * S && gate.size(0) == S, "dy, gate and indices_locations disagree");
  NEED(dy.scalar_type() == gate.scalar_type(), "dy takes the gate's dtype");
  if (!out.defined()) out = new_tensor(gate.sizes(), gate.scalar_type(), gate);
  NEED(out.scalar_type() == gate.scalar_type() && out.sizes() == gate.sizes() && out.is_contiguous(),
       "the gradient has the gate's shape and dtype");
  check(lancet_moe_encode_dgate(ptr(dy), ptr(gate), static_cast<const int32_t*>(ptr(il)), S, gate.size(1), static_cast<int>(top_k),
                                gate_dtype(gate), is_logits ? LANCET_GATE_IS_LOGITS : 0, ptr(out), current_stream()),
        "lancet_moe_encode_dgate");
  return out;
}

Tensor decode_dx(const Tensor& dy, const Tensor& gate, const Tensor& il, int64_t E, int64_t C, int64_t top_k, const Tensor& workspace,
                 Tensor out) {
  on_device(dy, "dy"), on_device(gate, "gate");
  NEED(dy.dim() == 2, "Input dy should be 2-D.");
  NEED(gate.dim() == 1, "gate must be 1-D");
  const int64_t S = mask_tokens(il, top_k);
  NEED(dy.size(0) == S && gate.size(0) == top_k * S, "dy, gate and indices_locations disagree");
  const int64_t M = dy.size(1);
  if (!out.defined()) out = new_tensor({E, C, M}, dy.scalar_type(), dy);
  const Tensor ws = scratch(lancet_moe_decode_dx_workspace_bytes(E, C), dy, workspace);
  check(lancet_moe_decode_dx(ptr(dy), ptr(gate), static_cast<const int32_t*>(ptr(il)), S, M, E, C, static_cast<int>(top_k),
                             rows_dtype(dy), gate_dtype(gate), ptr(out), ptr(ws), ws.numel(), current_stream()),
        "lancet_moe_decode_dx");
  return out;
}

Tensor decode_dg(const Tensor& dy, const Tensor& data, const Tensor& il, int64_t top_k, at::ScalarType gate_type, Tensor out) {
  on_device(dy, "dy"), on_device(data, "data");
  NEED(dy.dim() == 2 && data.dim() == 3 && dy.scalar_type() == data.scalar_type() && dy.size(1) == data.size(2),
       "dy must be [S,M] and data [E,C,M] of one dtype");
  const int64_t S = mask_tokens(il, top_k);
  NEED(dy.size(0) == S, "dy and indices_locations disagree");
  const int64_t E = data.size(0), C = data.size(1), M = data.size(2);
  if (!out.defined()) out = new_tensor({top_k * S}, gate_type, dy);
  check(lancet_moe_decode_dg(ptr(dy), ptr(data), static_cast<const int32_t*>(ptr(il)), S, M, E, C, static_cast<int>(top_k),
                             rows_dtype(dy), gate_dtype(out, "the gate gradient"), ptr(out), current_stream()),
        "lancet_moe_decode_dg");
  return out;
}

void decode_grad(const Tensor& dy, const Tensor& data, const Tensor& gate, const Tensor& il, int64_t top_k, const Tensor& workspace,
                 Tensor& d_data, Tensor& d_gate) {
  on_device(dy, "dy"), on_device(data, "data"), on_device(gate, "gate");
  NEED(dy.dim() == 2 && data.dim() == 3 && dy.scalar_type() == data.scalar_type() && dy.size(1) == data.size(2),
       "dy must be [S,M] and data [E,C,M] of one dtype");
  const int64_t S = mask_tokens(il, top_k);
  NEED(dy.size(0) == S && gate.dim() == 1 && gate.size(0) == top_k * S, "dy, gate and indices_locations disagree");
  const int64_t E = data.size(0), C = data.size(1), M = data.size(2);
  if (!d_data.defined()) {
    d_data = new_tensor(data.sizes(), data.scalar_type(), data), d_gate = new_tensor(gate.sizes(), gate.scalar_type(), gate);
  } else {
    on_device(d_data, "the expert rows' gradient"), on_device(d_gate, "the gate gradient");
    NEED(d_data.sizes() == data.sizes() && d_data.scalar_type() == data.scalar_type(), "the expert rows' gradient has the rows' shape and dtype");
    NEED(d_gate.sizes() == gate.sizes() && d_gate.scalar_type() == gate.scalar_type(), "the gate gradient has the gate's shape and dtype");
  }
  const Tensor ws = scratch(lancet_moe_decode_dx_workspace_bytes(E, C), dy, workspace);
  check(lancet_moe_decode_grad(ptr(dy), ptr(data), ptr(gate), static_cast<const int32_t*>(ptr(il)), S, M, E, C, static_cast<int>(top_k),
                               rows_dtype(dy), gate_dtype(gate), ptr(d_data), ptr(d_gate), ptr(ws), ws.numel(), current_stream()),
        "lancet_moe_decode_grad");
}

// ---- gradients ----------------------------------------------------------------------------------------------------
// A status that fails inside a backward pass travels through the engine as the Python exception it is.
template <typename F>
variable_list in_backward(F f) {
  try {
    return f();
  } catch (const Status& s) {
    pybind11::gil_scoped_acquire lock;
    set_lancet_error(s);
    python_error e;
    e.persist();
    throw e;
  }
}

struct EncodeFunction : torch::autograd::Function<EncodeFunction> {
  static variable_list forward(AutogradContext* ctx, const Tensor& data, const Tensor& gate, const std::optional<Tensor>& noise,
                               const std::optional<Tensor>& used, const EncodeArgs& a, int64_t cap) {
    const Encoded o = new_encoded(data, gate, cap, a);
    encode(data, gate, noise.value_or(Tensor()), used.value_or(Tensor()), cap, a, o);
    // the plain rule needs the mask only; the forms that transform the gate value need the gate too
    const bool logits = (a.flags & LANCET_GATE_IS_LOGITS) != 0, whole = a.top_k == 2 || logits;
    ctx->save_for_backward({o.indloc, whole ? gate : Tensor()});
    ctx->saved_data["args"] = std::vector<int64_t>{whole, logits, a.top_k, a.n_partitions, a.partition_id, cap, data.size(0), data.size(1),
                                                   gate.size(1), static_cast<int64_t>(data.scalar_type()), static_cast<int64_t>(gate.scalar_type())};
    ctx->mark_non_differentiable({o.indloc, o.used, o.elems});
    // gradients nobody sent arrive undefined: autograd would fill zeros for the three integer outputs too, which is
    // three launches per backward (14 of the 1430 us of a 65536 x 4096 bf16 top-2 pass)
    ctx->set_materialize_grads(false);
    return {o.gates_s, o.indloc, o.used, o.elems, o.disp};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    return in_backward([&]() -> variable_list {
      const auto saved = ctx->get_saved_variables();
      const auto v = ctx->saved_data["args"].toIntVector();
      const Tensor& il = saved[0];
      const bool whole = v[0], logits = v[1];
      const int64_t top_k = v[2], P = v[3], pid = v[4], cap = v[5], S0 = v[6], M = v[7], E = v[8];
      const auto type = static_cast<at::ScalarType>(v[9]), gate_type = static_cast<at::ScalarType>(v[10]);
      const auto options = at::TensorOptions().device(il.device());
      const int64_t S = P > 0 ? il.size(1) : S0;
      Tensor d_gates = grads[0].defined() ? grads[0].contiguous() : at::zeros({top_k * S}, options.dtype(gate_type));
      Tensor d_disp = grads[4].defined() ? grads[4].contiguous() : at::zeros({E, cap, M}, options.dtype(type));
      Tensor dx = encode_dx(d_disp, il, top_k, Tensor()), dg;
      if (!whole) dg = encode_dg(d_gates, il, E, 1, Tensor());
      else dg = encode_dgate(d_gates, P > 0 ? saved[1].narrow(0, pid * S, S) : saved[1], il, top_k, logits, Tensor());
      if (P > 0) {
        // the op saw the whole batch and encoded one partition of it: the other tokens get no gradient (the
        // reference's rule returns the partition-sized arrays as they are)
        Tensor full_x = at::zeros({S0, M}, options.dtype(type)), full_g = at::zeros({S0, E}, options.dtype(dg.scalar_type()));
        full_x.narrow(0, pid * S, S).copy_(dx), full_g.narrow(0, pid * S, S).copy_(dg);
        dx = full_x, dg = full_g;
      }
      return {dx, dg, Tensor(), Tensor(), Tensor(), Tensor()};
    });
  }
};

struct DecodeFunction : torch::autograd::Function<DecodeFunction> {
  static Tensor forward(AutogradContext* ctx, const Tensor& data, const Tensor& gate, const Tensor& il, int64_t top_k) {
    ctx->save_for_backward({data, gate, il});
    ctx->saved_data["top_k"] = top_k;
    return decode(data, gate, il, top_k, Tensor());
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    return in_backward([&]() -> variable_list {
      const auto saved = ctx->get_saved_variables();
      const int64_t top_k = ctx->saved_data["top_k"].toInt();
      const Tensor dy = grads[0].contiguous(), &data = saved[0], &gate = saved[1], &il = saved[2];
      Tensor d_data, d_gate;
      // both gradients in one pass over the rows, or the one that is asked for
      if (ctx->needs_input_grad(0) && ctx->needs_input_grad(1)) decode_grad(dy, data, gate, il, top_k, Tensor(), d_data, d_gate);
      else if (ctx->needs_input_grad(0)) d_data = decode_dx(dy, gate, il, data.size(0), data.size(1), top_k, Tensor(), Tensor());
      else if (ctx->needs_input_grad(1)) d_gate = decode_dg(dy, data, il, top_k, gate.scalar_type(), Tensor());
      return {d_data, d_gate, Tensor(), Tensor()};
    });
  }
};

// ---- Python entry points ------------------------------------------------------------------------------------------
typedef PyObject* const* Args;
PyObject* wrap(const Tensor& t) { return THPVariable_Wrap(t); }
PyObject* wrap_tuple(const variable_list& ts) {
  THPObjectPtr tuple(PyTuple_New(static_cast<Py_ssize_t>(ts.size())));
  if (!tuple) return nullptr;
  for (size_t i = 0; i < ts.size(); ++i) {
    PyObject* o = wrap(ts[i]);
    if (!o) return nullptr;
    PyTuple_SET_ITEM(tuple.get(), static_cast<Py_ssize_t>(i), o);
  }
  return tuple.release();
}

EncodeArgs encode_args(PyObject* factor, PyObject* capacity, PyObject* top_k, PyObject* flags) {
  EncodeArgs a;
  a.capacity_factor = float_arg(factor);
  if (capacity != Py_None) a.capacity = int_arg(capacity);
  a.top_k = int_arg(top_k), a.flags = static_cast<unsigned>(int_arg(flags));
  return a;
}
// out given: its five tensors, and the 64-bit counts seen as unsigned
PyObject* encode_into(const Tensor& data, const Tensor& gate, const Tensor& noise, const Tensor& used, int64_t cap, const EncodeArgs& a,
                      PyObject* out) {
  if (out == Py_None) {
    variable_list all;
    {
      pybind11::gil_scoped_release unlocked;
      const Encoded o = new_encoded(data, gate, cap, a);
      encode(data, gate, noise, used, cap, a, o);
      all = {o.gates_s, o.indloc, o.used, o.elems, o.disp};
    }
    return wrap_tuple(all);
  }
  const TensorSeq seq(out, "out must be a sequence of five tensors");
  NEED(seq.n == 5, "out must be a sequence of five tensors");
  const Encoded o = {seq.at(0, "gates_s"), seq.at(1, "indices_locations"), seq.at(2, "used_capacity"), seq.at(3, "elements_per_expert"), seq.at(4, "dispatched")};
  Tensor unsigned_elems;
  {
    pybind11::gil_scoped_release unlocked;
    encode(data, gate, noise, used, cap, a, o);
    if (o.elems.scalar_type() == at::kLong) unsigned_elems = o.elems.view(at::kUInt64);
  }
  return wrap_tuple({o.gates_s, o.indloc, o.used, unsigned_elems.defined() ? unsigned_elems : o.elems, o.disp});
}

// (data, gate, noise, used, capacity_factor, capacity, top_k, flags, workspace, out)
PyObject* py_encode(PyObject*, Args p, Py_ssize_t n) {
  LANCET_TRY
  need_args(n, 10, "moe_encode");
  const Tensor data = tensor_arg(p[0], "data"), gate = tensor_arg(p[1], "gate"), noise = optional_arg(p[2], "gate2_noise"),
               used = optional_arg(p[3], "used_capacity");
  EncodeArgs a = encode_args(p[4], p[5], p[6], p[7]);
  const int64_t cap = check_encode(data, gate, noise, used, a);
  a.workspace = scan_workspace(encode_workspace_bytes(gate, a), data, p[8]), a.kept_workspace = p[8] == Py_None;
  return encode_into(data, gate, noise, used, cap, a, p[9]);
  LANCET_CATCH
}
// (data, gate, n_partitions, partition_id, capacity_factor, flags, workspace, out)
PyObject* py_encode_bpr(PyObject*, Args p, Py_ssize_t n) {
  LANCET_TRY
  need_args(n, 8, "moe_encode_batch_prioritized");
  const Tensor data = tensor_arg(p[0], "data"), gate = tensor_arg(p[1], "gate");
  EncodeArgs a;
  a.capacity_factor = float_arg(p[4]), a.flags = static_cast<unsigned>(int_arg(p[5]));
  a.prioritized = true, a.n_partitions = int_arg(p[2]), a.partition_id = int_arg(p[3]);
  const int64_t cap = check_encode(data, gate, Tensor(), Tensor(), a);
  a.workspace = scan_workspace(encode_workspace_bytes(gate, a), data, p[6]), a.kept_workspace = p[6] == Py_None;
  return encode_into(data, gate, Tensor(), Tensor(), cap, a, p[7]);
  LANCET_CATCH
}
// (data, gate, noise, used, capacity_factor, capacity, top_k, flags, n_partitions or None, partition_id)
PyObject* py_encode_diff(PyObject*, Args p, Py_ssize_t n) {
  LANCET_TRY
  need_args(n, 10, "moe_encode");
  const Tensor data = tensor_arg(p[0], "data"), gate = tensor_arg(p[1], "gate"), noise = optional_arg(p[2], "gate2_noise"),
               used = optional_arg(p[3], "used_capacity");
  EncodeArgs a = encode_args(p[4], p[5], p[6], p[7]);
  if (p[8] != Py_None) a.prioritized = true, a.n_partitions = int_arg(p[8]), a.partition_id = int_arg(p[9]);
  const int64_t cap = check_encode(data, gate, noise, used, a);
  a.workspace = scan_workspace(encode_workspace_bytes(gate, a), data, Py_None), a.kept_workspace = true;
  const auto some = [](const Tensor& t) { return t.defined() ? std::optional<Tensor>(t) : std::nullopt; };
  variable_list all;
  {
    pybind11::gil_scoped_release unlocked;
    all = EncodeFunction::apply(data, gate, some(noise), some(used), a, cap);
  }
  return wrap_tuple(all);
  LANCET_CATCH
}
// (data, gate, indices_locations, top_k, out)
PyObject* py_decode(PyObject*, Args p, Py_ssize_t n) {
  LANCET_TRY
  need_args(n, 5, "moe_decode");
  const Tensor data = tensor_arg(p[0], "data"), gate = tensor_arg(p[1], "gate"), il = tensor_arg(p[2], "indices_locations");
  const int64_t k = int_arg(p[3]);
  Tensor out = optional_arg(p[4], "out");
  {
    pybind11::gil_scoped_release unlocked;
    out = decode(data, gate, il, k, out);
  }
  return wrap(out);
  LANCET_CATCH
}
// (data, gate, indices_locations, top_k)
PyObject* py_decode_diff(PyObject*, Args p, Py_ssize_t n) {
  LANCET_TRY
  need_args(n, 4, "moe_decode");
  const Tensor data = tensor_arg(p[0], "data"), gate = tensor_arg(p[1], "gate"), il = tensor_arg(p[2], "indices_locations");
  const int64_t k = int_arg(p[3]);
  Tensor out;
  {
    pybind11::gil_scoped_release unlocked;
    out = DecodeFunction::apply(data, gate, il, k);
  }
  return wrap(out);
  LANCET_CATCH
}
// (dy, indices_locations, top_k, out)
PyObject* py_encode_dx(PyObject*, Args p, Py_ssize_t n) {
  LANCET_TRY
  need_args(n, 4, "moe_encode_dx");
  const Tensor dy = tensor_arg(p[0], "dy"), il = tensor_arg(p[1], "indices_locations");
  const int64_t k = int_arg(p[2]);
  Tensor out = optional_arg(p[3], "out");
  {
    pybind11::gil_scoped_release unlocked;
    out = encode_dx(dy, il, k, out);
  }
  return wrap(out);
  LANCET_CATCH
}
// (dy, indices_locations, n_experts, top_k, out)
PyObject* py_encode_dg(PyObject*, Args p, Py_ssize_t n) {
  LANCET_TRY
  need_args(n, 5, "moe_encode_dg");
  const Tensor dy = tensor_arg(p[0], "dy"), il = tensor_arg(p[1], "indices_locations");
  const int64_t E = int_arg(p[2]), k = int_arg(p[3]);
  Tensor out = optional_arg(p[4], "out");
  {
    pybind11::gil_scoped_release unlocked;
    out = encode_dg(dy, il, E, k, out);
  }
  return wrap(out);
  LANCET_CATCH
}
// (dy, gate, indices_locations, top_k, gate_is_logits, out)
PyObject* py_encode_dgate(PyObject*, Args p, Py_ssize_t n) {
  LANCET_TRY
  need_args(n, 6, "moe_encode_dgate");
  const Tensor dy = tensor_arg(p[0], "dy"), gate = tensor_arg(p[1], "gate"), il = tensor_arg(p[2], "indices_locations");
  const int64_t k = int_arg(p[3]);
  const int logits = PyObject_IsTrue(p[4]);
  if (logits < 0) return nullptr;
  Tensor out = optional_arg(p[5], "out");
  {
    pybind11::gil_scoped_release unlocked;
    out = encode_dgate(dy, gate, il, k, logits != 0, out);
  }
  return wrap(out);
  LANCET_CATCH
}
// (dy, gate, indices_locations, n_experts, capacity, top_k, workspace, out)
PyObject* py_decode_dx(PyObject*, Args p, Py_ssize_t n) {
  LANCET_TRY
  need_args(n, 8, "moe_decode_dx");
  const Tensor dy = tensor_arg(p[0], "dy"), gate = tensor_arg(p[1], "gate"), il = tensor_arg(p[2], "indices_locations"),
               ws = optional_arg(p[6], "workspace");
  const int64_t E = int_arg(p[3]), C = int_arg(p[4]), k = int_arg(p[5]);
  Tensor out = optional_arg(p[7], "out");
  {
    pybind11::gil_scoped_release unlocked;
    out = decode_dx(dy, gate, il, E, C, k, ws, out);
  }
  return wrap(out);
  LANCET_CATCH
}
// (dy, data, indices_locations, top_k, an empty tensor of the gate gradient's dtype, out)
PyObject* py_decode_dg(PyObject*, Args p, Py_ssize_t n) {
  LANCET_TRY
  need_args(n, 6, "moe_decode_dg");
  const Tensor dy = tensor_arg(p[0], "dy"), data = tensor_arg(p[1], "data"), il = tensor_arg(p[2], "indices_locations");
  const int64_t k = int_arg(p[3]);
  TORCH_CHECK_TYPE(THPDtype_Check(p[4]), "gate_dtype must be a torch.dtype");
  const at::ScalarType gt = reinterpret_cast<THPDtype*>(p[4])->scalar_type;
  Tensor out = optional_arg(p[5], "out");
  {
    pybind11::gil_scoped_release unlocked;
    out = decode_dg(dy, data, il, k, gt, out);
  }
  return wrap(out);
  LANCET_CATCH
}
// (dy, data, gate, indices_locations, top_k, workspace, out)
PyObject* py_decode_grad(PyObject*, Args p, Py_ssize_t n) {
  LANCET_TRY
  need_args(n, 7, "moe_decode_grad");
  const Tensor dy = tensor_arg(p[0], "dy"), data = tensor_arg(p[1], "data"), gate = tensor_arg(p[2], "gate"),
               il = tensor_arg(p[3], "indices_locations"), ws = optional_arg(p[5], "workspace");
  const int64_t k = int_arg(p[4]);
  Tensor d_data, d_gate;
  if (p[6] != Py_None) {
    const TensorSeq seq(p[6], "out must be two tensors");
    NEED(seq.n == 2, "out must be two tensors");
    d_data = seq.at(0, "the expert rows' gradient"), d_gate = seq.at(1, "the gate gradient");
  }
  {
    pybind11::gil_scoped_release unlocked;
    decode_grad(dy, data, gate, il, k, ws, d_data, d_gate);
  }
  return wrap_tuple({d_data, d_gate});
  LANCET_CATCH
}

// (indices_locations, n_experts, workspace, out)
PyObject* py_merge_masks(PyObject*, Args p, Py_ssize_t n) {
  LANCET_TRY
  need_args(n, 4, "moe_merge_masks");
  const TensorSeq il(p[0], "indices_locations must be a sequence of tensors");
  const int64_t E = int_arg(p[1]);
  NEED(il.n >= 1, "need at least one partition");
  std::vector<const int32_t*> ptrs;
  const Tensor first = il.at(0, "indices_locations");
  for (Py_ssize_t i = 0; i < il.n; ++i) {
    const Tensor& t = il.at(i, "indices_locations");
    on_device(t, "indices_locations");
    NEED(t.dim() == 2 && t.sizes() == first.sizes() && t.scalar_type() == at::kInt, "Expected input indices_locations to be 2D int32 of equal shape.");
    ptrs.push_back(static_cast<const int32_t*>(ptr(t)));
  }
  const int64_t S = first.size(1);
  const Tensor given = optional_arg(p[2], "workspace");
  Tensor out = optional_arg(p[3], "out");
  {
    pybind11::gil_scoped_release unlocked;
    if (!out.defined()) out = new_tensor({2, static_cast<int64_t>(il.n) * S}, at::kInt, first);
    const Tensor ws = scratch(lancet_moe_merge_masks_workspace_bytes(static_cast<int>(il.n), E), first, given);
    check(lancet_moe_merge_masks(ptrs.data(), static_cast<int>(il.n), S, E, static_cast<int32_t*>(ptr(out)), ptr(ws), ws.numel(), current_stream()),
          "lancet_moe_merge_masks");
  }
  return wrap(out);
  LANCET_CATCH
}
// (data, indices_locations, workspace, out)
PyObject* py_redispatch(PyObject*, Args p, Py_ssize_t n) {
  LANCET_TRY
  need_args(n, 4, "moe_redispatch");
  const TensorSeq data(p[0], "data must be a sequence of tensors"), il(p[1], "indices_locations must be a sequence of tensors");
  NEED(il.n >= 1 && data.n == il.n, "data and indices_locations must have one entry per partition");
  std::vector<const void*> rows;
  std::vector<const int32_t*> masks;
  const Tensor first = data.at(0, "data");
  for (Py_ssize_t i = 0; i < data.n; ++i) {
    const Tensor& t = data.at(i, "data");
    on_device(t, "data");
    NEED((t.dim() == 3 || t.dim() == 4) && t.sizes() == first.sizes() && t.scalar_type() == first.scalar_type(),
         "Expected input data to be 3 or 4D of equal shape.");
    rows.push_back(ptr(t));
  }
  for (Py_ssize_t i = 0; i < il.n; ++i) {
    const Tensor& t = il.at(i, "indices_locations");
    on_device(t, "indices_locations");
    NEED(t.dim() == 2 && t.scalar_type() == at::kInt, "Expected input indices_locations to be 2D.");
    masks.push_back(static_cast<const int32_t*>(ptr(t)));
  }
  const bool four = first.dim() == 4;  // [G, LE, C, M]
  const int64_t E = four ? first.size(0) * first.size(1) : first.size(0), C = first.size(four ? 2 : 1), M = first.size(four ? 3 : 2);
  const int64_t S = il.at(0, "indices_locations").size(1);
  const int dt = rows_dtype(first), P = static_cast<int>(data.n);
  const Tensor given = optional_arg(p[2], "workspace");
  Tensor out = optional_arg(p[3], "out");
  {
    pybind11::gil_scoped_release unlocked;
    if (!out.defined()) out = new_tensor(first.sizes(), first.scalar_type(), first);
    const Tensor ws = scratch(lancet_moe_redispatch_workspace_bytes(P, E), first, given);
    check(lancet_moe_redispatch(rows.data(), masks.data(), P, S, M, C, E, dt, ptr(out), ptr(ws), ws.numel(), current_stream()),
          "lancet_moe_redispatch");
  }
  return wrap(out);
  LANCET_CATCH
}

// ---- the halves and token ranges of the operators (a caller with streams of its own names the stream) ---------------
// None: the current device's current stream; else the handle of one, for calls whose arrays are all given: what is allocated
// here, and the workspace kept, belong to the current stream, and could be handed on while the named one still uses them
void* stream_arg(PyObject* o, bool all_given) {
  if (o == Py_None) return current_stream();
  NEED(all_given, "a call on a named stream takes its outputs and its workspace from the caller");
  return reinterpret_cast<void*>(static_cast<intptr_t>(int_arg(o)));
}

// (gate, noise, used, M, capacity_factor, capacity, top_k, flags, workspace, out, stream)
PyObject* py_route(PyObject*, Args p, Py_ssize_t n) {
  LANCET_TRY
  need_args(n, 11, "moe_route");
  const Tensor gate = tensor_arg(p[0], "gate"), noise = optional_arg(p[1], "gate2_noise"), used = optional_arg(p[2], "used_capacity");
  const int64_t M = int_arg(p[3]);
  EncodeArgs a = encode_args(p[4], p[5], p[6], p[7]);
  on_device(gate, "gate");
  NEED(gate.dim() == 2, "gate must be 2-D");
  const int gd = gate_dtype(gate);
  const int64_t S = gate.size(0), E = gate.size(1);
  NEED(a.top_k == 1 || a.top_k == 2, "top_k must be 1 or 2");
  check_noise(noise, gate, a.top_k);
  const int64_t cap = a.capacity ? *a.capacity : capacity_of(S, E, a.capacity_factor * (a.top_k == 2 ? 2.0 : 1.0));
  void* const stream = stream_arg(p[10], p[8] != Py_None && p[9] != Py_None);
  Encoded o;
  if (p[9] == Py_None) {
    o = {new_tensor({a.top_k * S}, gate.scalar_type(), gate), new_tensor({2, a.top_k * S}, at::kInt, gate), new_tensor({E}, at::kInt, gate),
         new_tensor({E}, at::kLong, gate), Tensor()};
  } else {
    const TensorSeq seq(p[9], "out must be a sequence of four tensors");
    NEED(seq.n >= 4, "out must be a sequence of four tensors");
    o = {seq.at(0, "gates_s"), seq.at(1, "indices_locations"), seq.at(2, "used_capacity"), seq.at(3, "elements_per_expert"), Tensor()};
  }
  a.workspace = scan_workspace(encode_workspace_bytes(gate, a), gate, p[8]), a.kept_workspace = p[8] == Py_None;
  NEED(o.gates_s.scalar_type() == gate.scalar_type(), "gates_s takes the gate's dtype");
  {
    pybind11::gil_scoped_release unlocked;
    const auto lock = launches_on(a.workspace, a.kept_workspace);
    check(lancet_moe_route(ptr(gate), ptr(noise), static_cast<const int32_t*>(ptr(used)), S, M, E, cap, static_cast<int>(a.top_k), gd,
                           a.flags, ptr(o.gates_s), static_cast<int32_t*>(ptr(o.indloc)), static_cast<int32_t*>(ptr(o.used)),
                           static_cast<uint64_t*>(ptr(o.elems)), ptr(a.workspace), a.workspace.numel(), stream),
          "lancet_moe_route");
  }
  return wrap_tuple({o.gates_s, o.indloc, o.used, o.elems});
  LANCET_CATCH
}
// (data, indices_locations, used_in, used_out, token_first, n_experts, capacity, top_k, flags, out, stream)
PyObject* py_scatter_tokens(PyObject*, Args p, Py_ssize_t n) {
  LANCET_TRY
  need_args(n, 11, "moe_scatter_tokens");
  const Tensor data = tensor_arg(p[0], "data"), il = tensor_arg(p[1], "indices_locations"), used_in = optional_arg(p[2], "used_in"),
               used_out = optional_arg(p[3], "used_out");
  const int64_t first = int_arg(p[4]), E = int_arg(p[5]), C = int_arg(p[6]), k = int_arg(p[7]);
  const unsigned flags = static_cast<unsigned>(int_arg(p[8]));
  Tensor out = optional_arg(p[9], "out");
  on_device(data, "data");
  NEED(data.dim() == 2, "Expected input data to be 2D.");
  const int64_t total = mask_tokens(il, k), count = data.size(0), M = data.size(1);
  NEED(0 <= first && first + count <= total, "token range outside the routed batch");
  void* const stream = stream_arg(p[10], out.defined());
  {
    pybind11::gil_scoped_release unlocked;
    if (!out.defined()) out = new_tensor({E, C, M}, data.scalar_type(), data);
    check(lancet_moe_scatter_tokens(ptr(data), static_cast<const int32_t*>(ptr(il)), static_cast<const int32_t*>(ptr(used_in)),
                                    static_cast<const int32_t*>(ptr(used_out)), total, first, count, M, E, C, static_cast<int>(k),
                                    rows_dtype(data), flags, ptr(out), stream),
          "lancet_moe_scatter_tokens");
  }
  return wrap(out);
  LANCET_CATCH
}
// (data, gate, indices_locations, token_first, n_tokens, top_k, out, stream)
PyObject* py_decode_tokens(PyObject*, Args p, Py_ssize_t n) {
  LANCET_TRY
  need_args(n, 8, "moe_decode_tokens");
  const Tensor data = tensor_arg(p[0], "data"), gate = tensor_arg(p[1], "gate"), il = tensor_arg(p[2], "indices_locations");
  const int64_t first = int_arg(p[3]), count = int_arg(p[4]), k = int_arg(p[5]);
  Tensor out = optional_arg(p[6], "out");
  on_device(data, "data"), on_device(gate, "gate");
  NEED(data.dim() == 3, "Expected input data to be 3D.");
  NEED(gate.dim() == 1, "gate must be 1-D");
  const int64_t total = mask_tokens(il, k);
  NEED(gate.size(0) == k * total, "gate and indices_locations disagree on the token count");
  NEED(0 <= first && 0 <= count && first + count <= total, "token range outside the routed batch");
  const int64_t E = data.size(0), C = data.size(1), M = data.size(2);
  void* const stream = stream_arg(p[7], out.defined());
  {
    pybind11::gil_scoped_release unlocked;
    if (!out.defined()) out = new_tensor({count, M}, data.scalar_type(), data);
    check(lancet_moe_decode_tokens(ptr(data), ptr(gate), static_cast<const int32_t*>(ptr(il)), total, first, count, M, E, C,
                                   static_cast<int>(k), rows_dtype(data), gate_dtype(gate), ptr(out), stream),
          "lancet_moe_decode_tokens");
  }
  return wrap(out);
  LANCET_CATCH
}
// (indices_locations, n_partitions, n_experts, M, top_k, workspace, out, stream)
PyObject* py_partition_ranges(PyObject*, Args p, Py_ssize_t n) {
  LANCET_TRY
  need_args(n, 8, "moe_partition_ranges");
  const Tensor il = tensor_arg(p[0], "indices_locations"), given = optional_arg(p[5], "workspace");
  const int64_t P = int_arg(p[1]), E = int_arg(p[2]), M = int_arg(p[3]), k = int_arg(p[4]);
  const int64_t total = mask_tokens(il, k);
  NEED(P >= 1 && total % P == 0, "the token count must divide into n_partitions");
  Tensor starts, counts;
  if (p[6] != Py_None) {
    const TensorSeq seq(p[6], "out must be two tensors");
    NEED(seq.n == 2, "out must be two tensors");
    starts = seq.at(0, "starts"), counts = seq.at(1, "counts");
  }
  void* const stream = stream_arg(p[7], starts.defined() && given.defined());
  {
    pybind11::gil_scoped_release unlocked;
    if (!starts.defined()) starts = new_tensor({k * P, E}, at::kLong, il), counts = new_tensor({k * P, E}, at::kLong, il);
    const Tensor ws = scratch(lancet_moe_partition_ranges_workspace_bytes(static_cast<int>(k), static_cast<int>(P), E), il, given);
    check(lancet_moe_partition_ranges(static_cast<const int32_t*>(ptr(il)), total, static_cast<int>(k), static_cast<int>(P), E, M,
                                      static_cast<uint64_t*>(ptr(starts)), static_cast<uint64_t*>(ptr(counts)), ptr(ws), ws.numel(), stream),
          "lancet_moe_partition_ranges");
  }
  return wrap_tuple({starts, counts});
  LANCET_CATCH
}
// (src, dst, nelements_per_dim, starts_per_dim, stride, offset, axis, stream); PACK: src is the sparse buffer
template <bool PACK>
PyObject* py_sparse_ranges(PyObject*, Args p, Py_ssize_t n) {
  LANCET_TRY
  need_args(n, 8, "memcpy of sparse ranges");
  const Tensor src = tensor_arg(p[0], "src"), dst = tensor_arg(p[1], "dst"), count = tensor_arg(p[2], "nelements_per_dim"),
               start = tensor_arg(p[3], "starts_per_dim");
  const int64_t stride = int_arg(p[4]), offset = int_arg(p[5]), axis = int_arg(p[6]);
  const Tensor &buf = PACK ? src : dst, &packed = PACK ? dst : src;
  on_device(buf, "sparse buffer"), on_device(packed, "packed array"), on_device(count, "nelements_per_dim");
  NEED(buf.dim() == 3, "the sparse buffer must be 3-D");
  NEED(axis == 0 || axis == 1, "Axis ", axis, " not supported.");
  NEED(buf.scalar_type() == packed.scalar_type(), "dtype / layout mismatch");
  const auto wide = count.scalar_type();
  NEED(wide == at::kLong || wide == at::kUInt64, "nelements_per_dim must be contiguous 64-bit counts");
  on_device(start, "starts_per_dim");
  NEED(start.scalar_type() == wide && start.numel() == count.numel(), "starts_per_dim must match nelements_per_dim");
  void* const stream = stream_arg(p[7], true);
  {
    pybind11::gil_scoped_release unlocked;
    const auto copy = PACK ? lancet_memcpy_sparse_ranges_to_cont_3d : lancet_memcpy_cont_to_sparse_ranges_3d;
    check(copy(ptr(src), ptr(dst), static_cast<const uint64_t*>(ptr(count)), static_cast<const uint64_t*>(ptr(start)), count.numel(),
               static_cast<int>(stride), static_cast<int>(offset), static_cast<int>(axis), buf.size(0), buf.size(1), buf.size(2),
               packed.numel(), rows_dtype(buf), stream),
          PACK ? "lancet_memcpy_sparse_ranges_to_cont_3d" : "lancet_memcpy_cont_to_sparse_ranges_3d");
  }
  return wrap(dst);
  LANCET_CATCH
}

// ---- LANS ---------------------------------------------------------------------------------------------------------
// what ops.lans keeps its plans by: (the sizes of the T gradients, their device)
PyObject* py_lans_key(PyObject*, Args p, Py_ssize_t n) {
  LANCET_TRY
  need_args(n, 1, "lans_key");
  const TensorSeq g(p[0], "the gradients must be a sequence of tensors");
  NEED(g.n > 0, "tensor_list must hold 4 lists of equal length");
  THPObjectPtr sizes(PyTuple_New(g.n));
  if (!sizes) return nullptr;
  for (Py_ssize_t i = 0; i < g.n; ++i) {
    PyObject* size = PyLong_FromLongLong(g.at(i, "a gradient").numel());
    if (!size) return nullptr;
    PyTuple_SET_ITEM(sizes.get(), i, size);
  }
  const auto device = g.at(0, "a gradient").device();
  THPObjectPtr index(device.has_index() ? PyLong_FromLong(device.index()) : (Py_INCREF(Py_None), Py_None));
  return PyTuple_Pack(2, sizes.get(), index.get());
  LANCET_CATCH
}

// (plan handle, address of the planned sizes, T, g, p, m, v, p_lowp, step, step_dev, address of the lancet_lans_hyper, grad_norms)
PyObject* py_lans_step(PyObject*, Args a, Py_ssize_t n) {
  LANCET_TRY
  need_args(n, 12, "lans_step");
  const auto plan = reinterpret_cast<lancet_lans_plan_t>(int_arg(a[0]));
  const auto numels = reinterpret_cast<const int64_t*>(int_arg(a[1]));
  const Py_ssize_t T = static_cast<Py_ssize_t>(int_arg(a[2]));
  const Tensor grad_norms = optional_arg(a[11], "grad_norms"), step_dev = optional_arg(a[9], "step_dev");
  const auto hyper = reinterpret_cast<const lancet_lans_hyper*>(int_arg(a[10]));
  const int64_t step = int_arg(a[8]);
  if (grad_norms.defined())
    NEED(grad_norms.is_cuda() && grad_norms.scalar_type() == at::kFloat && grad_norms.numel() == T && grad_norms.is_contiguous(),
         "grad_norms must be a contiguous float32 GPU tensor of T values");
  const TensorSeq g(a[3], "g must be a sequence"), p(a[4], "p must be a sequence"), m(a[5], "m must be a sequence"), v(a[6], "v must be a sequence");
  NEED(g.n == T && p.n == T && m.n == T && v.n == T, "tensor lists must have one entry per planned tensor");
  std::optional<TensorSeq> low;
  if (a[7] != Py_None) {
    low.emplace(a[7], "p_lowp must be a sequence");
    NEED(low->n == T, "p_lowp must have one entry per planned tensor");
    if (low->n == 0) low.reset();
  }
  const at::ScalarType g_type = T ? g.at(0, "a gradient").scalar_type() : at::kFloat;
  NEED(dtype_code(g_type) >= 0, "gradients must be float32, bfloat16 or float16");
  const at::ScalarType low_type = low ? low->at(0, "a parameter copy").scalar_type() : at::kBFloat16;
  NEED(low_type == at::kBFloat16 || low_type == at::kHalf, "p_lowp must be bfloat16 or float16");
  std::vector<void*> ptrs(static_cast<size_t>(T) * 5);
  const auto take = [&](const TensorSeq& list, at::ScalarType type, void** to) {
    for (Py_ssize_t i = 0; i < T; ++i) {
      const Tensor& t = list.at(i, "a LANS tensor");
      NEED(t.is_cuda() && t.is_contiguous() && t.scalar_type() == type && t.numel() == numels[i],
           "LANS tensors must be contiguous GPU tensors of the planned sizes: p, m, v float32, every gradient of one type, every "
           "16-bit parameter copy of one type");
      to[i] = ptr(t);
    }
  };
  void** const at = ptrs.data();
  take(g, g_type, at), take(p, at::kFloat, at + T), take(m, at::kFloat, at + 2 * T), take(v, at::kFloat, at + 3 * T);
  if (low) take(*low, low_type, at + 4 * T);
  const auto floats = [&](int which) { return reinterpret_cast<float* const*>(at + which * T); };
  {
    pybind11::gil_scoped_release unlocked;
    const auto norms = static_cast<const float*>(ptr(grad_norms)), sd = static_cast<const float*>(ptr(step_dev));
    if (g_type == at::kFloat && !low) {
      check(lancet_lans_step(plan, floats(0), floats(1), floats(2), floats(3), static_cast<int>(step), sd, hyper, norms, current_stream()),
            "lancet_lans_step");
    } else {
      check(lancet_lans_step_mixed(plan, at, dtype_code(g_type), floats(1), floats(2), floats(3), low ? at + 4 * T : nullptr,
                                   dtype_code(low_type), static_cast<int>(step), sd, hyper, norms, current_stream()),
            "lancet_lans_step_mixed");
    }
  }
  Py_RETURN_NONE;
  LANCET_CATCH
}

// (capi.LancetError, ops._scan_pool, ops._scan_workspace)
PyObject* py_bind(PyObject*, Args p, Py_ssize_t n) {
  LANCET_TRY
  need_args(n, 3, "bind");
  TORCH_CHECK_TYPE(PyDict_Check(p[1]), "the pool must be a dict");
  g_lancet_error = Py_NewRef(p[0]), g_scan_pool = Py_NewRef(p[1]), g_scan_workspace = Py_NewRef(p[2]);
  Py_RETURN_NONE;
  LANCET_CATCH
}

#define ENTRY(name, fn) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(fn)), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {ENTRY("bind", py_bind),
                          ENTRY("moe_encode", py_encode),
                          ENTRY("moe_encode_bpr", py_encode_bpr),
                          ENTRY("moe_encode_diff", py_encode_diff),
                          ENTRY("moe_decode", py_decode),
                          ENTRY("moe_decode_diff", py_decode_diff),
                          ENTRY("moe_encode_dx", py_encode_dx),
                          ENTRY("moe_encode_dg", py_encode_dg),
                          ENTRY("moe_encode_dgate", py_encode_dgate),
                          ENTRY("moe_decode_dx", py_decode_dx),
                          ENTRY("moe_decode_dg", py_decode_dg),
                          ENTRY("moe_decode_grad", py_decode_grad),
                          ENTRY("moe_merge_masks", py_merge_masks),
                          ENTRY("moe_redispatch", py_redispatch),
                          ENTRY("moe_route", py_route),
                          ENTRY("moe_scatter_tokens", py_scatter_tokens),
                          ENTRY("moe_decode_tokens", py_decode_tokens),
                          ENTRY("moe_partition_ranges", py_partition_ranges),
                          ENTRY("memcpy_sparse_ranges_to_cont_3d", py_sparse_ranges<true>),
                          ENTRY("memcpy_cont_to_sparse_ranges_3d", py_sparse_ranges<false>),
                          ENTRY("lans_key", py_lans_key),
                          ENTRY("lans_step", py_lans_step),
                          {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "lancet_torch_host", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_lancet_torch_host(void) { return PyModule_Create(&kModule); }
