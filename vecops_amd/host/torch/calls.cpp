// The per-call work of the Python entry points in native code: vecops_amd.capi's products on torch tensors, and the device
// kernel of the operators that vecops_amd.torch_bridge registers.
//
// What bounds a small product's call is the host: describing three tensors, planning, finding the stream and the scratch
// through ctypes took 8 to 16 us in Python, and a registered operator 26 (the dispatcher into Python, a frame of ctypes
// records and a second call through the bridge), where the kernels take 4 to 10.
//
// A function here serves calls on plain device tensors (strided, with storage, of a known type, on no other dispatch
// layer's tensor) on the current stream and answers with the library's status; every other call it leaves to the Python
// form, which raises or runs what it always did.
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/jit/python/pybind_utils.h>
#include <torch/library.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>

#include <deque>
#include <memory>
#include <string>
#include <unordered_map>
#include <vector>

#include "vecops_hip.h"
#include "vecops_hip_host.h"
#include "vecops_rt/abi.h"

namespace {

constexpr int kNotPlain = -1;   // the Python form serves the call

// The VecopsDType number of a tensor's element type, 0 for a type outside the table.
uint32_t dtype_code(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kChar: return VECOPS_DTYPE_I8;
    case at::kByte: return VECOPS_DTYPE_U8;
    case at::kInt: return VECOPS_DTYPE_I32;
    case at::kHalf: return VECOPS_DTYPE_F16;
    case at::kBFloat16: return VECOPS_DTYPE_BF16;
    case at::kFloat: return VECOPS_DTYPE_F32;
    case at::kDouble: return VECOPS_DTYPE_F64;
    default: return 0;
  }
}

// A tensor whose address and strides are its own: no wrapper of vmap, functionalisation, a subclass or a tracing mode.
bool is_plain(const at::Tensor& t) {
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage()) return false;
  const c10::DispatchKeySet keys = t.key_set();
  return !keys.has(c10::DispatchKey::Python) && !keys.has(c10::DispatchKey::FuncTorchBatched) &&
         !keys.has(c10::DispatchKey::FuncTorchGradWrapper) && !keys.has(c10::DispatchKey::Functionalize) &&
         !keys.has(c10::DispatchKey::BatchedNestedTensor);
}

// The tensor behind a Python object, null if it is none or not plain.
const at::Tensor* plain_tensor(PyObject* object) {
  if (!THPVariable_CheckExact(object)) return nullptr;   // (a subclass may answer for its own address)
  const at::Tensor& t = THPVariable_Unpack(object);
  return is_plain(t) ? &t : nullptr;
}

bool describe(const at::Tensor& t, VecopsHipOperand* o) {
  const int64_t rank = t.dim();
  if (rank > 3) return false;
  memset(o, 0, sizeof(*o));
  o->dtype = dtype_code(t);
  if (o->dtype == 0) return false;
  o->data = t.data_ptr();
  o->rank = static_cast<uint32_t>(rank);
  for (int64_t i = 0; i < rank; ++i) {
    o->sizes[i] = t.size(i);
    o->strides[i] = t.stride(i);
  }
  return true;
}

bool describe(PyObject* object, VecopsHipOperand* o) {
  const at::Tensor* t = plain_tensor(object);
  return t != nullptr && describe(*t, o);
}

void* current_stream() { return c10::hip::getCurrentHIPStream().stream(); }

// The workspace a caller hands in, and the device of the output, where another one is allocated.
struct Given {
  void* data = nullptr;
  uint64_t size = 0;
  c10::Device device{c10::DeviceType::CPU};
  bool describe(PyObject* given, const at::Tensor& output) {
    device = output.device();
    if (given == Py_None) return true;
    const at::Tensor* t = plain_tensor(given);
    if (t == nullptr) return false;
    data = t->data_ptr();
    size = static_cast<uint64_t>(t->numel()) * t->element_size();
    return true;
  }
};

// The caller's workspace if it is large enough, else one from torch's allocator, which lives as long as this object: its
// reuse is ordered on the current stream, where the work goes.
struct Workspace {
  at::Tensor own;
  void* data;
  uint64_t size;
  Workspace(const Given& given, uint64_t need) : data(given.data), size(given.size) {
    if (need > 0 && (data == nullptr || size < need)) {
      own = at::empty({static_cast<int64_t>(need)}, at::TensorOptions().dtype(at::kByte).device(given.device));
      data = own.data_ptr();
      size = need;
    }
  }
};

// The library's part of a call, without the interpreter lock: a launch may wait for room in the queue or load code, the
// allocator may synchronise, and other threads' calls and host callbacks that need the lock must not wait for that (the lock
// is given back and taken again in about 0.1 us).  Whatever it needs of the Python objects has been read before; they live
// as long as the caller's references.
template <class Call>
int without_lock(Call&& call) {
  const pybind11::gil_scoped_release released;
  return call();
}

// An int argument that fits 64 bits; false (and no error set) otherwise.
bool integer(PyObject* object, int64_t* out) {
  if (!PyLong_Check(object)) return false;
  int overflow = 0;
  *out = PyLong_AsLongLongAndOverflow(object, &overflow);
  return overflow == 0;
}

// matmul(a, b, c, c_in, compute, workspace)  and, with an epilogue's address, matmul_fused
int product(PyObject* const* args, uint64_t epilogue_address) {
  VecopsHipOperand a, b, c, cin;
  int64_t compute = 0;
  const at::Tensor* out = plain_tensor(args[2]);
  if (out == nullptr || !describe(args[0], &a) || !describe(args[1], &b) || !describe(*out, &c) || !integer(args[4], &compute) ||
      compute < 0 || compute > UINT32_MAX)
    return kNotPlain;
  const VecopsHipOperand* ci = nullptr;
  if (args[3] != Py_None) {
    if (!describe(args[3], &cin)) return kNotPlain;
    ci = &cin;
  }
  Given given;
  if (!given.describe(args[5], *out)) return kNotPlain;
  const auto* epilogue = reinterpret_cast<const VecopsHipEpilogue*>(epilogue_address);
  const uint32_t how = static_cast<uint32_t>(compute);
  return without_lock([&]() -> int {
    VecopsHipPlan plan;
    int32_t rc = epilogue ? vecops_hip_plan_matmul_fused(&a, &b, ci, &c, how, epilogue, &plan) : vecops_hip_plan_matmul(&a, &b, ci, &c, how, &plan);
    if (rc != 0) return rc;
    const Workspace workspace(given, plan.slim_tile != 0 ? 0 : plan.workspace_bytes);
    return epilogue ? vecops_hip_matmul_fused(&a, &b, ci, &c, how, epilogue, workspace.data, workspace.size, current_stream())
                    : vecops_hip_matmul(&a, &b, ci, &c, how, workspace.data, workspace.size, current_stream());
  });
}

int matmul(PyObject* const* args) { return product(args, 0); }

// matmul_fused(a, b, c, c_in, compute, workspace, the epilogue record's address)
int matmul_fused(PyObject* const* args) {
  int64_t epilogue = 0;
  if (!integer(args[6], &epilogue) || epilogue == 0) return kNotPlain;
  return product(args, static_cast<uint64_t>(epilogue));
}

// Rank-2 tensors with contiguous rows, as the entry points on plain pointers take them.
const at::Tensor* matrix(PyObject* object) {
  const at::Tensor* t = plain_tensor(object);
  return t != nullptr && t->dim() == 2 && t->stride(1) == 1 ? t : nullptr;
}

// matmul_w8a16_group(x, w, scales, y, group)
int matmul_w8a16_group(PyObject* const* args) {
  const at::Tensor *x = matrix(args[0]), *w = matrix(args[1]), *scales = plain_tensor(args[2]), *y = matrix(args[3]);
  int64_t group = 0;
  if (x == nullptr || w == nullptr || scales == nullptr || y == nullptr || !scales->is_contiguous() || !integer(args[4], &group))
    return kNotPlain;
  const void* xv = x->data_ptr();
  const auto* wv = static_cast<const int8_t*>(w->data_ptr());
  const auto* sv = static_cast<const float*>(scales->data_ptr());
  void* yv = y->data_ptr();
  const int64_t ldx = x->stride(0), ldw = w->stride(0), ldy = y->stride(0), m = x->size(0), n = w->size(0), k = x->size(1);
  return without_lock([&] { return vecops_hip_matmul_w8a16_group(xv, ldx, wv, ldw, sv, yv, ldy, m, n, k, group, current_stream()); });
}

// matmul_i8_dequant(a, b or the packed storage, row_scales, column_scales, c, correction, workspace, n or -1): n < 0 says
// that b is the matrix itself
int matmul_i8_dequant(PyObject* const* args) {
  int64_t n = 0;
  if (!integer(args[7], &n)) return kNotPlain;
  const bool packed = n >= 0;
  const at::Tensor *a = matrix(args[0]), *b = packed ? plain_tensor(args[1]) : matrix(args[1]), *rows = plain_tensor(args[2]),
                   *columns = plain_tensor(args[3]), *c = matrix(args[4]), *correction = nullptr;
  if (a == nullptr || b == nullptr || rows == nullptr || columns == nullptr || c == nullptr) return kNotPlain;
  if (args[5] != Py_None && (correction = plain_tensor(args[5])) == nullptr) return kNotPlain;
  const int64_t m = a->size(0), k = a->size(1), lda = a->stride(0), ldb = packed ? 0 : b->stride(0), ldc = c->stride(0);
  if (!packed) n = b->size(0);
  Given given;
  if (!given.describe(args[6], *c)) return kNotPlain;
  const auto* av = static_cast<const int8_t*>(a->data_ptr());
  const void* bv = b->data_ptr();
  const auto *rv = static_cast<const float*>(rows->data_ptr()), *cv = static_cast<const float*>(columns->data_ptr());
  const auto* corr = correction ? static_cast<const int32_t*>(correction->data_ptr()) : nullptr;
  float* out = static_cast<float*>(c->data_ptr());
  return without_lock([&]() -> int {
    const Workspace workspace(given, vecops_hip_matmul_i8_dequant_workspace(m, n, k));
    return packed ? vecops_hip_matmul_i8_dequant_packed_b(av, lda, bv, rv, cv, corr, out, ldc, m, n, k, workspace.data,
                                                          workspace.size, current_stream())
                  : vecops_hip_matmul_i8_dequant(av, lda, static_cast<const int8_t*>(bv), ldb, rv, cv, corr, out, ldc, m, n, k,
                                                 workspace.data, workspace.size, current_stream());
  });
}

// matmul_runtime_quant(a, multipliers, zero_point, b or the packed storage, row_scales, column_scales, c, correction,
// workspace, n or -1)
int matmul_runtime_quant(PyObject* const* args) {
  int64_t n = 0, zero_point = 0;
  if (!integer(args[9], &n) || !integer(args[2], &zero_point) || zero_point < INT32_MIN || zero_point > INT32_MAX) return kNotPlain;
  const bool packed = n >= 0;
  VecopsHipOperand a, b, c;
  const at::Tensor *multipliers = plain_tensor(args[1]), *rows = plain_tensor(args[4]), *columns = plain_tensor(args[5]),
                   *out = plain_tensor(args[6]), *storage = plain_tensor(args[3]), *correction = nullptr;
  if (multipliers == nullptr || rows == nullptr || columns == nullptr || out == nullptr || storage == nullptr ||
      !describe(args[0], &a) || !describe(*out, &c) || (!packed && !describe(*storage, &b)))
    return kNotPlain;
  if (args[7] != Py_None && (correction = plain_tensor(args[7])) == nullptr) return kNotPlain;
  Given given;
  if (!given.describe(args[8], *out)) return kNotPlain;
  const auto *mv = static_cast<const float*>(multipliers->data_ptr()), *rv = static_cast<const float*>(rows->data_ptr()),
             *cv = static_cast<const float*>(columns->data_ptr());
  const auto* corr = correction ? static_cast<const int32_t*>(correction->data_ptr()) : nullptr;
  const int32_t zp = static_cast<int32_t>(zero_point);
  const void* weights = storage->data_ptr();
  return without_lock([&]() -> int {
    const Workspace workspace(given, packed ? vecops_hip_matmul_runtime_quant_packed_b_workspace(&a, n, &c)
                                            : vecops_hip_matmul_runtime_quant_workspace(&a, &b, &c));
    return packed ? vecops_hip_matmul_runtime_quant_packed_b(&a, mv, zp, weights, n, corr, rv, cv, &c, workspace.data,
                                                             workspace.size, current_stream())
                  : vecops_hip_matmul_runtime_quant(&a, mv, zp, &b, corr, rv, cv, &c, workspace.data, workspace.size, current_stream());
  });
}

// matmul_packed_b(a, storage, c, c_in, dtype, workspace, n)
int matmul_packed_b(PyObject* const* args) {
  VecopsHipOperand a, c, cin;
  int64_t dtype = 0, n = 0;
  const at::Tensor *storage = plain_tensor(args[1]), *out = plain_tensor(args[2]);
  if (storage == nullptr || out == nullptr || !describe(args[0], &a) || !describe(*out, &c) || !integer(args[4], &dtype) ||
      dtype < 0 || dtype > UINT32_MAX || !integer(args[6], &n))
    return kNotPlain;
  const VecopsHipOperand* ci = nullptr;
  if (args[3] != Py_None) {
    if (!describe(args[3], &cin)) return kNotPlain;
    ci = &cin;
  }
  Given given;
  if (!given.describe(args[5], *out)) return kNotPlain;
  const void* packed = storage->data_ptr();
  return without_lock([&]() -> int {
    VecopsHipPlan plan;
    int32_t rc = vecops_hip_plan_matmul_packed_b(&a, static_cast<uint32_t>(dtype), n, ci, &c, &plan);
    if (rc != 0) return rc;
    const Workspace workspace(given, plan.workspace_bytes);
    return vecops_hip_matmul_packed_b(&a, packed, static_cast<uint32_t>(dtype), n, ci, &c, workspace.data, workspace.size,
                                      current_stream());
  });
}

// A Python function of COUNT positional arguments around one of the above: no C++ exception leaves it.
template <int (*CALL)(PyObject* const*), int COUNT>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t count) {
  HANDLE_TH_ERRORS
  if (count != COUNT) {
    PyErr_Format(PyExc_TypeError, "expected %d arguments, got %zd", COUNT, count);
    return nullptr;
  }
  return PyLong_FromLong(CALL(args));
  END_HANDLE_TH_ERRORS
}

// ---- the device kernel of a registered operator -------------------------------------------------------------------

struct Parameter {
  enum Kind { kTensor, kInteger, kFloat } kind;
  bool output;
};
struct SpecializationName {
  std::string name;
  bool is_dtype;
};

// What a registration knows of its operator; the kernel below holds it for as long as the process runs.
struct Registered {
  uint64_t bridge = 0;               // the operator's handle with the process-local bridge
  void* host_operator = nullptr;     // the same operator, for its workspace query
  // the two entries of the host library that the operator came from (there may be several)
  decltype(&vecops_operator_bridge_invoke_v1) invoke = nullptr;
  decltype(&vecops_hip_host_operator_workspace) workspace = nullptr;
  std::vector<Parameter> parameters;
  std::vector<SpecializationName> specializations;
  bool return_outputs = false;
  PyObject* general = nullptr;       // the Python form: calls with host tensors or types outside the table
  PyObject* error = nullptr;         // HostError(code, message)
};

// Workspace sizes found for a thread's last call signatures (tensor kind, type, device, shape, strides, optional presence
// and specialization values, never addresses or scalar payloads).
constexpr size_t kPreparedCalls = 8;
using Signature = std::vector<int64_t>;
thread_local std::unordered_map<const Registered*, std::deque<std::pair<Signature, uint64_t>>> prepared;

class DeviceKernel final : public c10::OperatorKernel {
 public:
  explicit DeviceKernel(std::shared_ptr<const Registered> registered) : r_(std::move(registered)) {}

  void operator()(const c10::OperatorHandle&, c10::DispatchKeySet, torch::jit::Stack* stack) {
    const size_t tensors = r_->parameters.size(), count = tensors + r_->specializations.size();
    const size_t first = stack->size() - count;
    std::vector<VecopsValue> values(tensors);
    Signature signature;
    signature.reserve(8 * tensors + r_->specializations.size());
    const at::Tensor* on_device = nullptr;
    for (size_t i = 0; i < tensors; ++i) {
      const c10::IValue& arg = (*stack)[first + i];
      VecopsValue& v = values[i];
      memset(&v, 0, sizeof(v));
      v.struct_size = sizeof(v);
      const Parameter& p = r_->parameters[i];
      if (p.kind != Parameter::kTensor) {
        v.kind = VECOPS_VALUE_SCALAR;
        v.value.scalar.struct_size = sizeof(VecopsScalar);
        if (p.kind == Parameter::kInteger) {
          v.value.scalar.dtype = VECOPS_DTYPE_I64;
          v.value.scalar.value.i64 = arg.toInt();
        } else {
          v.value.scalar.dtype = VECOPS_DTYPE_F64;
          v.value.scalar.value.f64 = arg.toDouble();
        }
        signature.push_back(-2);
        continue;
      }
      if (arg.isNone()) {
        v.kind = VECOPS_VALUE_NONE;
        signature.push_back(-1);
        continue;
      }
      const at::Tensor& t = arg.toTensor();
      const uint32_t code = is_plain(t) ? dtype_code(t) : 0;
      if (code == 0 || code == VECOPS_DTYPE_F64) return general(stack, first);
      if (on_device == nullptr) on_device = &t;
      v.kind = VECOPS_VALUE_TENSOR;
      VecopsTensorView& view = v.value.tensor;
      view.struct_size = sizeof(view);
      view.data = t.data_ptr();
      view.device_type = VECOPS_DEVICE_PRIVATE;
      view.device_index = t.get_device();
      view.dtype = code;
      view.rank = static_cast<uint32_t>(t.dim());
      view.sizes = t.sizes().data();       // (the stack keeps the tensor until the call is over)
      view.strides = t.strides().data();
      view.flags = VECOPS_TENSOR_READ | (p.output ? VECOPS_TENSOR_WRITE : 0);
      signature.push_back(code);
      signature.push_back(view.device_index);
      signature.push_back(t.dim());
      signature.insert(signature.end(), t.sizes().begin(), t.sizes().end());
      signature.insert(signature.end(), t.strides().begin(), t.strides().end());
    }
    if (on_device == nullptr) return general(stack, first);
    std::vector<VecopsSpecializationArgument> bridge_specs;
    std::vector<VecopsHostSpecialization> host_specs;
    for (size_t i = 0; i < r_->specializations.size(); ++i) {
      const int64_t value = (*stack)[first + tensors + i].toInt();
      signature.push_back(value);
      if (value == -1) continue;   // not given
      const SpecializationName& s = r_->specializations[i];
      VecopsSpecializationArgument a;
      memset(&a, 0, sizeof(a));
      a.struct_size = sizeof(a);
      a.name = s.name.c_str();
      if (s.is_dtype) {
        a.kind = VECOPS_SPECIALIZATION_DTYPE;
        a.value.dtype = static_cast<uint32_t>(value);
      } else {
        a.kind = VECOPS_SPECIALIZATION_CONST_INT;
        a.value.integer = value;
      }
      bridge_specs.push_back(a);
      host_specs.push_back({s.name.c_str(), s.is_dtype ? 1 : 0, value});
    }
    char message[1024] = "";
    const c10::Device device = on_device->device();
    const uint64_t need = workspace_size(signature, values, host_specs, message);
    at::Tensor scratch;
    if (need > 0) scratch = at::empty({static_cast<int64_t>(need)}, at::TensorOptions().dtype(at::kByte).device(device));
    VecopsExecutionContext context;
    memset(&context, 0, sizeof(context));
    context.struct_size = sizeof(context);
    context.stream = c10::hip::getCurrentHIPStream(device.index()).stream();
    context.flags = VECOPS_HIP_CONTEXT_STREAM_ORDERED;   // (every tensor lives on the device)
    VecopsCall call;
    memset(&call, 0, sizeof(call));
    call.struct_size = sizeof(call);
    call.num_values = static_cast<uint32_t>(tensors);
    call.values = values.data();
    call.workspace = need > 0 ? scratch.data_ptr() : nullptr;
    call.workspace_size = need;
    call.context = &context;
    VecopsError error;
    memset(&error, 0, sizeof(error));
    error.struct_size = sizeof(error);
    error.message = message;
    error.message_capacity = sizeof(message);
    const int32_t rc = r_->invoke(r_->bridge, &call, static_cast<uint32_t>(bridge_specs.size()), bridge_specs.data(), &error);
    if (rc != 0) fail(rc, message);
    std::vector<c10::IValue> outputs;
    if (r_->return_outputs)
      for (size_t i = 0; i < tensors; ++i)
        if (r_->parameters[i].output) outputs.push_back((*stack)[first + i]);
    torch::jit::drop(*stack, count);
    for (c10::IValue& v : outputs) stack->push_back(std::move(v));
  }

 private:
  std::shared_ptr<const Registered> r_;

  uint64_t workspace_size(const Signature& signature, const std::vector<VecopsValue>& values,
                          const std::vector<VecopsHostSpecialization>& specs, char (&message)[1024]) const {
    auto& known = prepared[r_.get()];
    for (const auto& entry : known)
      if (entry.first == signature) return entry.second;
    uint64_t need = 0;
    const int32_t rc = r_->workspace(r_->host_operator, values.data(), static_cast<uint32_t>(values.size()), specs.data(),
                                     static_cast<uint32_t>(specs.size()), &need, message, sizeof(message));
    if (rc != 0) fail(rc, message);
    if (known.size() >= kPreparedCalls) known.pop_front();
    known.emplace_back(signature, need);
    return need;
  }

  [[noreturn]] void fail(int32_t code, const char* message) const {
    pybind11::gil_scoped_acquire gil;
    pybind11::object error = pybind11::reinterpret_borrow<pybind11::object>(r_->error)(code, message);
    PyErr_SetObject(r_->error, error.ptr());
    throw python_error();
  }

  // The call through the Python form, which takes host tensors too.
  void general(torch::jit::Stack* stack, size_t first) const {
    pybind11::gil_scoped_acquire gil;
    const size_t tensors = r_->parameters.size(), specs = r_->specializations.size();
    pybind11::tuple args(tensors);
    for (size_t i = 0; i < tensors; ++i) args[i] = torch::jit::toPyObject((*stack)[first + i]);
    pybind11::dict named;
    for (size_t i = 0; i < specs; ++i)
      named[pybind11::str(r_->specializations[i].name)] = (*stack)[first + tensors + i].toInt();
    pybind11::reinterpret_borrow<pybind11::object>(r_->general)(*args, **named);
    std::vector<c10::IValue> outputs;
    if (r_->return_outputs)
      for (size_t i = 0; i < tensors; ++i)
        if (r_->parameters[i].output) outputs.push_back((*stack)[first + i]);
    torch::jit::drop(*stack, tensors + specs);
    for (c10::IValue& v : outputs) stack->push_back(std::move(v));
  }
};

// register_device_kernel(library, name, bridge handle, host operator, the addresses of the host library's bridge entry and
// workspace query, parameter kinds, specializations, return_outputs, general form, error class): gives the operator, defined before, its kernel for device tensors.
void register_device_kernel(const std::string& library, const std::string& name, uint64_t bridge, uint64_t host_operator, uint64_t invoke,
                            uint64_t workspace, const std::vector<std::string>& kinds, const std::vector<std::pair<std::string, std::string>>& specs,
                            bool return_outputs, pybind11::object general, pybind11::object error) {
  auto r = std::make_shared<Registered>();
  r->bridge = bridge;
  r->host_operator = reinterpret_cast<void*>(host_operator);
  r->invoke = reinterpret_cast<decltype(r->invoke)>(invoke);
  r->workspace = reinterpret_cast<decltype(r->workspace)>(workspace);
  for (const std::string& kind : kinds)
    r->parameters.push_back({kind == "int" ? Parameter::kInteger : kind == "float" ? Parameter::kFloat : Parameter::kTensor,
                             kind == "out" || kind == "out?"});
  for (const auto& s : specs) r->specializations.push_back({s.first, s.second == "dtype"});
  r->return_outputs = return_outputs;
  r->general = general.release().ptr();   // (kept, like the registration, until the process ends)
  r->error = error.release().ptr();
  // registrations stay until the process ends: nothing is unregistered while other libraries are torn down
  auto* fragment = new torch::Library(torch::Library::FRAGMENT, library, std::nullopt, __FILE__, __LINE__);
  fragment->impl(name.c_str(), torch::dispatch(c10::DispatchKey::CUDA,
                                               torch::CppFunction::makeFromBoxedFunctor(std::make_unique<DeviceKernel>(std::move(r)))));
}

#define VECOPS_ENTRY(NAME, COUNT) \
  {#NAME, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<NAME, COUNT>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {VECOPS_ENTRY(matmul, 6),
                         VECOPS_ENTRY(matmul_fused, 7),
                         VECOPS_ENTRY(matmul_w8a16_group, 5),
                         VECOPS_ENTRY(matmul_i8_dequant, 8),
                         VECOPS_ENTRY(matmul_runtime_quant, 10),
                         VECOPS_ENTRY(matmul_packed_b, 7),
                         {nullptr, nullptr, 0, nullptr}};

}  // namespace

PYBIND11_MODULE(vecops_torch_calls, module) {
  module.def("register_device_kernel", &register_device_kernel);
  if (PyModule_AddFunctions(module.ptr(), methods) != 0) throw pybind11::error_already_set();
}
