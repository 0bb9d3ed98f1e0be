// Native call paths of the packed-weight operators.
//
// torch.ops.quantized.linear(x, packed, scale, zero_point) reaches the dispatcher
// through PyTorch's generic operator callable.  For an operator with a packed-weight
// object among its arguments that callable walks the arguments in Python and then
// converts the object through its script-class machinery: 9.7 us per call, measured
// with an operator that does nothing, against 0.55 us without the object and 2.3 us
// for a kernel launch.  The functions here take the same positional arguments, unwrap
// them directly and call the operator's typed dispatcher handle, so everything below
// the argument conversion (dispatch keys and modes, profiler records, autograd keys)
// is unchanged.
//
// A call that is not of the plain form -- keywords, another number of arguments,
// tensor subclasses, a torch-function mode, tracing, stand-in objects of the export
// machinery, numbers of other types -- goes to PyTorch's own callable, which is kept
// as `self` of the function, and has its results and its errors.  Some of PyTorch's modules
// are among those: quantized.dynamic.Linear passes reduce_range by name, QFunctional.add its
// scale and zero point.
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/api/object.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/pybind.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <ATen/native/quantized/PackedParams.h>

#include <cstring>
#include <optional>

namespace {

using LinearPtr = c10::intrusive_ptr<LinearPackedParamsBase>;
using ConvPtr = c10::intrusive_ptr<ConvPackedParamsBase<2>>;

PyTypeObject* g_script_object = nullptr;  // torch.ScriptObject

// Argument conversions: false where the plain form does not hold.
bool take(PyObject* o, at::Tensor* out) {
  // exactly torch.Tensor: subclasses may override the call
  if (reinterpret_cast<PyObject*>(Py_TYPE(o)) != THPVariableClass) return false;
  *out = THPVariable_Unpack(o);
  return true;
}
bool take(PyObject* o, double* out) {
  if (!PyFloat_CheckExact(o)) return false;
  *out = PyFloat_AS_DOUBLE(o);
  return true;
}
bool take(PyObject* o, int64_t* out) {
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  *out = PyLong_AsLongLongAndOverflow(o, &overflow);
  return overflow == 0;
}
bool take(PyObject* o, bool* out) {
  if (!PyBool_Check(o)) return false;
  *out = o == Py_True;
  return true;
}
bool take(PyObject* o, std::optional<at::Tensor>* out) {
  if (o == Py_None) {
    out->reset();
    return true;
  }
  at::Tensor t;
  if (!take(o, &t)) return false;
  *out = std::move(t);
  return true;
}
bool take(PyObject* o, std::optional<at::ScalarType>* out) {
  if (o == Py_None) {
    out->reset();
    return true;
  }
  if (!THPDtype_Check(o)) return false;
  *out = reinterpret_cast<THPDtype*>(o)->scalar_type;
  return true;
}
bool take(PyObject* o, c10::string_view* out) {  // a view into the string object, which the caller holds
  if (!PyUnicode_CheckExact(o)) return false;
  Py_ssize_t n = 0;
  const char* s = PyUnicode_AsUTF8AndSize(o, &n);
  if (s == nullptr) {
    PyErr_Clear();
    return false;
  }
  *out = c10::string_view(s, static_cast<size_t>(n));
  return true;
}
// The argument lists of post operations: only empty ones come this way.
struct NoScalars {
  torch::List<std::optional<at::Scalar>> list;
};
bool take(PyObject* o, NoScalars*) { return PyList_CheckExact(o) && PyList_GET_SIZE(o) == 0; }
template <typename T>
T& passed(T& v) { return v; }
torch::List<std::optional<at::Scalar>>& passed(NoScalars& v) { return v.list; }
template <typename Base>
bool take(PyObject* o, c10::intrusive_ptr<Base>* out) {
  if (Py_TYPE(o) != g_script_object) return false;
  const auto& held = py::cast<const torch::jit::Object&>(py::handle(o));
  const c10::IValue value(held._ivalue());
  static const auto type = c10::getCustomClassType<c10::intrusive_ptr<Base>>();
  if (*value.type() != *type) return false;
  *out = value.toCustomClass<Base>();
  return true;
}

template <typename... A, size_t... I>
bool take_all(PyObject* const* args, std::tuple<A...>* out, std::index_sequence<I...>) {
  return (take(args[I], &std::get<I>(*out)) && ...);
}

// One operator: `Values` are what its positional arguments convert to, `Sig` its registered
// C++ signature, `required` how many of them have no default (false is the only default here).
template <int ID, typename Sig, typename... Values>
struct Op {
  static std::optional<c10::TypedOperatorHandle<Sig>> handle;
  static Py_ssize_t required;
  static PyObject* call(PyObject* self, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
    HANDLE_TH_ERRORS
    constexpr Py_ssize_t kCount = sizeof...(Values);
    std::tuple<Values...> v{};
    if ((kwnames == nullptr || PyTuple_GET_SIZE(kwnames) == 0) && nargs <= kCount && nargs >= required &&
        !at::impl::torch_function_mode_enabled() && !torch::jit::tracer::isTracing()) {
      PyObject* filled[kCount];
      for (Py_ssize_t i = 0; i < kCount; ++i) filled[i] = i < nargs ? args[i] : Py_False;
      if (take_all(filled, &v, std::index_sequence_for<Values...>())) {
        at::Tensor result;
        {
          py::gil_scoped_release no_gil;
          result = std::apply([](auto&&... a) { return handle->call(passed(a)...); }, v);
        }
        return THPVariable_Wrap(std::move(result));
      }
    }
    return PyObject_Vectorcall(self, args, static_cast<size_t>(nargs), kwnames);
    END_HANDLE_TH_ERRORS
  }
  static PyObject* make(const char* name, const char* overload, Py_ssize_t need, PyMethodDef* def, PyObject* fallback) {
    handle = c10::Dispatcher::singleton().findSchemaOrThrow(name, overload).typed<Sig>();
    required = need;
    def->ml_meth = reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&call));
    def->ml_flags = METH_FASTCALL | METH_KEYWORDS;
    return PyCFunction_NewEx(def, fallback, nullptr);
  }
};
template <int ID, typename Sig, typename... Values>
std::optional<c10::TypedOperatorHandle<Sig>> Op<ID, Sig, Values...>::handle;
template <int ID, typename Sig, typename... Values>
Py_ssize_t Op<ID, Sig, Values...>::required = 0;

template <int ID>
using LinearOp = Op<ID, at::Tensor(at::Tensor, const LinearPtr&, double, int64_t), at::Tensor, LinearPtr, double, int64_t>;
template <int ID>
using DynamicOp = Op<ID, at::Tensor(at::Tensor, const LinearPtr&, bool), at::Tensor, LinearPtr, bool>;
template <int ID>
using ConvOp = Op<ID, at::Tensor(at::Tensor, const ConvPtr&, double, int64_t), at::Tensor, ConvPtr, double, int64_t>;
template <int ID>
using ConvAddOp = Op<ID, at::Tensor(at::Tensor, at::Tensor, const ConvPtr&, double, int64_t), at::Tensor, at::Tensor,
                     ConvPtr, double, int64_t>;
template <int ID>
using AddOp = Op<ID, at::Tensor(at::Tensor, at::Tensor, double, int64_t), at::Tensor, at::Tensor, double, int64_t>;

template <int ID>
using PlainLinearOp =
    Op<ID,
       at::Tensor(at::Tensor, double, int64_t, at::Tensor, at::Tensor, at::Tensor, std::optional<at::Tensor>, double,
                  int64_t, std::optional<at::ScalarType>, c10::string_view, torch::List<std::optional<at::Scalar>>,
                  c10::string_view),
       at::Tensor, double, int64_t, at::Tensor, at::Tensor, at::Tensor, std::optional<at::Tensor>, double, int64_t,
       std::optional<at::ScalarType>, c10::string_view, NoScalars, c10::string_view>;

struct Entry {
  PyMethodDef def;
  const char* qualified;
  const char* overload;
  Py_ssize_t required;
  PyObject* (*make)(const char*, const char*, Py_ssize_t, PyMethodDef*, PyObject*);
};
Entry g_entries[] = {
    {{"linear"}, "quantized::linear", "", 4, &LinearOp<0>::make},
    {{"linear_relu"}, "quantized::linear_relu", "", 4, &LinearOp<1>::make},
    {{"linear_dynamic"}, "quantized::linear_dynamic", "", 2, &DynamicOp<2>::make},
    {{"linear_relu_dynamic"}, "quantized::linear_relu_dynamic", "", 2, &DynamicOp<3>::make},
    {{"conv2d"}, "quantized::conv2d", "new", 4, &ConvOp<4>::make},
    {{"conv2d_relu"}, "quantized::conv2d_relu", "new", 4, &ConvOp<5>::make},
    {{"conv2d_silu"}, "quantized::conv2d_silu", "new", 4, &ConvOp<6>::make},
    {{"conv1d"}, "quantized::conv1d", "", 4, &ConvOp<7>::make},
    {{"conv1d_relu"}, "quantized::conv1d_relu", "", 4, &ConvOp<8>::make},
    {{"conv2d_add"}, "quantized::conv2d_add", "", 5, &ConvAddOp<9>::make},
    {{"conv2d_add_relu"}, "quantized::conv2d_add_relu", "", 5, &ConvAddOp<10>::make},
    {{"conv2d_add_silu"}, "quantized::conv2d_add_silu", "", 5, &ConvAddOp<11>::make},
    {{"add"}, "quantized::add", "", 4, &AddOp<12>::make},
    {{"add_relu"}, "quantized::add_relu", "", 4, &AddOp<13>::make},
    {{"linear_per_tensor"}, "quantized::linear_per_tensor", "", 13, &PlainLinearOp<14>::make},
};

// make(name, fallback) -> the native callable of quantized::<name>; `fallback` takes the same arguments
PyObject* make(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  const char* name = nullptr;
  PyObject* fallback = nullptr;
  if (!PyArg_ParseTuple(args, "sO", &name, &fallback)) return nullptr;
  for (Entry& e : g_entries)
    if (std::strcmp(e.def.ml_name, name) == 0) return e.make(e.qualified, e.overload, e.required, &e.def, fallback);
  PyErr_Format(PyExc_KeyError, "no native call path for quantized::%s", name);
  return nullptr;
  END_HANDLE_TH_ERRORS
}
PyObject* names(PyObject*, PyObject*) {
  PyObject* list = PyList_New(0);
  for (const Entry& e : g_entries) {
    PyObject* s = PyUnicode_FromString(e.def.ml_name);
    PyList_Append(list, s);
    Py_DECREF(s);
  }
  return list;
}

PyMethodDef g_methods[] = {{"make", make, METH_VARARGS, nullptr},
                           {"names", names, METH_NOARGS, nullptr},
                           {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_fastcall", nullptr, -1, g_methods};

}  // namespace

PyMODINIT_FUNC PyInit__fastcall() {
  PyObject* torch = PyImport_ImportModule("torch");
  if (torch == nullptr) return nullptr;
  PyObject* type = PyObject_GetAttrString(torch, "ScriptObject");
  Py_DECREF(torch);
  if (type == nullptr) return nullptr;
  g_script_object = reinterpret_cast<PyTypeObject*>(type);  // kept for the life of the process
  return PyModule_Create(&g_module);
}
