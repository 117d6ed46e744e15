// The host side of the flow._C functions: argument checks, output and workspace tensors, the
// current stream and the call into the C ABI, for torch tensors, as a CPython extension module.
//
// Why it is native: a decode-sized kernel takes 3 to 6 us, and the same steps written in Python
// (checks, torch.empty, torch.cuda.current_stream, a ctypes call with 18 arguments) took 13 us a
// call, so a loop of such calls was bound by the interpreter.  Here a call is its checks
// (< 0.2 us), one allocation per output from the caching allocator and the launch itself
// (2.3 us in the HIP runtime, which is then what bounds back-to-back small calls).
//
// Functions take positional arguments only: names, defaults and documentation live in
// functional.py, which forwards to them.  The checks and their messages are those of the
// reference functors (oneflow/core/functional/impl/quantization.cpp:34-372); a failed one raises
// functional.CheckFailedError, a non-zero ofq_status raises _lib.OfqError.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/DynamicTypes.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>

#include <string>
#include <vector>

#include "ofq.h"

namespace {

using at::ScalarType;
using at::Tensor;

PyObject* check_failed_error = nullptr;  // functional.CheckFailedError
PyObject* ofq_error = nullptr;           // _lib.OfqError(fn, status, text)

// ---- errors -------------------------------------------------------------------------------------
struct CheckFailed {
  std::string msg;
};
struct StatusFailed {
  const char* fn;
  int status;
};
struct PythonError {};  // already set

#define OFQ_CHECK(cond, ...)                               \
  do {                                                 \
    if (__builtin_expect(!(cond), 0)) throw CheckFailed{(__VA_ARGS__)}; \
  } while (0)

inline std::string str(int64_t v) { return std::to_string(v); }

std::string dtype_name(ScalarType t) {
  return std::string("torch.") + torch::getTHPDtype(t)->name;
}

// ---- arguments ----------------------------------------------------------------------------------
const Tensor& tensor_arg(PyObject* o, const char* name) {
  if (!THPVariable_Check(o)) {
    PyErr_Format(PyExc_TypeError, "%s should be a tensor, not %s", name, Py_TYPE(o)->tp_name);
    throw PythonError{};
  }
  return THPVariable_Unpack(o);
}

// an undefined tensor for None
const Tensor& optional_arg(PyObject* o, const char* name) {
  static const Tensor none;
  return o == Py_None ? none : tensor_arg(o, name);
}

int64_t int_arg(PyObject* o) {
  const int64_t v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) throw PythonError{};
  return v;
}

double double_arg(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw PythonError{};
  return v;
}

bool bool_arg(PyObject* o) {
  const int v = PyObject_IsTrue(o);
  if (v < 0) throw PythonError{};
  return v != 0;
}

// a str's text; "" (which no table holds) for anything else
const char* text_arg(PyObject* o) {
  if (!PyUnicode_Check(o)) return "";
  const char* s = PyUnicode_AsUTF8(o);
  if (s == nullptr) throw PythonError{};
  return s;
}

inline bool same(const char* a, const char* b) { return strcmp(a, b) == 0; }

ScalarType dtype_arg(PyObject* o) {
  if (!THPDtype_Check(o)) {
    PyErr_Format(PyExc_TypeError, "a torch.dtype is expected, not %s", Py_TYPE(o)->tp_name);
    throw PythonError{};
  }
  return reinterpret_cast<THPDtype*>(o)->scalar_type;
}

int code_of(ScalarType t) {
  switch (t) {
    case at::kFloat: return OFQ_F32;
    case at::kHalf: return OFQ_F16;
    case at::kBFloat16: return OFQ_BF16;
    case at::kDouble: return OFQ_F64;
    case at::kChar: return OFQ_I8;
    case at::kByte: return OFQ_U8;
    default: throw CheckFailed{"unsupported dtype " + dtype_name(t)};
  }
}
inline int code_of(const Tensor& t) { return code_of(t.scalar_type()); }

inline bool is_code_dtype(const Tensor& t) {
  return t.scalar_type() == at::kChar || t.scalar_type() == at::kByte;
}
inline bool is_linear_dtype(ScalarType t) {
  return t == at::kHalf || t == at::kFloat || t == at::kBFloat16;
}

template<typename... Ts>
void require_gpu(const Ts&... ts) {
  OFQ_CHECK(((!ts.defined() || ts.is_cuda()) && ...),
        "tensors must live on the GPU: this build has no CPU kernels");
}

inline void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

// The runtime hands kernels contiguous inputs (op_interpreter_util.cpp:156) in buffers of its own
// allocator (512-byte aligned); a view that starts off a 16-byte boundary is copied, since the
// kernels use 128-bit accesses.  `hold` keeps a copy alive until the launch has been enqueued.
const Tensor& contig(const Tensor& t, Tensor& hold) {
  if (!t.defined()) return t;
  if (__builtin_expect(t.is_contiguous(), 1)) {
    if (__builtin_expect((reinterpret_cast<uintptr_t>(t.data_ptr()) & 15u) == 0, 1)) return t;
    hold = t.clone();
    return hold;
  }
  hold = t.contiguous();
  return hold;
}

Tensor empty(at::IntArrayRef size, ScalarType dtype, const Tensor& like) {
  return Tensor(at::detail::empty_cuda(size, dtype, like.device(), std::nullopt));
}

// workspaces come from torch's caching allocator: stream-ordered, shared with every other tensor
// of the program, returned to it when the call is over
Tensor workspace(size_t nbytes, const Tensor& like) {
  return empty({(int64_t)(nbytes < 16 ? 16 : nbytes)}, at::kByte, like);
}

inline void* stream_of(const Tensor& t) {
  return c10::hip::getCurrentHIPStream(t.get_device()).stream();
}

// A call into the library.  The interpreter lock is released, since a launch waits when the stream's
// queue is full.  The arguments are evaluated before that: taking a tensor's pointer can throw (a
// tensor of a function transform has no storage), and the error has to be set under the lock.
class Unlocked {
 public:
  Unlocked() : save_(PyEval_SaveThread()) {}
  ~Unlocked() { PyEval_RestoreThread(save_); }
  Unlocked(const Unlocked&) = delete;

 private:
  PyThreadState* save_;
};

template<typename... Params, typename... Args>
int unlocked(int (*fn)(Params...), Args... args) {
  const Unlocked released;
  return fn(args...);
}

void check_status(const char* fn, int st) {
  if (__builtin_expect(st != OFQ_OK, 0)) throw StatusFailed{fn, st};
}

PyObject* wrap(Tensor&& t) { return THPVariable_Wrap(std::move(t)); }

PyObject* tuple_of(PyObject* a, PyObject* b, PyObject* c = nullptr) {
  PyObject* t = PyTuple_New(c == nullptr ? 2 : 3);
  PyTuple_SET_ITEM(t, 0, a);
  PyTuple_SET_ITEM(t, 1, b);
  if (c != nullptr) PyTuple_SET_ITEM(t, 2, c);
  return t;
}

PyObject* none() { return Py_NewRef(Py_None); }

// every entry: argument count, C++ exceptions -> Python exceptions
template<int N, PyObject* (*BODY)(PyObject* const*)>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != N) {
    PyErr_Format(PyExc_TypeError, "%d positional arguments are expected, %zd were given", N, nargs);
    return nullptr;
  }
  try {
    return BODY(args);
  } catch (const CheckFailed& e) {
    PyErr_SetString(check_failed_error, e.msg.c_str());
  } catch (const StatusFailed& e) {
    PyObject* err = PyObject_CallFunction(ofq_error, "sis", e.fn, e.status,
                                          ofq_status_string(e.status));
    if (err != nullptr) {
      PyErr_SetObject(ofq_error, err);
      Py_DECREF(err);
    }
  } catch (const PythonError&) {
  } catch (python_error& e) {
    e.restore();
  } catch (const c10::Error& e) {
    // out of memory and the like: torch's own exception types
    torch::translate_exception_to_python(std::current_exception());
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
  }
  return nullptr;
}

// ---- groupwise_dequantize: GroupwiseDequantizeFunctor, quantization.cpp:155-220 -----------------
// (in, scale, zero, num_bits, symmetric, group_dim, group_size)
PyObject* groupwise_dequantize(PyObject* const* args) {
  const Tensor& in = tensor_arg(args[0], "in");
  const Tensor& scale = tensor_arg(args[1], "scale");
  const Tensor& zero = optional_arg(args[2], "zero");
  const int64_t num_bits = int_arg(args[3]);
  const bool symmetric = bool_arg(args[4]);
  const int64_t group_dim = int_arg(args[5]);
  const int64_t group_size = int_arg(args[6]);
  OFQ_CHECK(num_bits == 4 || num_bits == 8, "num_bits should be 4 or 8.");
  const int64_t nd = in.dim();
  OFQ_CHECK(nd >= 1, "The number of dimensions for tensor in should be greater than or equal to 1.");
  const int64_t gd = group_dim < 0 ? nd + group_dim : group_dim;
  OFQ_CHECK(0 <= gd && gd < nd, "group_dim should be in range [-" + str(nd) + "," + str(nd) + ").");
  const int64_t per = 8 / num_bits;
  const int64_t dim_size = in.size(gd) * (gd == nd - 1 ? per : 1);
  const int64_t gs = group_size < 0 ? dim_size : group_size;
  OFQ_CHECK(0 < gs && gs <= dim_size, "group_size should be in range (0," + str(dim_size) + "].");
  OFQ_CHECK(dim_size % gs == 0, "group_size should be a divisor of " + str(dim_size) + ".");
  const int64_t num_groups = dim_size / gs;
  if (symmetric) {
    OFQ_CHECK(is_code_dtype(in), "The dtype of tensor in should be int8 or uint8.");
  } else {
    OFQ_CHECK(in.scalar_type() == at::kByte, "The dtype of tensor in should be uint8.");
  }
  OFQ_CHECK(scale.dim() == nd,
        "The number of dimensions of tensor scale should be equal to tensor in.");
  for (int64_t i = 0; i < nd; ++i) {
    if (i == gd) {
      OFQ_CHECK(scale.size(i) == num_groups, "The size of the " + str(i)
            + "-th dimension of tensor scale should be equal to " + str(num_groups));
    } else if (i == nd - 1) {
      OFQ_CHECK(scale.size(i) == in.size(i) * per, "The size of the " + str(i)
            + "-th dimension of tensor scale should be equal to " + str(in.size(i) * per) + ".");
    } else {
      OFQ_CHECK(scale.size(i) == in.size(i), "The size of the " + str(i)
            + "-th dimension of tensor scale should be equal to tensor in.");
    }
  }
  if (!symmetric) {
    OFQ_CHECK(zero.defined(), "When symmetric is False, tensor zero should be specified.");
    OFQ_CHECK(zero.scalar_type() == scale.scalar_type(),
          "The dtype of the zero tensor should be the same as the scale tensor.");
    OFQ_CHECK(zero.sizes() == scale.sizes(), "The shape of zero tensor should be equal to tensor scale.");
  } else {
    OFQ_CHECK(!zero.defined(), "When symmetric is True, tensor zero should be None.");
  }
  // kernels are registered on the dtype of scale (groupwise_quantization_kernels.cu:456-463);
  // bf16 is added here
  OFQ_CHECK(is_linear_dtype(scale.scalar_type()),
        "no groupwise_dequantize kernel for scale dtype " + dtype_name(scale.scalar_type()));
  require_gpu(in, scale, zero);
  Tensor h0, h1, h2;
  const Tensor& i_ = contig(in, h0);
  const Tensor& s_ = contig(scale, h1);
  const Tensor& z_ = contig(zero, h2);
  at::DimVector shape(in.sizes().begin(), in.sizes().end());
  shape.back() *= per;
  Tensor out = empty(shape, scale.scalar_type(), in);
  int64_t outer = num_groups, inner = 1;
  for (int64_t d = 0; d < gd; ++d) outer *= shape[d];
  for (int64_t d = gd + 1; d < nd; ++d) inner *= shape[d];
  void* st = stream_of(in);
  check_status("ofq_groupwise_dequantize", unlocked(
      ofq_groupwise_dequantize, st, ptr(i_), ptr(s_), ptr(z_), ptr(out), code_of(i_), code_of(s_),
      (int)num_bits, symmetric, outer, gs, inner));
  return wrap(std::move(out));
}

// ---- fused linear: FusedLinearWithGroupwiseQuantizedWeightFunctor, quantization.cpp:264-372 -----
struct LinearDims {
  int64_t m, n, k;
  int64_t gd, gs;
};

LinearDims check_linear(const Tensor& x, const Tensor& w, const Tensor& w_scale,
                        const Tensor& w_zero, const Tensor& b, int64_t num_bits, bool symmetric,
                        int64_t group_dim, int64_t group_size) {
  LinearDims d;
  OFQ_CHECK(x.dim() >= 2,
        "The number of dimensions for tensor x should be greater than or equal to 2.");
  d.k = x.size(-1);
  d.m = d.k != 0 ? x.numel() / d.k : 0;
  OFQ_CHECK(num_bits == 4 || num_bits == 8, "num_bits should be 4 or 8.");
  OFQ_CHECK(w.dim() == 2, "The number of dimensions for tensor w should be equal to 2.");
  const int64_t per = 8 / num_bits;
  OFQ_CHECK(d.k % per == 0, "The size of the last dimension of x should be a multiple of (8/num_bits).");
  OFQ_CHECK(w.size(1) == d.k / per,
        "The size of second dimension of tensor w should be equal to " + str(d.k / per));
  d.n = w.size(0);
  d.gd = group_dim < 0 ? 2 + group_dim : group_dim;
  OFQ_CHECK(d.gd == 0 || d.gd == 1, "group_dim should be in range [-2,2).");
  const int64_t dim_size = d.gd == 0 ? d.n : d.k;
  d.gs = group_size < 0 ? dim_size : group_size;
  OFQ_CHECK(0 < d.gs && d.gs <= dim_size, "group_size should be in range (0," + str(dim_size) + "].");
  OFQ_CHECK(dim_size % d.gs == 0, "group_size should be a divisor of " + str(dim_size) + ".");
  const int64_t num_groups = dim_size / d.gs;
  if (symmetric) {
    OFQ_CHECK(is_code_dtype(w), "The dtype of tensor w should be int8 or uint8.");
  } else {
    OFQ_CHECK(w.scalar_type() == at::kByte, "The dtype of tensor w should be uint8.");
  }
  OFQ_CHECK(w_scale.dim() == 2,
        "The number of dimensions of tensor w_scale should be equal to 2.");
  for (int64_t i = 0; i < 2; ++i) {
    if (i == d.gd) {
      OFQ_CHECK(w_scale.size(i) == num_groups, "The size of the " + str(i)
            + "-th dimension of tensor w_scale should be equal to " + str(num_groups));
    } else if (i == 1) {
      OFQ_CHECK(w_scale.size(i) == d.k, "The size of the " + str(i)
            + "-th dimension of tensor w_scale should be equal to " + str(d.k) + ".");
    } else {
      OFQ_CHECK(w_scale.size(i) == w.size(i), "The size of the " + str(i)
            + "-th dimension of tensor w_scale should be equal to tensor w.");
    }
  }
  OFQ_CHECK(w_scale.scalar_type() == x.scalar_type(),
        "The dtype of the w_scale tensor should be the same as the x tensor.");
  if (!symmetric) {
    OFQ_CHECK(w_zero.defined(), "When symmetric is False, tensor w_zero should be specified.");
    OFQ_CHECK(w_zero.scalar_type() == w_scale.scalar_type(),
          "The dtype of the w_zero tensor should be the same as the w_scale tensor.");
    OFQ_CHECK(w_zero.sizes() == w_scale.sizes(),
          "The shape of w_zero tensor should be equal to tensor w_scale.");
  } else {
    OFQ_CHECK(!w_zero.defined(), "When symmetric is True, tensor w_zero should be None.");
  }
  if (b.defined()) {
    OFQ_CHECK(b.scalar_type() == x.scalar_type(),
          "The dtype of the b tensor should be the same as the x tensor.");
    OFQ_CHECK(b.dim() == 1, "The number of dimensions for tensor b should be equal to 1.");
    OFQ_CHECK(b.size(0) == d.n,
          "The size of first dimension of tensor b should be equal to the size of first dimension "
          "of tensor w");
  }
  OFQ_CHECK(is_linear_dtype(x.scalar_type()),
        "no fused_linear_with_groupwise_quantized_weight kernel for dtype "
            + dtype_name(x.scalar_type()));
  return d;
}

// x.shape[:-1] + (n,)
at::DimVector linear_shape(const Tensor& x, int64_t n) {
  at::DimVector shape(x.sizes().begin(), x.sizes().end());
  shape.back() = n;
  return shape;
}

// (x, w, w_scale, w_zero, b, num_bits, symmetric, group_dim, group_size)
PyObject* fused_linear(PyObject* const* args) {
  const Tensor& x = tensor_arg(args[0], "x");
  const Tensor& w = tensor_arg(args[1], "w");
  const Tensor& w_scale = tensor_arg(args[2], "w_scale");
  const Tensor& w_zero = optional_arg(args[3], "w_zero");
  const Tensor& b = optional_arg(args[4], "b");
  const int num_bits = (int)int_arg(args[5]);
  const bool symmetric = bool_arg(args[6]);
  const LinearDims d = check_linear(x, w, w_scale, w_zero, b, num_bits, symmetric,
                                    int_arg(args[7]), int_arg(args[8]));
  require_gpu(x, w, w_scale, w_zero, b);
  Tensor h0, h1, h2, h3, h4;
  const Tensor& x_ = contig(x, h0);
  const Tensor& w_ = contig(w, h1);
  const Tensor& s_ = contig(w_scale, h2);
  const Tensor& z_ = contig(w_zero, h3);
  const Tensor& b_ = contig(b, h4);
  Tensor out = empty(linear_shape(x, d.n), x.scalar_type(), x);
  const int wd = code_of(w), td = code_of(x), gd = (int)d.gd;
  const size_t ws_bytes = ofq_fused_linear_gq_workspace_bytes(wd, td, num_bits, symmetric, gd, d.gs,
                                                              d.m, d.n, d.k);
  Tensor ws;
  if (ws_bytes != 0) ws = workspace(ws_bytes, x);
  void* st = stream_of(x);
  check_status("ofq_fused_linear_gq", unlocked(
      ofq_fused_linear_gq, st, ptr(x_), ptr(w_), ptr(s_), ptr(z_), ptr(b_), ptr(out), wd, td,
      num_bits, symmetric, gd, d.gs, d.m, d.n, d.k, ptr(ws), ws_bytes));
  return wrap(std::move(out));
}

// (w, num_bits)
PyObject* groupwise_repack(PyObject* const* args) {
  const Tensor& w = tensor_arg(args[0], "w");
  const int64_t num_bits = int_arg(args[1]);
  OFQ_CHECK(w.dim() == 2 && is_code_dtype(w), "w should be 2-D int8 / uint8 codes");
  OFQ_CHECK(num_bits == 4, "only 4-bit codes have a tile-major form");
  require_gpu(w);
  Tensor h0;
  const Tensor& w_ = contig(w, h0);
  const int64_t n = w.size(0), k = w.size(1) * 2;
  const size_t nbytes = ofq_groupwise_repack_bytes((int)num_bits, n, k);
  OFQ_CHECK(nbytes > 0, "no tile-major form for n=" + str(n) + ", k=" + str(k)
        + " (k should be a multiple of 128)");
  Tensor tiled = empty({(int64_t)nbytes}, w.scalar_type(), w);
  void* st = stream_of(w);
  check_status("ofq_groupwise_repack", unlocked(
      ofq_groupwise_repack, st, ptr(w_), ptr(tiled), (int)num_bits, n, k));
  return wrap(std::move(tiled));
}

// (x, w_tiled, w_scale, w_zero, b, num_bits, symmetric, group_dim, group_size)
PyObject* fused_linear_tiled(PyObject* const* args) {
  const Tensor& x = tensor_arg(args[0], "x");
  const Tensor& w_tiled = tensor_arg(args[1], "w_tiled");
  const Tensor& w_scale = tensor_arg(args[2], "w_scale");
  const Tensor& w_zero = optional_arg(args[3], "w_zero");
  const Tensor& b = optional_arg(args[4], "b");
  const int num_bits = (int)int_arg(args[5]);
  const bool symmetric = bool_arg(args[6]);
  const int64_t group_dim = int_arg(args[7]), group_size = int_arg(args[8]);
  OFQ_CHECK(x.dim() >= 1, "x should have at least one dimension");
  const int64_t k = x.size(-1);
  const int64_t m = k != 0 ? x.numel() / k : 0;
  OFQ_CHECK(w_scale.dim() >= 1, "w_scale should have at least one dimension");
  const int64_t n = w_scale.size(0);
  const int64_t gd = group_dim >= 0 ? group_dim : group_dim + 2;
  OFQ_CHECK(gd == 1, "the tile-major copy serves groups along K only");
  const int64_t gs = group_size >= 0 ? group_size : k;
  OFQ_CHECK(w_tiled.dim() == 1 && is_code_dtype(w_tiled),
        "w_tiled should be the flat tensor groupwise_repack returns");
  OFQ_CHECK(!w_zero.defined() == symmetric, "w_zero is given exactly when symmetric is False");
  require_gpu(x, w_tiled, w_scale, w_zero, b);
  OFQ_CHECK((size_t)w_tiled.numel() == ofq_groupwise_repack_bytes(num_bits, n, k),
        "w_tiled does not have the size of the tile-major copy of an [n, k] weight");
  Tensor h0, h2, h3, h4;
  const Tensor& x_ = contig(x, h0);
  const Tensor& s_ = contig(w_scale, h2);
  const Tensor& z_ = contig(w_zero, h3);
  const Tensor& b_ = contig(b, h4);
  Tensor out = empty(linear_shape(x, n), x.scalar_type(), x);
  const int wd = code_of(w_tiled), td = code_of(x);
  void* st = stream_of(x);
  check_status("ofq_fused_linear_gq_tiled", unlocked(
      ofq_fused_linear_gq_tiled, st, ptr(x_), ptr(w_tiled), ptr(s_), ptr(z_), ptr(b_), ptr(out),
      wd, td, num_bits, symmetric, 1, gs, m, n, k));
  return wrap(std::move(out));
}

// the items of a list or tuple argument (held by `fast`)
struct Sequence {
  PyObject* fast;
  explicit Sequence(PyObject* o) : fast(PySequence_Fast(o, "a sequence of tensors is expected")) {
    if (fast == nullptr) throw PythonError{};
  }
  ~Sequence() { Py_DECREF(fast); }
  Sequence(const Sequence&) = delete;
  int64_t size() const { return PySequence_Fast_GET_SIZE(fast); }
  PyObject* operator[](int64_t i) const { return PySequence_Fast_GET_ITEM(fast, i); }
};

// (xs, ws, w_scales, w_zeros | None, bs | None, num_bits, symmetric, group_dim, group_size)
PyObject* grouped_linear(PyObject* const* args) {
  constexpr int kMost = 64;
  Sequence xs(args[0]), ws(args[1]), w_scales(args[2]);
  const int64_t count = xs.size();
  OFQ_CHECK(count > 0, "xs should not be empty");
  OFQ_CHECK(count <= kMost, "at most 64 problems per call");
  OFQ_CHECK(ws.size() == count && w_scales.size() == count,
        "xs, ws and w_scales should have the same length");
  const bool zeros = args[3] != Py_None, biases = args[4] != Py_None;
  Sequence w_zeros(zeros ? args[3] : args[0]), bs(biases ? args[4] : args[0]);
  OFQ_CHECK(!zeros || w_zeros.size() == count, "w_zeros should have the length of xs");
  OFQ_CHECK(!biases || bs.size() == count, "bs should have the length of xs");
  const int num_bits = (int)int_arg(args[5]);
  const bool symmetric = bool_arg(args[6]);
  const int64_t group_dim = int_arg(args[7]), group_size = int_arg(args[8]);
  LinearDims dims[kMost];
  const auto z_at = [&](int64_t i) -> const Tensor& {
    return optional_arg(zeros ? w_zeros[i] : Py_None, "w_zeros");
  };
  const auto b_at = [&](int64_t i) -> const Tensor& {
    return optional_arg(biases ? bs[i] : Py_None, "bs");
  };
  for (int64_t i = 0; i < count; ++i) {
    dims[i] = check_linear(tensor_arg(xs[i], "xs"), tensor_arg(ws[i], "ws"),
                           tensor_arg(w_scales[i], "w_scales"), z_at(i), b_at(i), num_bits,
                           symmetric, group_dim, group_size);
  }
  const Tensor& x0 = THPVariable_Unpack(xs[0]);
  const Tensor& w0 = THPVariable_Unpack(ws[0]);
  for (int64_t i = 1; i < count; ++i) {
    OFQ_CHECK(THPVariable_Unpack(xs[i]).scalar_type() == x0.scalar_type()
              && THPVariable_Unpack(ws[i]).scalar_type() == w0.scalar_type(),
          "all problems should share the dtypes of x and w");
  }
  for (int64_t i = 1; i < count; ++i) {
    OFQ_CHECK(dims[i].gd == dims[0].gd && dims[i].gs == dims[0].gs,
          "all problems should share group_dim and group_size");
  }
  const void *px[kMost], *pw[kMost], *ps[kMost], *pz[kMost], *pb[kMost];
  void* po[kMost];
  int64_t ms[kMost], ns[kMost], ks[kMost];
  std::vector<Tensor> outs(count);
  std::vector<Tensor> hold;  // copies of inputs that were not contiguous
  const auto device_ptr = [&](const Tensor& t) -> const void* {
    Tensor h;
    const void* p = ptr(contig(t, h));
    if (h.defined()) hold.push_back(std::move(h));
    return p;
  };
  for (int64_t i = 0; i < count; ++i) {
    require_gpu(THPVariable_Unpack(xs[i]), THPVariable_Unpack(ws[i]),
                THPVariable_Unpack(w_scales[i]), z_at(i), b_at(i));
  }
  for (int64_t i = 0; i < count; ++i) {
    const Tensor& x = THPVariable_Unpack(xs[i]);
    px[i] = device_ptr(x);
    pw[i] = device_ptr(THPVariable_Unpack(ws[i]));
    ps[i] = device_ptr(THPVariable_Unpack(w_scales[i]));
    pz[i] = device_ptr(z_at(i));
    pb[i] = device_ptr(b_at(i));
    outs[i] = empty(linear_shape(x, dims[i].n), x.scalar_type(), x);
    po[i] = ptr(outs[i]);
    ms[i] = dims[i].m;
    ns[i] = dims[i].n;
    ks[i] = dims[i].k;
  }
  const int wd = code_of(w0), td = code_of(x0);
  void* st = stream_of(x0);
  check_status("ofq_grouped_linear_gq", unlocked(
      ofq_grouped_linear_gq, st, (int)count, px, pw, ps, symmetric ? nullptr : pz, pb, po, ms, ns,
      ks, wd, td, num_bits, symmetric, (int)dims[0].gd, dims[0].gs));
  PyObject* list = PyList_New(count);
  for (int64_t i = 0; i < count; ++i) PyList_SET_ITEM(list, i, wrap(std::move(outs[i])));
  return list;
}

int activation_code(const char* name) {
  if (same(name, "silu")) return OFQ_ACT_SILU;
  if (same(name, "none")) return OFQ_ACT_NONE;
  if (same(name, "sigmoid")) return OFQ_ACT_SIGMOID;
  if (same(name, "relu")) return OFQ_ACT_RELU;
  if (same(name, "gelu")) return OFQ_ACT_GELU;
  if (same(name, "fast_gelu")) return OFQ_ACT_FAST_GELU;
  throw CheckFailed{std::string("unsupported activation '") + name + "'"};
}

// FusedGluFunctor's rules (nn_functor.cpp:3724-3800)
// (x, w, w_scale, w_zero, b, v, v_scale, v_zero, c, activation, num_bits, symmetric, group_dim,
//  group_size)
PyObject* fused_glu(PyObject* const* args) {
  const Tensor& x = tensor_arg(args[0], "x");
  const Tensor& w = tensor_arg(args[1], "w");
  const Tensor& w_scale = tensor_arg(args[2], "w_scale");
  const Tensor& w_zero = optional_arg(args[3], "w_zero");
  const Tensor& b = optional_arg(args[4], "b");
  const Tensor& v = optional_arg(args[5], "v");
  const Tensor& v_scale = optional_arg(args[6], "v_scale");
  const Tensor& v_zero = optional_arg(args[7], "v_zero");
  const Tensor& c = optional_arg(args[8], "c");
  const int act = activation_code(text_arg(args[9]));
  const int num_bits = (int)int_arg(args[10]);
  const bool symmetric = bool_arg(args[11]);
  const int64_t group_dim = int_arg(args[12]), group_size = int_arg(args[13]);
  const bool split = v.defined();
  if (b.defined()) {
    OFQ_CHECK(!split || c.defined(), "expected existance of c, when provide tensors w, v and b");
  } else {
    OFQ_CHECK(!c.defined(), "expected existance of b while providing c");
  }
  const LinearDims d =
      check_linear(x, w, w_scale, w_zero, b, num_bits, symmetric, group_dim, group_size);
  int64_t n = d.n;
  if (split) {
    OFQ_CHECK(v_scale.defined(), "v_scale should be specified with v");
    OFQ_CHECK(v.sizes() == w.sizes() && v.scalar_type() == w.scalar_type(),
          "v should have the shape and dtype of w");
    check_linear(x, v, v_scale, v_zero, c, num_bits, symmetric, group_dim, group_size);
  } else {
    OFQ_CHECK(!v_scale.defined() && !v_zero.defined() && !c.defined(),
          "v_scale, v_zero and c belong to v");
    OFQ_CHECK(d.n % 2 == 0, "dimension 0 of 'w' is not divisible by 2");
    n = d.n / 2;
  }
  require_gpu(x, w, w_scale, w_zero, b, v, v_scale, v_zero, c);
  Tensor h[9];
  const Tensor& x_ = contig(x, h[0]);
  const Tensor& w_ = contig(w, h[1]);
  const Tensor& ws_ = contig(w_scale, h[2]);
  const Tensor& wz_ = contig(w_zero, h[3]);
  const Tensor& b_ = contig(b, h[4]);
  const Tensor& v_ = contig(v, h[5]);
  const Tensor& vs_ = contig(v_scale, h[6]);
  const Tensor& vz_ = contig(v_zero, h[7]);
  const Tensor& c_ = contig(c, h[8]);
  Tensor y = empty(linear_shape(x, n), x.scalar_type(), x);
  // matmul_wx and matmul_vx (in this function scratch: the caller gets y only) in one allocation,
  // the second one 16-byte aligned
  const int64_t esize = (int64_t)x.element_size();
  const int64_t wx_bytes = (d.m * d.n * esize + 15) / 16 * 16;
  const Tensor scratch = workspace((size_t)(wx_bytes + (split ? d.m * n * esize : 0)), x);
  char* wx = static_cast<char*>(ptr(scratch));
  void* vx = split ? wx + wx_bytes : nullptr;
  const int wd = code_of(w), td = code_of(x);
  void* st = stream_of(x);
  check_status("ofq_fused_glu_gq", unlocked(
      ofq_fused_glu_gq, st, ptr(x_), ptr(w_), ptr(ws_), ptr(wz_), ptr(b_), ptr(v_), ptr(vs_),
      ptr(vz_), ptr(c_), ptr(y), wx, vx, act, wd, td, num_bits, symmetric, (int)d.gd, d.gs, d.m, n,
      d.k));
  return wrap(std::move(y));
}

// ---- min_max_observer / quantization / fake_quantization: quantization.cpp:34-153; attribute ----
// checks oneflow/user/ops/min_max_observer_op.cpp:58-70, quantization_op.cpp:92-104
struct QuantAttrs {
  int bit, scheme, formula;
};

void check_bit(int64_t bit) {
  OFQ_CHECK(1 < bit && bit <= 8, "quantization_bit should be in range (1, 8].");
}

QuantAttrs quant_attrs(PyObject* formula, PyObject* bit, PyObject* scheme) {
  const int64_t b = int_arg(bit);
  check_bit(b);
  const char* s = text_arg(scheme);
  const char* f = text_arg(formula);
  OFQ_CHECK(same(s, "symmetric") || same(s, "affine"),
        "quantization_scheme should be symmetric or affine.");
  OFQ_CHECK(same(f, "google") || same(f, "cambricon"),
        "quantization_formula should be google or cambricon.");
  return {(int)b, same(s, "affine") ? OFQ_SCHEME_AFFINE : OFQ_SCHEME_SYMMETRIC,
          same(f, "google") ? OFQ_FORMULA_GOOGLE : OFQ_FORMULA_CAMBRICON};
}

// (in, formula, bit, scheme, per_layer)
PyObject* min_max_observer(PyObject* const* args) {
  const Tensor& in = tensor_arg(args[0], "in");
  const QuantAttrs q = quant_attrs(args[1], args[2], args[3]);
  const bool per_layer = bool_arg(args[4]);
  const ScalarType t = in.scalar_type();
  OFQ_CHECK(t == at::kFloat || t == at::kDouble, "no min_max_observer kernel for dtype " + dtype_name(t));
  OFQ_CHECK(q.formula != OFQ_FORMULA_CAMBRICON || per_layer,
        " per-channel mode is not supported in cambricon scheme");
  require_gpu(in);
  Tensor h0;
  const Tensor& i_ = contig(in, h0);
  const int64_t channels = per_layer ? 1 : in.size(0);
  Tensor scale = empty({channels}, t, in), zero_point = empty({channels}, t, in);
  const size_t ws_bytes = ofq_min_max_observer_workspace_bytes(code_of(t), in.numel(), channels);
  const Tensor ws = workspace(ws_bytes, in);
  void* st = stream_of(in);
  check_status("ofq_min_max_observer", unlocked(
      ofq_min_max_observer, st, ptr(i_), ptr(scale), ptr(zero_point), code_of(t), i_.numel(),
      channels, q.bit, q.scheme, q.formula, ptr(ws), ws_bytes));
  return tuple_of(wrap(std::move(scale)), wrap(std::move(zero_point)));
}

// (in, current_train_step, moving_max, moving_min, training, stop_update_after_iters, formula,
//  bit, scheme, momentum)
PyObject* moving_average_min_max_observer(PyObject* const* args) {
  const Tensor& in = tensor_arg(args[0], "in");
  const Tensor& step = tensor_arg(args[1], "current_train_step");
  const Tensor& moving_max = tensor_arg(args[2], "moving_max");
  const Tensor& moving_min = tensor_arg(args[3], "moving_min");
  const bool training = bool_arg(args[4]);
  const int64_t stop = int_arg(args[5]);
  const QuantAttrs q = quant_attrs(args[6], args[7], args[8]);
  const double momentum = double_arg(args[9]);
  OFQ_CHECK(stop > 0, "stop_update_after_iters should be greater than 0");
  const ScalarType t = in.scalar_type();
  OFQ_CHECK(t == at::kFloat || t == at::kDouble,
        "no moving_average_min_max_observer kernel for dtype " + dtype_name(t));
  // shape rules of moving_average_min_max_observer_op.cpp:29-32
  const auto one = [](const Tensor& v) { return v.dim() == 1 && v.size(0) == 1; };
  OFQ_CHECK(one(moving_max), "moving_max should have shape [1]");
  OFQ_CHECK(one(moving_min), "moving_min should have shape [1]");
  OFQ_CHECK(one(step), "current_train_step should have shape [1]");
  OFQ_CHECK(moving_max.scalar_type() == t && moving_min.scalar_type() == t,
        "moving_max and moving_min should have the dtype of in");
  OFQ_CHECK(step.scalar_type() == at::kLong, "current_train_step should be int64");
  require_gpu(in, step, moving_max, moving_min);
  OFQ_CHECK(moving_max.is_contiguous() && moving_min.is_contiguous(),
        "moving_max and moving_min are updated in place and must be contiguous");
  Tensor h0;
  const Tensor& i_ = contig(in, h0);
  Tensor scale = empty({1}, t, in), zero_point = empty({1}, t, in);
  const size_t ws_bytes = ofq_moving_average_min_max_observer_workspace_bytes(code_of(t), in.numel());
  const Tensor ws = workspace(ws_bytes, in);
  void* st = stream_of(in);
  check_status("ofq_moving_average_min_max_observer", unlocked(
      ofq_moving_average_min_max_observer, st, ptr(i_), static_cast<const int64_t*>(ptr(step)),
      ptr(moving_max), ptr(moving_min), ptr(scale), ptr(zero_point), code_of(t), i_.numel(), q.bit,
      q.scheme, q.formula, (float)momentum, stop, training, ptr(ws), ws_bytes));
  return tuple_of(wrap(std::move(scale)), wrap(std::move(zero_point)));
}

int zp_mode_code(PyObject* o) {
  const char* s = text_arg(o);
  if (same(s, "float")) return OFQ_ZP_FLOAT;
  if (same(s, "uint8")) return OFQ_ZP_UINT8;
  PyErr_SetObject(PyExc_KeyError, o);
  throw PythonError{};
}

void check_quant_tensors(const char* fn, const Tensor& in, const Tensor& scale,
                         const Tensor& zero_point) {
  const ScalarType t = in.scalar_type();
  OFQ_CHECK(t == at::kFloat || t == at::kDouble || t == at::kHalf || t == at::kBFloat16,
        std::string("no ") + fn + " kernel for dtype " + dtype_name(t));
  const ScalarType p = t == at::kDouble ? at::kDouble : at::kFloat;
  OFQ_CHECK(scale.scalar_type() == p, "scale should have dtype " + dtype_name(p));
  OFQ_CHECK(!zero_point.defined() || zero_point.scalar_type() == p,
        "zero_point should have dtype " + dtype_name(p));
  // per-channel iff scale has more than one element (quantization_op.cpp:66-69)
  if (scale.numel() > 1) {
    OFQ_CHECK(in.dim() > 0 && scale.numel() == in.size(0), "scale.elem_cnt() should equal in.shape[0]");
    OFQ_CHECK(!zero_point.defined() || zero_point.numel() == in.size(0),
          "zero_point.elem_cnt() should equal in.shape[0]");
  }
  require_gpu(in, scale, zero_point);
}

// (in, scale, zero_point, formula, bit, scheme, out_dtype | None, zp_mode)
PyObject* quantization(PyObject* const* args) {
  const Tensor& in = tensor_arg(args[0], "in");
  const Tensor& scale = tensor_arg(args[1], "scale");
  const Tensor& zero_point = optional_arg(args[2], "zero_point");
  const QuantAttrs q = quant_attrs(args[3], args[4], args[5]);
  check_quant_tensors("quantization", in, scale, zero_point);
  const ScalarType to = args[6] == Py_None ? in.scalar_type() : dtype_arg(args[6]);
  const int zp_mode = zp_mode_code(args[7]);
  Tensor h0, h1, h2;
  const Tensor& i_ = contig(in, h0);
  const Tensor& s_ = contig(scale, h1);
  const Tensor& z_ = contig(zero_point, h2);
  Tensor out = empty(in.sizes(), to, in);
  const int id = code_of(in), od = code_of(to);
  void* st = stream_of(in);
  check_status("ofq_quantization", unlocked(
      ofq_quantization, st, ptr(i_), ptr(s_), ptr(z_), ptr(out), id, od, i_.numel(), s_.numel(),
      q.bit, q.scheme, q.formula, zp_mode));
  return wrap(std::move(out));
}

// The reference's gradient of fake_quantization: the output gradient passes to `in` unchanged,
// scale and zero_point get none (oneflow/core/autograd/gradient_funcs/fake_quantization.cpp:36-42).
// Forward mode is the same rule: the tangent of `in` is the tangent of the result.
struct FakeQuantizationBackward : public torch::autograd::Node {
  torch::autograd::variable_list apply(torch::autograd::variable_list&& grads) override {
    return std::move(grads);
  }
  std::string name() const override { return "FakeQuantizationBackward"; }
};

// (in, scale, zero_point, formula, bit, scheme, zp_mode)
PyObject* fake_quantization(PyObject* const* args) {
  const Tensor& in = tensor_arg(args[0], "in");
  const Tensor& scale = tensor_arg(args[1], "scale");
  const Tensor& zero_point = optional_arg(args[2], "zero_point");
  const QuantAttrs q = quant_attrs(args[3], args[4], args[5]);
  check_quant_tensors("fake_quantization", in, scale, zero_point);
  const int zp_mode = zp_mode_code(args[6]);
  Tensor out;
  {
    at::NoGradGuard no_grad;  // a copy made here is not part of the graph
    Tensor h0, h1, h2;
    const Tensor& i_ = contig(in, h0);
    const Tensor& s_ = contig(scale, h1);
    const Tensor& z_ = contig(zero_point, h2);
    out = empty(in.sizes(), in.scalar_type(), in);
    const int id = code_of(in);
    void* st = stream_of(in);
    check_status("ofq_fake_quantization", unlocked(
        ofq_fake_quantization, st, ptr(i_), ptr(s_), ptr(z_), ptr(out), id, i_.numel(), s_.numel(),
        q.bit, q.scheme, q.formula, zp_mode));
  }
  if (in.requires_grad() && at::GradMode::is_enabled()) {
    auto node = std::shared_ptr<FakeQuantizationBackward>(new FakeQuantizationBackward(),
                                                          torch::autograd::deleteNode);
    node->set_next_edges(torch::autograd::collect_next_edges(in));
    torch::autograd::set_history(out, node);
  }
  const Tensor& tangent = in._fw_grad(/*level=*/0);  // undefined where forward mode is off
  if (tangent.defined()) {
    out._set_fw_grad(tangent.clone(), /*level=*/0, /*is_inplace_op=*/false);
  }
  return wrap(std::move(out));
}

// ---- LayerNorm + observer / quantisation, matmul_quant (absent from the reference tree) ---------
void check_layer_norm_dtype(const char* fn, const Tensor& x) {
  OFQ_CHECK(is_linear_dtype(x.scalar_type()),
        std::string("no ") + fn + " kernel for dtype " + dtype_name(x.scalar_type()));
}

void check_affine(const Tensor& x, int64_t cols, const Tensor& gamma, const Tensor& beta) {
  const auto fits = [&](const Tensor& p) {
    return !p.defined() || (p.scalar_type() == x.scalar_type() && p.numel() == cols);
  };
  OFQ_CHECK(fits(gamma), "gamma should have the dtype of x and x.shape[-1] elements");
  OFQ_CHECK(fits(beta), "beta should have the dtype of x and x.shape[-1] elements");
}

// (x, gamma, beta, epsilon, bit, exact_statistics)
PyObject* layer_norm_observer(PyObject* const* args) {
  const Tensor& x = tensor_arg(args[0], "x");
  const Tensor& gamma = optional_arg(args[1], "gamma");
  const Tensor& beta = optional_arg(args[2], "beta");
  const double epsilon = double_arg(args[3]);
  const int64_t bit = int_arg(args[4]);
  const bool exact = bool_arg(args[5]);
  check_bit(bit);
  check_layer_norm_dtype("fused_layer_norm_min_max_observer", x);
  OFQ_CHECK(x.dim() >= 1, "number of axes of x should be greater than or equal to 1");
  const int64_t cols = x.size(-1);
  check_affine(x, cols, gamma, beta);
  require_gpu(x, gamma, beta);
  Tensor h0, h1, h2;
  const Tensor& x_ = contig(x, h0);
  const Tensor& g_ = contig(gamma, h1);
  const Tensor& b_ = contig(beta, h2);
  const int64_t rows = cols != 0 ? x.numel() / cols : 0;
  Tensor y = empty(x.sizes(), x.scalar_type(), x);
  Tensor scale = empty({1}, at::kFloat, x), zero_point = empty({1}, at::kFloat, x);
  const int td = code_of(x);
  const size_t ws_bytes = ofq_fused_layer_norm_min_max_observer_workspace_bytes(td, rows, cols);
  const Tensor ws = workspace(ws_bytes, x);
  void* st = stream_of(x);
  float* ps = static_cast<float*>(ptr(scale));
  float* pz = static_cast<float*>(ptr(zero_point));
  check_status("ofq_fused_layer_norm_min_max_observer", unlocked(
      ofq_fused_layer_norm_min_max_observer_stats, st, ptr(x_), nullptr, nullptr, 0.0, 0, ptr(g_),
      ptr(b_), ptr(y), ps, pz, td, rows, cols, epsilon, (int)bit,
      exact ? OFQ_LN_STATS_FP64 : OFQ_LN_STATS_FP32, ptr(ws), ws_bytes));
  return tuple_of(wrap(std::move(y)), wrap(std::move(scale)), wrap(std::move(zero_point)));
}

// (x, gamma, beta, bias, skip, epsilon, alpha, bit, exact_statistics)
PyObject* skip_layer_norm_observer(PyObject* const* args) {
  const Tensor& x = tensor_arg(args[0], "x");
  const Tensor& gamma = optional_arg(args[1], "gamma");
  const Tensor& beta = optional_arg(args[2], "beta");
  const Tensor& bias = optional_arg(args[3], "bias");
  const Tensor& skip = optional_arg(args[4], "skip");
  const double epsilon = double_arg(args[5]), alpha = double_arg(args[6]);
  const int64_t bit = int_arg(args[7]);
  const bool exact = bool_arg(args[8]);
  check_bit(bit);
  check_layer_norm_dtype("fused_skip_layer_norm_min_max_observer", x);
  OFQ_CHECK(x.dim() >= 2, "number of axes of x should be greater than or equal to 2");
  const int64_t cols = x.size(-1);
  const auto fits = [&](const Tensor& p) {
    return !p.defined()
           || (p.scalar_type() == x.scalar_type() && p.dim() == 1 && p.numel() == cols);
  };
  OFQ_CHECK(fits(gamma), "gamma should be 1-D with the dtype of x and x.shape[-1] elements");
  OFQ_CHECK(fits(beta), "beta should be 1-D with the dtype of x and x.shape[-1] elements");
  OFQ_CHECK(fits(bias), "bias should be 1-D with the dtype of x and x.shape[-1] elements");
  OFQ_CHECK(!skip.defined() || (skip.scalar_type() == x.scalar_type() && skip.sizes() == x.sizes()),
        "skip should have the shape and dtype of x");
  require_gpu(x, gamma, beta, bias, skip);
  Tensor h[5];
  const Tensor& x_ = contig(x, h[0]);
  const Tensor& g_ = contig(gamma, h[1]);
  const Tensor& b_ = contig(beta, h[2]);
  const Tensor& p_ = contig(bias, h[3]);
  const Tensor& s_ = contig(skip, h[4]);
  const int64_t rows = cols != 0 ? x.numel() / cols : 0;
  Tensor y = empty(x.sizes(), x.scalar_type(), x);
  Tensor scale = empty({1}, at::kFloat, x), zero_point = empty({1}, at::kFloat, x);
  const int td = code_of(x);
  const size_t ws_bytes = ofq_fused_layer_norm_min_max_observer_workspace_bytes(td, rows, cols);
  const Tensor ws = workspace(ws_bytes, x);
  void* st = stream_of(x);
  float* ps = static_cast<float*>(ptr(scale));
  float* pz = static_cast<float*>(ptr(zero_point));
  check_status("ofq_fused_skip_layer_norm_min_max_observer", unlocked(
      ofq_fused_layer_norm_min_max_observer_stats, st, ptr(x_), ptr(p_), ptr(s_), alpha, 1,
      ptr(g_), ptr(b_), ptr(y), ps, pz, td, rows, cols, epsilon, (int)bit,
      exact ? OFQ_LN_STATS_FP64 : OFQ_LN_STATS_FP32, ptr(ws), ws_bytes));
  return tuple_of(wrap(std::move(y)), wrap(std::move(scale)), wrap(std::move(zero_point)));
}

// (x, gamma, beta, epsilon, bit, exact_statistics)
PyObject* layer_norm_quantization(PyObject* const* args) {
  const Tensor& x = tensor_arg(args[0], "x");
  const Tensor& gamma = optional_arg(args[1], "gamma");
  const Tensor& beta = optional_arg(args[2], "beta");
  const double epsilon = double_arg(args[3]);
  const int64_t bit = int_arg(args[4]);
  const int stats = bool_arg(args[5]) ? OFQ_LN_STATS_FP64 : OFQ_LN_STATS_FP32;
  check_bit(bit);
  check_layer_norm_dtype("fused_layer_norm_quantization", x);
  OFQ_CHECK(x.dim() >= 1, "number of axes of x should be greater than or equal to 1");
  const int64_t cols = x.size(-1);
  check_affine(x, cols, gamma, beta);
  require_gpu(x, gamma, beta);
  Tensor h0, h1, h2;
  const Tensor& x_ = contig(x, h0);
  const Tensor& g_ = contig(gamma, h1);
  const Tensor& b_ = contig(beta, h2);
  const int64_t rows = cols != 0 ? x.numel() / cols : 0;
  Tensor codes = empty(x.sizes(), at::kChar, x);
  Tensor scale = empty({1}, at::kFloat, x), zero_point = empty({1}, at::kFloat, x);
  const int td = code_of(x);
  const size_t ws_bytes = ofq_fused_layer_norm_quantization_workspace_bytes(td, rows, cols);
  void* st = stream_of(x);
  float* ps = static_cast<float*>(ptr(scale));
  float* pz = static_cast<float*>(ptr(zero_point));
  int rc;
  {
    const Tensor ws = workspace(ws_bytes, x);
    rc = unlocked(
        ofq_fused_layer_norm_quantization_any_row, st, ptr(x_), ptr(g_), ptr(b_), ptr(codes), ps, pz, td,
        rows, cols, epsilon, (int)bit, stats, ptr(ws), ws_bytes);
  }
  if (rc == OFQ_ERR_UNSUPPORTED) {
    // the two ops in a row
    const Tensor y = empty(x.sizes(), x.scalar_type(), x);
    const size_t ws2_bytes = ofq_fused_layer_norm_min_max_observer_workspace_bytes(td, rows, cols);
    const Tensor ws2 = workspace(ws2_bytes, x);
    check_status("ofq_fused_layer_norm_min_max_observer", unlocked(
        ofq_fused_layer_norm_min_max_observer_stats, st, ptr(x_), nullptr, nullptr, 0.0, 0,
        ptr(g_), ptr(b_), ptr(y), ps, pz, td, rows, cols, epsilon, (int)bit, stats, ptr(ws2),
        ws2_bytes));
    check_status("ofq_quantization", unlocked(
        ofq_quantization, st, ptr(y), ps, pz, ptr(codes), td, OFQ_I8, y.numel(), 1, (int)bit,
        OFQ_SCHEME_SYMMETRIC, OFQ_FORMULA_GOOGLE, OFQ_ZP_FLOAT));
  } else {
    check_status("ofq_fused_layer_norm_quantization_any_row", rc);
  }
  return tuple_of(wrap(std::move(codes)), wrap(std::move(scale)), wrap(std::move(zero_point)));
}

// (a, b, a_scale, b_scale, bias, out_dtype)
PyObject* matmul_quant(PyObject* const* args) {
  const Tensor& a = tensor_arg(args[0], "a");
  const Tensor& b = tensor_arg(args[1], "b");
  const Tensor& a_scale = tensor_arg(args[2], "a_scale");
  const Tensor& b_scale = tensor_arg(args[3], "b_scale");
  const Tensor& bias = optional_arg(args[4], "bias");
  const ScalarType to = dtype_arg(args[5]);
  OFQ_CHECK(a.scalar_type() == at::kChar && b.scalar_type() == at::kChar, "a and b should be int8");
  OFQ_CHECK(a.dim() == 2 && b.dim() == 2 && a.size(1) == b.size(1), "a should be [m,k] and b [n,k]");
  OFQ_CHECK(a_scale.scalar_type() == at::kFloat && a_scale.numel() == 1,
        "a_scale should be one float32");
  OFQ_CHECK(b_scale.scalar_type() == at::kFloat && b_scale.numel() == b.size(0),
        "b_scale should be float32 with b.shape[0] elements");
  OFQ_CHECK(!bias.defined() || (bias.scalar_type() == to && bias.numel() == b.size(0)),
        "bias should have the output dtype and b.shape[0] elements");
  require_gpu(a, b, a_scale, b_scale, bias);
  Tensor h[5];
  const Tensor& a_ = contig(a, h[0]);
  const Tensor& b_ = contig(b, h[1]);
  const Tensor& as_ = contig(a_scale, h[2]);
  const Tensor& bs_ = contig(b_scale, h[3]);
  const Tensor& bias_ = contig(bias, h[4]);
  const int64_t m = a.size(0), k = a.size(1), n = b.size(0);
  Tensor out = empty({m, n}, to, a);
  const int od = code_of(to);
  const size_t ws_bytes = ofq_matmul_quant_workspace_bytes(m, n, k);
  Tensor ws;
  if (ws_bytes != 0) ws = workspace(ws_bytes, a);
  void* st = stream_of(a);
  check_status("ofq_matmul_quant_ws", unlocked(
      ofq_matmul_quant_ws, st, ptr(a_), ptr(b_), static_cast<const float*>(ptr(as_)),
      static_cast<const float*>(ptr(bs_)), ptr(bias_), ptr(out), od, m, n, k, ptr(ws), ws_bytes));
  return wrap(std::move(out));
}

// ---- weight quantiser: python/oneflow/test/modules/test_groupwise_quantization.py:26-81 ---------
// (x, num_bits, symmetric, group_dim, group_size, quant_type)
PyObject* groupwise_quantize(PyObject* const* args) {
  const Tensor& x = tensor_arg(args[0], "x");
  const int64_t num_bits = int_arg(args[1]);
  const bool symmetric = bool_arg(args[2]);
  const int64_t group_dim = int_arg(args[3]), group_size = int_arg(args[4]);
  OFQ_CHECK(num_bits == 4 || num_bits == 8, "num_bits should be 4 or 8.");
  OFQ_CHECK(x.dim() == 2, "x should be a 2-D weight [n, k].");
  const int64_t gd = group_dim < 0 ? group_dim + 2 : group_dim;
  OFQ_CHECK(gd == 0 || gd == 1, "group_dim should be in range [-2,2).");
  const int64_t n = x.size(0), k = x.size(1), dim = x.size(gd);
  const int64_t gs = group_size < 0 ? dim : group_size;
  OFQ_CHECK(0 < gs && gs <= dim, "group_size should be in range (0," + str(dim) + "].");
  OFQ_CHECK(dim % gs == 0, "group_size should be a divisor of " + str(dim) + ".");
  const ScalarType qt = THPDtype_Check(args[5]) ? dtype_arg(args[5]) : ScalarType::Undefined;
  OFQ_CHECK(qt == at::kChar || qt == at::kByte, "quant_type should be int8 or uint8.");
  OFQ_CHECK(symmetric || qt == at::kByte, "asymmetric codes are uint8.");
  OFQ_CHECK(is_linear_dtype(x.scalar_type()), "x should be float16, bfloat16 or float32.");
  OFQ_CHECK(num_bits != 4 || (k % 2 == 0 && (gd == 0 || gs % 2 == 0)),
        "4-bit codes are packed in pairs along k.");
  require_gpu(x);
  Tensor h0;
  const Tensor& x_ = contig(x, h0);
  const ScalarType t = x.scalar_type();
  Tensor q = empty({n, k * num_bits / 8}, qt, x);
  const int64_t sn = gd == 0 ? n / gs : n, sk = gd == 0 ? k : k / gs;
  Tensor scale = empty({sn, sk}, t, x), zero;
  if (!symmetric) zero = empty({sn, sk}, t, x);
  void* st = stream_of(x);
  check_status("ofq_groupwise_quantize", unlocked(
      ofq_groupwise_quantize, st, ptr(x_), ptr(q), ptr(scale), ptr(zero), code_of(t), code_of(qt),
      (int)num_bits, symmetric, (int)gd, gs, n, k));
  return tuple_of(wrap(std::move(q)), wrap(std::move(scale)),
                  symmetric ? none() : wrap(std::move(zero)));
}

// (CheckFailedError, OfqError): called once by _lib.native()
PyObject* set_errors(PyObject* const* args) {
  Py_XSETREF(check_failed_error, Py_NewRef(args[0]));
  Py_XSETREF(ofq_error, Py_NewRef(args[1]));
  return none();
}

#define ENTRY(N, FN) \
  {#FN, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(entry<N, FN>)), METH_FASTCALL, nullptr}

PyMethodDef methods[] = {
    ENTRY(2, set_errors),
    ENTRY(7, groupwise_dequantize),
    ENTRY(9, fused_linear),
    ENTRY(2, groupwise_repack),
    ENTRY(9, fused_linear_tiled),
    ENTRY(9, grouped_linear),
    ENTRY(14, fused_glu),
    ENTRY(5, min_max_observer),
    ENTRY(10, moving_average_min_max_observer),
    ENTRY(8, quantization),
    ENTRY(7, fake_quantization),
    ENTRY(6, layer_norm_observer),
    ENTRY(9, skip_layer_norm_observer),
    ENTRY(6, layer_norm_quantization),
    ENTRY(6, matmul_quant),
    ENTRY(6, groupwise_quantize),
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "ofq_torch", nullptr, -1, methods, nullptr, nullptr,
                      nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_ofq_torch() { return PyModule_Create(&module); }
