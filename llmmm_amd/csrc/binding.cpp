// llmmm_amd._native: the Python entry points' host work -- argument checks, output and workspace allocation, the current stream,
// the call into the C ABI -- as one CPython extension.
//
// What bounds a decode step through these entry points is the host: one decoder layer at M = 1 is nine kernels, about 40 us of GPU
// time, and took 99 us when every argument went through Python checks and ctypes (about 17 us per call); the same six calls here
// keep ahead of the GPU (50 us a layer; batched decode at M = 16 / 100: 98 -> 83, 99 -> 73; one product at M = 1: 11.2 -> 6.1; the
// FP16 product 1024^3: 8.7 -> 6.4).  The checks, their order and the exceptions are those the Python module documents: a CUDA tensor (TypeError),
// contiguous (ValueError), of a supported type (RuntimeError "T is not supported."), large enough (ValueError).  Outputs are
// allocated through torch's dispatcher, so its modes see them as they see torch.empty.  No state is kept between calls.
#include <Python.h>

#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/Exceptions.h>
#include <ATen/ATen.h>
#include <c10/core/impl/VirtualGuardImpl.h>

#include <climits>

#include "../../include/llmmm.h"

namespace {

enum : unsigned { T_F32 = 1, T_F16 = 2, T_BF16 = 4, T_FP8 = 8, T_I32 = 16, T_ANY = 0 };

unsigned type_bit(const at::Tensor& t)
{
  switch (t.scalar_type()) {
    case at::kFloat: return T_F32;
    case at::kHalf: return T_F16;
    case at::kBFloat16: return T_BF16;
    case at::kByte:
    case at::kFloat8_e4m3fn: return T_FP8;  // e4m3 codes travel as either type
    case at::kInt: return T_I32;
    default: return 0;
  }
}

struct Refused {};  // a Python exception has been set

// Without the interpreter lock, as torch.empty and ctypes go about it: other Python threads run while the allocator has to go to
// the device, and while a launch waits for a full hardware queue.
struct Unlocked {
  PyThreadState* const state = PyEval_SaveThread();
  Unlocked() = default;
  Unlocked(const Unlocked&) = delete;
  ~Unlocked() { PyEval_RestoreThread(state); }
};

[[noreturn]] void refuse(PyObject* type, const char* fmt, ...)
{
  va_list ap;
  va_start(ap, fmt);
  PyErr_FormatV(type, fmt, ap);
  va_end(ap);
  throw Refused();
}
[[noreturn]] void not_supported() { refuse(PyExc_RuntimeError, "T is not supported."); }

const at::Tensor& tensor(PyObject* o, const char* what)
{
  if (!THPVariable_Check(o)) refuse(PyExc_TypeError, "%s must be a CUDA tensor", what);
  return THPVariable_Unpack(o);
}

// The device address of a tensor argument; `types` = the element types it may have (T_ANY: all), `numel` = elements needed.
void* ptr(PyObject* o, const char* what, unsigned types, int64_t numel)
{
  const at::Tensor& t = tensor(o, what);
  if (!t.is_cuda()) refuse(PyExc_TypeError, "%s must be a CUDA tensor", what);
  if (!t.is_contiguous()) refuse(PyExc_ValueError, "%s must be contiguous", what);
  if (types != T_ANY && !(type_bit(t) & types)) not_supported();
  if (t.numel() < numel) refuse(PyExc_ValueError, "%s holds %lld elements, %lld needed", what, (long long)t.numel(), (long long)numel);
  return t.data_ptr();
}
void* ptr_or_null(PyObject* o, const char* what, unsigned types, int64_t numel) { return o == Py_None ? nullptr : ptr(o, what, types, numel); }

int as_int(PyObject* o)
{
  const long v = PyLong_AsLong(o);
  if (v == -1 && PyErr_Occurred()) throw Refused();
  if (v < INT_MIN || v > INT_MAX) refuse(PyExc_OverflowError, "%ld does not fit an int", v);
  return (int)v;
}
float as_float(PyObject* o)
{
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw Refused();
  return (float)v;
}
bool as_bool(PyObject* o)
{
  const int v = PyObject_IsTrue(o);
  if (v < 0) throw Refused();
  return v != 0;
}

// A Python object that is dropped with its scope; null: a Python exception has been set.
struct Owned {
  PyObject* o;
  explicit Owned(PyObject* o) : o(o)
  {
    if (!o) throw Refused();
  }
  Owned(const Owned&) = delete;
  ~Owned() { Py_DECREF(o); }
};
void* as_pointer(PyObject* o)
{
  void* p = PyLong_AsVoidPtr(o);
  if (!p && PyErr_Occurred()) throw Refused();
  return p;
}
int64_t int_attribute(PyObject* o, const char* name)
{
  const Owned     a(PyObject_GetAttrString(o, name));
  const long long v = PyLong_AsLongLong(a.o);
  if (v == -1 && PyErr_Occurred()) throw Refused();
  return v;
}

PyObject *current_raw_stream, *external_stream;  // torch._C._cuda_getCurrentRawStream(device index), torch.cuda.ExternalStream

// The stream a call runs on.  Its tensors -- the private workspace, which the caller never sees and nobody else can protect, and the
// returned outputs -- belong to that stream: the allocator hands a block freed there only to work ordered behind this call.  From the
// current stream's blocks they would be taken while that stream may still use them, and given back while this call still runs.
struct Launch {
  void*       handle;
  bool        foreign = false;                                                     // not torch's current stream
  c10::Stream current = c10::Stream(c10::Stream::DEFAULT, c10::Device(c10::kCUDA, 0)), stream = current;  // set where foreign

  template <typename Make>
  at::Tensor allocate(Make&& make) const
  {
    const Unlocked unlocked;
    if (!foreign) return make();
    const c10::impl::VirtualGuardImpl impl(c10::DeviceType::CUDA);
    struct Restore {
      const c10::impl::VirtualGuardImpl& impl;
      c10::Stream                        previous;
      ~Restore() { impl.exchangeStream(previous); }
    } restore{impl, impl.exchangeStream(stream)};
    return make();
  }
  at::Tensor empty(at::IntArrayRef sizes, at::ScalarType type, const at::Device& device) const
  {
    return allocate([&] { return at::empty(sizes, at::TensorOptions().dtype(type).device(device)); });
  }
  // A tensor that goes back to the caller, who goes on with it on the current stream.
  const at::Tensor& returned(const at::Tensor& t) const
  {
    if (foreign) t.record_stream(current);
    return t;
  }
};
// None: torch's current stream; a torch stream: its handle; anything else: the handle as an integer.
Launch launch(PyObject* o)
{
  const c10::impl::VirtualGuardImpl impl(c10::DeviceType::CUDA);
  const c10::Device                 device = impl.getDevice();
  const Owned                       index(PyLong_FromLong(device.index())), raw(PyObject_CallOneArg(current_raw_stream, index.o));
  Launch                            on{as_pointer(raw.o)};
  if (o == Py_None) return on;
  PyObject* attribute = PyLong_Check(o) ? nullptr : PyObject_GetAttrString(o, "cuda_stream");
  if (!attribute) PyErr_Clear();
  const bool named  = attribute != nullptr;
  PyObject*  number = PyNumber_Long(named ? attribute : o);
  Py_XDECREF(attribute);
  const Owned handle(number);
  void* const p = as_pointer(handle.o);
  if (p == on.handle) return on;
  on.handle  = p;
  on.foreign = true;
  on.current = impl.getStream(device);
  if (named)
    on.stream = c10::Stream::unpack3(int_attribute(o, "stream_id"), (c10::DeviceIndex)int_attribute(o, "device_index"), c10::DeviceType::CUDA);
  else if ((uintptr_t)p > 1) {
    const Owned s(PyObject_CallOneArg(external_stream, handle.o));
    on.stream = c10::Stream::unpack3(int_attribute(s.o, "stream_id"), (c10::DeviceIndex)int_attribute(s.o, "device_index"), c10::DeviceType::CUDA);
  }
  else  // 0 and 1 (the legacy handle): the device's default stream
    on.stream = c10::Stream(c10::Stream::DEFAULT, device);
  return on;
}

int64_t blocks(int64_t n) { return (n + 127) / 128; }
int64_t whole_blocks(int64_t n) { return n % 128 == 0 ? n / 128 : 0; }

PyObject* tuple2(const at::Tensor& a, const at::Tensor& b)
{
  PyObject* r = PyTuple_New(2);
  if (!r) throw Refused();
  PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(a));
  PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(b));
  return r;
}

// The call itself.  The text of a failure is the calling thread's, so it is fetched before anything else runs on this thread.
template <typename F>
void call(F&& f)
{
  int rc;
  {
    const Unlocked unlocked;
    rc = f();
  }
  if (rc == LLMMM_OK) return;
  const char *text = llmmm_error_string(rc), *detail = llmmm_last_error();
  if (rc == LLMMM_ERR_NOT_ALIGNED || rc == LLMMM_ERR_UNSUPPORTED_TYPE)
    refuse(PyExc_RuntimeError, "%s", *detail ? detail : text);  // the detail is the reference's text for the entry point that failed
  if (*detail) refuse(PyExc_RuntimeError, "%s: %s", text, detail);
  refuse(PyExc_RuntimeError, "%s", text);
}

int hidden_dtype(const at::Tensor& t)
{
  switch (type_bit(t)) {
    case T_F32: return LLMMM_DTYPE_F32;
    case T_BF16: return LLMMM_DTYPE_BF16;
    case T_F16: return LLMMM_DTYPE_F16;
    default: not_supported();
  }
}
void shape2(const at::Tensor& t, const char* what, int& rows, int& cols)
{
  if (t.dim() != 2) refuse(PyExc_ValueError, "%s must have two dimensions", what);
  if (t.size(0) > INT_MAX || t.size(1) > INT_MAX) refuse(PyExc_OverflowError, "%s is too large", what);
  rows = (int)t.size(0), cols = (int)t.size(1);
}

// The A operand of an FP8 product by layout: quantised codes with their scales, the fp32 gate_up result [M, 2K], or the host
// address of an llmmm_a_planes_rmsnorm.
struct AOperand {
  const void*  a;
  const float* as;
};
AOperand a_operand(PyObject* A, PyObject* As, int layout, int64_t M, int64_t K)
{
  if (layout == LLMMM_FP8_A_PLANES_RMSNORM) {
    void* p = PyLong_AsVoidPtr(A);
    if (!p) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null A operand");
      throw Refused();
    }
    return {p, nullptr};
  }
  if (layout == LLMMM_FP8_A_SWIGLU_F32) return {ptr(A, "A (fp32 gate_up result)", T_F32, M * 2 * K), nullptr};
  const void* a = ptr(A, "A", T_FP8, M * K);
  return {a, (const float*)ptr(As, "A_scale_transposed", T_F32, whole_blocks(K) * M)};
}
size_t a_workspace_bytes(int layout, int M, int N, int K)
{
  if (layout == LLMMM_FP8_A_PLANES_RMSNORM) return llmmm_fp8_planes_rmsnorm_a_workspace(M, N, K);
  return layout == LLMMM_FP8_A_SWIGLU_F32 ? llmmm_fp8_swiglu_a_workspace(M, N, K) : 0;
}
struct Workspace {
  at::Tensor own;
  void*      p = nullptr;
  size_t     n = 0;
};
// The caller's workspace, if there is one.
Workspace workspace(PyObject* o)
{
  Workspace w;
  if (o == Py_None) return w;
  if (!THPVariable_Check(o)) refuse(PyExc_TypeError, "workspace must be a tensor");
  const at::Tensor& t = THPVariable_Unpack(o);
  w.p = t.data_ptr(), w.n = (size_t)t.numel() * t.element_size();
  return w;
}
// The caller's workspace, or one of own() bytes, at least 16.
template <typename Bytes>
Workspace workspace(PyObject* o, Bytes&& own, const Launch& on, const at::Device& device)
{
  if (o != Py_None) return workspace(o);
  Workspace     w;
  const int64_t n = (int64_t)own();
  w.own = on.empty({n > 16 ? n : 16}, at::kByte, device);
  w.p = w.own.data_ptr(), w.n = (size_t)w.own.numel();
  return w;
}

// Planes for the split the library chooses for an FP16 / BF16 product, if it chooses one; dropped with the call, in stream order.
Workspace fp16_workspace(bool automatic, int M, int N, int K, const Launch& on, const at::Device& device)
{
  Workspace    w;
  const size_t n = automatic ? llmmm_fp16_gemm_workspace(M, N, K) : 0;
  if (n) w.own = on.empty({(int64_t)n}, at::kByte, device), w.p = w.own.data_ptr(), w.n = n;
  return w;
}

// ---------------------------------------------------------------------------------------------- entry points
typedef PyObject* const* Args;

// (A, B, C or None, b_transposed, tile, stream) -> C
PyObject* fp16_gemm(Args v)
{
  const at::Tensor &A = tensor(v[0], "A"), &B = tensor(v[1], "B");
  const unsigned    t = type_bit(A);
  if (t != T_F16 && t != T_BF16) not_supported();
  int M, K;
  shape2(A, "A", M, K);
  if (B.dim() < 2) refuse(PyExc_IndexError, "B must have two dimensions");  // (more are taken: the first two are its shape)
  if (B.size(0) > INT_MAX || B.size(1) > INT_MAX) refuse(PyExc_OverflowError, "B is too large");
  const int  b0 = (int)B.size(0), b1 = (int)B.size(1);
  const bool bt = as_bool(v[3]);
  const int  N  = bt ? b0 : b1;
  if ((bt ? b1 : b0) != K || B.scalar_type() != A.scalar_type()) refuse(PyExc_ValueError, "shape or dtype mismatch between A and B");
  const llmmm_gemm_cfg cfg = {as_int(v[4]), 0, 0, 0};
  const void *         a = ptr(v[0], "A", T_ANY, 0), *b = ptr(v[1], "B", T_ANY, 0);
  void*                c = v[2] == Py_None ? nullptr : ptr(v[2], "C", t, (int64_t)M * N);
  const Launch         on = launch(v[5]);
  at::Tensor           own;
  if (!c) own = on.empty({M, N}, A.scalar_type(), A.device()), c = own.data_ptr();
  const Workspace ws = fp16_workspace(cfg.tile == LLMMM_TILE_AUTO, M, N, K, on, A.device());
  call([&] {
    return llmmm_fp16_gemm_ws(t == T_F16 ? LLMMM_DTYPE_F16 : LLMMM_DTYPE_BF16, a, b, c, M, N, K, bt ? LLMMM_B_TRANSPOSED : LLMMM_B_ROW_MAJOR, ws.p, ws.n, &cfg,
                              on.handle);
  });
  if (own.defined()) return THPVariable_Wrap(on.returned(own));
  Py_INCREF(v[2]);
  return v[2];
}

// (A, B, C, M, N, K, stream): the reference's launcher
PyObject* fp16_mm(Args v)
{
  const at::Tensor &A = tensor(v[0], "A"), &B = tensor(v[1], "B"), &C = tensor(v[2], "C");
  const unsigned    t = type_bit(A);
  if ((t != T_F16 && t != T_BF16) || B.scalar_type() != A.scalar_type() || C.scalar_type() != A.scalar_type()) not_supported();
  const int M = as_int(v[3]), N = as_int(v[4]), K = as_int(v[5]);
  if (M % 256 || N % 256 || K % 16) refuse(PyExc_RuntimeError, "M or N or K are not aligned.");
  const void* a = ptr(v[0], "A", T_ANY, (int64_t)M * K);
  const void* b = ptr(v[1], "B", T_ANY, (int64_t)K * N);
  void*       c = ptr(v[2], "C", T_ANY, (int64_t)M * N);
  const Launch on = launch(v[6]);
  const Workspace ws = fp16_workspace(true, M, N, K, on, A.device());
  call([&] {
    return llmmm_fp16_gemm_ws(t == T_F16 ? LLMMM_DTYPE_F16 : LLMMM_DTYPE_BF16, a, b, c, M, N, K, LLMMM_B_ROW_MAJOR, ws.p, ws.n, nullptr, on.handle);
  });
  Py_RETURN_NONE;
}

int64_t scale_count(int kind, int64_t M, int64_t N)
{
  switch (kind) {
    case LLMMM_QUANT_1x128_T:
    case LLMMM_QUANT_128x128_T: return blocks(N) * M;
    case LLMMM_QUANT_1x128: return M * blocks(N);
    default: return blocks(M) * blocks(N);
  }
}

// (x, q, scale, M, N, kind, stream)
PyObject* quantize_into(Args v)
{
  const int    M = as_int(v[3]), N = as_int(v[4]), kind = as_int(v[5]);
  const float* x = (const float*)ptr(v[0], "x", T_F32, (int64_t)M * N);
  void*        q = ptr(v[1], "q", T_FP8, (int64_t)M * N);
  float*       c = (float*)ptr(v[2], "scale", T_F32, scale_count(kind, M, N));
  const Launch on = launch(v[6]);
  call([&] { return llmmm_quant_fp8(kind, x, q, c, M, N, on.handle); });
  Py_RETURN_NONE;
}

// (x, kind, stream) -> (codes, scales); kind 1x128 transposed (activations) or 128x128 (weights)
PyObject* quantize(Args v)
{
  const at::Tensor& X = tensor(v[0], "x");
  const int         kind = as_int(v[1]);
  int               M, N;
  shape2(X, "x", M, N);
  const float*     x  = (const float*)ptr(v[0], "x", T_F32, (int64_t)M * N);
  const Launch     on = launch(v[2]);
  const at::Tensor q  = on.empty({M, N}, at::kByte, X.device());
  const at::Tensor c =
      kind == LLMMM_QUANT_1x128_T ? on.empty({blocks(N), M}, at::kFloat, X.device()) : on.empty({blocks(M), blocks(N)}, at::kFloat, X.device());
  call([&] { return llmmm_quant_fp8(kind, x, q.data_ptr(), (float*)c.data_ptr(), M, N, on.handle); });
  return tuple2(on.returned(q), on.returned(c));
}

// (x, weight, eps, stream) -> (codes, scales)
PyObject* rmsnorm_quantize(Args v)
{
  const at::Tensor& X = tensor(v[0], "x");
  int               M, K;
  shape2(X, "x", M, K);
  const int        code = hidden_dtype(X);
  const void*      x    = ptr(v[0], "x", T_ANY, 0);
  const float*     w    = (const float*)ptr(v[1], "weight", T_F32, K);
  const float      eps  = as_float(v[2]);
  const Launch     on   = launch(v[3]);
  const at::Tensor q = on.empty({M, K}, at::kByte, X.device()), c = on.empty({blocks(K), M}, at::kFloat, X.device());
  call([&] { return llmmm_rmsnorm_quant_fp8(code, x, w, eps, q.data_ptr(), (float*)c.data_ptr(), M, K, on.handle); });
  return tuple2(on.returned(q), on.returned(c));
}

// (out_kind, A, As, Bt, Bs, C, Cs, M, N, K, workspace, tile, split_k, b_preshuffled, a_layout, stream)
PyObject* fp8_gemm(Args v)
{
  const int      kind = as_int(v[0]), M = as_int(v[7]), N = as_int(v[8]), K = as_int(v[9]), layout = as_int(v[14]);
  const int64_t  n_out = kind == LLMMM_OUT_FP8Q_SWIGLU ? N / 2 : N;  // SwiGLU halves the width
  const unsigned types = kind == LLMMM_OUT_F32 ? T_F32 : kind == LLMMM_OUT_BF16 ? T_BF16 : T_FP8;
  const bool     fp8   = types == T_FP8;
  const AOperand a     = a_operand(v[1], v[2], layout, M, K);
  const void*    b     = ptr(v[3], "B_transposed", T_FP8, (int64_t)N * K);
  const float*   bs    = (const float*)ptr(v[4], "B_scale_transposed", T_F32, blocks(N) * whole_blocks(K));
  void*          c     = ptr(v[5], "C", types, M * n_out);
  float*         cs    = fp8 ? (float*)ptr(v[6], "C_scale_transposed", T_F32, blocks(n_out) * M) : nullptr;
  const Workspace      w   = workspace(v[10]);
  const llmmm_gemm_cfg cfg = {as_int(v[11]), as_int(v[12]), as_bool(v[13]) ? LLMMM_FP8_B_PRESHUFFLED : LLMMM_FP8_B_ROWS, layout};
  const Launch         on  = launch(v[15]);
  call([&] { return llmmm_fp8_gemm_ex(kind, a.a, a.as, b, bs, c, cs, M, N, K, w.p, w.n, &cfg, on.handle); });
  Py_RETURN_NONE;
}

// (A, As, Bt, Bs, residual, hidden_out, norm_weight, eps, M, N, K, workspace, tile, split_k, b_preshuffled, a_layout, stream) -> (codes, scales)
PyObject* fp8_gemm_add_rmsnorm_quant(Args v)
{
  const at::Tensor &R = tensor(v[4], "residual"), &H = tensor(v[5], "hidden_out");
  const int         code = hidden_dtype(R);
  if (H.scalar_type() != R.scalar_type()) not_supported();
  const int        M = as_int(v[8]), N = as_int(v[9]), K = as_int(v[10]), layout = as_int(v[15]);
  const AOperand   a  = a_operand(v[0], v[1], layout, M, K);
  const void*      b  = ptr(v[2], "B_transposed", T_FP8, (int64_t)N * K);
  const float*     bs = (const float*)ptr(v[3], "B_scale_transposed", T_F32, blocks(N) * whole_blocks(K));
  const void*      r  = ptr(v[4], "residual", T_ANY, (int64_t)M * N);
  void*            h  = ptr(v[5], "hidden_out", T_ANY, (int64_t)M * N);
  const float*     nw = (const float*)ptr(v[6], "norm_weight", T_F32, N);
  const float      eps = as_float(v[7]);
  const llmmm_gemm_cfg cfg = {as_int(v[12]), as_int(v[13]), as_bool(v[14]) ? LLMMM_FP8_B_PRESHUFFLED : LLMMM_FP8_B_ROWS, layout};
  const Launch         on  = launch(v[16]);
  const Workspace  w = workspace(
      v[11], [&] { return llmmm_fp8_gemm_add_rmsnorm_quant_workspace(M, N, K) + a_workspace_bytes(layout, M, N, K); }, on, R.device());
  const at::Tensor q = on.empty({M, N}, at::kByte, R.device()), c = on.empty({blocks(N), M}, at::kFloat, R.device());
  call([&] {
    return llmmm_fp8_gemm_add_rmsnorm_quant(a.a, a.as, b, bs, code, r, h, nw, eps, q.data_ptr(), (float*)c.data_ptr(), M, N, K, w.p, w.n, &cfg, on.handle);
  });
  return tuple2(on.returned(q), on.returned(c));
}

// (A, As, Bt, Bs, q_norm, k_norm, eps, cos, sin, positions, n_q, n_kv, M, N, K, out_fp8, workspace, tile, split_k, b_preshuffled, a_layout, stream)
// -> out or (codes, scales)
PyObject* fp8_gemm_qkv_rope(Args v)
{
  const at::Tensor &B = tensor(v[2], "B_transposed"), &T = tensor(v[7], "cos_table");
  const int         n_q = as_int(v[10]), n_kv = as_int(v[11]), M = as_int(v[12]), N = as_int(v[13]), K = as_int(v[14]), layout = as_int(v[20]);
  const bool        fp8 = as_bool(v[15]);
  if (T.dim() < 1) refuse(PyExc_IndexError, "cos_table must have rows");
  if (T.size(0) > INT_MAX) refuse(PyExc_OverflowError, "cos_table is too large");
  const int      rows = (int)T.size(0);
  const AOperand a    = a_operand(v[0], v[1], layout, M, K);
  const void*    b    = ptr(v[2], "B_transposed", T_FP8, (int64_t)N * K);
  const float*   bs   = (const float*)ptr(v[3], "B_scale_transposed", T_F32, blocks(N) * whole_blocks(K));
  const float*   qn   = (const float*)ptr_or_null(v[4], "q_norm_weight", T_F32, 128);
  const float*   kn   = (const float*)ptr_or_null(v[5], "k_norm_weight", T_F32, 128);
  const float    eps  = as_float(v[6]);
  const float*   ct   = (const float*)ptr(v[7], "cos_table", T_F32, (int64_t)rows * 64);
  const float*   st   = (const float*)ptr(v[8], "sin_table", T_F32, (int64_t)rows * 64);
  const int*     pos  = (const int*)ptr(v[9], "positions", T_I32, M);
  const llmmm_gemm_cfg cfg = {as_int(v[17]), as_int(v[18]), as_bool(v[19]) ? LLMMM_FP8_B_PRESHUFFLED : LLMMM_FP8_B_ROWS, layout};
  const Launch         on  = launch(v[21]);
  const Workspace  w   = workspace(
      v[16], [&] { return llmmm_fp8_gemm_qkv_rope_workspace(M, N, K) + a_workspace_bytes(layout, M, N, K); }, on, B.device());
  const at::Tensor out = on.empty({M, N}, fp8 ? at::kByte : at::kBFloat16, B.device());
  at::Tensor       sc;
  if (fp8) sc = on.empty({blocks(N), M}, at::kFloat, B.device());
  call([&] {
    return llmmm_fp8_gemm_qkv_rope(fp8 ? LLMMM_OUT_FP8Q : LLMMM_OUT_BF16, a.a, a.as, b, bs, out.data_ptr(), fp8 ? (float*)sc.data_ptr() : nullptr, qn, kn, eps, ct, st,
                                   rows, pos, n_q, n_kv, M, N, K, w.p, w.n, &cfg, on.handle);
  });
  return fp8 ? tuple2(on.returned(out), on.returned(sc)) : THPVariable_Wrap(on.returned(out));
}

// (codes, stream) -> the pre-shuffled image, a new tensor of the same shape and type
PyObject* preshuffle(Args v)
{
  const at::Tensor& Q = tensor(v[0], "src_transposed");
  int               N, K;
  shape2(Q, "src_transposed", N, K);
  const void*      q   = ptr(v[0], "src_transposed", T_FP8, (int64_t)N * K);
  const Launch     on  = launch(v[1]);
  const at::Tensor out = on.allocate([&] { return at::empty_like(Q); });
  call([&] { return llmmm_fp8_preshuffle_b(q, out.data_ptr(), N, K, on.handle); });
  return THPVariable_Wrap(on.returned(out));
}

template <PyObject* (*F)(Args), Py_ssize_t COUNT>
PyObject* entry(PyObject*, Args v, Py_ssize_t n)
{
  HANDLE_TH_ERRORS
  if (n != COUNT) {
    PyErr_Format(PyExc_TypeError, "%zd arguments expected, got %zd", COUNT, n);
    return nullptr;
  }
  try {
    return F(v);
  }
  catch (const Refused&) {
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}

#define LLMMM_ENTRY(NAME, COUNT) {#NAME, (PyCFunction)(void*)&entry<NAME, COUNT>, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {LLMMM_ENTRY(fp16_gemm, 6),        LLMMM_ENTRY(fp16_mm, 7),   LLMMM_ENTRY(quantize_into, 7),
                         LLMMM_ENTRY(quantize, 3),         LLMMM_ENTRY(rmsnorm_quantize, 4),
                         LLMMM_ENTRY(fp8_gemm, 16),        LLMMM_ENTRY(fp8_gemm_add_rmsnorm_quant, 17),
                         LLMMM_ENTRY(fp8_gemm_qkv_rope, 22), LLMMM_ENTRY(preshuffle, 2),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void)
{
  PyObject* torch_c  = PyImport_ImportModule("torch._C");
  current_raw_stream = torch_c ? PyObject_GetAttrString(torch_c, "_cuda_getCurrentRawStream") : nullptr;
  Py_XDECREF(torch_c);
  PyObject* cuda  = current_raw_stream ? PyImport_ImportModule("torch.cuda") : nullptr;
  external_stream = cuda ? PyObject_GetAttrString(cuda, "ExternalStream") : nullptr;
  Py_XDECREF(cuda);
  return external_stream ? PyModule_Create(&module) : nullptr;
}
