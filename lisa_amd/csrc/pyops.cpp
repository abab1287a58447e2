// Native side of lisa_amd/ops.py: the checks, output allocation and C-ABI call
// of one op in one C++ call.  In Python a call cost ~14 us of host time
// (attribute reads, torch.empty, the current stream, a 14-argument ctypes
// call), more than most decode kernels take (a 3072 x 1024 matvec: 3.2 us).
// Calls in a row, Python -> here: that matvec 13.7 -> 4.7 us, one token of a
// 128-expert block 19.0 -> 10.7, of a dense MLP block 49.5 -> 42.4.
//
// Every function returns None where the arguments are not the plain case --
// exactly torch.Tensor (or Parameter) on one GPU, contiguous, of the dtypes
// and shapes that the op takes, no tensor-subclass, vmap or dispatch mode in
// the way -- or where the C ABI reports an error; ops.py then takes its own
// path, which converts, raises the op's errors, or hands the mode what it
// expects.  Nothing is kept between calls.  Split-K partials come from torch's
// allocator and go back when the call returns, in the order of the caller's
// stream.  A captured call's replays write them again, and only a capture that
// torch began keeps freed memory to itself: under any capture they share the
// output's storage and live as long as it does.  The GIL is released over
// allocation and launch, as a ctypes call does: either can wait for the driver
// or for room in a full queue.
#include <Python.h>
#include <ATen/TensorSubclassLikeUtils.h>
#include <ATen/core/TensorBase.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <mutex>

#include "../../include/lisaq.h"

namespace {

using at::Tensor;

bool modes_active() {
  return c10::impl::dispatch_mode_enabled() || at::impl::torch_function_mode_enabled();
}

// Argument i as a plain contiguous GPU tensor
bool plain(PyObject* o, const Tensor** out) {
  if (!THPVariable_CheckExact(o)) return false;
  const Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != c10::kStrided || !t.is_contiguous() || t.is_neg() ||
      at::isTensorSubclassLike(t))
    return false;
  *out = &t;
  return true;
}

bool integer(PyObject* o, int64_t* out) {
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  *out = PyLong_AsLongLongAndOverflow(o, &overflow);
  return overflow == 0;
}

bool codes(const Tensor& w) { return w.scalar_type() == at::kInt || w.scalar_type() == at::kUInt32; }

// (w, scales, biases) as `lead` + [N, Kq] / [N, G] of one quantized matrix or stack
struct Packed {
  const Tensor *w, *s, *b;
  bool read(PyObject* const* a, int dim, at::ScalarType dt, c10::Device dev) {
    return plain(a[0], &w) && plain(a[1], &s) && plain(a[2], &b) && codes(*w) && s->scalar_type() == dt &&
           b->scalar_type() == dt && w->dim() == dim && s->dim() == dim && w->device() == dev && s->device() == dev &&
           b->device() == dev && s->sizes() == b->sizes();
  }
  // rows N and columns K of the matrix at this group size and width
  bool shape(int64_t N, int64_t K, int64_t gs, int64_t bits) const {
    const int d = (int)w->dim();
    if (d == 3 && s->size(0) != w->size(0)) return false;
    return w->size(d - 2) == N && w->size(d - 1) * 32 / bits == K && s->size(d - 2) == N && s->size(d - 1) == K / gs;
  }
  const uint32_t* codes_ptr() const { return static_cast<const uint32_t*>(w->data_ptr()); }
};

bool format(PyObject* g, PyObject* b, int64_t* gs, int64_t* bits) {
  return integer(g, gs) && integer(b, bits) && *gs > 0 && *gs <= 4096 && (*bits == 2 || *bits == 4 || *bits == 8);
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

Tensor output(const Tensor& x, int64_t N) {
  c10::SmallVector<int64_t, 5> sizes(x.sizes().begin(), x.sizes().end());
  sizes.back() = N;
  return at::empty(sizes, x.options());
}

// The output [..., N] of x and `bytes` of scratch for the call's launches
struct Outputs {
  Tensor y, ws;
  void* wp = nullptr;
  Outputs(const Tensor& x, int64_t N, size_t bytes, void* stream) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    // (the null stream is never captured, and asking takes ~0.5 us)
    if (bytes && stream && hipStreamIsCapturing(static_cast<hipStream_t>(stream), &st) == hipSuccess &&
        st != hipStreamCaptureStatusNone) {
      c10::SmallVector<int64_t, 5> sizes(x.sizes().begin(), x.sizes().end());
      sizes.back() = N;
      const int64_t ybytes = (x.numel() / x.size(-1) * N * (int64_t)x.element_size() + 255) / 256 * 256;
      ws = at::empty({ybytes + (int64_t)bytes}, x.options().dtype(at::kByte));
      wp = static_cast<char*>(ws.data_ptr()) + ybytes;
      y = at::empty({0}, x.options());
      y.set_(ws.storage(), 0, sizes);
      return;
    }
    if (bytes) {
      ws = at::empty({(int64_t)bytes}, x.options().dtype(at::kByte));
      wp = ws.data_ptr();
    }
    y = output(x, N);
  }
};

// The arguments' tensors stay alive without the GIL: the caller's frame holds them.
class NoGil {
  PyThreadState* const state_ = PyEval_SaveThread();

 public:
  NoGil() = default;
  NoGil(const NoGil&) = delete;
  ~NoGil() { PyEval_RestoreThread(state_); }
};

#define LISAQ_NONE_UNLESS(cond) \
  if (!(cond)) Py_RETURN_NONE

// linear(x, w, scales, biases, group_size, bits, serial_rows) -> y [..., N]
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int64_t gs, bits, serial;
  const Tensor* x;
  Packed q;
  LISAQ_NONE_UNLESS(n == 7 && format(a[4], a[5], &gs, &bits) && integer(a[6], &serial) && plain(a[0], &x) &&
                    x->dim() >= 1);
  const at::ScalarType dt = x->scalar_type();
  const int code = dt == at::kBFloat16 ? LISAQ_DTYPE_BF16 : dt == at::kHalf ? LISAQ_DTYPE_F16
                   : dt == at::kFloat  ? LISAQ_DTYPE_F32
                                       : -1;
  LISAQ_NONE_UNLESS(code >= 0 && q.read(a + 1, 2, dt, x->device()) && !modes_active());
  const int64_t K = x->size(-1), N = q.w->size(0);
  LISAQ_NONE_UNLESS(K > 0 && N > 0 && x->numel() > 0 && q.shape(N, K, gs, bits));
  const int64_t M = x->numel() / K;
  const bool typed = code != LISAQ_DTYPE_BF16 || bits == 8;
  LISAQ_NONE_UNLESS(!(typed && serial));
  Tensor y;
  int rc;
  {
    NoGil nogil;
    size_t bytes = 0;
    if (!typed || (code != LISAQ_DTYPE_F32 && M >= lisaq_qmv_batch_limit(K, N)))
      bytes = lisaq_quantized_matmul_workspace(M, N, K, (int)gs, (int)bits);
    void* const st = stream_of(*x);
    Outputs o(*x, N, bytes, st);
    if (typed)
      rc = lisaq_quantized_matmul_typed(st, x->data_ptr(), q.codes_ptr(), q.s->data_ptr(), q.b->data_ptr(),
                                        o.y.data_ptr(), M, N, K, 1, (int)gs, (int)bits, code, o.wp, bytes);
    else if (serial)
      rc = lisaq_quantized_matmul_serial_rows(st, x->data_ptr(), q.codes_ptr(), q.s->data_ptr(), q.b->data_ptr(),
                                              o.y.data_ptr(), M, N, K, 1, (int)gs, (int)bits, o.wp, bytes);
    else
      rc = lisaq_quantized_matmul(st, x->data_ptr(), q.codes_ptr(), q.s->data_ptr(), q.b->data_ptr(), o.y.data_ptr(),
                                  M, N, K, 1, (int)gs, (int)bits, o.wp, bytes);
    y = std::move(o.y);
  }
  LISAQ_NONE_UNLESS(rc == LISAQ_OK);
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// addnorm(x, r, norm_weight, w, scales, biases, eps, group_size, bits) -> (y, sum, normed)
PyObject* addnorm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int64_t gs, bits;
  const Tensor *x, *r, *nw;
  Packed q;
  LISAQ_NONE_UNLESS(n == 9 && format(a[7], a[8], &gs, &bits) && PyFloat_CheckExact(a[6]) && plain(a[0], &x) &&
                    plain(a[1], &r) && plain(a[2], &nw) && x->dim() == 2 && r->sizes() == x->sizes() &&
                    x->scalar_type() == at::kBFloat16 && r->scalar_type() == at::kBFloat16 &&
                    nw->scalar_type() == at::kBFloat16 && r->device() == x->device() && nw->device() == x->device() &&
                    q.read(a + 3, 2, at::kBFloat16, x->device()) && !modes_active());
  const int64_t M = x->size(0), K = x->size(1), N = q.w->size(0);
  LISAQ_NONE_UNLESS(M > 0 && K > 0 && N > 0 && nw->numel() == K && q.shape(N, K, gs, bits));
  Tensor y, sum, normed;
  int rc;
  {
    NoGil nogil;
    const size_t bytes = lisaq_quantized_matmul_workspace(M, N, K, (int)gs, (int)bits);
    void* const st = stream_of(*x);
    Outputs o(*x, N, bytes, st);
    sum = output(*x, K);
    normed = output(*x, K);
    rc = lisaq_qmv_addnorm(st, x->data_ptr(), r->data_ptr(), nw->data_ptr(), q.codes_ptr(), q.s->data_ptr(),
                           q.b->data_ptr(), sum.data_ptr(), normed.data_ptr(), o.y.data_ptr(), M, N, K,
                           (float)PyFloat_AS_DOUBLE(a[6]), (int)gs, (int)bits, o.wp, bytes);
    y = std::move(o.y);
  }
  LISAQ_NONE_UNLESS(rc == LISAQ_OK);
  PyObject* out = PyTuple_New(3);
  if (!out) return nullptr;
  PyTuple_SET_ITEM(out, 0, THPVariable_Wrap(std::move(y)));
  PyTuple_SET_ITEM(out, 1, THPVariable_Wrap(std::move(sum)));
  PyTuple_SET_ITEM(out, 2, THPVariable_Wrap(std::move(normed)));
  return out;
  END_HANDLE_TH_ERRORS
}

// swiglu(gate, up) -> act
PyObject* swiglu(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const Tensor *g, *u;
  LISAQ_NONE_UNLESS(n == 2 && plain(a[0], &g) && plain(a[1], &u) && g->sizes() == u->sizes() &&
                    g->scalar_type() == at::kBFloat16 && u->scalar_type() == at::kBFloat16 &&
                    g->device() == u->device() && g->numel() > 0 && !modes_active());
  Tensor act;
  int rc;
  {
    NoGil nogil;
    act = at::empty(g->sizes(), g->options());
    rc = lisaq_swiglu(stream_of(*g), g->data_ptr(), u->data_ptr(), act.data_ptr(), g->numel());
  }
  LISAQ_NONE_UNLESS(rc == LISAQ_OK);
  return THPVariable_Wrap(std::move(act));
  END_HANDLE_TH_ERRORS
}

// moe(x, logits, gate w/s/b, up w/s/b, down w/s/b, top_k, group_size, bits, workspace) -> y, the shape of x.
// The workspace is the op's own zeroed buffer (its decode flags outlive a call); None where it is too small.
PyObject* moe(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int64_t k, gs, bits;
  const Tensor *x, *lg, *ws;
  Packed g, u, d;
  LISAQ_NONE_UNLESS(n == 15 && integer(a[11], &k) && format(a[12], a[13], &gs, &bits) && bits != 8 &&
                    plain(a[0], &x) && plain(a[1], &lg) && plain(a[14], &ws) && x->scalar_type() == at::kBFloat16 &&
                    lg->scalar_type() == at::kFloat && ws->scalar_type() == at::kByte && x->dim() >= 1 &&
                    lg->dim() >= 1 && x->numel() > 0 && lg->numel() > 0 && lg->device() == x->device() &&
                    ws->device() == x->device() && g.read(a + 2, 3, at::kBFloat16, x->device()) &&
                    u.read(a + 5, 3, at::kBFloat16, x->device()) && d.read(a + 8, 3, at::kBFloat16, x->device()) &&
                    !modes_active());
  const int64_t H = x->size(-1), T = x->numel() / H, E = lg->size(-1), I = g.w->size(1);
  LISAQ_NONE_UNLESS(k >= 1 && k <= E && E <= 1024 && I > 0 && lg->numel() == T * E && g.w->size(0) == E &&
                    u.w->size(0) == E && d.w->size(0) == E && H % gs == 0 && I % gs == 0 && g.shape(I, H, gs, bits) &&
                    u.shape(I, H, gs, bits) && d.shape(H, I, gs, bits));
  LISAQ_NONE_UNLESS((size_t)ws->numel() >= lisaq_moe_workspace(T, H, I, (int)E, (int)k, (int)gs, (int)bits));
  Tensor out;
  int rc;
  {
    NoGil nogil;
    out = at::empty(x->sizes(), x->options());
    // the launches of one call stay together on a stream: the next call's use the same workspace
    static std::mutex mu;
    std::lock_guard<std::mutex> lock(mu);
    rc = lisaq_moe_forward(
        stream_of(*x), x->data_ptr(), static_cast<const float*>(lg->data_ptr()), g.codes_ptr(), g.s->data_ptr(),
        g.b->data_ptr(), u.codes_ptr(), u.s->data_ptr(), u.b->data_ptr(), d.codes_ptr(), d.s->data_ptr(),
        d.b->data_ptr(), out.data_ptr(), T, H, I, (int)E, (int)k, (int)gs, (int)bits, nullptr, nullptr, ws->data_ptr(),
        (size_t)ws->numel());
  }
  LISAQ_NONE_UNLESS(rc == LISAQ_OK);
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// dequantize(w, scales, biases, group_size, bits) -> bf16 [..., K]
PyObject* dequantize(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int64_t gs, bits;
  const Tensor *w, *s, *b;
  LISAQ_NONE_UNLESS(n == 5 && format(a[3], a[4], &gs, &bits) && plain(a[0], &w) && plain(a[1], &s) &&
                    plain(a[2], &b) && codes(*w) && s->scalar_type() == at::kBFloat16 &&
                    b->scalar_type() == at::kBFloat16 && w->dim() >= 1 && w->numel() > 0 &&
                    s->device() == w->device() && b->device() == w->device() && !modes_active());
  const int64_t K = w->size(-1) * 32 / bits, rows = w->numel() / w->size(-1);
  LISAQ_NONE_UNLESS(K % gs == 0 && s->numel() == rows * (K / gs) && b->numel() == s->numel());
  c10::SmallVector<int64_t, 5> sizes(w->sizes().begin(), w->sizes().end());
  sizes.back() = K;
  Tensor out;
  int rc;
  {
    NoGil nogil;
    out = at::empty(sizes, s->options());
    rc = lisaq_dequantize(stream_of(*w), static_cast<const uint32_t*>(w->data_ptr()), s->data_ptr(), b->data_ptr(),
                          out.data_ptr(), rows, K, (int)gs, (int)bits);
  }
  LISAQ_NONE_UNLESS(rc == LISAQ_OK);
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// quantize(w, group_size, bits) -> (codes, scales, biases)
PyObject* quantize(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int64_t gs, bits;
  const Tensor* w;
  LISAQ_NONE_UNLESS(n == 3 && format(a[1], a[2], &gs, &bits) && plain(a[0], &w) && w->dim() >= 1 && w->numel() > 0 &&
                    (w->scalar_type() == at::kBFloat16 || w->scalar_type() == at::kFloat) && !modes_active());
  const int64_t K = w->size(-1), rows = w->numel() / K;
  LISAQ_NONE_UNLESS(K % gs == 0 && gs % (32 / bits) == 0);
  c10::SmallVector<int64_t, 5> sizes(w->sizes().begin(), w->sizes().end());
  sizes.back() = K * bits / 32;
  Tensor wq, s, b;
  int rc;
  {
    NoGil nogil;
    wq = at::empty(sizes, w->options().dtype(at::kInt));
    sizes.back() = K / gs;
    s = at::empty(sizes, w->options());
    b = at::empty(sizes, w->options());
    rc = lisaq_quantize(stream_of(*w), w->data_ptr(),
                        w->scalar_type() == at::kFloat ? LISAQ_DTYPE_F32 : LISAQ_DTYPE_BF16,
                        static_cast<uint32_t*>(wq.data_ptr()), s.data_ptr(), b.data_ptr(), rows, K, (int)gs, (int)bits);
  }
  LISAQ_NONE_UNLESS(rc == LISAQ_OK);
  PyObject* out = PyTuple_New(3);
  if (!out) return nullptr;
  PyTuple_SET_ITEM(out, 0, THPVariable_Wrap(std::move(wq)));
  PyTuple_SET_ITEM(out, 1, THPVariable_Wrap(std::move(s)));
  PyTuple_SET_ITEM(out, 2, THPVariable_Wrap(std::move(b)));
  return out;
  END_HANDLE_TH_ERRORS
}

PyMethodDef kMethods[] = {
    {"dequantize", (PyCFunction)(void (*)(void))dequantize, METH_FASTCALL, nullptr},
    {"quantize", (PyCFunction)(void (*)(void))quantize, METH_FASTCALL, nullptr},
    {"linear", (PyCFunction)(void (*)(void))linear, METH_FASTCALL, nullptr},
    {"addnorm", (PyCFunction)(void (*)(void))addnorm, METH_FASTCALL, nullptr},
    {"swiglu", (PyCFunction)(void (*)(void))swiglu, METH_FASTCALL, nullptr},
    {"moe", (PyCFunction)(void (*)(void))moe, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_pyops", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__pyops(void) { return PyModule_Create(&kModule); }
