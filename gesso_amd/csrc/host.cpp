// The launches that a prompt's step makes most, without the interpreter between the check of an operand and the launch.
//
// A short prompt's step is some 115 calls, and what stands between two of them is the host: a call of the Python functions takes some
// 10 us, of which the launch itself is 2 (LFM2-350M sizes, 13 tokens 1,620 us a step on the host, with these functions 880 to 980;
// 333 tokens with all logits 1,550 and 1,100 to 1,220, of which the device needs 1,100).  A function here takes the operands of one call in its
// plainest form (ordinary tensors, a result made here or room for it), checks all that the Python function of the same name checks,
// makes the result and launches.  Whatever is in another form, or wrong, comes back as False, and the Python function goes on: it
// handles the other forms and words the errors.
#include <Python.h>

#include <ATen/ATen.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include <dlfcn.h>

#include "native_calls.h"

namespace {

typedef hipStream_t stream_t;
enum { F32 = 0, BF16 = 1 };

PyObject* kernel_error;

// The library's entry points, found by name.
decltype(&gs_last_error) last_error;
#define ENTRY(name) decltype(&gs_##name) name##_
ENTRY(add_rmsnorm);
ENTRY(gemm_skinny);
ENTRY(gemm_mid_takes);
ENTRY(gemm_mid);
ENTRY(gemm_mid_swiglu_scaled);
ENTRY(gemm_mid_residual_sums);
ENTRY(gemm_mid_residual);
ENTRY(gemm_mid_parts);
ENTRY(residual_from_parts);
ENTRY(short_conv);
ENTRY(qknorm_rope_kv);
ENTRY(attention_prefill);
#undef ENTRY

// ------------------------------------------------------------------ arguments and results

const at::Tensor no_tensor;

// A tensor on the GPU, or one that is not defined (None, or anything else: `other` is set for that).
const at::Tensor& tensor(PyObject* o, bool& other) {
  if (o == Py_None) return no_tensor;
  if (THPVariable_Check(o)) {
    const at::Tensor& t = THPVariable_Unpack(o);
    if (t.is_cuda()) return t;
  }
  other = true;
  return no_tensor;
}

bool is(const at::Tensor& t, at::ScalarType type) { return t.defined() && t.scalar_type() == type; }
bool vector(const at::Tensor& t, int64_t n) { return is(t, at::kFloat) && t.dim() == 1 && t.size(0) == n && t.is_contiguous(); }
bool matrix(const at::Tensor& t, at::ScalarType type) { return is(t, type) && t.dim() == 2; }
bool indices(const at::Tensor& t, int64_t least) { return is(t, at::kInt) && t.numel() >= least && t.is_contiguous(); }
bool activations(const at::Tensor& t) { return is(t, at::kBFloat16) || is(t, at::kFloat); }
int kind(const at::Tensor& t) { return t.scalar_type() == at::kBFloat16 ? BF16 : F32; }
bool aligned(const at::Tensor& t) { return ((uintptr_t)t.data_ptr() & 15) == 0; }
void* at_(const at::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
float* floats(const at::Tensor& t) { return (float*)at_(t); }
const int* ints(const at::Tensor& t) { return (const int*)at_(t); }
at::Tensor make(const at::Tensor& like, at::IntArrayRef sizes, at::ScalarType type) { return at::empty(sizes, like.options().dtype(type)); }

// Numbers as the interpreter holds them (a wrong type leaves a Python error, which `call` turns into "another form").
int number(PyObject* o) { return (int)PyLong_AsLong(o); }
float real(PyObject* o) { return (float)PyFloat_AsDouble(o); }
stream_t stream(PyObject* o) { return (stream_t)PyLong_AsVoidPtr(o); }

PyObject* other_form() {
  PyErr_Clear();
  Py_RETURN_FALSE;
}

// A tensor as Python's.  It is made before the launch: nothing may fail behind one, or the Python function would make it once more.
THPObjectPtr result(const at::Tensor& t) {
  THPObjectPtr y(THPVariable_Wrap(t));
  if (!y) throw std::bad_alloc();
  return y;
}

struct Failed {};                       // an entry point refused: its message is the error

// The interpreter's lock let go of, and taken back however the block ends.
struct Unlocked {
  PyThreadState* const held = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(held); }
};

// A launch without the lock.  The operands' addresses are this function's arguments: asking for one can throw (a tensor that has no
// memory), and does so while the lock is still held.
template <typename... P, typename... A>
void launch(int (*entry)(P...), A... a) {
  int rc;
  {
    const Unlocked unlocked;
    rc = entry(a...);
  }
  if (rc != 0) throw Failed();
}

// One function as Python calls it: `N` arguments; an exception of torch's is another form too (a tensor without memory, say).
template <PyObject* (*BODY)(PyObject* const*), int N>
PyObject* call(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != N) {
    PyErr_Format(PyExc_TypeError, "%d arguments, %d given", N, (int)n);
    return nullptr;
  }
  try {
    PyObject* r = BODY(a);
    if (PyErr_Occurred()) {
      Py_XDECREF(r);
      return other_form();
    }
    return r;
  } catch (const Failed&) {
    PyErr_SetString(kernel_error, last_error());
    return nullptr;
  } catch (const std::exception&) {
    return other_form();
  }
}

// ------------------------------------------------------------------ the launches

// res, delta or None, weight, eps, whether the result is bfloat16, stream
PyObject* add_rmsnorm(PyObject* const* a) {
  bool other = false;
  const at::Tensor &res = tensor(a[0], other), &delta = tensor(a[1], other), &w = tensor(a[2], other);
  const float eps = real(a[3]);
  const int type = number(a[4]);
  const stream_t s = stream(a[5]);
  if (other || PyErr_Occurred() || !matrix(res, at::kFloat) || !res.is_contiguous() || !vector(w, res.size(1))) return other_form();
  if (delta.defined() && !(activations(delta) && delta.is_contiguous() && delta.sizes() == res.sizes())) return other_form();
  const int T = (int)res.size(0), H = (int)res.size(1);
  at::Tensor out = make(res, {T, H}, type == BF16 ? at::kBFloat16 : at::kFloat);
  THPObjectPtr y = result(out);
  launch(add_rmsnorm_, floats(res), at_(delta), delta.defined() ? kind(delta) : type, floats(w), eps, out.data_ptr(), type, nullptr, T, H, s);
  return y.release();
}

// x, w, its tile-major copy or None, whether the result is bfloat16, whether SwiGLU, stream
PyObject* gemm_skinny(PyObject* const* a) {
  bool other = false;
  const at::Tensor &x = tensor(a[0], other), &w = tensor(a[1], other), &wt = tensor(a[2], other);
  const int type = number(a[3]), swiglu = number(a[4]);
  const stream_t s = stream(a[5]);
  if (other || PyErr_Occurred() || !matrix(x, at::kBFloat16) || !matrix(w, at::kBFloat16)) return other_form();
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  if (M > 64 || K % 8 != 0 || w.size(1) != K || x.stride(1) != 1 || (M > 1 && x.stride(0) % 8 != 0) || !w.is_contiguous() || !aligned(x) ||
      !aligned(w))
    return other_form();
  const int64_t cols = swiglu ? N / 2 : N;
  at::Tensor out = make(x, {M, cols}, type == BF16 ? at::kBFloat16 : at::kFloat);
  THPObjectPtr y = result(out);
  launch(gemm_skinny_, x.data_ptr(), M > 1 ? (int)x.stride(0) : (int)K, 0, nullptr, nullptr, 0, nullptr, 0.f, w.data_ptr(), at_(wt),
         out.data_ptr(), type, (int)cols, (int)M, (int)N, (int)K, swiglu, 0, s);
  return y.release();
}

// bfloat16 rows that do not overlap and the whole weight with its tile-major copy, as the products of some hundred rows take them
bool mid_operands(const at::Tensor& x, const at::Tensor& w, const at::Tensor& wt) {
  if (!matrix(x, at::kBFloat16) || !matrix(w, at::kBFloat16) || !matrix(wt, at::kBFloat16)) return false;
  const int64_t K = x.size(1), ld = x.stride(0);
  return x.stride(1) == 1 && ld >= K && ld % 8 == 0 && aligned(x) && K == w.size(1) && wt.sizes() == w.sizes() && w.is_contiguous() &&
         wt.is_contiguous();
}

// x, w, its tile-major copy, whether SwiGLU, stream
PyObject* gemm_mid(PyObject* const* a) {
  bool other = false;
  const at::Tensor &x = tensor(a[0], other), &w = tensor(a[1], other), &wt = tensor(a[2], other);
  const int swiglu = number(a[3]);
  const stream_t s = stream(a[4]);
  if (other || PyErr_Occurred() || !mid_operands(x, w, wt)) return other_form();
  const int M = (int)x.size(0), K = (int)x.size(1), N = (int)w.size(0), cols = swiglu ? N / 2 : N;
  if (!gemm_mid_takes_(M, N, K, swiglu)) return other_form();
  at::Tensor out = make(x, {M, cols}, at::kBFloat16);
  THPObjectPtr y = result(out);
  launch(gemm_mid_, x.data_ptr(), (int)x.stride(0), wt.data_ptr(), out.data_ptr(), cols, M, N, K, swiglu, s);
  return y.release();
}

bool stream_of(const at::Tensor& res, const at::Tensor& x, const at::Tensor& w) {
  return matrix(res, at::kFloat) && res.size(0) == x.size(0) && res.size(1) == w.size(0) && res.is_contiguous();
}

// x, w, its tile-major copy, the stream, the next norm's weight, stream: the weighted rows and their partial sums of squares
PyObject* gemm_mid_residual(PyObject* const* a) {
  bool other = false;
  const at::Tensor &x = tensor(a[0], other), &w = tensor(a[1], other), &wt = tensor(a[2], other), &res = tensor(a[3], other),
                   &nw = tensor(a[4], other);
  const stream_t s = stream(a[5]);
  if (other || PyErr_Occurred() || !mid_operands(x, w, wt) || !stream_of(res, x, w) || !vector(nw, w.size(0))) return other_form();
  const int M = (int)x.size(0), K = (int)x.size(1), N = (int)w.size(0), sums = gemm_mid_residual_sums_(M, N, K);
  if (sums <= 0) return other_form();
  at::Tensor rows = make(x, {M, N}, at::kBFloat16), ssq = make(x, {M, sums}, at::kFloat);
  const THPObjectPtr first = result(rows), second = result(ssq);
  THPObjectPtr y(Py_BuildValue("(OO)", first.get(), second.get()));
  if (!y) return nullptr;
  launch(gemm_mid_residual_, x.data_ptr(), (int)x.stride(0), wt.data_ptr(), floats(res), floats(nw), rows.data_ptr(), floats(ssq), M, N, K, s);
  return y.release();
}

// weighted rows, their partial sums of squares, eps, gate's and up's weight, its tile-major copy, stream
PyObject* gemm_mid_swiglu_scaled(PyObject* const* a) {
  bool other = false;
  const at::Tensor &x = tensor(a[0], other), &ssq = tensor(a[1], other), &w = tensor(a[3], other), &wt = tensor(a[4], other);
  const float eps = real(a[2]);
  const stream_t s = stream(a[5]);
  if (other || PyErr_Occurred() || !mid_operands(x, w, wt) || !matrix(ssq, at::kFloat) || !ssq.is_contiguous()) return other_form();
  const int M = (int)x.size(0), K = (int)x.size(1), N = (int)w.size(0), sums = (int)ssq.size(1);
  if (ssq.size(0) != M || sums > 128 || sums % 4 != 0 || !gemm_mid_takes_(M, N, K, 1)) return other_form();
  at::Tensor out = make(x, {M, N / 2}, at::kBFloat16);
  THPObjectPtr y = result(out);
  launch(gemm_mid_swiglu_scaled_, x.data_ptr(), (int)x.stride(0), floats(ssq), sums, eps, wt.data_ptr(), out.data_ptr(), N / 2, M, N, K, s);
  return y.release();
}

// x, w, its tile-major copy, the stream, the next norm's weight, eps, parts of K (more than none), stream: the normed rows
PyObject* gemm_mid_residual_parts(PyObject* const* a) {
  bool other = false;
  const at::Tensor &x = tensor(a[0], other), &w = tensor(a[1], other), &wt = tensor(a[2], other), &res = tensor(a[3], other),
                   &nw = tensor(a[4], other);
  const float eps = real(a[5]);
  const int parts = number(a[6]);
  const stream_t s = stream(a[7]);
  if (other || PyErr_Occurred() || parts <= 0 || !mid_operands(x, w, wt) || !stream_of(res, x, w) || !vector(nw, w.size(0))) return other_form();
  const int M = (int)x.size(0), K = (int)x.size(1), N = (int)w.size(0);
  const int64_t sheet = (int64_t)parts * M * N;
  at::Tensor sheets = make(x, {sheet + M}, at::kFloat), normed = make(x, {M, N}, at::kBFloat16);       // (and the new rows' sums of squares)
  THPObjectPtr y = result(normed);
  float *part = floats(sheets), *stream_at = floats(res), *next = floats(nw);
  launch(gemm_mid_parts_, x.data_ptr(), (int)x.stride(0), wt.data_ptr(), part, parts, M, N, K, s);
  launch(residual_from_parts_, part, parts, stream_at, part + sheet, next, eps, normed.data_ptr(), BF16, 0, M, N, s);
  return y.release();
}

// bcx, taps, bias or None, state, seq_of_token, q_start, slots, sequences, whether all bring one token, stream
PyObject* short_conv(PyObject* const* a) {
  bool other = false;
  const at::Tensor &bcx = tensor(a[0], other), &taps = tensor(a[1], other), &bias = tensor(a[2], other), &state = tensor(a[3], other),
                   &seq = tensor(a[4], other), &start = tensor(a[5], other), &slots = tensor(a[6], other);
  const int nseq = number(a[7]), single = number(a[8]);
  const stream_t s = stream(a[9]);
  if (other || PyErr_Occurred() || !activations(bcx) || bcx.dim() != 2 || !bcx.is_contiguous() || bcx.size(1) % 3 != 0) return other_form();
  const int T = (int)bcx.size(0), H = (int)bcx.size(1) / 3;
  if (!matrix(taps, at::kFloat) || !taps.is_contiguous() || taps.size(0) != H || (bias.defined() && !vector(bias, H))) return other_form();
  const int W = (int)taps.size(1);
  if (!is(state, at::kFloat) || state.dim() != 3 || state.size(1) != H || state.size(2) != W - 1 || !state.is_contiguous()) return other_form();
  if (!indices(seq, T) || !indices(start, nseq + 1) || !indices(slots, nseq)) return other_form();
  at::Tensor out = make(bcx, {T, H}, bcx.scalar_type());
  THPObjectPtr y = result(out);
  launch(short_conv_, bcx.data_ptr(), kind(bcx), floats(taps), floats(bias), floats(state), ints(seq), ints(start), ints(slots), out.data_ptr(),
         T, nseq, H, W, single ? 1 : 0, s);
  return y.release();
}

// caches (pages, nkv, page_size, d) of one type and one shape
bool caches(const at::Tensor& k, const at::Tensor& v, at::ScalarType type, int64_t nkv, int64_t page, int64_t d) {
  return is(k, type) && is(v, type) && k.dim() == 4 && k.size(1) == nkv && k.size(2) == page && k.size(3) == d && v.sizes() == k.sizes() &&
         k.is_contiguous() && v.is_contiguous();
}

// qkv, q's and k's head norm or None, eps, cos, sin, rotary_dim, positions, seq_of_token, block_table, page_size, caches, nh, nkv, d,
// whether k and v are written, whether pairs are interleaved, stream
PyObject* qknorm_rope_kv(PyObject* const* a) {
  bool other = false;
  const at::Tensor &qkv = tensor(a[0], other), &qw = tensor(a[1], other), &kw = tensor(a[2], other), &cos = tensor(a[4], other),
                   &sin = tensor(a[5], other), &pos = tensor(a[7], other), &seq = tensor(a[8], other), &table = tensor(a[9], other),
                   &kc = tensor(a[11], other), &vc = tensor(a[12], other);
  const float eps = real(a[3]);
  const int rot = number(a[6]), page = number(a[10]), nh = number(a[13]), nkv = number(a[14]), d = number(a[15]), write = number(a[16]),
            pairs = number(a[17]);
  const stream_t s = stream(a[18]);
  if (other || PyErr_Occurred() || !activations(qkv) || qkv.dim() != 2 || !qkv.is_contiguous() || qkv.size(1) < (int64_t)(nh + 2 * nkv) * d) return other_form();
  if ((qw.defined() && !vector(qw, d)) || (kw.defined() && !vector(kw, d))) return other_form();
  if ((cos.defined() && !cos.is_contiguous()) || (sin.defined() && !sin.is_contiguous())) return other_form();
  const int T = (int)qkv.size(0);
  int most = 0;
  if (rot) {
    if (!matrix(cos, at::kFloat) || !matrix(sin, at::kFloat) || cos.sizes() != sin.sizes() || cos.size(1) != rot / 2)
      return other_form();
    most = (int)cos.size(0);
  }
  if (!indices(pos, T) || !indices(seq, T) || !matrix(table, at::kInt) || !table.is_contiguous()) return other_form();
  if (!caches(kc, vc, qkv.scalar_type(), nkv, page, d)) return other_form();
  launch(qknorm_rope_kv_, qkv.data_ptr(), kind(qkv), floats(qw), floats(kw), eps, floats(cos), floats(sin), rot, pairs ? 1 : 0, most, ints(pos),
         ints(seq), ints(table), (int)table.size(1), page, kc.data_ptr(), vc.data_ptr(), T, nh, nkv, d, write ? 1 : 0, d, nullptr,
         nullptr, (int)qkv.size(1), 0, nullptr, 0, nullptr, 1, s);
  Py_RETURN_NONE;
}

// q, q_stride, caches, positions, tiles (3, n), block_table, page_size, window or 0, scale, nh, nkv, d, tokens, rows a tile, the result's
// room or None, stream
PyObject* attention_prefill(PyObject* const* a) {
  bool other = false;
  const at::Tensor &q = tensor(a[0], other), &kc = tensor(a[2], other), &vc = tensor(a[3], other), &pos = tensor(a[4], other),
                   &tiles = tensor(a[5], other), &table = tensor(a[6], other), &room = tensor(a[15], other);
  const int ld = number(a[1]), page = number(a[7]), window = number(a[8]), nh = number(a[10]), nkv = number(a[11]), d = number(a[12]),
            tokens = number(a[13]), rows = number(a[14]);
  const float scale = real(a[9]);
  const stream_t s = stream(a[16]);
  if (other || PyErr_Occurred() || !is(q, at::kBFloat16) || !q.is_contiguous() || !caches(kc, vc, at::kBFloat16, nkv, page, d)) return other_form();
  if (tokens < 1 || q.numel() < (int64_t)(tokens - 1) * ld + (int64_t)nh * d || !indices(pos, tokens) || !matrix(tiles, at::kInt) ||
      tiles.size(0) != 3 || !tiles.is_contiguous() || !matrix(table, at::kInt) || !table.is_contiguous())
    return other_form();
  if (room.defined() && !(matrix(room, at::kBFloat16) && room.size(0) == tokens && room.size(1) == (int64_t)nh * d && room.is_contiguous()))
    return other_form();
  const int n = (int)tiles.size(1);
  const int* at = ints(tiles);
  at::Tensor out = room.defined() ? room : make(q, {tokens, (int64_t)nh * d}, at::kBFloat16);
  THPObjectPtr y = result(out);
  launch(attention_prefill_, q.data_ptr(), ld, kc.data_ptr(), vc.data_ptr(), ints(pos), at, at + n, at + 2 * n, n, ints(table), (int)table.size(1),
         page, window, scale, out.data_ptr(), nh, nkv, d, rows, 0, 0, 0.f, 0, nullptr, s);
  return y.release();
}

// ------------------------------------------------------------------ the module

// The library's path and the class of its errors: once, before any other call.
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 2 || !PyUnicode_Check(a[0])) {
    PyErr_SetString(PyExc_TypeError, "bind(path, error class)");
    return nullptr;
  }
  void* lib = dlopen(PyUnicode_AsUTF8(a[0]), RTLD_NOW | RTLD_LOCAL);
  if (!lib) {
    PyErr_SetString(PyExc_OSError, dlerror());
    return nullptr;
  }
  bool all = true;
  auto get = [&](const char* name) {
    void* f = dlsym(lib, name);
    all = all && f;
    return f;
  };
#define GET(name) name##_ = (decltype(name##_))get("gs_" #name)
  GET(add_rmsnorm); GET(gemm_skinny); GET(gemm_mid_takes); GET(gemm_mid); GET(gemm_mid_swiglu_scaled); GET(gemm_mid_residual_sums);
  GET(gemm_mid_residual); GET(gemm_mid_parts); GET(residual_from_parts); GET(short_conv); GET(qknorm_rope_kv); GET(attention_prefill);
#undef GET
  last_error = (decltype(last_error))get("gs_last_error");
  const auto version = (decltype(&gs_abi_version))get("gs_abi_version");
  if (!all || version() != GS_ABI_VERSION) {
    PyErr_SetString(PyExc_OSError, all ? "module and kernel library have other interface versions; build them again" : "the kernel library lacks an entry point");
    return nullptr;
  }
  Py_INCREF(a[1]);
  kernel_error = a[1];
  Py_RETURN_NONE;
}

#define METHOD(name, n) {#name, (PyCFunction)(void*)(&call<name, n>), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {{"bind", (PyCFunction)(void*)(&bind), METH_FASTCALL, nullptr},
                         METHOD(add_rmsnorm, 6), METHOD(gemm_skinny, 6), METHOD(gemm_mid, 5), METHOD(gemm_mid_residual, 6),
                         METHOD(gemm_mid_swiglu_scaled, 6), METHOD(gemm_mid_residual_parts, 8), METHOD(short_conv, 10),
                         METHOD(qknorm_rope_kv, 19), METHOD(attention_prefill, 17), {nullptr, nullptr, 0, nullptr}};
PyModuleDef definition = {PyModuleDef_HEAD_INIT, "gesso_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_gesso_host() { return PyModule_Create(&definition); }
