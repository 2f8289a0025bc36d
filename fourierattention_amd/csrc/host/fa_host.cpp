// The host side of the calls a decode step makes, as a CPython module on torch tensors (fourierattention_amd._fa_host).
//
// A decode step of one layer is three launches of a few microseconds each; filling the argument blocks of the C ABI
// field by field from Python took longer than the launches (53 us of host work per layer for 35 us of kernels at 2600
// tokens).  The functions below take the tensors themselves on every call, check them, fill the argument block and
// launch on the caller's stream; they keep nothing between calls.
#include <Python.h>

#include <ATen/ATen.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <vector>

#include "../../../include/fourier_attn_hip.h"

namespace {

PyObject* g_stream_fn = nullptr;      // device index -> raw handle of torch's current stream
PyObject* g_check_fn = nullptr;       // status -> raises the package's exception
PyObject* g_workspace_fn = nullptr;   // (device, bytes, tag) -> uint8 tensor of at least that size

// interned attribute names of a page store
PyObject *s_data, *s_cap_pages, *s_batch_stride, *s_pad_h32, *s_max_pad, *s_pad_h_host, *s_n_list32, *s_n_h32, *s_Cn, *s_Hkv, *s_decode;

struct PyError {};   // a Python exception is set

[[noreturn]] void fail(PyObject* type, const char* msg) {
  PyErr_SetString(type, msg);
  throw PyError{};
}
#define CHECK(cond, msg) do { if (!(cond)) fail(PyExc_AssertionError, msg); } while (0)

// owns one reference
struct Ref {
  PyObject* p;
  explicit Ref(PyObject* o) : p(o) { if (!o) throw PyError{}; }
  ~Ref() { Py_DECREF(p); }
  Ref(const Ref&) = delete;
};

// a sequence of any kind, held as a list or tuple
struct Items : Ref {
  Items(PyObject* o, const char* msg) : Ref(sequence(o, msg)) {}
  Py_ssize_t size() const { return PySequence_Fast_GET_SIZE(p); }
  PyObject* operator[](Py_ssize_t i) const { return PySequence_Fast_GET_ITEM(p, i); }
  static PyObject* sequence(PyObject* o, const char* msg) {
    PyObject* r = PySequence_Fast(o, msg);
    if (!r) {   // (what is no sequence is refused like every other operand)
      PyErr_Clear();
      fail(PyExc_AssertionError, msg);
    }
    return r;
  }
};

const at::Tensor& tensor(PyObject* o, const char* what) {
  if (!THPVariable_Check(o)) {
    PyErr_Format(PyExc_TypeError, "%s must be a tensor", what);
    throw PyError{};
  }
  return THPVariable_Unpack(o);
}
const at::Tensor& gpu_tensor(PyObject* o, const char* what) {
  const at::Tensor& t = tensor(o, what);
  if (!t.is_cuda()) {
    PyErr_Format(PyExc_RuntimeError, "%s must be a GPU tensor: the HIP kernels are the only implementation", what);
    throw PyError{};
  }
  return t;
}
int64_t integer(PyObject* o) {
  const long long v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) throw PyError{};
  return v;
}
// what int() makes of it
int64_t whole(PyObject* o) {
  if (PyLong_CheckExact(o)) return integer(o);
  return integer(Ref(PyNumber_Long(o)).p);
}
double real(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw PyError{};
  return v;
}
bool truth(PyObject* o) {
  const int v = PyObject_IsTrue(o);
  if (v < 0) throw PyError{};
  return v != 0;
}
int64_t int_attr(PyObject* o, PyObject* name) { return integer(Ref(PyObject_GetAttr(o, name)).p); }
// (the store keeps its own reference to the tensor: it outlives the call)
const at::Tensor& tensor_attr(PyObject* o, PyObject* name, const char* what) { return tensor(Ref(PyObject_GetAttr(o, name)).p, what); }

int dtype_code(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kBFloat16: return FA_BF16;
    case at::kHalf: return FA_FP16;
    case at::kFloat: return FA_FP32;
    default: fail(PyExc_TypeError, "unsupported dtype; expected bfloat16, float16 or float32");
  }
}
template <typename T = void>
T* ptr(const at::Tensor& t) { return t.numel() == 0 ? nullptr : static_cast<T*>(t.data_ptr()); }

fa_stream_t stream_of(const at::Tensor& t) {
  Ref idx(PyLong_FromLong(t.device().index()));
  Ref s(PyObject_CallOneArg(g_stream_fn, idx.p));
  return reinterpret_cast<fa_stream_t>(PyLong_AsVoidPtr(s.p));
}
void check_status(int rc) {
  if (rc == FA_OK) return;
  Ref code(PyLong_FromLong(rc));
  Ref none(PyObject_CallOneArg(g_check_fn, code.p));
  fail(PyExc_RuntimeError, "a HIP call failed");
}

// Runs f without the interpreter lock: a launch waits where the queue is full, an allocation or a copy to the host may wait for
// everything queued, and other Python threads go on meanwhile.  Whatever f needs of Python is taken beforehand, and the
// tensors behind its pointers are held.
template <typename F>
auto unlocked(F&& f) {
  struct Guard {
    PyThreadState* state = PyEval_SaveThread();
    ~Guard() { PyEval_RestoreThread(state); }
  } guard;
  return f();
}
#define LAUNCH(call) check_status(unlocked([&] { return call; }))

#define FA_BEGIN HANDLE_TH_ERRORS try {
#define FA_END } catch (const PyError&) { return nullptr; } END_HANDLE_TH_ERRORS

// (B, width) rows, or the one new token (B, heads, 1, D) of a decode step whose heads lie side by side
void token_rows(const at::Tensor& t, int64_t& batch, int64_t& width, int64_t& batch_stride) {
  batch = t.size(0);
  batch_stride = t.stride(0);
  if (t.dim() == 2) {
    CHECK(t.stride(1) == 1, "rows must be contiguous");
    width = t.size(1);
  } else {
    CHECK(t.dim() == 4 && t.size(2) == 1 && t.stride(3) == 1 && t.stride(1) == t.size(3), "the heads of a token must lie side by side");
    width = t.size(1) * t.size(3);
  }
}

// stream_update(k_new, v_new, k_ring, v_ring, evict_slot, write_slot, k_coef, v_coef, kc_list, vc_list, phase, T,
//               k_mid, v_mid, mid_pos, skip_coef)
// fills `s` from them and returns the window buffer of K; held: the memory of the page stores, which grow by replacing it
const at::Tensor& stream_args(PyObject* const* a, fa_stream_args& s, at::Tensor (&held)[2]) {
  const at::Tensor &k_new = tensor(a[0], "k_new"), &v_new = tensor(a[1], "v_new");
  const at::Tensor &k_ring = gpu_tensor(a[2], "k_ring"), &v_ring = gpu_tensor(a[3], "v_ring");
  const at::Tensor &k_coef = tensor(a[6], "k_coef"), &v_coef = tensor(a[7], "v_coef");
  const at::Tensor &kc = tensor(a[8], "kc_list"), &vc = tensor(a[9], "vc_list");
  PyObject *k_mid = a[12], *v_mid = a[13];
  int64_t B, width, vB, v_width, v_stride;
  token_rows(k_new, B, width, s.new_batch_stride);
  token_rows(v_new, vB, v_width, v_stride);
  CHECK(vB == B && v_width == width && v_stride == s.new_batch_stride, "k_new and v_new must share shape and strides");
  CHECK(k_ring.dim() == 3 && k_ring.stride(2) == 1 && v_ring.strides() == k_ring.strides() && v_ring.sizes() == k_ring.sizes() &&
        k_ring.size(0) == B && k_ring.size(2) == width, "k_ring and v_ring must share shape and strides");
  CHECK(k_new.scalar_type() == k_ring.scalar_type() && v_new.scalar_type() == k_ring.scalar_type() && k_new.is_cuda() && v_new.is_cuda(),
        "the new token must have the type of the window and be on the GPU");
  CHECK(k_coef.scalar_type() == at::kFloat && v_coef.scalar_type() == at::kFloat && kc.scalar_type() == at::kInt && vc.scalar_type() == at::kInt,
        "coefficients are float32, column lists int32");
  s.k_new = k_new.data_ptr(); s.v_new = v_new.data_ptr();
  s.k_ring = k_ring.data_ptr(); s.v_ring = v_ring.data_ptr();
  s.ring_batch_stride = k_ring.stride(0); s.ring_row_stride = k_ring.stride(1);
  s.evict_slot = (int32_t)whole(a[4]); s.write_slot = (int32_t)whole(a[5]);
  CHECK(s.evict_slot != s.write_slot && s.evict_slot < k_ring.size(1) && s.write_slot < k_ring.size(1), "window slots");
  s.k_coef = ptr<float>(k_coef); s.v_coef = ptr<float>(v_coef);
  s.kc_list = ptr<int32_t>(kc); s.vc_list = ptr<int32_t>(vc);
  s.Ck = (int32_t)kc.numel(); s.Cv = (int32_t)vc.numel();
  s.N = (int32_t)(k_coef.size(1) / 2); s.phase = whole(a[10]); s.T = (int32_t)whole(a[11]);
  held[0] = tensor_attr(k_mid, s_data, "k_mid.data"); held[1] = tensor_attr(v_mid, s_data, "v_mid.data");
  s.k_mid = held[0].data_ptr(); s.v_mid = held[1].data_ptr();
  s.k_mid_batch_stride = int_attr(k_mid, s_batch_stride); s.v_mid_batch_stride = int_attr(v_mid, s_batch_stride);
  s.cap_pages = (int32_t)int_attr(k_mid, s_cap_pages); s.mid_pos = whole(a[14]);
  CHECK(s.cap_pages == int_attr(v_mid, s_cap_pages), "the page stores of K and V must have the same capacity");
  s.kn_list = ptr<int32_t>(tensor_attr(k_mid, s_n_list32, "n_list32")); s.vn_list = ptr<int32_t>(tensor_attr(v_mid, s_n_list32, "n_list32"));
  s.kn_h_list = ptr<int32_t>(tensor_attr(k_mid, s_n_h32, "n_h32")); s.vn_h_list = ptr<int32_t>(tensor_attr(v_mid, s_n_h32, "n_h32"));
  s.k_pad_h_list = ptr<int32_t>(tensor_attr(k_mid, s_pad_h32, "pad_h32")); s.v_pad_h_list = ptr<int32_t>(tensor_attr(v_mid, s_pad_h32, "pad_h32"));
  s.Cnk = (int32_t)int_attr(k_mid, s_Cn); s.Cnv = (int32_t)int_attr(v_mid, s_Cn);
  s.B = (int32_t)B; s.Hkv = (int32_t)int_attr(k_mid, s_Hkv); s.width = (int32_t)width; s.dtype = dtype_code(k_ring);
  s.skip_coef = truth(a[15]);
  return k_ring;
}

PyObject* stream_update(PyObject*, PyObject* const* a, Py_ssize_t n) {
  FA_BEGIN
  CHECK(n == 16, "stream_update takes 16 arguments");
  fa_stream_args s{};
  at::Tensor held[2];
  const at::Tensor& k_ring = stream_args(a, s, held);
  const fa_stream_t st = stream_of(k_ring);
  LAUNCH(fa_stream_update(&s, st));
  Py_RETURN_NONE;
  FA_END
}

// one (rows, Hkv*D) segment of sink / window rows
void il_segment(fa_decode_args& d, int i, const at::Tensor& k, const at::Tensor& v, int64_t row0, int64_t rows, at::ScalarType dt) {
  if (rows <= 0) return;
  CHECK(k.dim() == 3 && k.stride(2) == 1 && v.strides() == k.strides() && v.sizes() == k.sizes(), "sink/window rows of K and V must share shape and strides");
  CHECK(k.scalar_type() == dt && v.scalar_type() == dt && k.is_cuda() && v.is_cuda(), "sink/window rows must have the type of q and be on the GPU");
  const int64_t off = row0 * k.stride(1) * (int64_t)k.element_size();
  d.k_il[i] = (const char*)k.data_ptr() + off; d.v_il[i] = (const char*)v.data_ptr() + off;
  d.il_rows[i] = (int32_t)rows; d.il_batch_stride[i] = k.stride(0); d.il_row_stride[i] = k.stride(1);
}

const float* stat(const Items& stats, Py_ssize_t i) {
  const at::Tensor& t = tensor(stats[i], "statistics");
  CHECK(t.scalar_type() == at::kFloat && t.is_contiguous(), "statistics must be contiguous float32");
  return ptr<const float>(t);
}

// decode_attn(q, il, k_mc, v_mc, k_mn, v_mn, stats_k, stats_v, lists, Hq, Hkv, L_m, T, sm_scale, out, cast, tables,
//             force_generic, balance_heads, no_fuse, pending, no_alloc, timings[, step]) -> out
// step: the arguments of stream_update as a tuple, or that in a list, which loses it when the update is launched; the update
// comes in front of the attention
// q (B, 1, Hq*D) or (B, Hq, 1, D), contiguous.  il: a sequence of up to two (k, v) pairs of row views, or (k, v, r): the
// rows of one buffer in front of and behind row r.  Sequences of any kind; whole numbers as int() takes them.
PyObject* decode_attn(PyObject*, PyObject* const* a, Py_ssize_t n) {
  FA_BEGIN
  CHECK(n == 23 || n == 24, "decode_attn takes 23 or 24 arguments");
  PyObject* step = n == 24 && a[23] != Py_None ? a[23] : nullptr;
  PyObject* step_list = step && PyList_Check(step) ? step : nullptr;
  if (step_list) {
    CHECK(PyList_GET_SIZE(step_list) == 1, "step: a list of one tuple");
    step = PyList_GET_ITEM(step_list, 0);
  }
  Ref step_held(step ? (Py_INCREF(step), step) : (Py_INCREF(Py_None), Py_None));
  CHECK(!step || (PyTuple_Check(step) && PyTuple_GET_SIZE(step) == 16 && a[20] == Py_None && !truth(a[21]) && a[22] == Py_None),
        "step: the 16 arguments of stream_update, with a workspace, no pending update and no timings");
  fa_stream_args su{};
  at::Tensor held[2], step_mem[2];
  if (step) stream_args(&PyTuple_GET_ITEM(step, 0), su, step_mem);
  const at::Tensor& q = gpu_tensor(a[0], "q");
  fa_decode_args d{};
  d.Hq = (int32_t)integer(a[9]); d.Hkv = (int32_t)integer(a[10]);
  CHECK(q.is_contiguous() && (q.dim() == 3 || q.dim() == 4) && d.Hq > 0, "q must be contiguous, (B, 1, Hq*D) or (B, Hq, 1, D)");
  const at::ScalarType dt = q.scalar_type();
  d.B = (int32_t)q.size(0);
  d.q_len = (int32_t)(q.dim() == 3 ? q.size(1) : q.size(2));
  d.D = (int32_t)(q.dim() == 3 ? q.size(2) / d.Hq : q.size(3));
  CHECK(q.dim() == 3 || q.size(1) == d.Hq, "q has another number of heads");
  d.q = q.data_ptr();
  d.dtype = dtype_code(q);
  const Items il(a[1], "il: (k, v) pairs");
  if (il.size() == 3 && THPVariable_Check(il[0])) {
    const at::Tensor &k = tensor(il[0], "k"), &v = tensor(il[1], "v");
    const int64_t cut = integer(il[2]);
    CHECK(k.dim() == 3 && cut >= 0 && cut < k.size(1), "row to leave out");
    il_segment(d, 0, k, v, 0, cut, dt);
    il_segment(d, 1, k, v, cut + 1, k.size(1) - cut - 1, dt);
  } else {
    for (Py_ssize_t i = 0; i < 2 && i < il.size(); ++i) {
      if (il[i] == Py_None) continue;
      const Items pair(il[i], "il: (k, v) pairs");
      CHECK(pair.size() == 2, "il: (k, v) pairs");
      const at::Tensor& k = tensor(pair[0], "k");
      il_segment(d, (int)i, k, tensor(pair[1], "v"), 0, k.dim() == 3 ? k.size(1) : 0, dt);
    }
  }
  d.L_m = (int32_t)whole(a[11]); d.T = (int32_t)whole(a[12]);
  const Items lists(a[8], "lists: eight int32 tensors");
  CHECK(lists.size() == 8, "lists: eight int32 tensors");
  const int32_t* lp[8];
  int32_t ln[8];
  for (int i = 0; i < 8; ++i) {
    const at::Tensor& t = tensor(lists[i], "list");
    CHECK(t.scalar_type() == at::kInt && t.is_contiguous(), "lists: contiguous int32 tensors");
    lp[i] = static_cast<const int32_t*>(t.data_ptr());
    ln[i] = (int32_t)t.numel();
  }
  d.kc_list = lp[0]; d.kc_h_list = lp[1]; d.kn_list = lp[2]; d.kn_h_list = lp[3];
  d.vc_list = lp[4]; d.vc_h_list = lp[5]; d.vn_list = lp[6]; d.vn_h_list = lp[7];
  d.Ck = ln[0]; d.Cnk = ln[2]; d.Cv = ln[4]; d.Cnv = ln[6];
  std::vector<int32_t> kpad, vpad;
  if (d.L_m > 0) {
    const at::Tensor &k_mc = tensor(a[2], "k_mc"), &v_mc = tensor(a[3], "v_mc");
    CHECK(k_mc.scalar_type() == at::kFloat && k_mc.is_contiguous() && v_mc.scalar_type() == at::kFloat && v_mc.is_contiguous() &&
          k_mc.dim() == 3 && v_mc.dim() == 3, "coefficients must be contiguous float32");
    d.N = (int32_t)((d.Ck ? k_mc : v_mc).size(1) / 2);
    d.k_mc = ptr<const float>(k_mc); d.v_mc = ptr<const float>(v_mc);
    if (THPVariable_Check(a[4])) {
      const at::Tensor &k_mn = tensor(a[4], "k_mn"), &v_mn = tensor(a[5], "v_mn");
      CHECK(k_mn.dim() == 3 && v_mn.dim() == 3 && k_mn.stride(2) == 1 && v_mn.stride(2) == 1 && k_mn.scalar_type() == dt && v_mn.scalar_type() == dt,
            "stored dims must have contiguous rows of the type of q");
      d.mid_layout = FA_MID_TOKEN_MAJOR;
      d.k_mn = ptr<>(k_mn); d.v_mn = ptr<>(v_mn);
      d.k_mn_batch_stride = k_mn.stride(0); d.k_mn_row_stride = k_mn.stride(1);
      d.v_mn_batch_stride = v_mn.stride(0); d.v_mn_row_stride = v_mn.stride(1);
    } else {
      const at::Tensor &kd = held[0] = tensor_attr(a[4], s_data, "k_mn.data"), &vd = held[1] = tensor_attr(a[5], s_data, "v_mn.data");
      CHECK(kd.scalar_type() == dt && vd.scalar_type() == dt && int_attr(a[4], s_cap_pages) == int_attr(a[5], s_cap_pages),
            "the page stores must have the type of q and one capacity");
      d.mid_layout = FA_MID_PAGED;
      d.mid_cap_pages = (int32_t)int_attr(a[4], s_cap_pages);
      d.k_mn = kd.data_ptr(); d.v_mn = vd.data_ptr();
      d.k_mn_batch_stride = int_attr(a[4], s_batch_stride); d.v_mn_batch_stride = int_attr(a[5], s_batch_stride);
      d.k_pad_h_list = ptr<const int32_t>(tensor_attr(a[4], s_pad_h32, "pad_h32"));
      d.v_pad_h_list = ptr<const int32_t>(tensor_attr(a[5], s_pad_h32, "pad_h32"));
      d.mid_max_k_pad = (int32_t)int_attr(a[4], s_max_pad); d.mid_max_v_pad = (int32_t)int_attr(a[5], s_max_pad);
      if (truth(a[18])) {
        auto host_list = [&](PyObject* store, std::vector<int32_t>& out) {
          Ref attr(PyObject_GetAttr(store, s_pad_h_host));
          Ref seq(PySequence_Fast(attr.p, "pad_h_host"));
          const Py_ssize_t len = PySequence_Fast_GET_SIZE(seq.p);
          CHECK(len == d.Hkv + 1, "pad_h_host: one entry per head and one more");
          out.resize(len);
          for (Py_ssize_t i = 0; i < len; ++i) out[i] = (int32_t)integer(PySequence_Fast_GET_ITEM(seq.p, i));
        };
        host_list(a[4], kpad);
        host_list(a[5], vpad);
        d.k_pad_h_host = kpad.data(); d.v_pad_h_host = vpad.data();
      }
    }
    const Items stats_k(a[6], "statistics: (avg_u, avg_d, scale)"), stats_v(a[7], "statistics: (avg_u, avg_d, scale)");
    CHECK(stats_k.size() == 3 && stats_v.size() == 3, "statistics: (avg_u, avg_d, scale)");
    d.avg_k_u = stat(stats_k, 0); d.avg_k_d = stat(stats_k, 1); d.scale_k = stat(stats_k, 2);
    d.avg_v_u = stat(stats_v, 0); d.avg_v_d = stat(stats_v, 1); d.scale_v = stat(stats_v, 2);
    if (a[16] != Py_None) d.tables = tensor(a[16], "tables").data_ptr();
  }
  if (a[20] != Py_None) {
    CHECK(d.L_m > 0, "a layer without mid rows has no coefficients to update");
    const Items pending(a[20], "pending: (k_row, v_row, phase, T)");
    CHECK(pending.size() == 4, "pending: (k_row, v_row, phase, T)");
    const at::Tensor &uk = tensor(pending[0], "k_row"), &uv = tensor(pending[1], "v_row");
    CHECK(uk.dim() == 2 && uk.stride(1) == 1 && uv.strides() == uk.strides() && uk.scalar_type() == dt && uv.scalar_type() == dt, "pending rows");
    d.upd_k_row = uk.data_ptr(); d.upd_v_row = uv.data_ptr(); d.upd_batch_stride = uk.stride(0);
    d.upd_phase = whole(pending[2]); d.upd_T = (int32_t)whole(pending[3]);
  }
  d.sm_scale = (float)real(a[13]);
  d.force_generic = truth(a[17]);
  d.no_fuse = (int32_t)whole(a[19]);
  at::Tensor out;
  if (a[14] != Py_None) {
    out = gpu_tensor(a[14], "out");
    CHECK(out.is_contiguous() && out.numel() == q.numel(), "out must be contiguous and as large as q");
  } else {
    const auto options = q.options().dtype(truth(a[15]) ? dt : at::kFloat);
    out = unlocked([&] { return at::empty({d.B, d.Hq, 1, d.D}, options); });
  }
  if (out.scalar_type() == at::kFloat) d.out = static_cast<float*>(out.data_ptr());
  else {
    CHECK(out.scalar_type() == dt, "out must be float32 or have the type of q");
    d.out_cast = out.data_ptr();
  }
  const fa_stream_t st = stream_of(q);
  if (truth(a[21])) {
    LAUNCH(fa_decode_attn_noalloc(&d, st));
    return a[14] != Py_None ? (Py_INCREF(a[14]), a[14]) : THPVariable_Wrap(out);
  }
  const size_t need = fa_decode_attn_workspace_bytes(d.B, d.Hq, d.Hkv, d.D, d.N, d.il_rows[0] + d.il_rows[1], d.L_m);
  Ref device(THPVariable_Check(a[0]) ? PyObject_GetAttrString(a[0], "device") : nullptr), bytes(PyLong_FromSize_t(need));
  PyObject* wargs[3] = {device.p, bytes.p, s_decode};
  Ref ws(PyObject_Vectorcall(g_workspace_fn, wargs, 3, nullptr));
  const at::Tensor& w = gpu_tensor(ws.p, "workspace");
  d.workspace = w.data_ptr(); d.workspace_bytes = (size_t)w.numel();
  if (a[22] != Py_None) {
    float ms[4];
    LAUNCH(fa_decode_attn_timed(&d, st, ms));
    Ref list(PyList_New(4));
    for (int i = 0; i < 4; ++i) PyList_SET_ITEM(list.p, i, PyFloat_FromDouble(ms[i]));
    Ref all(PySlice_New(nullptr, nullptr, nullptr));
    if (PyObject_SetItem(a[22], all.p, list.p) < 0) throw PyError{};   // timings[:] = list
  } else if (step) {
    // (the library launches the update even where it refuses the attention)
    if (step_list && PyList_SetSlice(step_list, 0, 1, nullptr) < 0) throw PyError{};
    LAUNCH(fa_decode_step(&su, &d, st));
  } else {
    LAUNCH(fa_decode_attn(&d, st));
  }
  return a[14] != Py_None ? (Py_INCREF(a[14]), a[14]) : THPVariable_Wrap(out);
  FA_END
}

// add_rmsnorm(h, delta or None, weight, eps) -> y
PyObject* add_rmsnorm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  FA_BEGIN
  CHECK(n == 4, "add_rmsnorm takes 4 arguments");
  const at::Tensor &h = gpu_tensor(a[0], "h"), &w = tensor(a[2], "weight");
  CHECK(h.is_contiguous() && w.is_contiguous() && w.scalar_type() == h.scalar_type() && h.dim() >= 1 && w.numel() == h.size(-1) && h.size(-1) > 0,
        "add_rmsnorm: h and weight contiguous, of one type, weight as long as a row");
  const void* delta = nullptr;
  if (a[1] != Py_None) {
    const at::Tensor& t = tensor(a[1], "delta");
    CHECK(t.is_contiguous() && t.sizes() == h.sizes() && t.scalar_type() == h.scalar_type(), "add_rmsnorm: delta must match h");
    delta = ptr<>(t);
  }
  at::Tensor y = unlocked([&] { return at::empty_like(h); });
  const int64_t hidden = h.size(-1);
  const float eps = (float)real(a[3]);
  const int dtype = dtype_code(h);
  const fa_stream_t st = stream_of(h);
  LAUNCH(fa_add_rmsnorm(h.data_ptr(), delta, w.data_ptr(), y.data_ptr(), (int)(h.numel() / hidden), (int)hidden, eps, dtype, st));
  return THPVariable_Wrap(y);
  FA_END
}

// distance of the rows of a (..., width) tensor whose rows are evenly spaced (the width for a single row, whatever its
// view reports)
int64_t row_stride(const at::Tensor& t) {
  CHECK(t.stride(-1) == 1 || t.size(-1) == 1, "rows must be contiguous");
  int64_t step = 0, span = 0;
  for (int64_t i = t.dim() - 2; i >= 0; --i) {
    if (t.size(i) == 1) continue;
    if (step == 0) step = t.stride(i);
    else CHECK(t.stride(i) == span, "rows are not evenly spaced");
    span = t.stride(i) * t.size(i);
  }
  return step == 0 ? t.size(-1) : step;
}

// linear_packed(x, packed weight, k, n_out[, norm weight or None, eps, residual or None, gated]) -> (..., n_out), or
// (..., n_out / 2) when gated, or the residual, added to in place
PyObject* linear_packed(PyObject*, PyObject* const* a, Py_ssize_t n) {
  FA_BEGIN
  CHECK(n == 4 || n == 8, "linear_packed takes 4 or 8 arguments");
  const at::Tensor &x = gpu_tensor(a[0], "x"), &w = gpu_tensor(a[1], "weight");
  const int64_t k = integer(a[2]), n_out = integer(a[3]);
  CHECK(x.scalar_type() == w.scalar_type() && x.dim() >= 1 && k > 0 && x.size(-1) == k && w.numel() == k * n_out, "linear_packed: x does not fit the weight");
  const int rows = (int)(x.numel() / k), dtype = dtype_code(x);
  const int64_t stride = row_stride(x);
  const fa_stream_t st = stream_of(x);
  const void* norm = nullptr;
  float eps = 0.f;
  bool gated = false;
  at::DimVector shape(x.sizes().begin(), x.sizes().end());
  shape.back() = n_out;
  if (n == 8) {
    if (a[4] != Py_None) {
      const at::Tensor& nw = gpu_tensor(a[4], "norm weight");
      CHECK(nw.scalar_type() == x.scalar_type() && nw.is_contiguous() && nw.numel() == k, "linear_packed: the norm weight must match the rows of x");
      norm = nw.data_ptr();
      eps = (float)real(a[5]);
    }
    gated = truth(a[7]);
    if (a[6] != Py_None) {
      const at::Tensor& res = gpu_tensor(a[6], "residual");
      CHECK(!gated && res.is_contiguous() && res.scalar_type() == x.scalar_type() && res.sizes() == at::IntArrayRef(shape),
            "linear_packed: the residual must be contiguous and have the type and shape of the result");
      LAUNCH(fa_linear_packed_step(x.data_ptr(), stride, norm, eps, w.data_ptr(), res.data_ptr(), rows, (int)k, (int)n_out, 1, dtype, st));
      Py_INCREF(a[6]);
      return a[6];
    }
  }
  if (gated) shape.back() = n_out / 2;
  at::Tensor out = unlocked([&] { return at::empty(shape, x.options()); });
  LAUNCH(fa_linear_packed_step(x.data_ptr(), stride, norm, eps, w.data_ptr(), out.data_ptr(), rows, (int)k, (int)n_out, gated ? 2 : 0, dtype, st));
  return THPVariable_Wrap(out);
  FA_END
}

// linear_packed_qkv(x (B, q_len, k), packed weight, norm weight or None, eps, cos, sin, Hq, Hkv, D) -> q, k, v (B, heads, q_len, D)
PyObject* linear_packed_qkv(PyObject*, PyObject* const* a, Py_ssize_t n) {
  FA_BEGIN
  CHECK(n == 9, "linear_packed_qkv takes 9 arguments");
  const at::Tensor &x = gpu_tensor(a[0], "x"), &w = gpu_tensor(a[1], "weight"), &cos = gpu_tensor(a[4], "cos"), &sin = gpu_tensor(a[5], "sin");
  const int64_t Hq = integer(a[6]), Hkv = integer(a[7]), D = integer(a[8]);
  CHECK(x.dim() == 3 && x.scalar_type() == w.scalar_type() && x.size(2) > 0 && Hq > 0 && Hkv > 0 && D > 0 &&
        w.numel() == x.size(2) * (Hq + 2 * Hkv) * D, "linear_packed_qkv: x (B, q_len, k) does not fit the weight");
  const int64_t B = x.size(0), q_len = x.size(1), k = x.size(2), rows = B * q_len;
  for (const at::Tensor* t : {&cos, &sin})
    CHECK(t->is_contiguous() && t->scalar_type() == x.scalar_type() && (B == 1 ? t->numel() >= rows * D : t->numel() == rows * D),
          "linear_packed_qkv: one row of cos and sin per token, of the type of x");
  const void* norm = nullptr;
  if (a[2] != Py_None) {
    const at::Tensor& nw = gpu_tensor(a[2], "norm weight");
    CHECK(nw.scalar_type() == x.scalar_type() && nw.is_contiguous() && nw.numel() == k, "linear_packed_qkv: the norm weight must match the rows of x");
    norm = nw.data_ptr();
  }
  const float eps = (float)real(a[3]);
  const int64_t stride = row_stride(x);
  const int dtype = dtype_code(x);
  const fa_stream_t st = stream_of(x);
  at::Tensor q, kv;
  unlocked([&] {
    q = at::empty({B, q_len, Hq, D}, x.options());
    kv = at::empty({B, q_len, 2 * Hkv, D}, x.options());
    return 0;
  });
  LAUNCH(fa_linear_packed_qkv(x.data_ptr(), stride, norm, eps, w.data_ptr(), cos.data_ptr(), sin.data_ptr(), q.data_ptr(), kv.data_ptr(),
                              (int)rows, (int)k, (int)Hq, (int)Hkv, (int)D, dtype, st));
  const auto heads = kv.transpose(1, 2);
  PyObject* out[3] = {THPVariable_Wrap(q.transpose(1, 2)), THPVariable_Wrap(heads.narrow(1, 0, Hkv)), THPVariable_Wrap(heads.narrow(1, Hkv, Hkv))};
  PyObject* t = PyTuple_New(3);
  for (int i = 0; i < 3; ++i) {
    if (t && out[i]) PyTuple_SET_ITEM(t, i, out[i]);
    else { Py_CLEAR(t); Py_XDECREF(out[i]); }
  }
  return t;
  FA_END
}

// silu_mul(gate, up) -> dense
PyObject* silu_mul(PyObject*, PyObject* const* a, Py_ssize_t n) {
  FA_BEGIN
  CHECK(n == 2, "silu_mul takes 2 arguments");
  const at::Tensor &g = gpu_tensor(a[0], "gate"), &u = gpu_tensor(a[1], "up");
  CHECK(g.sizes() == u.sizes() && g.scalar_type() == u.scalar_type() && g.strides() == u.strides() && g.dim() >= 1 && g.stride(-1) == 1,
        "silu_mul: gate and up must share shape, type and strides");
  const int64_t cols = g.size(-1), rows = g.numel() / (cols > 0 ? cols : 1), stride = row_stride(g), es = g.element_size();
  const auto options = g.options().memory_format(at::MemoryFormat::Contiguous);
  at::Tensor out = unlocked([&] { return at::empty(g.sizes(), options); });
  const fa_stream_t st = stream_of(g);
  const int dtype = dtype_code(g);
  for (int64_t r0 = 0; r0 < rows; r0 += 65535)   // the row index is the launch's second grid dimension
    LAUNCH(fa_silu_mul((const char*)g.data_ptr() + r0 * stride * es, (const char*)u.data_ptr() + r0 * stride * es,
                       (char*)out.data_ptr() + r0 * cols * es, (int)std::min<int64_t>(65535, rows - r0), (int)cols, stride, dtype, st));
  return THPVariable_Wrap(out);
  FA_END
}

// rope_qk(q, k, cos, sin, head_dim) -> q rotated, dense (q itself when it was dense); k in place.  cos, sin: one row per token
PyObject* rope_qk(PyObject*, PyObject* const* a, Py_ssize_t n) {
  FA_BEGIN
  CHECK(n == 5, "rope_qk takes 5 arguments");
  const at::Tensor &q = gpu_tensor(a[0], "q"), &k = gpu_tensor(a[1], "k"), &cos = gpu_tensor(a[2], "cos"), &sin = gpu_tensor(a[3], "sin");
  const int64_t D = integer(a[4]);
  CHECK(q.dim() == 3 && k.dim() == 3 && q.scalar_type() == k.scalar_type() && q.size(0) == k.size(0) && q.size(1) == k.size(1) && D > 0,
        "rope_qk: q and k (B, q_len, heads * D) of one type");
  const int64_t rows = q.size(0) * q.size(1);
  // (one sequence may bring longer tables, of which the first rows are its own)
  auto fits = [&](const at::Tensor& t) { return q.size(0) == 1 ? t.numel() >= rows * D : t.numel() == rows * D; };
  CHECK(cos.is_contiguous() && sin.is_contiguous() && cos.scalar_type() == q.scalar_type() && sin.scalar_type() == q.scalar_type() &&
        fits(cos) && fits(sin), "rope_qk: one row of cos and sin per token, of the type of q");
  const bool dense = q.is_contiguous();
  const auto options = q.options().memory_format(at::MemoryFormat::Contiguous);
  at::Tensor out = dense ? q : unlocked([&] { return at::empty(q.sizes(), options); });
  const int64_t q_stride = row_stride(q), k_stride = row_stride(k);
  const int dtype = dtype_code(q);
  const fa_stream_t st = stream_of(q);
  LAUNCH(fa_rope_qk(q.data_ptr(), q_stride, out.data_ptr(), k.data_ptr(), k_stride, cos.data_ptr(), sin.data_ptr(), (int)rows,
                    (int)(q.size(2) / D), (int)(k.size(2) / D), (int)D, dtype, st));
  return dense ? (Py_INCREF(a[0]), a[0]) : THPVariable_Wrap(out);
  FA_END
}

// append_rows(k, v, k_dst, v_dst, pos): rows of K and V (B, rows, width) to row pos of the buffers
PyObject* append_rows(PyObject*, PyObject* const* a, Py_ssize_t n) {
  FA_BEGIN
  CHECK(n == 5, "append_rows takes 5 arguments");
  const at::Tensor &k = gpu_tensor(a[0], "k"), &v = gpu_tensor(a[1], "v"), &kd = gpu_tensor(a[2], "k_dst"), &vd = gpu_tensor(a[3], "v_dst");
  const int64_t pos = integer(a[4]);
  CHECK(k.dim() == 3 && k.sizes() == v.sizes() && k.strides() == v.strides() && k.stride(2) == 1 && kd.dim() == 3 && kd.sizes() == vd.sizes() &&
        kd.strides() == vd.strides() && kd.stride(2) == 1 && kd.size(0) == k.size(0) && kd.size(2) == k.size(2), "append_rows: shapes and strides");
  CHECK(v.scalar_type() == k.scalar_type() && kd.scalar_type() == k.scalar_type() && vd.scalar_type() == k.scalar_type() && pos >= 0 &&
        pos + k.size(1) <= kd.size(1), "append_rows: types, rows past the end");
  const int dtype = dtype_code(k);
  const fa_stream_t st = stream_of(kd);
  LAUNCH(fa_append_rows(k.data_ptr(), v.data_ptr(), k.stride(0), k.stride(1), kd.data_ptr(), vd.data_ptr(), kd.stride(0), kd.stride(1),
                        pos, (int)k.size(0), (int)k.size(1), (int)k.size(2), dtype, st));
  Py_RETURN_NONE;
  FA_END
}

// operands(lists, stats, k_unit, v_unit) -> (lists, stats, paging)
// The index lists (a tuple of eight: kc, kc_h, kn, kn_h, vc, vc_h, vn, vn_h) as int32 and the statistics (a tuple) as
// contiguous float32, those that are not of these types already in one launch and one allocation.  With k_unit > 0 also
// what a page store of the stored dims needs: paging = (kn_h, vn_h on the host, padded offsets of K and V on the device),
// one copy and one wait for it; None otherwise.
PyObject* operands(PyObject*, PyObject* const* a, Py_ssize_t n) {
  FA_BEGIN
  CHECK(n == 4 && PyTuple_Check(a[0]) && PyTuple_GET_SIZE(a[0]) == 8 && PyTuple_Check(a[1]), "operands takes 4 arguments");
  const Py_ssize_t n_st = PyTuple_GET_SIZE(a[1]);
  CHECK(n_st <= 6, "operands: at most six statistics");
  const int32_t k_unit = (int32_t)integer(a[2]), v_unit = (int32_t)integer(a[3]);
  const at::Tensor& first = gpu_tensor(PyTuple_GET_ITEM(a[0], 0), "list");
  const at::Device dev = first.device();
  at::Tensor lists[8], stats[6];
  fa_convert_item items[16];
  int64_t at_item[16];
  int n_items = 0;
  int64_t used = 0;                                      // in 4-byte elements, every piece at a multiple of 16 bytes
  auto add = [&](const at::Tensor& src, int64_t count, int kind, int unit) {
    items[n_items] = fa_convert_item{src.numel() ? src.data_ptr() : nullptr, nullptr, count, kind, unit};
    at_item[n_items] = used;
    used += (count + 3) / 4 * 4;
    return n_items++;
  };
  int list_item[8], stat_item[6], pad_item[2] = {-1, -1};
  // (the per-head offsets first: they go to the host in one piece)
  static const int order[8] = {3, 7, 0, 1, 2, 4, 5, 6};
  for (int o : order) {
    const at::Tensor& t = tensor(PyTuple_GET_ITEM(a[0], o), "list");
    list_item[o] = -1;
    if (t.scalar_type() == at::kInt) lists[o] = t;
    else if (t.scalar_type() == at::kLong && t.is_contiguous() && t.device() == dev) list_item[o] = add(t, t.numel(), FA_CONVERT_I64_I32, 1);
    else lists[o] = unlocked([&] { return t.to(at::kInt); });
  }
  for (Py_ssize_t i = 0; i < n_st; ++i) {
    const at::Tensor& t = tensor(PyTuple_GET_ITEM(a[1], i), "statistics");
    stat_item[i] = -1;
    const bool here = t.is_contiguous() && t.device() == dev;
    if (here && t.scalar_type() == at::kBFloat16) stat_item[i] = add(t, t.numel(), FA_CONVERT_BF16_F32, 1);
    else if (here && t.scalar_type() == at::kHalf) stat_item[i] = add(t, t.numel(), FA_CONVERT_F16_F32, 1);
    else stats[i] = unlocked([&] { return t.to(at::kFloat).contiguous(); });
  }
  if (k_unit > 0) {
    for (int i = 0; i < 2; ++i) {
      const int o = i ? 7 : 3;
      const at::Tensor& t = tensor(PyTuple_GET_ITEM(a[0], o), "list");
      const bool wide = list_item[o] >= 0;
      const at::Tensor& src = wide ? t : lists[o];
      CHECK(src.is_contiguous() && src.device() == dev && src.numel() >= 1, "per-head offsets: contiguous, on the GPU");
      pad_item[i] = add(src, src.numel(), wide ? FA_CONVERT_PAD_I64 : FA_CONVERT_PAD_I32, i ? v_unit : k_unit);
    }
  }
  at::Tensor arena;
  if (n_items > 0) {   // (empty items are views of it too)
    arena = unlocked([&] { return at::empty({used}, at::TensorOptions().dtype(at::kInt).device(dev)); });
    for (int i = 0; i < n_items; ++i) items[i].dst = static_cast<int32_t*>(arena.data_ptr()) + at_item[i];
    const fa_stream_t st = stream_of(arena);
    LAUNCH(fa_convert(items, n_items, st));
  }
  auto part = [&](int item) { return arena.narrow(0, at_item[item], items[item].count); };
  Ref out(PyTuple_New(3));
  PyObject* ls = PyTuple_New(8);
  PyTuple_SET_ITEM(out.p, 0, ls);
  for (int o = 0; o < 8; ++o) {
    if (list_item[o] >= 0) lists[o] = part(list_item[o]);
    PyTuple_SET_ITEM(ls, o, THPVariable_Wrap(lists[o]));
  }
  PyObject* ss = PyTuple_New(n_st);
  PyTuple_SET_ITEM(out.p, 1, ss);
  for (Py_ssize_t i = 0; i < n_st; ++i) {
    const at::Tensor& t = tensor(PyTuple_GET_ITEM(a[1], i), "statistics");
    if (stat_item[i] >= 0) stats[i] = part(stat_item[i]).view(at::kFloat).view(t.sizes());
    PyTuple_SET_ITEM(ss, i, THPVariable_Wrap(stats[i]));
  }
  if (k_unit <= 0) {
    Py_INCREF(Py_None);
    PyTuple_SET_ITEM(out.p, 2, Py_None);
    Py_INCREF(out.p);
    return out.p;
  }
  PyObject* paging = PyTuple_New(4);
  PyTuple_SET_ITEM(out.p, 2, paging);
  const bool one = list_item[3] == 0 && list_item[7] == 1;
  at::Tensor host[2];
  if (one) {
    const at::Tensor both = unlocked([&] { return arena.narrow(0, 0, at_item[1] + items[1].count).cpu(); });
    for (int i = 0; i < 2; ++i) host[i] = both.narrow(0, at_item[i], items[i].count);
  } else {
    unlocked([&] {
      host[0] = lists[3].cpu();
      host[1] = lists[7].cpu();
    });
  }
  for (int i = 0; i < 2; ++i) {
    const int64_t len = host[i].numel();
    PyObject* l = PyList_New(len);
    PyTuple_SET_ITEM(paging, i, l);
    const int32_t* v = static_cast<const int32_t*>(host[i].data_ptr());
    for (int64_t j = 0; j < len; ++j) PyList_SET_ITEM(l, j, PyLong_FromLong(v[j]));
    PyTuple_SET_ITEM(paging, 2 + i, THPVariable_Wrap(part(pad_item[i])));
  }
  Py_INCREF(out.p);
  return out.p;
  FA_END
}

// layout() -> (ABI version, sizes of the argument structs) this module was compiled with
PyObject* layout(PyObject*, PyObject* const*, Py_ssize_t) {
  return Py_BuildValue("(inn)", FA_ABI_VERSION, (Py_ssize_t)sizeof(fa_decode_args), (Py_ssize_t)sizeof(fa_stream_args));
}

// init(stream_fn, check_fn, workspace_fn)
PyObject* init(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 3) {
    PyErr_SetString(PyExc_TypeError, "init takes 3 arguments");
    return nullptr;
  }
  PyObject** slots[3] = {&g_stream_fn, &g_check_fn, &g_workspace_fn};
  for (int i = 0; i < 3; ++i) {
    Py_INCREF(a[i]);
    Py_XDECREF(*slots[i]);
    *slots[i] = a[i];
  }
  Py_RETURN_NONE;
}

#define FN(name) {#name, (PyCFunction)(void*)name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FN(init), FN(layout), FN(stream_update), FN(decode_attn), FN(add_rmsnorm), FN(linear_packed), FN(linear_packed_qkv), FN(silu_mul), FN(rope_qk), FN(operands), FN(append_rows),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_fa_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fa_host() {
  struct { PyObject** at; const char* name; } names[] = {
      {&s_data, "data"}, {&s_cap_pages, "cap_pages"}, {&s_batch_stride, "batch_stride"}, {&s_pad_h32, "pad_h32"}, {&s_max_pad, "max_pad"},
      {&s_pad_h_host, "pad_h_host"}, {&s_n_list32, "n_list32"}, {&s_n_h32, "n_h32"}, {&s_Cn, "Cn"}, {&s_Hkv, "Hkv"}, {&s_decode, "decode"}};
  for (auto& e : names)
    if (!(*e.at = PyUnicode_InternFromString(e.name))) return nullptr;
  return PyModule_Create(&module_def);
}
