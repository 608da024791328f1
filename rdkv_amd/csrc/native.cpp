// Host side of the entry points that a prefill or a decode loop calls once a layer, in C++: argument checks, output
// tensors and library calls of the plain forms (dense fp16 K / V on one device, fp32 scores, no taps).  Interpreted, the
// checks and 25 tensors of a layer's selection took 165 us where its launches take 40 and the device 75; a decode
// step's checks and call 9 us next to 7.4 of launches.
//
// Every function returns None, before it has launched or allocated anything, when its arguments are of any other form:
// the Python code it was called from then takes them, with its own conversions and its own errors.  Nothing is kept
// from one call for the next but the addresses of the library's functions.
#include <Python.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/_to_copy.h>
#include <ATen/ops/cat.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/full.h>

#include <algorithm>
#include <initializer_list>
#include <string>
#include <utility>
#include <vector>

#include "rdkv.h"

namespace {

// ---- the library's functions, by the addresses the ctypes binding has ------------------------------------------
#define RDKV_NATIVE_FUNCTIONS(X)                                                                                  \
  X(rdkv_pool_scores) X(rdkv_knapsack_batched_value) X(rdkv_pack_layer_plan_ints) X(rdkv_pack_layer_plan_start)  \
  X(rdkv_pack_layers_k_minmax) X(rdkv_pack_layer_v_rows) X(rdkv_pack_layer_tables) X(rdkv_pack_layer_k_rows)     \
  X(rdkv_decode_fused) X(rdkv_decode_fused_zone_c) X(rdkv_decode_fused_workspace_bytes)                           \
  X(rdkv_unpack_layer) X(rdkv_stream_plan_layer) X(rdkv_pack_layer) X(rdkv_plan_layers)                                                           \
  X(rdkv_select_layer_start) X(rdkv_pack_layers_stream)
struct Library {
#define X(name) decltype(&::name) name = nullptr;
  RDKV_NATIVE_FUNCTIONS(X)
#undef X
  PyObject *check = nullptr;     // _lib.check: raises what a status code stands for
} lib;

struct PythonError {};           // the Python error is set
struct NotPlain {};              // arguments of another form: None

void status(int rc) {
  if (rc == RDKV_OK) return;
  PyObject *r = PyObject_CallFunction(lib.check, "i", rc);
  Py_XDECREF(r);
  if (r) PyErr_Format(PyExc_RuntimeError, "rdkv HIP backend error %d", rc);
  throw PythonError{};
}

// Without the interpreter lock, as ctypes calls the library: a launch can wait for a full queue.
struct Unlocked {
  PyThreadState *state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};

// ---- arguments ---------------------------------------------------------------------------------------------------
void plain(bool ok) {
  if (!ok) throw NotPlain{};
}
const at::Tensor &tensor(PyObject *o) {
  plain(THPVariable_Check(o));
  return THPVariable_Unpack(o);
}
int64_t integer(PyObject *o) {
  const long long v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) throw PythonError{};
  return v;
}
int64_t whole(PyObject *o) {      // a field or an option: other numbers are another form
  plain(PyIndex_Check(o));
  const long long v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    throw NotPlain{};
  }
  return v;
}
double real(PyObject *o) {
  plain(PyFloat_Check(o) || PyLong_Check(o));
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw PythonError{};
  return v;
}
void *address(PyObject *o) { return reinterpret_cast<void *>(integer(o)); }
std::vector<float> reals(PyObject *list) {
  plain(PyList_Check(list));
  std::vector<float> v(PyList_GET_SIZE(list));
  for (size_t i = 0; i < v.size(); ++i) v[i] = (float)real(PyList_GET_ITEM(list, i));
  return v;
}
int dtype_code(const at::Tensor &t) {
  switch (t.scalar_type()) {
    case at::kFloat: return RDKV_DTYPE_F32;
    case at::kHalf: return RDKV_DTYPE_F16;
    case at::kBFloat16: return RDKV_DTYPE_BF16;
    default: return -1;
  }
}
bool shape_is(const at::Tensor &t, std::initializer_list<int64_t> s) { return t.sizes() == at::IntArrayRef(s.begin(), s.size()); }
template <typename T = void>
T *data(const at::Tensor &t) {
  return t.defined() && t.numel() ? reinterpret_cast<T *>(t.data_ptr()) : nullptr;
}

PyObject *wrap(const at::Tensor &t) {
  if (!t.defined()) Py_RETURN_NONE;
  PyObject *o = THPVariable_Wrap(t);
  if (!o) throw PythonError{};
  return o;
}

struct Ref {                      // an owned reference
  PyObject *o;
  explicit Ref(PyObject *p) : o(p) {
    if (!o) throw PythonError{};
  }
  Ref(const Ref &) = delete;
  ~Ref() { Py_XDECREF(o); }
  PyObject *release() { return std::exchange(o, nullptr); }
};

void put(PyObject *dict, const char *name, PyObject *value) {      // takes the value's reference
  Ref v(value);
  if (PyDict_SetItemString(dict, name, v.o)) throw PythonError{};
}
PyObject *ints(std::initializer_list<int64_t> v) {
  Ref t(PyTuple_New(v.size()));
  Py_ssize_t i = 0;
  for (int64_t x : v) {
    Ref n(PyLong_FromLongLong(x));
    PyTuple_SET_ITEM(t.o, i++, n.release());
  }
  return t.release();
}

// The entry points: a function of (args, count) that returns a new reference.  Errors of torch's own come out as torch's
// bindings raise them (an allocation that fails: torch.OutOfMemoryError, which callers catch to free memory).
template <PyObject *(*F)(PyObject *const *, Py_ssize_t), int N>
PyObject *entry(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != N) return PyErr_Format(PyExc_TypeError, "%d arguments expected, got %zd", N, n);
  HANDLE_TH_ERRORS
  try {
    return F(args, n);
  } catch (const NotPlain &) {
    Py_RETURN_NONE;
  } catch (const PythonError &) {
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}

// ---- packing of a planned layer (packing._pack_planned_layer) -----------------------------------------------------
// K, V, k_bits, order, rank3, plan, min / max or None, counts rows, info rows, first head, heads of the plan, G, stream
PyObject *pack_layer(PyObject *const *a, Py_ssize_t) {
  const at::Tensor &K = tensor(a[0]), &V = tensor(a[1]), &kb = tensor(a[2]), &order = tensor(a[3]), &rank3 = tensor(a[4]),
                   &plan = tensor(a[5]);
  const at::Tensor mm_all = a[6] == Py_None ? at::Tensor() : tensor(a[6]);
  const int64_t first = integer(a[9]), n_total = integer(a[10]), G = integer(a[11]);
  void *stream = address(a[12]);
  plain(K.is_cuda() && V.device() == K.device() && K.scalar_type() == at::kHalf && V.scalar_type() == at::kHalf);
  plain(K.dim() == 4 && K.size(0) == 1 && V.sizes() == K.sizes() && K.stride(3) == 1 && V.stride(3) == 1 &&
        K.stride(1) == V.stride(1) && K.stride(2) == V.stride(2));
  const int64_t H = K.size(1), T = K.size(2), D = K.size(3);
  plain(H >= 1 && D >= 1 && D <= 1024 && G >= 1 && first >= 0 && first + H <= n_total);
  plain(kb.dim() == 2 && kb.size(0) == n_total && kb.size(1) == D && kb.device() == K.device());
  plain(shape_is(order, {n_total, T}) && shape_is(rank3, {n_total, T}) && order.stride(1) == 1 && rank3.stride(1) == 1);
  // the class sizes, as the launches sent them
  plain(PyList_Check(a[7]) && PyList_Check(a[8]) && PyList_GET_SIZE(a[7]) == n_total && PyList_GET_SIZE(a[8]) == n_total);
  auto row = [&](PyObject *rows, int64_t h, Py_ssize_t width, int64_t *out) {
    PyObject *r = PyList_GET_ITEM(rows, first + h);
    plain(PyList_Check(r) && PyList_GET_SIZE(r) == width);
    for (Py_ssize_t i = 0; i < width; ++i) out[i] = integer(PyList_GET_ITEM(r, i));
  };
  int64_t mN[3] = {0, 0, 0}, m[3] = {0, 0, 0}, max_tv = 0, max_n16 = 0, kept_max = 0, ref = -1, tv_ref = 0;
  Ref host_tokens(PyList_New(H)), host_channels(PyList_New(H));
  for (int64_t h = 0; h < H; ++h) {
    int64_t c[4], f[8];
    row(a[7], h, 4, c);
    row(a[8], h, 8, f);
    const int64_t tv = c[0] + c[1] + c[2];
    for (int i = 0; i < 3; ++i) {
      mN[i] = std::max(mN[i], c[i]);
      m[i] = std::max(m[i], f[2 + i]);
    }
    kept_max = std::max(kept_max, f[2] + f[3] + f[4]);
    max_tv = std::max(max_tv, tv);
    max_n16 = std::max(max_n16, c[3]);
    if (h == 0) tv_ref = tv;
    if (ref < 0 && tv + c[3] > 0) {
      ref = h;
      tv_ref = tv;
    }
    PyList_SET_ITEM(host_tokens.o, h, ints({c[0], c[1], c[2], c[3]}));
    PyList_SET_ITEM(host_channels.o, h, ints({f[2], f[3], f[4]}));
  }
  ref = std::max<int64_t>(ref, 0);
  const int64_t max_tk = max_tv + max_n16, sub2 = (m[0] + 3) / 4, sub4 = (m[1] + 1) / 2, Dp = 4 * sub2 + 2 * sub4 + m[2];
  plain(max_tk > 0 && Dp > 0);       // (nothing kept, or no channel: the composed path)

  const bool early = mm_all.defined();
  const int32_t *order_l = data<int32_t>(order) + first * order.stride(0), *rank3_l = data<int32_t>(rank3) + first * rank3.stride(0);
  const int32_t *counts4 = data<int32_t>(plan) + 4 * first, *info = data<int32_t>(plan) + 4 * n_total + 8 * first;
  const uint8_t *kb_l = data<uint8_t>(kb) + first * kb.stride(0) * kb.element_size();
  const auto dev = K.options();
  auto make = [&](at::IntArrayRef s, at::ScalarType t) { return at::empty(s, dev.dtype(t)); };
  auto bytes = [&](int64_t n, int64_t w) { return n > 0 && w > 0 ? make({1, H, n, w}, at::kByte) : at::Tensor(); };
  at::Tensor V2, V4, V8, vs, vz, v16, mm, slot_ch, perm, perm_q, sort_ph, seg_ph, seg_tok, t_eff, t_eff_k, n_v16, sort_idx,
      mask, K2, K4, K8, ks, kz, sort0, perm0;
  int rc;
  {
    Unlocked u;
    V2 = bytes(mN[0], D / 4), V4 = bytes(mN[1], D / 2), V8 = bytes(mN[2], D);
    vs = make({1, H, max_tv, 1}, at::kHalf), vz = make({1, H, max_tv, 1}, at::kHalf);
    if (max_n16 > 0) v16 = make({1, H, max_n16, D}, at::kHalf);
    auto tables = [&] {
      perm = make({H, Dp}, at::kLong), perm_q = make({H * G, Dp}, at::kLong);
      sort_ph = make({H, kept_max}, at::kLong), seg_ph = make({H, 3}, at::kInt), seg_tok = make({H, 3}, at::kInt);
      t_eff = make({H}, at::kInt), t_eff_k = make({H}, at::kInt), n_v16 = make({H}, at::kInt);
      sort_idx = make({tv_ref}, at::kLong), mask = make({H * G, max_tk}, at::kFloat);
    };
    auto k_outputs = [&] {
      K2 = bytes(max_tk, sub2), K4 = bytes(max_tk, sub4), K8 = bytes(max_tk, m[2]);
      ks = make({1, H, 1, Dp}, at::kHalf), kz = make({1, H, 1, Dp}, at::kHalf);
    };
    const float *mm_at = early ? data<float>(mm_all) + first * 2 * D : nullptr;
    const uintptr_t at16 = reinterpret_cast<uintptr_t>(K.data_ptr()) | reinterpret_cast<uintptr_t>(V.data_ptr());
    if (early && D == 128 && Dp <= 512 && at16 % 16 == 0 && K.stride(1) % 8 == 0 && K.stride(2) % 8 == 0 &&
        max_tk < 0x7fff0000 && mN[0] + mN[1] + mN[2] + max_n16 < 0x7fff0000) {
      // one launch (the lines that rdkv_pack_layer requires)
      tables();
      k_outputs();
      RdkvPackLayer y{};
      y.K_f16 = K.data_ptr(), y.V_f16 = V.data_ptr(), y.stride_h = K.stride(1), y.stride_t = K.stride(2);
      y.k_bits = kb_l, y.kb_elem_size = kb.element_size(), y.kb_stride_h = kb.stride(0);
      y.order = order_l, y.order_stride_h = order.stride(0), y.rank3 = rank3_l, y.rank3_stride_h = rank3.stride(0);
      y.counts = counts4, y.info = info, y.minmax = mm_at, y.max_tv = max_tv, y.tv_ref = tv_ref;
      y.V2 = data<uint8_t>(V2), y.V4 = data<uint8_t>(V4), y.V8 = data<uint8_t>(V8);
      y.K2 = data<uint8_t>(K2), y.K4 = data<uint8_t>(K4), y.K8 = data<uint8_t>(K8);
      y.V_scale_f16 = data(vs), y.V_zp_f16 = data(vz), y.V16_f16 = data(v16), y.K_scale_f16 = data(ks), y.K_zp_f16 = data(kz);
      y.perm = data<int64_t>(perm), y.perm_for_q = data<int64_t>(perm_q), y.sort_ch = data<int64_t>(sort_ph);
      y.sort_idx = data<int64_t>(sort_idx), y.softmax_mask = data<float>(mask);
      y.seg_ch = data<int32_t>(seg_ph), y.seg_tok = data<int32_t>(seg_tok), y.t_eff = data<int32_t>(t_eff);
      y.t_eff_k = data<int32_t>(t_eff_k), y.n_v16 = data<int32_t>(n_v16);
      y.H_kv = H, y.G = G, y.max_n16 = max_n16, y.n2p = 4 * sub2, y.n4p = 2 * sub4, y.n8 = m[2];
      for (int i = 0; i < 3; ++i) y.mN[i] = mN[i];
      y.kept_max = kept_max, y.ref_head = ref;
      rc = lib.rdkv_pack_layer(&y, stream);
    } else {
      // V rows first: they need neither the channel tables nor the K outputs
      if (!early) mm = make({H * 2 * D}, at::kFloat);
      float *mm_ws = early ? const_cast<float *>(mm_at) : data<float>(mm);
      rc = lib.rdkv_pack_layer_v_rows(V.data_ptr(), K.stride(1), K.stride(2), H, D, order_l, order.stride(0), counts4, mN[0],
                                      mN[1], mN[2], max_tv, max_n16, data<uint8_t>(V2), data<uint8_t>(V4), data<uint8_t>(V8),
                                      data(vs), data(vz), data(v16), early ? nullptr : mm_ws, stream);
      if (rc == RDKV_OK) {
        tables();
        slot_ch = make({H, Dp}, at::kInt);
        rc = lib.rdkv_pack_layer_tables(kb_l, kb.element_size(), kb.stride(0), H, D, G, counts4, info, 4 * sub2, 2 * sub4,
                                        m[2], kept_max, max_tv, max_n16, order_l, order.stride(0), rank3_l, rank3.stride(0),
                                        ref, tv_ref, data<int32_t>(slot_ch), data<int64_t>(perm), data<int64_t>(perm_q),
                                        data<int64_t>(sort_ph), data<int32_t>(seg_ph), data<int32_t>(seg_tok),
                                        data<int32_t>(t_eff), data<int32_t>(t_eff_k), data<int32_t>(n_v16),
                                        data<int64_t>(sort_idx), data<float>(mask), stream);
      }
      if (rc == RDKV_OK) {
        k_outputs();
        rc = lib.rdkv_pack_layer_k_rows(K.data_ptr(), K.stride(1), K.stride(2), H, D, order_l, order.stride(0), counts4,
                                        max_tv, max_n16, data<int32_t>(slot_ch), 4 * sub2, 2 * sub4, m[2], data<uint8_t>(K2),
                                        data<uint8_t>(K4), data<uint8_t>(K8), data(ks), data(kz), mm_ws,
                                        early ? 2 : mN[0] + mN[1] + mN[2] + max_n16 > 0 ? 1 : 0, stream);
      }
    }
    if (rc == RDKV_OK) sort0 = sort_ph.select(0, 0), perm0 = perm.select(0, 0);
  }
  status(rc);
  Ref d(PyDict_New());
  for (auto &f : std::initializer_list<std::pair<const char *, const at::Tensor &>>{
           {"K_2bit", K2}, {"K_4bit", K4}, {"K_8bit", K8}, {"K_ch_scale", ks}, {"K_ch_zp", kz}, {"K_ch_sort_idx", sort0},
           {"K_ch_perm_padded_idx", perm0}, {"V_2bit", V2}, {"V_4bit", V4}, {"V_8bit", V8}, {"V_scale", vs}, {"V_zp", vz},
           {"sort_idx", sort_idx}, {"seg_bounds_per_head", seg_tok}, {"T_eff_per_head", t_eff}, {"softmax_mask", mask},
           {"K_ch_sort_idx_per_head", sort_ph}, {"K_ch_perm_padded_idx_per_head", perm}, {"K_ch_seg_bounds_per_head", seg_ph},
           {"K_ch_perm_padded_idx_for_Q", perm_q}, {"T_eff_k_per_head", t_eff_k}, {"n_v16_per_head", n_v16}})
    put(d.o, f.first, wrap(f.second));
  put(d.o, "K_ch_seg_bounds", ints({m[0], m[1], m[2]}));
  put(d.o, "seg_bounds", ints({mN[0], mN[1], mN[2]}));
  put(d.o, "T_eff", PyLong_FromLongLong(max_tv));
  put(d.o, "T_eff_k", PyLong_FromLongLong(max_tk));
  put(d.o, "n_v16", PyLong_FromLongLong(max_n16));
  put(d.o, "_host_counts", PyTuple_Pack(2, host_tokens.o, host_channels.o));
  Ref v(wrap(v16));
  return Ref(PyTuple_Pack(2, d.o, v.o)).release();
}

// ---- a layer's selection up to its token order (obkv_fast._perhead_select_and_pack_joint) --------------------------
// K, V, token scores, channel scores, (kernel, average, reflect, iterations, tolerance), V widths, V errors, V budget, K widths, K errors, K bits
// of a head, the column of the V width 0, tokens from which K min / max go ahead, keep the widths, host words, tag,
// workspace, its bytes, stream
PyObject *select_layer(PyObject *const *a, Py_ssize_t) {
  const at::Tensor &K = tensor(a[0]), &V = tensor(a[1]), &scores = tensor(a[2]), &channels = tensor(a[3]);
  plain(K.is_cuda() && V.device() == K.device() && scores.device() == K.device() && channels.device() == K.device());
  plain(K.dim() == 4 && K.size(0) == 1 && V.sizes() == K.sizes() && K.scalar_type() == at::kHalf && V.scalar_type() == at::kHalf);
  const int64_t H = K.size(1), T = K.size(2), D = K.size(3);
  plain(H >= 1 && H <= 65535 && T >= 1 && T <= (1 << 20) && D >= 1);
  plain(scores.scalar_type() == at::kFloat && shape_is(scores, {H, T}) && scores.stride(1) == 1);
  plain(channels.scalar_type() == at::kFloat && shape_is(channels, {H, D}) && channels.stride(1) == 1);
  plain(PyTuple_Check(a[4]) && PyTuple_GET_SIZE(a[4]) == 5);
  const int64_t kernel = integer(PyTuple_GET_ITEM(a[4], 0)), average = integer(PyTuple_GET_ITEM(a[4], 1)),
                reflect = integer(PyTuple_GET_ITEM(a[4], 2)), iters = integer(PyTuple_GET_ITEM(a[4], 3));
  const float tol = (float)real(PyTuple_GET_ITEM(a[4], 4));
  const std::vector<float> v_bits = reals(a[5]), v_eps = reals(a[6]), k_bits = reals(a[8]), k_eps = reals(a[9]);
  plain(v_bits.size() >= 1 && v_bits.size() <= 8 && k_bits.size() >= 1 && k_bits.size() <= 8);
  const double v_avg = real(a[7]), k_kept = real(a[10]);
  const int64_t zero_col = integer(a[11]), early_from = integer(a[12]);
  const bool keep = PyObject_IsTrue(a[13]) == 1;
  auto *words = static_cast<uint64_t *>(address(a[14]));
  const uint32_t tag = (uint32_t)integer(a[15]);
  void *ws = address(a[16]), *stream = address(a[18]);
  const int64_t ws_bytes = integer(a[17]);
  const int64_t k_clipped = reflect ? std::min(kernel, 2 * T - 1) : kernel;
  plain(kernel <= 1 || T + 2 * (k_clipped / 2) - k_clipped + 1 == T);        // (an even kernel changes the length)
  const bool early = T >= early_from && K.stride(3) == 1 && D % 4 == 0 && D <= 1024 && K.stride(1) % 2 == 0 &&
                     K.stride(2) % 2 == 0 && reinterpret_cast<uintptr_t>(K.data_ptr()) % 4 == 0;
  const auto dev = K.options();
  auto make = [&](at::IntArrayRef s, at::ScalarType t) { return at::empty(s, dev.dtype(t)); };
  at::Tensor pooled, vb, counts, kb, order, rank3, plan, mm, v16, k16;
  int rc = RDKV_OK;
  {
    Unlocked u;
    const float *rows = data<float>(scores);
    int64_t row_stride = scores.stride(0);
    const bool together = H <= 16 && T <= 65536 && D <= 256 && channels.stride(0) >= D;      // (rdkv_select_layer_start)
    if (together) {
      const int64_t T16 = (T + 15) / 16 * 16;
      if (kernel > 1) pooled = make({H, T}, at::kFloat);
      vb = make({H, T16}, at::kByte), counts = make({H, (int64_t)v_bits.size()}, at::kInt), kb = make({H, D}, at::kByte);
      order = make({H, T}, at::kInt), rank3 = make({H, T}, at::kInt);
      plan = make({lib.rdkv_pack_layer_plan_ints(H, T)}, at::kInt);
      if (early) mm = make({H * 2 * D}, at::kFloat);
      if (keep) v16 = make({H, T}, at::kShort), k16 = make({H, D}, at::kShort);
      rc = lib.rdkv_select_layer_start(rows, row_stride, H, T, kernel, average, reflect, data<float>(pooled), (float)v_avg,
                                       v_bits.data(), v_eps.data(), v_bits.size(), zero_col, data<uint8_t>(vb), T16,
                                       data<int32_t>(counts), data<float>(channels), channels.stride(0), D, (float)k_kept,
                                       k_bits.data(), k_eps.data(), k_bits.size(), data<uint8_t>(kb), iters, tol, data<int32_t>(order),
                                       data<int32_t>(rank3), data<int32_t>(plan), data<float>(mm), early ? 2 * D : 0,
                                       data<int16_t>(v16), data<int16_t>(k16), words, tag, ws, ws_bytes, stream);
      vb = vb.narrow(1, 0, T);
    } else if (kernel > 1) {
      pooled = make({H, T}, at::kFloat);
      rc = lib.rdkv_pool_scores(rows, row_stride, H, T, kernel, average, reflect, data<float>(pooled), T, stream);
      rows = data<float>(pooled);
      row_stride = T;
    }
    if (rc == RDKV_OK && !together) {
      vb = make({H, T}, at::kByte), counts = make({H, (int64_t)v_bits.size()}, at::kInt);
      rc = lib.rdkv_knapsack_batched_value(rows, row_stride, H, T, (float)v_avg, nullptr, 0, 0, 0, 0, v_bits.data(), v_eps.data(),
                                           v_bits.size(), iters, tol, 0, data(vb), 1, T, data<int32_t>(counts), ws, ws_bytes,
                                           stream);
    }
    if (rc == RDKV_OK && !together) {
      kb = make({H, D}, at::kByte);
      rc = lib.rdkv_knapsack_batched_value(data<float>(channels), channels.stride(0), H, D, (float)k_kept, data<int32_t>(counts),
                                           v_bits.size(), zero_col, T, D, k_bits.data(), k_eps.data(), k_bits.size(), iters, tol,
                                           0, data(kb), 1, D, nullptr, ws, ws_bytes, stream);
    }
    if (rc == RDKV_OK && !together) {
      order = make({H, T}, at::kInt), rank3 = make({H, T}, at::kInt);
      plan = make({lib.rdkv_pack_layer_plan_ints(H, T)}, at::kInt);
      if (early) mm = make({H * 2 * D}, at::kFloat);
      rc = lib.rdkv_pack_layer_plan_start(data(vb), 1, T, data(kb), 1, D, H, T, D, data<int32_t>(order), T, data<int32_t>(rank3),
                                          T, data<int32_t>(plan), data<float>(mm), early ? 2 * D : 0, words, tag, stream);
    }
    if (rc == RDKV_OK && early) {
      const void *K_at = K.data_ptr();
      const int64_t strides[2] = {K.stride(1), K.stride(2)};
      rc = lib.rdkv_pack_layers_k_minmax(&K_at, strides, 1, H, T, D, data<int32_t>(order), T, data<int32_t>(plan),
                                         data<float>(mm), 2 * H * D, stream);
    }
    if (rc == RDKV_OK && keep && !together) v16 = at::_to_copy(vb, at::kShort), k16 = at::_to_copy(kb, at::kShort);
  }
  status(rc);
  Ref r(PyTuple_New(8));
  Py_ssize_t i = 0;
  for (const at::Tensor *t : {&vb, &kb, &order, &rank3, &plan, &mm, &v16, &k16}) PyTuple_SET_ITEM(r.o, i++, wrap(*t));
  return r.release();
}

// ---- layers straight to the streaming format (stream_cache._pack_entries_direct) ------------------------------------
struct Buffer {                   // an array's memory, as long as the call lasts
  Py_buffer view{};
  explicit Buffer(PyObject *array, bool write = false) {
    if (PyObject_GetBuffer(array, &view, write ? PyBUF_WRITABLE : PyBUF_SIMPLE)) {
      PyErr_Clear();
      throw NotPlain{};
    }
  }
  Buffer(const Buffer &) = delete;
  ~Buffer() { PyBuffer_Release(&view); }
  template <typename T>
  T *of(int64_t n) const {
    plain(view.len >= n * (int64_t)sizeof(T));
    return static_cast<T *>(view.buf);
  }
};
std::vector<at::Tensor> tensors(PyObject *list) {
  plain(PyList_Check(list) && PyList_GET_SIZE(list) > 0);
  std::vector<at::Tensor> v;
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(list); ++i) v.push_back(tensor(PyList_GET_ITEM(list, i)));
  return v;
}

// K, V, V widths, K widths (lists: an entry each), words, tag, stream
PyObject *stream_order(PyObject *const *a, Py_ssize_t) {
  const std::vector<at::Tensor> Ks = tensors(a[0]), Vs = tensors(a[1]);
  std::vector<at::Tensor> vbs = tensors(a[2]), kbs = tensors(a[3]);
  const int64_t n = Ks.size();
  auto *words = static_cast<uint64_t *>(address(a[4]));
  const uint32_t tag = (uint32_t)integer(a[5]);
  void *stream = address(a[6]);
  plain((int64_t)Vs.size() == n && (int64_t)vbs.size() == n && (int64_t)kbs.size() == n && Ks[0].is_cuda() && Ks[0].dim() == 4);
  const auto dev = Ks[0].device();
  const int64_t H = Ks[0].size(1), T = Ks[0].size(2);
  plain(H >= 1 && T >= 1 && T <= (1 << 30) && n * H <= 65535 && H <= 8191);
  auto widths = [&](const std::vector<at::Tensor> &ts, int64_t w) {
    const auto type = ts[0].scalar_type();
    plain(type == at::kByte || type == at::kShort || type == at::kInt || type == at::kLong);
    for (const auto &t : ts)
      plain(t.device() == dev && t.scalar_type() == type && shape_is(t, {H, w}) && t.is_contiguous());
  };
  widths(vbs, T);
  widths(kbs, 128);
  std::vector<const void *> K_at;
  std::vector<int64_t> strides;
  for (int64_t i = 0; i < n; ++i) {
    const at::Tensor &K = Ks[i], &V = Vs[i];
    plain(shape_is(K, {1, H, T, 128}) && V.sizes() == K.sizes() && K.device() == dev && V.device() == dev &&
          K.scalar_type() == at::kHalf && V.scalar_type() == at::kHalf && K.strides() == V.strides() && K.stride(3) == 1 &&
          K.stride(2) % 8 == 0 && K.stride(1) % 8 == 0 && reinterpret_cast<uintptr_t>(K.data_ptr()) % 16 == 0 &&
          reinterpret_cast<uintptr_t>(V.data_ptr()) % 16 == 0);
    K_at.push_back(K.data_ptr());
    strides.insert(strides.end(), {K.stride(1), K.stride(2)});
  }
  std::vector<const void *> vb_at, kb_at;
  for (int64_t i = 0; i < n; ++i) vb_at.push_back(vbs[i].data_ptr()), kb_at.push_back(kbs[i].data_ptr());
  at::Tensor kb, order, plan, mm;
  int rc;
  {
    Unlocked u;
    auto make = [&](at::IntArrayRef s, at::ScalarType t) { return at::empty(s, Ks[0].options().dtype(t)); };
    kb = make({n * H, 128}, at::kByte), order = make({n * H, T}, at::kInt);
    plan = make({lib.rdkv_pack_layer_plan_ints(n * H, T)}, at::kInt);
    mm = make({n * H * 768}, at::kFloat);
    rc = lib.rdkv_plan_layers(vb_at.data(), vbs[0].element_size(), kb_at.data(), kbs[0].element_size(), n, H, T, 128,
                              data<int32_t>(order), data<int32_t>(plan), data<float>(mm), 768, data<uint8_t>(kb), words, tag,
                              stream);
    if (rc == RDKV_OK)
      rc = lib.rdkv_pack_layers_k_minmax(K_at.data(), strides.data(), n, H, T, 128, data<int32_t>(order), T, data<int32_t>(plan),
                                         data<float>(mm), 768 * H, stream);
  }
  status(rc);
  Ref o(wrap(order)), p(wrap(plan)), k(wrap(kb)), w(wrap(mm));
  return Ref(PyTuple_Pack(4, o.o, p.o, k.o, w.o)).release();
}

// Unit descriptors, sizes [n][4] and dimensions [n][5] of the entries, into the arrays given; None if an
// entry keeps nothing.  Counts rows, info rows, first query rows, heads, G, units, sizes, dimensions
PyObject *stream_tables(PyObject *const *a, Py_ssize_t) {
  plain(PyList_Check(a[0]) && PyList_Check(a[1]) && PyList_Check(a[2]));
  const int64_t n = PyList_GET_SIZE(a[2]), H = integer(a[3]), G = integer(a[4]);
  plain(n >= 1 && H >= 1 && PyList_GET_SIZE(a[0]) == n * H && PyList_GET_SIZE(a[1]) == n * H);
  Buffer units(a[5], true), sizes(a[6], true), dims(a[7], true);
  auto *unit_p = units.of<RdkvUnit>(n * H);
  auto *size_p = sizes.of<int64_t>(4 * n);
  auto *dim_p = dims.of<int32_t>(5 * n);
  std::vector<int32_t> tok(4 * H), ch(3 * H);
  for (int64_t e = 0; e < n; ++e) {
    int32_t m[3] = {0, 0, 0}, max_tv = 0, max_n16 = 0;
    for (int64_t h = 0; h < H; ++h) {
      PyObject *c = PyList_GET_ITEM(a[0], e * H + h), *f = PyList_GET_ITEM(a[1], e * H + h);
      plain(PyList_Check(c) && PyList_GET_SIZE(c) == 4 && PyList_Check(f) && PyList_GET_SIZE(f) == 8);
      for (int i = 0; i < 4; ++i) tok[4 * h + i] = (int32_t)integer(PyList_GET_ITEM(c, i));
      for (int i = 0; i < 3; ++i) {
        ch[3 * h + i] = (int32_t)integer(PyList_GET_ITEM(f, 2 + i));
        m[i] = std::max(m[i], ch[3 * h + i]);
      }
      max_tv = std::max(max_tv, tok[4 * h] + tok[4 * h + 1] + tok[4 * h + 2]);
      max_n16 = std::max(max_n16, tok[4 * h + 3]);
    }
    plain(max_tv + max_n16 > 0 && m[0] + m[1] + m[2] > 0);
    int32_t *d = dim_p + 5 * e;
    d[0] = (m[0] + 3) / 4 * 4, d[1] = (m[1] + 1) / 2 * 2, d[2] = m[2], d[3] = max_tv, d[4] = max_n16;
    status(lib.rdkv_stream_plan_layer(tok.data(), 4, ch.data(), 3, H, d[0], d[1], (int)integer(PyList_GET_ITEM(a[2], e)), G,
                                      unit_p + e * H, nullptr, 0, size_p + 4 * e));
  }
  Py_RETURN_TRUE;
}

// The entries' blobs, packed; the units' offsets become addresses.  K, V, order, plan, K widths, min / max, units
// (host), sizes, dimensions, largest scales [n][2][H], whether every byte of the blobs is set beforehand, stream
PyObject *stream_pack(PyObject *const *a, Py_ssize_t) {
  const std::vector<at::Tensor> Ks = tensors(a[0]), Vs = tensors(a[1]);
  const at::Tensor &order = tensor(a[2]), &plan = tensor(a[3]), &kb = tensor(a[4]), &mm = tensor(a[5]), &scales = tensor(a[9]);
  const bool poison = PyObject_IsTrue(a[10]) == 1;      // (tests: a byte that the launches leave out cannot pass for a right one)
  void *stream = address(a[11]);
  const int64_t n = Ks.size(), H = Ks[0].size(1), T = Ks[0].size(2);
  Buffer host(a[6], true), sizes(a[7]), dims(a[8]);
  auto *unit_p = host.of<RdkvUnit>(n * H);
  const auto *size_p = sizes.of<int64_t>(4 * n);
  const auto *dim_p = dims.of<int32_t>(5 * n);
  plain(shape_is(order, {n * H, T}) && shape_is(scales, {n, 2, H}) && shape_is(kb, {n * H, 128}) && kb.is_contiguous());
  plain(mm.numel() >= n * H * 768 && plan.numel() >= 12 * n * H);
  std::vector<at::Tensor> blobs;
  std::vector<RdkvStreamLayer> layers;
  std::vector<int32_t> tiles(n * H, 0);
  for (int64_t i = 0; i < n * H; ++i)
    for (const int32_t tokens : unit_p[i].n_tok) tiles[i] += (tokens + 63) / 64;      // (a tile: 64 tokens)
  int rc = RDKV_OK;
  {
    Unlocked u;
    for (int64_t e = 0; e < n; ++e) {
      const int32_t *d = dim_p + 5 * e;
      // (256 bytes of slack for 16-byte reads at the end; the launches write every other byte)
      const int64_t bytes = std::max<int64_t>(size_p[4 * e], 256) + 256;
      const auto options = Ks[e].options().dtype(at::kByte);
      blobs.push_back(poison ? at::full({bytes}, 0xAB, options) : at::empty({bytes}, options));
      layers.push_back({Ks[e].data_ptr(), Vs[e].data_ptr(), Ks[e].stride(1), Ks[e].stride(2), data<uint8_t>(blobs.back()), bytes,
                        d[3], d[0], d[1], d[2], d[4], (int32_t)size_p[4 * e + 1], 0, tiles.data() + e * H});
    }
    const at::Tensor units = at::empty({n * H * (int64_t)sizeof(RdkvUnit)}, kb.options().dtype(at::kByte));
    rc = lib.rdkv_pack_layers_stream(layers.data(), n, H, data<int32_t>(order), T, data<int32_t>(plan),
                                     data<int32_t>(plan) + 4 * n * H, data<uint8_t>(kb), kb.element_size(), 128,
                                     data<RdkvUnit>(units), data<float>(mm), data<float>(scales), stream);
    for (int64_t e = 0; e < n && rc == RDKV_OK; ++e) {
      const uint64_t base = reinterpret_cast<uintptr_t>(layers[e].blob);
      for (RdkvUnit *p = unit_p + e * H; p < unit_p + (e + 1) * H; ++p) {
        p->k_off += base, p->sz_off += base, p->qtab_off += base;
        for (auto &v : p->v_off) v += base;
      }
    }
  }
  status(rc);
  Ref list(PyList_New(n));
  for (int64_t e = 0; e < n; ++e) PyList_SET_ITEM(list.o, e, wrap(blobs[e]));
  return list.release();
}

// ---- a decode step's attention (stream_cache.decode_attn_fused) -----------------------------------------------------
PyObject *field(PyObject *dict, const char *name) {
  PyObject *o = PyDict_GetItemString(dict, name);
  plain(o != nullptr);
  return o;
}

// cache fields, host units, q, out or None, lse or None, cos, sin or None, zone C K, V or None, counts or None, step k, v,
// row or None, workspace, its bytes, stream
PyObject *decode_attn(PyObject *const *a, Py_ssize_t) {
  PyObject *c = a[0];
  plain(PyDict_Check(c));
  // (what is reached through a dictionary is held: another thread may replace it while the lock is released)
  const at::Tensor &q = tensor(a[2]), units = tensor(field(c, "units")), work = tensor(field(c, "work"));
  const int64_t n_units = whole(field(c, "n_units")), n_work = whole(field(c, "n_work")), G = whole(field(c, "G")),
                rows = whole(field(c, "rows")), n_groups = whole(field(c, "n_groups"));
  const int row_dwords = (int)(whole(field(c, "max_row_dwords")) | whole(field(c, "row_shape")) << 8);
  const at::Tensor group_table = n_groups != n_work ? tensor(field(c, "groups")) : at::Tensor();
  const int32_t *groups = data<int32_t>(group_table);
  const auto dev = q.device();
  const int q_dt = dtype_code(q);
  plain(q.is_cuda() && q_dt >= 0 && shape_is(q, {rows, 128}) && q.stride(1) == 1 && units.device() == dev && work.device() == dev);
  plain(G >= 1 && rows % G == 0 && n_units > 0 && n_work > 0);
  auto fp32 = [&](const at::Tensor &t) { return t.device() == dev && t.scalar_type() == at::kFloat; };
  at::Tensor out, lse;
  if (a[3] != Py_None) {
    out = tensor(a[3]);
    plain(fp32(out) && shape_is(out, {rows, 128}) && out.stride(1) == 1);
  }
  if (a[4] != Py_None) {
    lse = tensor(a[4]);
    plain(fp32(lse) && shape_is(lse, {rows}) && lse.stride(0) == 1);
  }
  const void *cos = nullptr, *sin = nullptr;
  int rope_dt = 0;
  if (a[5] != Py_None) {
    const at::Tensor &rc = tensor(a[5]), &rs = tensor(a[6]);
    rope_dt = dtype_code(rc);
    plain(rope_dt >= 0 && rc.device() == dev && rs.device() == dev && rs.scalar_type() == rc.scalar_type() && rc.numel() == 64 &&
          rs.numel() == 64 && rc.is_contiguous() && rs.is_contiguous());
    cos = rc.data_ptr();
    sin = rs.data_ptr();
  }
  void *ws = address(a[13]), *stream = address(a[15]);
  const int64_t ws_bytes = integer(a[14]);
  plain(ws_bytes >= lib.rdkv_decode_fused_workspace_bytes(n_work, G));       // (it is grown there)
  at::Tensor kn, vn, counts, ks, vs, row;
  if (a[7] != Py_None) {
    kn = tensor(a[7]);
    vn = tensor(a[8]);
    plain(fp32(kn) && fp32(vn) && kn.dim() == 3 && kn.size(0) == rows / G && kn.size(1) > 0 && kn.size(2) == 128 &&
          kn.stride(2) == 1 && vn.sizes() == kn.sizes() && vn.strides() == kn.strides());
    if (a[9] != Py_None) {
      counts = tensor(a[9]);
      plain(counts.device() == dev && counts.scalar_type() == at::kInt && counts.numel() == rows / G && counts.is_contiguous());
    }
    if (a[10] != Py_None) {
      ks = tensor(a[10]), vs = tensor(a[11]), row = tensor(a[12]);
      plain(counts.defined() && ks.device() == dev && vs.device() == dev && row.device() == dev && dtype_code(ks) >= 0 &&
            vs.scalar_type() == ks.scalar_type() && shape_is(ks, {rows / G, 128}) && shape_is(vs, {rows / G, 128}) &&
            ks.stride(1) == 1 && vs.stride(1) == 1 && row.scalar_type() == at::kLong && row.numel() == 1);
    }
  } else {
    plain(a[9] == Py_None && a[10] == Py_None);
  }
  Buffer host(a[1]);
  const auto *units_host = host.of<RdkvUnit>(n_units);
  int rc;
  {
    Unlocked u;
    if (!out.defined()) out = at::empty({rows, 128}, q.options().dtype(at::kFloat));
    if (!lse.defined()) lse = at::empty({rows}, q.options().dtype(at::kFloat));
    auto *units_p = data<RdkvUnit>(units);
    auto *work_p = data<RdkvWork>(work);
    if (!kn.defined()) {
      rc = lib.rdkv_decode_fused(nullptr, units_p, n_units, work_p, n_work, groups, groups ? n_groups : 0, row_dwords, q.data_ptr(),
                                 q_dt, q.stride(0), G, cos, sin, rope_dt, data<float>(out), out.stride(0), data<float>(lse), ws,
                                 ws_bytes, stream);
    } else {
      rc = lib.rdkv_decode_fused_zone_c(
          units_p, units_host, n_units, work_p, n_work, groups, groups ? n_groups : 0,
          row_dwords, G, q.data_ptr(), q_dt, q.stride(0), cos, sin, rope_dt, data<float>(kn), data<float>(vn), kn.stride(0),
          kn.stride(1), kn.size(1), data<int32_t>(counts), data(ks), ks.defined() ? ks.stride(0) : 0, data(vs),
          vs.defined() ? vs.stride(0) : 0, ks.defined() ? dtype_code(ks) : 0, data<int64_t>(row), data<float>(out), out.stride(0),
          data<float>(lse), nullptr, 0, nullptr, 0, nullptr, ws, ws_bytes, stream);
    }
  }
  status(rc);
  if (a[3] != Py_None && a[4] != Py_None) return Ref(PyTuple_Pack(2, a[3], a[4])).release();
  Ref o(wrap(out)), l(wrap(lse));
  return Ref(PyTuple_Pack(2, o.o, l.o)).release();
}

// ---- a packed layer back to dense K and V (trizone_decompress) -------------------------------------------------------
// layer fields, fp16-kept V rows or None, head dimension, words for K, words for V, tag, stream
PyObject *dense_layer(PyObject *const *a, Py_ssize_t) {
  PyObject *f = a[0];
  plain(PyDict_Check(f));
  const int64_t D = integer(a[2]);
  auto *k_words = static_cast<uint64_t *>(address(a[3])), *v_words = static_cast<uint64_t *>(address(a[4]));
  const uint32_t tag = (uint32_t)integer(a[5]);
  void *stream = address(a[6]);
  // the fp16 rows, or (the fp16 rows, the mask, zeros behind its rows)
  PyObject *rows_b = a[1], *mask_o = Py_None;
  int64_t extra = 0;
  if (PyTuple_Check(rows_b)) {
    plain(PyTuple_GET_SIZE(a[1]) == 3);
    rows_b = PyTuple_GET_ITEM(a[1], 0), mask_o = PyTuple_GET_ITEM(a[1], 1);
    extra = std::max<int64_t>(whole(PyTuple_GET_ITEM(a[1], 2)), 0);
  }
  auto maybe = [&](const char *name) {
    PyObject *o = field(f, name);
    return o == Py_None ? at::Tensor() : tensor(o);
  };
  // (held, not referred to: another thread may replace a field while the lock is released)
  const at::Tensor ks = tensor(field(f, "K_ch_scale")), kz = tensor(field(f, "K_ch_zp")),
                   sort = tensor(field(f, "K_ch_sort_idx_per_head")), k_counts = tensor(field(f, "K_ch_seg_bounds_per_head")),
                   vs = tensor(field(f, "V_scale")), vz = tensor(field(f, "V_zp")),
                   v_counts = tensor(field(f, "seg_bounds_per_head")), totals = tensor(field(f, "T_eff_per_head"));
  const auto dev = ks.device();
  const int64_t T_v = whole(field(f, "T_eff")), T_k = whole(field(f, "T_eff_k")), n16 = whole(field(f, "n_v16"));
  plain(ks.is_cuda() && ks.dim() == 4 && T_v > 0 && T_k == T_v + n16 && n16 >= 0);
  const int64_t H = ks.size(1);
  auto three = [&](const char *name, int64_t *out) {
    PyObject *t = field(f, name);
    plain(PyTuple_Check(t) && PyTuple_GET_SIZE(t) == 3);
    for (int i = 0; i < 3; ++i) out[i] = whole(PyTuple_GET_ITEM(t, i));
  };
  auto dense = [&](const at::Tensor &t, at::ScalarType type, std::initializer_list<int64_t> s) {
    plain(t.device() == dev && t.scalar_type() == type && shape_is(t, s) && t.is_contiguous());
  };
  int64_t m[3], mv[3];
  three("K_ch_seg_bounds", m);
  three("seg_bounds", mv);
  const int64_t w[3] = {(m[0] + 3) / 4 * 4, (m[1] + 1) / 2 * 2, m[2]}, Dp = w[0] + w[1] + w[2];
  plain(m[0] >= 0 && m[1] >= 0 && m[2] >= 0 && Dp > 0 && H >= 1);
  at::Tensor K[3] = {maybe("K_2bit"), maybe("K_4bit"), maybe("K_8bit")}, V[3] = {maybe("V_2bit"), maybe("V_4bit"), maybe("V_8bit")};
  int64_t rows[3];
  for (int i = 0; i < 3; ++i) {
    plain(K[i].defined() == (w[i] > 0));
    if (w[i]) dense(K[i], at::kByte, {1, H, T_k, w[i] * (2 << i) / 8});
    rows[i] = V[i].defined() ? V[i].size(2) : 0;
    plain(rows[i] == mv[i]);
    if (V[i].defined()) dense(V[i], at::kByte, {1, H, rows[i], D * (2 << i) / 8});
  }
  plain(D % 4 == 0 && D > 0);
  dense(ks, at::kHalf, {1, H, 1, Dp});
  dense(kz, at::kHalf, {1, H, 1, Dp});
  plain(sort.dim() == 2 && sort.device() == dev && sort.scalar_type() == at::kLong && sort.size(0) == H && sort.is_contiguous());
  dense(k_counts, at::kInt, {H, 3});
  dense(vs, at::kHalf, {1, H, T_v, 1});
  dense(vz, at::kHalf, {1, H, T_v, 1});
  dense(v_counts, at::kInt, {H, 3});
  dense(totals, at::kInt, {H});
  at::Tensor zone_b;
  if (n16 > 0) {
    zone_b = tensor(rows_b);
    dense(zone_b, at::kHalf, {1, H, n16, D});
  }
  at::Tensor mask;
  if (mask_o != Py_None) {
    mask = tensor(mask_o);
    plain(mask.device() == dev && mask.scalar_type() == at::kFloat && mask.dim() == 2 && mask.is_contiguous() && mask.numel() > 0 &&
          !mask.requires_grad() && extra < (1 << 30) && mask.size(0) * (mask.size(1) + extra) < (int64_t(1) << 31));
  }
  at::Tensor Kd, Vd, Md;
  int rc;
  {
    Unlocked u;
    Kd = at::empty({1, H, T_k, D}, ks.options()), Vd = at::empty({1, H, T_k, D}, ks.options());
    RdkvDenseLayer y{};
    for (int i = 0; i < 3; ++i) {
      y.K[i] = data<uint8_t>(K[i]), y.V[i] = data<uint8_t>(V[i]);
      if (K[i].defined()) y.k_stride_h[i] = K[i].stride(1), y.k_stride_t[i] = K[i].stride(2);
      if (V[i].defined()) y.v_stride_h[i] = V[i].stride(1);
      y.n[i] = m[i], y.np[i] = w[i], y.m[i] = mv[i];
    }
    y.k_scale_f16 = data(ks), y.k_zp_f16 = data(kz), y.ks_stride_h = ks.stride(1);
    y.sort_idx = data<int64_t>(sort), y.sort_stride_h = sort.stride(0), y.sort_n = sort.size(1), y.k_counts = data<int32_t>(k_counts);
    y.v_scale_f16 = data(vs), y.v_zp_f16 = data(vz), y.vs_stride_h = vs.stride(1);
    y.v_counts = data<int32_t>(v_counts), y.totals = data<int32_t>(totals);
    y.V16_f16 = data(zone_b), y.v16_stride_h = n16 ? zone_b.stride(1) : 0, y.n16 = n16;
    y.H_kv = H, y.D = D, y.T = T_k, y.max_tv = T_v;
    y.K_out_f16 = data(Kd), y.V_out_f16 = data(Vd);
    y.k_words = k_words, y.v_words = v_words, y.tag = tag;
    if (mask.defined()) {
      Md = at::empty({1, mask.size(0), 1, mask.size(1) + extra}, ks.options());
      y.mask = data<float>(mask), y.mask_out_f16 = data(Md);
      y.mask_rows = mask.size(0), y.mask_width = mask.size(1), y.mask_extra = extra;
    }
    rc = lib.rdkv_unpack_layer(&y, stream);
  }
  status(rc);
  Ref k(wrap(Kd)), v(wrap(Vd));
  if (!mask.defined()) return Ref(PyTuple_Pack(2, k.o, v.o)).release();
  Ref additive(wrap(Md));
  return Ref(PyTuple_Pack(3, k.o, v.o, additive.o)).release();
}

// {name: address of the function}, check
PyObject *bind(PyObject *const *a, Py_ssize_t) {
  Library l;
#define X(name) l.name = reinterpret_cast<decltype(l.name)>(address(field(a[0], #name)));
  RDKV_NATIVE_FUNCTIONS(X)
#undef X
  Py_INCREF(a[1]);
  l.check = a[1];
  lib = l;
  Py_RETURN_TRUE;
}
PyObject *names(PyObject *, PyObject *) {
  std::string s;
#define X(name) s += #name " ";
  RDKV_NATIVE_FUNCTIONS(X)
#undef X
  return PyUnicode_FromString(s.c_str());
}

#define ENTRY(f, n, doc) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(entry<f, n>)), METH_FASTCALL, doc}
PyMethodDef kMethods[] = {
    ENTRY(bind, 2, "Takes the library's function addresses and the function that raises for a status code."),
    {"names", names, METH_NOARGS, "The library functions that bind asks for."},
    ENTRY(pack_layer, 13, "The tensors of a planned layer: (fields of the layer, fp16-kept V rows), or None."),
    ENTRY(select_layer, 19, "Widths and token order of a layer: (v_bits, k_bits, order, rank3, plan, min / max, int16 widths), or None."),
    ENTRY(stream_order, 7, "Token order of the layers: (order, plan, K widths, min / max), or None."),
    ENTRY(stream_tables, 8, "Fills the units, sizes and dimensions of the layers: True, or None."),
    ENTRY(stream_pack, 12, "The blobs of the layers, or None."),
    ENTRY(decode_attn, 16, "(out, lse) of a decode step, or None."),
    ENTRY(dense_layer, 7, "Dense (K, V) of a packed layer, with its additive mask where one is given; or None."),
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_native", "Host side of the per-layer entry points.", -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};
}  // namespace

PyMODINIT_FUNC PyInit__native() { return PyModule_Create(&kModule); }
