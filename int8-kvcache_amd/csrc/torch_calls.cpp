// CPython calls into libkvq_int8.so for torch tensors: the operators' argument checks and the C ABI call in one
// native function, in place of ~40 attribute reads, ctypes conversions and formatted messages per call (18-30 us
// of host time, more than a decode-sized kernel takes).
//
// Each function returns 0 after the launch, the library's status if it refused the call, or DECLINED without
// having done anything when the arguments are not the plain form it knows (an exact torch.Tensor of dense GPU
// memory in every place, the documented shapes, layouts and dtypes). The caller then takes kvq.cuda_kernels'
// Python path, which repeats the checks, raises what is wrong or serves the form: nothing is accepted, refused
// or reported differently here. No C++ exception leaves a function.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <cstdlib>

#include "../../include/kvq_int8.h"

#ifndef KVQ_TORCH_VERSION
#error "KVQ_TORCH_VERSION: torch.__version__ of the headers in use (int8-kvcache_amd/build.py passes it)"
#endif
#define KVQ_TEXT_(x) #x
#define KVQ_TEXT(x) KVQ_TEXT_(x)

namespace {

constexpr long DECLINED = -1;

// What this file's calls were compiled against: the library's signatures, torch's tensor layout, the interpreter's
// objects. kvq._native binds the module only where all three are the running ones.
constexpr char BUILT_FOR[] = "abi " KVQ_TEXT(KVQ_ABI_VERSION) ", torch " KVQ_TORCH_VERSION ", python " KVQ_TEXT(
    PY_MAJOR_VERSION) "." KVQ_TEXT(PY_MINOR_VERSION);

// the library's entry points, by address (bind): whichever library file the package loaded
decltype(&kvq_quant_cache) p_quant_cache;
decltype(&kvq_int8_decode_attention) p_decode;
decltype(&kvq_int8_decode_attention_ex) p_decode_ex;
decltype(&kvq_dequant_pages) p_dequant;
decltype(&kvq_paged_prefill_attention_ex) p_prefill;
decltype(&kvq_int8_prefill_attention_ex) p_prefill_i8;

// A tensor argument this file may read: exactly torch.Tensor (or Parameter), dense GPU memory, no wrapper
// (functorch, functionalization, fake or subclass tensors go to the Python path).
const at::Tensor* tensor(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda()) return nullptr;
  static const c10::DispatchKeySet plain({c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA,
                                          c10::DispatchKey::AutocastCUDA, c10::DispatchKey::ADInplaceOrView});
  if (!((t.key_set() | plain) == plain)) return nullptr;
  return &t;
}

bool as_int(PyObject* o, int64_t& v) {
  if (!PyLong_CheckExact(o)) return false;
  v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

// K / V scale tables: contiguous float32 [heads, 1 or d]; their columns, or 0
int64_t scale_cols(const at::Tensor& s, int64_t heads, int64_t d) {
  if (s.scalar_type() != at::kFloat || s.dim() != 2 || !s.is_contiguous() || s.size(0) != heads ||
      (s.size(1) != 1 && s.size(1) != d))
    return 0;
  return s.size(1);
}

template <typename... T>
bool one_device(const at::Tensor& first, const T&... rest) {
  return ((rest.device() == first.device()) && ...);
}

bool bf16_rows(const at::Tensor& t) { return t.dim() == 3 && t.scalar_type() == at::kBFloat16 && t.stride(2) == 1; }
bool int8_cache(const at::Tensor& k, const at::Tensor& v) {
  return k.dim() == 4 && v.dim() == 4 && k.scalar_type() == at::kChar && v.scalar_type() == at::kChar &&
         k.sizes() == v.sizes() && k.stride(3) == 1 && v.stride(3) == 1;
}
bool index_vector(const at::Tensor& t) { return t.dim() == 1 && t.scalar_type() == at::kInt && t.is_contiguous(); }

void* stream_of(const at::Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// The entry point this thread's last call went to (its own record: the interpreter lock is not held meanwhile).
thread_local const char* entry = "";

// The C call with the interpreter lock released (as ctypes does): a full launch queue blocks this thread alone.
template <typename F>
long launch(const char* name, F&& f) {
  long rc;
  entry = name;
  Py_BEGIN_ALLOW_THREADS
  rc = f();
  Py_END_ALLOW_THREADS
  return rc;
}

template <typename F>
PyObject* guarded(F&& f) {
  long rc = DECLINED;
  try {
    rc = f();
  } catch (...) {
    rc = DECLINED;   // the Python path meets the same condition and reports it
  }
  return PyLong_FromLong(rc);
}

// (key, value, k_cache, v_cache, slots, k_scale, v_scale, k_mu)
PyObject* quant_cache(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> long {
    if (n != 8 || !p_quant_cache) return DECLINED;
    const at::Tensor* t[8];
    for (int i = 0; i < 8; ++i)
      if (!(t[i] = tensor(a[i]))) return DECLINED;
    const at::Tensor &key = *t[0], &value = *t[1], &kc = *t[2], &vc = *t[3], &slots = *t[4], &ks = *t[5], &vs = *t[6], &mu = *t[7];
    if (!bf16_rows(key) || !bf16_rows(value) || !int8_cache(kc, vc) || slots.dim() != 1 ||
        slots.scalar_type() != at::kLong || slots.stride(0) != 1 ||
        !one_device(key, value, kc, vc, slots, ks, vs, mu))
      return DECLINED;
    const int64_t T = slots.size(0), H = key.size(1), D = key.size(2);
    if (T == 0 || value.size(2) != D || kc.size(3) != D || kc.size(2) != H || key.size(0) < T || value.size(0) < T)
      return DECLINED;
    const int64_t kcols = scale_cols(ks, H, D), vcols = scale_cols(vs, H, D);
    if (!kcols || !vcols || mu.scalar_type() != at::kFloat || mu.dim() != 2 || !mu.is_contiguous() || mu.size(0) != H ||
        mu.size(1) != D)
      return DECLINED;
    void *kp = key.data_ptr(), *vp = value.data_ptr(), *st = stream_of(key);
    auto *kcp = (int8_t*)kc.data_ptr(), *vcp = (int8_t*)vc.data_ptr();
    auto* sp = (const int64_t*)slots.data_ptr();
    auto *ksp = (const float*)ks.data_ptr(), *vsp = (const float*)vs.data_ptr(), *mup = (const float*)mu.data_ptr();
    return launch("kvq_quant_cache", [&] {
      return p_quant_cache(kp, key.stride(0), key.stride(1), vp, value.stride(0), value.stride(1), kcp, kc.stride(0),
                           kc.stride(1), kc.stride(2), vcp, vc.stride(0), vc.stride(1), vc.stride(2), sp, T, H, D,
                           kc.size(0), kc.size(1), ksp, kcols, vsp, vcols, mup, st);
    });
  });
}

// (q, k_cache, v_cache, out, cu_seqlens_q, seq_lens, block_table, k_scale, v_scale, softmax_scale,
//  segm_out | None, segm_max | None, segm_sum | None, max_query_len, qmax, q_group | None, max_splits)
PyObject* decode_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> long {
    if (n != 17 || !p_decode || !p_decode_ex || getenv("KVQ_TARGET_WAVES")) return DECLINED;
    const at::Tensor* t[9];
    for (int i = 0; i < 9; ++i)
      if (!(t[i] = tensor(a[i]))) return DECLINED;
    const at::Tensor &q = *t[0], &kc = *t[1], &vc = *t[2], &out = *t[3], &cu = *t[4], &sl = *t[5], &bt = *t[6], &ks = *t[7], &vs = *t[8];
    if (!PyFloat_CheckExact(a[9])) return DECLINED;
    const double scale = PyFloat_AS_DOUBLE(a[9]);
    int64_t maxq, qmax, max_splits, group = 0;
    if (!as_int(a[13], maxq) || !as_int(a[14], qmax) || !as_int(a[16], max_splits)) return DECLINED;
    if (!bf16_rows(q) || !bf16_rows(out) || !int8_cache(kc, vc) || !index_vector(cu) || !index_vector(sl) || bt.dim() != 2 ||
        bt.scalar_type() != at::kInt || bt.stride(1) != 1 || !one_device(q, kc, vc, out, cu, sl, bt, ks, vs))
      return DECLINED;
    const int64_t B = cu.size(0) - 1, T = q.size(0), Hq = q.size(1), D = q.size(2), bs = kc.size(1), Hkv = kc.size(2);
    if (B <= 0 || kc.size(3) != D || bs < 16 || (bs & (bs - 1)) || out.size(0) < T || out.size(1) != Hq || out.size(2) != D ||
        sl.size(0) < B || bt.size(0) < B || Hkv <= 0 || Hq % Hkv)
      return DECLINED;
    if (a[15] != Py_None && !as_int(a[15], group)) return DECLINED;
    if (a[15] == Py_None) group = D;
    if (group != D && group != 32) return DECLINED;
    const int64_t kcols = scale_cols(ks, Hkv, D), vcols = scale_cols(vs, Hkv, D);
    if (!kcols || !vcols) return DECLINED;
    int64_t S = 1, rows = 0, seg_st = 0, seg_sh = 0;
    float *sop = nullptr, *smp = nullptr, *ssp = nullptr;
    if (a[11] != Py_None) {
      const at::Tensor *so = tensor(a[10]), *sm = tensor(a[11]), *ss = tensor(a[12]);
      if (!so || !sm || !ss || so->dim() != 4 || sm->dim() != 3 || ss->dim() != 3 || !one_device(q, *so, *sm, *ss)) return DECLINED;
      S = sm->size(2);
      rows = sm->size(0);
      for (const at::Tensor* x : {so, sm, ss})
        if (x->scalar_type() != at::kFloat || x->size(0) != rows || x->size(1) != Hq || x->size(2) != S) return DECLINED;
      seg_st = sm->stride(0);
      seg_sh = sm->stride(1);
      if (S > max_splits || sm->stride(2) != 1 || ss->strides() != sm->strides() || so->size(3) != D || so->stride(3) != 1 ||
          so->stride(2) != D || so->stride(1) != seg_sh * D || so->stride(0) != seg_st * D)
        return DECLINED;
      sop = (float*)so->data_ptr();
      smp = (float*)sm->data_ptr();
      ssp = (float*)ss->data_ptr();
    } else if (a[10] != Py_None || a[12] != Py_None) {
      return DECLINED;
    }
    void *qp = q.data_ptr(), *op = out.data_ptr(), *st = stream_of(q);
    auto *kp = (const int8_t*)kc.data_ptr(), *vp = (const int8_t*)vc.data_ptr();
    auto *cup = (const int32_t*)cu.data_ptr(), *slp = (const int32_t*)sl.data_ptr(), *btp = (const int32_t*)bt.data_ptr();
    auto *ksp = (const float*)ks.data_ptr(), *vsp = (const float*)vs.data_ptr();
    const bool ex = group != D || rows < T;   // tokens past the buffers' rows are never cut
    return launch(ex ? "kvq_int8_decode_attention_ex" : "kvq_int8_decode_attention", [&] {
      if (ex)
        return p_decode_ex(qp, q.stride(0), q.stride(1), kp, kc.stride(0), kc.stride(1), kc.stride(2), vp, vc.stride(0),
                           vc.stride(1), vc.stride(2), kc.size(0), bs, Hkv, D, op, out.stride(0), out.stride(1), cup, slp,
                           btp, bt.stride(0), B, Hq, ksp, kcols, vsp, vcols, scale, sop, smp, ssp, seg_st, seg_sh, S, rows,
                           0, maxq, qmax, group, st);
      return p_decode(qp, q.stride(0), q.stride(1), kp, kc.stride(0), kc.stride(1), kc.stride(2), vp, vc.stride(0),
                      vc.stride(1), vc.stride(2), kc.size(0), bs, Hkv, D, op, out.stride(0), out.stride(1), cup, slp, btp,
                      bt.stride(0), B, Hq, ksp, kcols, vsp, vcols, scale, sop, smp, ssp, seg_st, seg_sh, S, 0, maxq, qmax,
                      st);
    });
  });
}

// (q, k_cache, v_cache, out, cu_seqlens_q, seq_lens, block_table, k_scale, v_scale, softmax_scale, mode,
//  rows_per_tile, tile_req, tile_row, tile_piece | None, tile_slot | None, merge | None, slots,
//  src_req, src_j, temporary block table)
// The long requests' attention with its scratch: mode 0 dequantizes their pages into a temporary bf16 cache and
// runs the bf16 prefill on it (the last three arguments), 1 and 2 read the INT8 pages (2: scales folded).
PyObject* long_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> long {
    if (n != 21 || !p_dequant || !p_prefill || !p_prefill_i8) return DECLINED;
    const at::Tensor* t[9];
    for (int i = 0; i < 9; ++i)
      if (!(t[i] = tensor(a[i]))) return DECLINED;
    const at::Tensor &q = *t[0], &kc = *t[1], &vc = *t[2], &out = *t[3], &cu = *t[4], &sl = *t[5], &bt = *t[6], &ks = *t[7], &vs = *t[8];
    if (!PyFloat_CheckExact(a[9])) return DECLINED;
    const double scale = PyFloat_AS_DOUBLE(a[9]);
    int64_t mode, rows, slots;
    if (!as_int(a[10], mode) || !as_int(a[11], rows) || !as_int(a[17], slots) || mode < 0 || mode > 2) return DECLINED;
    const at::Tensor *treq = tensor(a[12]), *trow = tensor(a[13]);
    if (!treq || !trow || !index_vector(*treq) || !index_vector(*trow)) return DECLINED;
    const int64_t tiles = treq->size(0);
    if (!bf16_rows(q) || !bf16_rows(out) || !int8_cache(kc, vc) || cu.scalar_type() != at::kInt || sl.scalar_type() != at::kInt ||
        bt.dim() != 2 || bt.scalar_type() != at::kInt || bt.stride(1) != 1 || trow->size(0) != tiles || tiles == 0 ||
        !one_device(q, kc, vc, out, cu, sl, bt, ks, vs, *treq, *trow))
      return DECLINED;
    const int64_t Hq = q.size(1), D = q.size(2), nb = kc.size(0), bs = kc.size(1), H = kc.size(2);
    if (kc.size(3) != D || out.size(1) != Hq || out.size(2) != D || out.size(0) != q.size(0) || H <= 0) return DECLINED;
    const int64_t kcols = scale_cols(ks, H, D), vcols = scale_cols(vs, H, D);
    if (!kcols || !vcols) return DECLINED;
    const int32_t *pp = nullptr, *sp = nullptr, *mp = nullptr;
    int64_t nm = 0;
    at::Tensor part_out, part_ml;
    const auto f32 = q.options().dtype(at::kFloat);
    if (a[14] != Py_None) {
      const at::Tensor *piece = tensor(a[14]), *slot = tensor(a[15]), *merge = tensor(a[16]);
      if (!piece || !slot || !merge || !index_vector(*piece) || !index_vector(*slot) || piece->size(0) != tiles ||
          slot->size(0) != tiles || merge->scalar_type() != at::kInt || merge->dim() != 2 || !merge->is_contiguous() ||
          merge->size(1) != 4 || !one_device(q, *piece, *slot, *merge))
        return DECLINED;
      pp = (const int32_t*)piece->data_ptr();
      sp = (const int32_t*)slot->data_ptr();
      mp = (const int32_t*)merge->data_ptr();
      nm = merge->size(0);
      part_out = at::empty({slots, H, rows, D}, f32);
      part_ml = at::empty({slots, H, rows, 2}, f32);
    }
    float *pop = pp ? (float*)part_out.data_ptr() : nullptr, *pmp = pp ? (float*)part_ml.data_ptr() : nullptr;
    void *qp = q.data_ptr(), *op = out.data_ptr(), *st = stream_of(q);
    auto *kp = (const int8_t*)kc.data_ptr(), *vp = (const int8_t*)vc.data_ptr();
    auto *cup = (const int32_t*)cu.data_ptr(), *slp = (const int32_t*)sl.data_ptr(), *btp = (const int32_t*)bt.data_ptr();
    auto *ksp = (const float*)ks.data_ptr(), *vsp = (const float*)vs.data_ptr();
    auto *rp = (const int32_t*)treq->data_ptr(), *wp = (const int32_t*)trow->data_ptr();
    if (mode) {
      return launch(pp ? "kvq_int8_prefill_attention_ex" : "kvq_int8_prefill_attention", [&] {
        return p_prefill_i8(qp, q.stride(0), q.stride(1), kp, kc.stride(0), kc.stride(1), kc.stride(2), vp, vc.stride(0),
                            vc.stride(1), vc.stride(2), nb, bs, H, D, op, out.stride(0), out.stride(1), cup, slp, btp,
                            bt.stride(0), Hq, rp, wp, tiles, rows, scale, ksp, kcols, vsp, vcols, mode == 2, pp, sp, mp, nm,
                            pop, pmp, st);
      });
    }
    const at::Tensor *sreq = tensor(a[18]), *sj = tensor(a[19]), *tbt = tensor(a[20]);
    if (!sreq || !sj || !tbt || !index_vector(*sreq) || !index_vector(*sj) || sreq->size(0) == 0 ||
        sj->size(0) != sreq->size(0) || tbt->dim() != 2 || tbt->scalar_type() != at::kInt || tbt->stride(1) != 1 ||
        !one_device(q, *sreq, *sj, *tbt))
      return DECLINED;
    const int64_t P = sreq->size(0);
    const at::Tensor kt = at::empty({P, bs, H, D}, q.options()), vt = at::empty({P, bs, H, D}, q.options());
    void *ktp = kt.data_ptr(), *vtp = vt.data_ptr();
    auto *rqp = (const int32_t*)sreq->data_ptr(), *jp = (const int32_t*)sj->data_ptr(), *tbp = (const int32_t*)tbt->data_ptr();
    return launch("kvq_dequant_pages", [&] {
      const int rc = p_dequant(kp, kc.stride(0), kc.stride(1), kc.stride(2), vp, vc.stride(0), vc.stride(1), vc.stride(2), nb,
                               bs, H, D, ktp, vtp, btp, bt.stride(0), rqp, jp, P, ksp, kcols, vsp, vcols, st);
      if (rc) return rc;
      entry = pp ? "kvq_paged_prefill_attention_ex" : "kvq_paged_prefill_attention";
      return p_prefill(qp, q.stride(0), q.stride(1), ktp, bs * H * D, H * D, D, vtp, bs * H * D, H * D, D, P, bs, H, D, op,
                       out.stride(0), out.stride(1), cup, slp, tbp, tbt->stride(0), Hq, rp, wp, tiles, rows, scale, pp, sp, mp,
                       nm, pop, pmp, st);
    });
  });
}

// (): the entry point of this thread's last call, as the Python path names it in its error
PyObject* last_entry(PyObject*, PyObject*) { return PyUnicode_FromString(entry); }

// ({name: address}): the library's entry points
PyObject* bind(PyObject*, PyObject* d) {
  auto at_name = [&](const char* nm) -> void* {
    PyObject* v = PyDict_Check(d) ? PyDict_GetItemString(d, nm) : nullptr;
    return v ? PyLong_AsVoidPtr(v) : nullptr;
  };
  p_quant_cache = (decltype(p_quant_cache))at_name("kvq_quant_cache");
  p_decode = (decltype(p_decode))at_name("kvq_int8_decode_attention");
  p_decode_ex = (decltype(p_decode_ex))at_name("kvq_int8_decode_attention_ex");
  p_dequant = (decltype(p_dequant))at_name("kvq_dequant_pages");
  p_prefill = (decltype(p_prefill))at_name("kvq_paged_prefill_attention_ex");
  p_prefill_i8 = (decltype(p_prefill_i8))at_name("kvq_int8_prefill_attention_ex");
  if (PyErr_Occurred()) return nullptr;
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", bind, METH_O, "bind({entry point: address})"},
    {"quant_cache", (PyCFunction)(void (*)(void))quant_cache, METH_FASTCALL, "kvq_quant_cache on torch tensors"},
    {"decode_attention", (PyCFunction)(void (*)(void))decode_attention, METH_FASTCALL,
     "kvq_int8_decode_attention on torch tensors"},
    {"long_attention", (PyCFunction)(void (*)(void))long_attention, METH_FASTCALL,
     "the long requests' attention on torch tensors"},
    {"last_entry", last_entry, METH_NOARGS, "the entry point of this thread's last call"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_torch_calls", "kvq operators on torch tensors", -1, methods, nullptr, nullptr,
                      nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__torch_calls(void) {
  PyObject* m = PyModule_Create(&module);
  if (m) PyModule_AddIntConstant(m, "DECLINED", DECLINED);
  if (m) PyModule_AddStringConstant(m, "BUILT_FOR", BUILT_FOR);
  return m;
}
