// Host side of the plugin steps: walks the engine's ParamRecords once, in
// native code, and hands the whole step to one kernel launch per pass.
//
// What bounds a small model's step is this walk: 45 records of a 1.15 M-element
// bucket took 0.9 ms per step in Python (attribute reads, a tensor view and a
// dict per record, one ctypes call per norm and per scale) against 0.1 ms of
// GPU work.  Here a record costs well under a microsecond.
//
// Every function answers None / False when it meets anything but the ordinary
// case (flat contiguous fp32 device tensors, uint8 masks); the Python callers
// then take the general route, which also raises the errors.  Nothing has been
// launched at that point.
//
// Tables travel through torch's caching allocators: a pinned block and a device
// block per call, both returned when the call is over, ordered on the current
// stream by torch itself -- nothing here outlives a call or is shared between
// threads or streams.  A captured graph would read the pinned block again at its
// replay: the callers keep captures away from here.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/core/CachingHostAllocator.h>
#include <c10/core/impl/VirtualGuardImpl.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <chrono>
#include <cmath>
#include <utility>
#include <vector>

#include "../../include/sga_hip.h"

namespace {

// entry points of libsga_hip.so, handed over once by the ctypes loader
decltype(&sga_adamw_grad_correct_multi) f_gc_multi = nullptr;
decltype(&sga_adamw_grad_correct_compact_multi) f_gcc_multi = nullptr;
decltype(&sga_norm_sq_multi) f_norm_multi = nullptr;
decltype(&sga_scale_multi) f_scale_multi = nullptr;

PyObject* record_type = nullptr;   // adamw.ParamRecord: what it computes from its fields is known here

// interned attribute names
PyObject *s_main_param, *s_grad, *s_data, *s_state, *s_exp_avg, *s_exp_avg_sq, *s_bucket_state, *s_mask,
    *s_start, *s_end, *s_lr, *s_beta1, *s_beta2, *s_eps, *s_wd, *s_step, *s_support_index,
    *s_buckets, *s_idx, *s_dir_table;

struct Ref {                       // owned reference
  PyObject* o;
  explicit Ref(PyObject* p = nullptr) : o(p) {}
  Ref(const Ref&) = delete;
  Ref& operator=(const Ref&) = delete;
  ~Ref() { Py_XDECREF(o); }
  operator PyObject*() const { return o; }
};

// The interpreter lock is released while one of these lives: also where what runs under it throws
// (a device error surfaces at the next read from the device) the handler holds the lock again.
struct Unlocked {
  PyThreadState* state = PyEval_SaveThread();
  Unlocked() = default;
  Unlocked(const Unlocked&) = delete;
  Unlocked& operator=(const Unlocked&) = delete;
  ~Unlocked() { PyEval_RestoreThread(state); }
};

bool number(PyObject* obj, PyObject* name, double* out) {
  Ref v(PyObject_GetAttr(obj, name));
  if (!v.o) return false;
  *out = PyFloat_AsDouble(v);
  return !(*out == -1.0 && PyErr_Occurred());
}
bool integer(PyObject* obj, PyObject* name, int64_t* out) {
  Ref v(PyObject_GetAttr(obj, name));
  if (!v.o) return false;
  *out = PyLong_AsLongLong(v);
  return !(*out == -1 && PyErr_Occurred());
}

// A flat fp32 device tensor behind `o` (a tensor, or an object with .data): address and length.
bool flat32(PyObject* o, float** ptr, int64_t* n) {
  Ref held;
  if (!THPVariable_Check(o)) {
    held.o = PyObject_GetAttr(o, s_data);
    if (!held.o || !THPVariable_Check(held)) return false;
    o = held;
  }
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.scalar_type() != at::kFloat || !t.is_contiguous()) return false;
  *ptr = static_cast<float*>(t.data_ptr());
  *n = t.numel();
  return true;
}

// The record's slice of its bucket's mask: 1 a mask, 0 none, -1 not the ordinary case.
int mask_of(PyObject* rec, int64_t n, const uint8_t** mask) {
  *mask = nullptr;
  Ref bs(PyObject_GetAttr(rec, s_bucket_state));
  if (!bs.o) return -1;
  if (bs.o == Py_None) return 0;
  Ref mk(PyObject_GetAttr(bs, s_mask));
  if (!mk.o) return -1;
  if (mk.o == Py_None) return 0;
  int64_t a, b;
  if (!THPVariable_Check(mk) || !integer(rec, s_start, &a) || !integer(rec, s_end, &b)) return -1;
  const at::Tensor& t = THPVariable_Unpack(mk.o);
  if (!t.is_cuda() || t.scalar_type() != at::kByte || t.dim() != 1 || !t.is_contiguous() || a < 0 ||
      b - a != n || b > t.numel())
    return -1;
  *mask = static_cast<const uint8_t*>(t.data_ptr()) + a;
  return 1;
}

constexpr int64_t kSpan = 4096;    // elements per workgroup of the table-driven kernels

// A table of plain structs on the device of `like`, uploaded on the current stream.
template <class T>
at::Tensor to_device(const std::vector<T>& rows, c10::Device dev) {
  const int64_t bytes = (int64_t)(rows.size() * sizeof(T));
  at::Tensor host = at::empty({bytes}, at::TensorOptions().dtype(at::kByte).pinned_memory(true));
  memcpy(host.data_ptr(), rows.data(), (size_t)bytes);
  at::Tensor out = at::empty({bytes}, at::TensorOptions().dtype(at::kByte).device(dev));
  out.copy_(host, /*non_blocking=*/true);
  return out;
}

struct Walk {                      // a list / tuple of records; n < 0: anything else, left untouched
  PyObject* seq;
  Py_ssize_t n;
  explicit Walk(PyObject* records) : seq(records) {
    n = PyList_Check(records) || PyTuple_Check(records) ? PySequence_Fast_GET_SIZE(records) : -1;
  }
  PyObject* at(Py_ssize_t i) { return PySequence_Fast_GET_ITEM(seq, i); }
};

PyObject* not_ordinary() {
  PyErr_Clear();
  Py_RETURN_FALSE;
}

c10::Device device_of(PyObject* rec) {
  Ref mp(PyObject_GetAttr(rec, s_main_param));
  Ref d(THPVariable_Check(mp.o) ? (Py_INCREF(mp.o), mp.o) : PyObject_GetAttr(mp, s_data));
  return THPVariable_Unpack(d.o).device();
}

// p, g, m, v and the hyper-parameters of one record.
struct Common {
  float *p, *g, *m, *v;
  int64_t n;
  double lr, b1, b2, eps, wd;
  int64_t step;
};
bool common_of(PyObject* rec, Common* c) {
  if ((PyObject*)Py_TYPE(rec) != record_type) return false;
  Ref mp(PyObject_GetAttr(rec, s_main_param)), st(PyObject_GetAttr(rec, s_state));
  if (!mp.o || !st.o || !PyDict_Check(st.o)) return false;
  Ref g(PyObject_GetAttr(mp, s_grad));
  PyObject* m = PyDict_GetItem(st, s_exp_avg);        // borrowed
  PyObject* v = PyDict_GetItem(st, s_exp_avg_sq);
  if (!g.o || !m || !v) return false;
  int64_t ng, nm, nv;
  return flat32(mp, &c->p, &c->n) && flat32(g, &c->g, &ng) && flat32(m, &c->m, &nm) &&
         flat32(v, &c->v, &nv) && ng == c->n && nm == c->n && nv == c->n && number(rec, s_lr, &c->lr) &&
         number(rec, s_beta1, &c->b1) && number(rec, s_beta2, &c->b2) && number(rec, s_eps, &c->eps) &&
         number(rec, s_wd, &c->wd) && integer(rec, s_step, &c->step);
}
template <class E>
void hyper_into(E& e, const Common& c, bool adams) {
  e.lr = (float)c.lr; e.beta1 = (float)c.b1; e.om1 = (float)(1.0 - c.b1);
  e.beta2 = (float)c.b2; e.om2 = (float)(1.0 - c.b2); e.eps = (float)c.eps; e.wd = (float)c.wd;
  e.bc1 = adams ? 1.0f : (float)(1.0 - std::pow(c.b1, (double)c.step));
  e.bc2 = adams ? 1.0f : (float)(1.0 - std::pow(c.b2, (double)c.step));
}

// commit(records, use_mask, emit_id, coeff, clear, fold, interval, inactive_lr_scale, adams, stream)
PyObject* commit(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject* records;
  int use_mask, emit, clear, fold, adams;
  double coeff, interval, inactive;
  unsigned long long stream;
  if (!PyArg_ParseTuple(args, "OpidppddpK", &records, &use_mask, &emit, &coeff, &clear, &fold, &interval,
                        &inactive, &adams, &stream))
    return nullptr;
  Walk w(records);
  if (w.n < 0) return not_ordinary();
  std::vector<sga_gc_record> rows;
  rows.reserve((size_t)w.n);
  int64_t spans = 0;
  for (Py_ssize_t i = 0; i < w.n; ++i) {
    PyObject* rec = w.at(i);
    Common c;
    if (!common_of(rec, &c)) return not_ordinary();
    const uint8_t* mask = nullptr;
    const int has = use_mask ? mask_of(rec, c.n, &mask) : 0;
    if (has < 0) return not_ordinary();
    if (c.n == 0) continue;
    sga_gc_record e = {};
    e.p = c.p; e.g = c.g; e.m = c.m; e.v = c.v; e.mask = mask;
    e.n = c.n; e.first_span = spans;
    hyper_into(e, c, adams);
    // a record without a mask takes none of the sparse step's knobs
    e.lr_inactive = (float)(c.lr * (has ? inactive : 1.0));
    e.flags = (adams ? SGA_GC_ADAMS : 0);
    if (has)
      e.flags |= SGA_GC_HAS_MASK | (coeff != 1.0 ? SGA_GC_APPLY_COEFF : 0) | (clear ? SGA_GC_CLEAR : 0) |
                 (fold ? SGA_GC_FOLD : 0) | (inactive != 1.0 ? SGA_GC_LR_SPLIT : 0);
    rows.push_back(e);
    spans += (c.n + kSpan - 1) / kSpan;
  }
  if (rows.empty()) return PyLong_FromLong(0);
  const at::Tensor table = to_device(rows, device_of(w.at(0)));
  return PyLong_FromLong(f_gc_multi(static_cast<const sga_gc_record*>(table.data_ptr()), (int)rows.size(),
                                    spans, (float)coeff, (float)interval, emit, (void*)stream));
  END_HANDLE_TH_ERRORS
}

// commit_compact(records, compact_values, support, use_table, coeff, fold, interval, adams, stream):
// every record's bucket must have communicated values of one dtype
PyObject* commit_compact(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject *records, *values_of, *support;
  int use_table, fold, adams;
  double coeff, interval;
  unsigned long long stream;
  if (!PyArg_ParseTuple(args, "OOOpdpdpK", &records, &values_of, &support, &use_table, &coeff, &fold, &interval,
                        &adams, &stream))
    return nullptr;
  Walk w(records);
  if (w.n < 0) return not_ordinary();
  if (!PyDict_Check(values_of)) return not_ordinary();
  std::vector<sga_gcc_record> rows;
  rows.reserve((size_t)w.n);
  int64_t spans = 0;
  PyObject* last = nullptr;                            // the bucket looked up last (borrowed)
  const int32_t *idx = nullptr, *table = nullptr;
  const void* vals = nullptr;
  int64_t k_total = 0, n_table = -1;                   // n_table < 0: no table to search by
  int dtype = -1;
  for (Py_ssize_t i = 0; i < w.n; ++i) {
    PyObject* rec = w.at(i);
    Common c;
    int64_t start;
    Ref bs(PyObject_GetAttr(rec, s_bucket_state));
    if (!bs.o || !common_of(rec, &c) || !integer(rec, s_start, &start) || start < 0) return not_ordinary();
    if (bs.o != last) {
      Ref id(PyLong_FromVoidPtr(bs.o));
      PyObject* v = PyDict_GetItem(values_of, id);     // borrowed
      if (!v || !THPVariable_Check(v)) return not_ordinary();
      Ref si(PyObject_GetAttr(bs, s_support_index)), bl(PyObject_GetAttr(support, s_buckets));
      if (!si.o || !bl.o) return not_ordinary();
      Ref bucket(PyObject_GetItem(bl, si));
      if (!bucket.o) return not_ordinary();
      Ref ix(PyObject_GetAttr(bucket, s_idx)), dt(PyObject_GetAttr(bucket, s_dir_table));
      if (!ix.o || !THPVariable_Check(ix.o)) return not_ordinary();
      const at::Tensor& tv = THPVariable_Unpack(v);
      const at::Tensor& ti = THPVariable_Unpack(ix.o);
      const int code = tv.scalar_type() == at::kFloat ? SGA_F32 : tv.scalar_type() == at::kBFloat16 ? SGA_BF16 : -2;
      if (!tv.is_cuda() || !tv.is_contiguous() || code < 0 || (dtype >= 0 && code != dtype) || !ti.is_cuda() ||
          !ti.is_contiguous() || ti.scalar_type() != at::kInt)
        return not_ordinary();
      dtype = code;
      idx = static_cast<const int32_t*>(ti.data_ptr());
      vals = tv.data_ptr();
      k_total = ti.numel();
      table = nullptr;
      n_table = -1;
      if (use_table && dt.o && dt.o != Py_None) {
        if (!THPVariable_Check(dt.o)) return not_ordinary();
        const at::Tensor& tt = THPVariable_Unpack(dt.o);
        if (!tt.is_cuda() || !tt.is_contiguous() || tt.scalar_type() != at::kInt) return not_ordinary();
        table = static_cast<const int32_t*>(tt.data_ptr());
        n_table = tt.numel();
      } else if (use_table && !dt.o) {
        return not_ordinary();
      }
      PyErr_Clear();
      last = bs.o;
    }
    if (c.n == 0) continue;
    const int64_t lim = (int64_t)1 << 31;
    if (k_total + 1024 >= lim || start + c.n + 1024 >= lim || (n_table >= 0 && n_table < ((start + c.n - 1) >> 10) + 2))
      return not_ordinary();
    sga_gcc_record e = {};
    e.p = c.p; e.g = c.g; e.m = c.m; e.v = c.v;
    e.idx = idx; e.values = vals; e.table = table;
    e.rec_start = start; e.n = c.n; e.k_total = k_total; e.n_table = table ? n_table : 0; e.first_span = spans;
    hyper_into(e, c, adams);
    e.flags = (coeff != 1.0 ? SGA_GC_APPLY_COEFF : 0) | (fold ? SGA_GC_FOLD : 0) | (adams ? SGA_GC_ADAMS : 0);
    rows.push_back(e);
    spans += (c.n + kSpan - 1) / kSpan;
  }
  if (rows.empty()) return PyLong_FromLong(0);
  const at::Tensor dev = to_device(rows, device_of(w.at(0)));
  return PyLong_FromLong(f_gcc_multi(static_cast<const sga_gcc_record*>(dev.data_ptr()), (int)rows.size(), spans,
                                     dtype, (float)coeff, (float)interval, (void*)stream));
  END_HANDLE_TH_ERRORS
}

// norm_table(records, was_full): the gradients (and masks) of every record as one device
// table.  -> (table tensor, n_rows, spans, any_maskless), None for an empty set, False otherwise
PyObject* norm_table(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject* records;
  int was_full;
  if (!PyArg_ParseTuple(args, "Op", &records, &was_full)) return nullptr;
  Walk w(records);
  if (w.n < 0) return not_ordinary();
  std::vector<sga_span_record> rows;
  rows.reserve((size_t)w.n);
  int64_t spans = 0;
  bool maskless = false;
  c10::Device dev(c10::kCPU);
  for (Py_ssize_t i = 0; i < w.n; ++i) {
    PyObject* rec = w.at(i);
    if ((PyObject*)Py_TYPE(rec) != record_type) return not_ordinary();
    Ref mp(PyObject_GetAttr(rec, s_main_param));
    if (!mp.o) return not_ordinary();
    Ref g(PyObject_GetAttr(mp, s_grad));
    sga_span_record e = {};
    if (!g.o || !THPVariable_Check(g.o) || !flat32(g, &e.g, &e.n)) return not_ordinary();
    if (dev.is_cpu()) dev = THPVariable_Unpack(g.o).device();
    const int has = was_full ? 0 : mask_of(rec, e.n, &e.mask);
    if (has < 0) return not_ordinary();
    maskless = maskless || has == 0;
    if (e.n == 0) continue;
    e.first_span = spans;
    rows.push_back(e);
    spans += (e.n + kSpan - 1) / kSpan;
  }
  if (rows.empty()) Py_RETURN_NONE;
  at::Tensor table = to_device(rows, dev);
  return Py_BuildValue("(NnLO)", THPVariable_Wrap(table), (Py_ssize_t)rows.size(), (long long)spans,
                       maskless ? Py_True : Py_False);
  END_HANDLE_TH_ERRORS
}

// Results that the host waits for come into words of its own, which the kernel writes one by one (st_host): a copy and
// the stream's end behind it were 5 to 15 us of every wait, and what follows the kernel on the stream runs on.  With a
// copy -> so, us: mask layout step on 1.15 M coordinates 122 -> 106, dense replay step and two configurations of 1.5 M
// 1,930 -> 1,783, full step on 63 M 854 -> 835.  A block is one call's, from torch's
// pool.  It goes back with the tensor once all of its words have been written; a tensor that dies before (an error or
// an interrupt between the launch and the wait) leaves it with an event of the stream, behind which nothing writes there.
// words(n, wide): n results of 32 bits, or of 64, in pinned host memory, all bits set: none of them has arrived.
// A result of 64 bits is stored and looked at in one piece: its halves may well have all bits set (2^53 - 1 as a
// double), the whole of it never has.
template <class W>
bool written(const W* w, int64_t n) {
  for (int64_t i = 0; i < n; ++i)
    if (__atomic_load_n(w + i, __ATOMIC_ACQUIRE) == (W)~(W)0) return false;
  return true;
}
struct Words {
  at::DataPtr block;
  int64_t n;
  bool wide;
  c10::Stream stream;
  bool all_written() const {
    return wide ? written(static_cast<uint64_t*>(block.get()), n) : written(static_cast<uint32_t*>(block.get()), n);
  }
  // of the tensor, on whichever thread drops it
  static void release(void* ctx) {
    auto* w = static_cast<Words*>(ctx);
    bool ours = w->all_written();
    try {
      if (!ours) ours = at::getHostAllocator(at::kCUDA)->record_event(w->block.get(), w->block.get_context(), w->stream);
    } catch (...) {
    }
    if (ours) delete w;                                // otherwise (a lost device) nobody gets the block any more
  }
};
at::Tensor blank_words(int64_t n, bool wide = false) {
  const size_t bytes = (size_t)n * (wide ? 8 : 4);
  const c10::impl::VirtualGuardImpl gpu(c10::DeviceType::CUDA);
  auto* w = new Words{at::getHostAllocator(at::kCUDA)->allocate(bytes), n, wide, gpu.getStream(gpu.getDevice())};
  void* at = w->block.get();
  if (bytes) memset(at, 0xFF, bytes);
  c10::Storage mem(c10::Storage::use_byte_size_t(), bytes, at::DataPtr(at, w, &Words::release, at::kCPU), nullptr, false);
  at::Tensor t = at::detail::make_tensor<c10::TensorImpl>(std::move(mem), c10::DispatchKeySet(c10::DispatchKey::CPU),
                                                          caffe2::TypeMeta::fromScalarType(wide ? at::kLong : at::kInt));
  t.unsafeGetTensorImpl()->set_sizes_contiguous({n});
  return t;
}
PyObject* words(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  long long n;
  int wide = 0;
  if (!PyArg_ParseTuple(args, "L|p", &n, &wide)) return nullptr;
  return THPVariable_Wrap(blank_words(n, wide != 0));
  END_HANDLE_TH_ERRORS
}
// True when all of them have been written; looks for kLook at most.
constexpr std::chrono::milliseconds kLook(20);
template <class W>
bool all_arrived(const W* w, int64_t n) {
  const auto end = std::chrono::steady_clock::now() + kLook;
  for (;;) {
    for (int i = 0; i < 64; ++i) {
      if (written(w, n)) return true;
      __builtin_ia32_pause();
    }
    if (std::chrono::steady_clock::now() > end) return written(w, n);
  }
}
// arrived(words) -> their values, or None where they have not come for some time
PyObject* arrived(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject* t;
  if (!PyArg_ParseTuple(args, "O", &t)) return nullptr;
  if (!THPVariable_Check(t)) {
    PyErr_SetString(PyExc_TypeError, "arrived: a tensor of words");
    return nullptr;
  }
  const at::Tensor held = THPVariable_Unpack(t);
  const bool wide = held.scalar_type() == at::kLong;
  if (held.is_cuda() || (!wide && held.scalar_type() != at::kInt) || !held.is_contiguous()) {
    PyErr_SetString(PyExc_TypeError, "arrived: words of 32 or 64 bits in host memory");
    return nullptr;
  }
  const uint32_t* w = static_cast<const uint32_t*>(held.data_ptr());
  const uint64_t* w64 = static_cast<const uint64_t*>(held.data_ptr());
  const int64_t n = held.numel();
  const bool there = [&] {
    Unlocked released;
    return wide ? all_arrived(w64, n) : all_arrived(w, n);
  }();
  if (!there) Py_RETURN_NONE;
  PyObject* out = PyTuple_New(n);
  for (int64_t i = 0; out && i < n; ++i) PyTuple_SET_ITEM(out, i, PyLong_FromUnsignedLongLong(wide ? w64[i] : w[i]));
  return out;
  END_HANDLE_TH_ERRORS
}

// norm(table, n_rows, spans, stream) -> sqrt of the sum of squares (waits for the stream)
PyObject* norm(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject* t;
  int n_rows;
  long long spans;
  unsigned long long stream;
  if (!PyArg_ParseTuple(args, "OiLK", &t, &n_rows, &spans, &stream)) return nullptr;
  const at::Tensor& table = THPVariable_Unpack(t);
  // the partials, fp32; every slot that is read is written first.  The total comes into host memory (a copy of it is
  // a launch, and 3 us of the wait).
  at::Tensor buf = at::empty({spans}, at::TensorOptions().dtype(at::kFloat).device(table.device()));
  const at::Tensor word = table.is_cuda() ? blank_words(1) : at::full({1}, -1, at::kInt);
  const int rc = f_norm_multi(static_cast<const sga_span_record*>(table.data_ptr()), n_rows, spans,
                              static_cast<float*>(buf.data_ptr()), static_cast<float*>(word.data_ptr()), (void*)stream);
  if (rc != 0) return PyLong_FromLong(rc);
  const uint32_t* w = static_cast<const uint32_t*>(word.data_ptr());
  const bool there = [&] {
    Unlocked released;
    // not there in time: a read from the device waits for the stream, and raises its errors
    if (!table.is_cuda() || !all_arrived(w, 1)) (void)buf[0].item<float>();
    return written(w, 1);
  }();
  if (!there) {
    PyErr_SetString(PyExc_RuntimeError, "norm: a result that its kernel should have written has not arrived");
    return nullptr;
  }
  const double total = *static_cast<const float*>(word.data_ptr());
  return PyFloat_FromDouble((double)(float)std::sqrt(total));
  END_HANDLE_TH_ERRORS
}

// scale(table, n_rows, spans, coeff, stream)
PyObject* scale(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject* t;
  int n_rows;
  long long spans;
  double coeff;
  unsigned long long stream;
  if (!PyArg_ParseTuple(args, "OiLdK", &t, &n_rows, &spans, &coeff, &stream)) return nullptr;
  const at::Tensor& table = THPVariable_Unpack(t);
  return PyLong_FromLong(f_scale_multi(static_cast<const sga_span_record*>(table.data_ptr()), n_rows, spans,
                                       (float)coeff, (void*)stream));
  END_HANDLE_TH_ERRORS
}

// bind(record type, gc_multi, gcc_multi, norm_multi, scale_multi): addresses of the entry points
PyObject* bind(PyObject*, PyObject* args) {
  unsigned long long a, b, c, d;
  PyObject* type;
  if (!PyArg_ParseTuple(args, "OKKKK", &type, &a, &b, &c, &d)) return nullptr;
  Py_INCREF(type);
  record_type = type;
  f_gc_multi = reinterpret_cast<decltype(f_gc_multi)>(a);
  f_gcc_multi = reinterpret_cast<decltype(f_gcc_multi)>(b);
  f_norm_multi = reinterpret_cast<decltype(f_norm_multi)>(c);
  f_scale_multi = reinterpret_cast<decltype(f_scale_multi)>(d);
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"words", words, METH_VARARGS, nullptr},
                         {"arrived", arrived, METH_VARARGS, nullptr},
                         {"bind", bind, METH_VARARGS, nullptr},
                         {"commit", commit, METH_VARARGS, nullptr},
                         {"commit_compact", commit_compact, METH_VARARGS, nullptr},
                         {"norm_table", norm_table, METH_VARARGS, nullptr},
                         {"norm", norm, METH_VARARGS, nullptr},
                         {"scale", scale, METH_VARARGS, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
  const struct { PyObject** at; const char* name; } names[] = {
      {&s_main_param, "main_param"}, {&s_grad, "grad"}, {&s_data, "data"}, {&s_state, "_state"},
      {&s_exp_avg, "exp_avg"}, {&s_exp_avg_sq, "exp_avg_sq"}, {&s_bucket_state, "bucket_state"},
      {&s_mask, "active_mask_u8"}, {&s_start, "start"}, {&s_end, "end"}, {&s_lr, "lr"}, {&s_beta1, "beta1"},
      {&s_beta2, "beta2"}, {&s_eps, "eps"}, {&s_wd, "weight_decay"}, {&s_step, "step"},
      {&s_support_index, "support_index"}, {&s_buckets, "buckets"}, {&s_idx, "idx"},
      {&s_dir_table, "dir_table"}};
  for (const auto& s : names) *s.at = PyUnicode_InternFromString(s.name);
  return PyModule_Create(&module);
}
