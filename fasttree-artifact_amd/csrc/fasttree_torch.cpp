// Python binding of the calls a serving loop makes once per layer: decode and the store of the
// step's K/V rows.  It reads the tensors' addresses, strides and types itself and calls the C ABI
// of include/fasttree_hip.h.
//
// Why it exists: a decode call of a few requests takes the device about 11 us, and marshalling its
// 21 arguments in Python (some thirty data_ptr() / stride() calls, as many checks, 45 ctypes
// conversions) took the host 16 us, so small calls ran at the speed of the interpreter.
//
// The checks, their order and the exceptions are those the Python wrapper documents: AssertionError
// for head dimensions that differ, FastTreeLibraryError otherwise.  Functions return the C ABI's code.

#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/fasttree_hip.h"

namespace {

PyObject* g_library_error = nullptr;   // fasttree_hip._lib.FastTreeLibraryError
// attribute names of a launch-order plan's phase list, interned once
PyObject *g_prog_table, *g_narrow_table, *g_prog_records, *g_req_table, *g_num_programs, *g_narrow_in_programs, *g_wave_records, *g_records_version;

// what decode_layer reads from a FastTreeMetadata, in the order of the decode call's arguments
constexpr int kMetaAttributes = 14;
const char* const kMetaNames[kMetaAttributes] = {
    "vnode_to_kv_offs", "vnode_to_kv_lens", "vnode_to_q_entries", "vnode_to_q_offs", "vnode_to_q_lens", "req_to_vnode_entries",
    "req_to_vnode_offs", "req_to_vnode_lens", "mid_o", "mid_lse", "phase_node_nums", "phase_node_offsets", "phase_q_tile_sizes",
    "phase_kv_tile_sizes"};
PyObject* g_meta_attributes[kMetaAttributes];

struct PyFailure {};   // thrown with a Python exception set

[[noreturn]] void refuse(const char* message) {
  PyErr_SetString(g_library_error, message);
  throw PyFailure{};
}

const at::Tensor& tensor(PyObject* o) {
  if (!THPVariable_Check(o)) {
    PyErr_Format(PyExc_TypeError, "expected a tensor, got %s", Py_TYPE(o)->tp_name);
    throw PyFailure{};
  }
  return THPVariable_Unpack(o);
}

void need_gpu(const at::Tensor& t) {
  if (!t.is_cuda()) refuse("fasttree_decode needs device tensors; there is no CPU path");
}
void need_i32(const at::Tensor& t) {
  if (t.scalar_type() != at::kInt || !t.is_contiguous()) refuse("index tensors must be contiguous int32");
}
void need_inner_contiguous(const at::Tensor& t) {
  if (t.stride(-1) != 1) refuse("the last dimension of q, k, v, o and the scratch must be contiguous");
}

int dtype_code(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kHalf: return FT_DTYPE_F16;
    case at::kBFloat16: return FT_DTYPE_BF16;
    default: break;
  }
  refuse("unsupported dtype: fp16 and bf16 only");
}

ft_stream_t stream_of(const at::Tensor& t) {
  return reinterpret_cast<ft_stream_t>(c10::hip::getCurrentHIPStream(t.device().index()).stream());
}

int64_t integer(PyObject* o) {
  PyObject* n = PyNumber_Long(o);
  if (!n) throw PyFailure{};
  const long long v = PyLong_AsLongLong(n);
  Py_DECREF(n);
  if (v == -1 && PyErr_Occurred()) throw PyFailure{};
  return v;
}

struct Pair { int32_t v[2]; };
Pair int32_pair(PyObject* o) {
  const Py_ssize_t n = PySequence_Size(o);
  if (n == -1) throw PyFailure{};
  if (n != 2) {
    PyErr_SetString(PyExc_ValueError, "expected a sequence of two integers");
    throw PyFailure{};
  }
  Pair p;
  for (int i = 0; i < 2; ++i) {
    PyObject* item = PySequence_GetItem(o, i);
    if (!item) throw PyFailure{};
    int64_t v;
    try {
      v = integer(item);
    } catch (...) {
      Py_DECREF(item);
      throw;
    }
    Py_DECREF(item);
    p.v[i] = (int32_t)v;
  }
  return p;
}

// Gives the interpreter up around a launch (a full queue makes it wait).
struct Unlocked {
  PyThreadState* state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};

// What a launch-order plan's phase list carries besides its two counts (null / 0: not there).
struct PlanTables {
  const int32_t *prog_table = nullptr, *narrow_table = nullptr, *prog_records = nullptr, *req_table = nullptr;
  int num_programs = 0, narrow_in_programs = 0;
  const int32_t* wave_records = nullptr;   // of a plan of whole paths whose lists nobody has written to
  int64_t wave_ints = 0;
};

struct Held {   // a new reference that is dropped at the end of the scope
  PyObject* o;
  explicit Held(PyObject* p) : o(p) {}
  Held(const Held&) = delete;
  ~Held() { Py_XDECREF(o); }
};

PyObject* attribute_or_null(PyObject* o, PyObject* name) {
  PyObject* a = PyObject_GetAttr(o, name);
  if (!a) {
    if (!PyErr_ExceptionMatches(PyExc_AttributeError)) throw PyFailure{};
    PyErr_Clear();
  }
  return a;
}
// The records of a plan of whole paths, if they still say what its lists do (launch_schedule.whole_paths asks the same).
void find_wave_records(PyObject* phases, PlanTables& t) {
  Held records(attribute_or_null(phases, g_wave_records));
  if (!records.o || records.o == Py_None) return;
  Held narrow(attribute_or_null(phases, g_narrow_table)), version(attribute_or_null(phases, g_records_version));
  if (!narrow.o || narrow.o == Py_None || !version.o || version.o == Py_None) return;
  const at::Tensor& table = tensor(narrow.o);
  if (table.is_inference() || (int64_t)table._version() != integer(version.o)) return;
  const at::Tensor& r = tensor(records.o);
  t.wave_records = static_cast<const int32_t*>(r.data_ptr());
  t.wave_ints = r.numel();
}
// (the plan's list keeps the tensor alive past this call)
const int32_t* table_address(PyObject* phases, PyObject* name) {
  Held a(attribute_or_null(phases, name));
  if (!a.o || a.o == Py_None) return nullptr;
  return static_cast<const int32_t*>(tensor(a.o).data_ptr());
}
int count_of(PyObject* phases, PyObject* name) {
  Held a(attribute_or_null(phases, name));
  return a.o ? (int)integer(a.o) : 0;
}

PlanTables plan_tables(PyObject* phases) {
  PlanTables t;
  if (PyList_CheckExact(phases) || PyTuple_CheckExact(phases)) return t;
  t.narrow_table = table_address(phases, g_narrow_table);
  t.req_table = table_address(phases, g_req_table);
  t.prog_table = table_address(phases, g_prog_table);
  if (t.prog_table) {
    t.prog_records = table_address(phases, g_prog_records);
    t.num_programs = count_of(phases, g_num_programs);
    t.narrow_in_programs = count_of(phases, g_narrow_in_programs);
  } else {
    find_wave_records(phases, t);
  }
  return t;
}

// Sizes and element strides of a [tokens, heads, dim] tensor.
struct Rows {
  int64_t n, heads, dim, s0, s1;
};
Rows rows_of(const at::Tensor& t) { return Rows{t.size(0), t.size(1), t.size(-1), t.stride(0), t.stride(1)}; }

int32_t* i32(const at::Tensor& t) { return static_cast<int32_t*>(t.data_ptr()); }

// [tokens, heads * dim] or [tokens, heads, dim] as [tokens, heads, dim], without making a view of it.
Rows rows_as(const at::Tensor& t, int64_t heads, int64_t dim) {
  if (t.dim() == 3 && t.size(1) == heads && t.size(2) == dim) return rows_of(t);
  if (t.dim() == 2 && t.size(1) == heads * dim) return Rows{t.size(0), heads, dim, t.stride(0), dim * t.stride(1)};
  return rows_of(t.view({-1, heads, dim}));   // (raises where the shape does not fit)
}

// The checks and the call shared by decode and decode_layer.  `index`: the nine index tensors.
int decode_call(const at::Tensor& q, const Rows& qr, const at::Tensor& k, const at::Tensor& v, const at::Tensor& o, const Rows& orow,
                const at::Tensor* const (&index)[9], const at::Tensor& mid_o, const at::Tensor& mid_lse, PyObject* phase_nums,
                PyObject* phase_offs, PyObject* phase_q_tiles, PyObject* phase_kv_tiles, PyObject* sm_scale) {
  if (qr.dim != k.size(-1)) {   // fasttree.py:437-438
    PyErr_SetNone(PyExc_AssertionError);
    throw PyFailure{};
  }
  for (const at::Tensor* t : {&q, &k, &v, &o, &mid_o, &mid_lse, index[0]}) need_gpu(*t);
  for (const at::Tensor* t : {&q, &k, &v, &o, &mid_o, &mid_lse}) need_inner_contiguous(*t);
  for (const at::Tensor* t : index) need_i32(*t);
  if (k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type() || o.scalar_type() != q.scalar_type())
    refuse("q, k, v and o must share one dtype");
  if (mid_o.scalar_type() != at::kFloat || mid_lse.scalar_type() != at::kFloat) refuse("mid_o and mid_lse must be float32");

  PlanTables plan = plan_tables(phase_nums);
  const Pair nums = int32_pair(phase_nums), offs = int32_pair(phase_offs);
  const double scale = PyFloat_AsDouble(sm_scale);
  if (scale == -1.0 && PyErr_Occurred()) throw PyFailure{};
  const int d = (int)qr.dim, dtype = dtype_code(q);
  const ft_stream_t stream = stream_of(q);
  const int heads_kv = (int)k.size(1);
  // (laid out for other rows, as for a plan made for another head_dim, they are not for this call)
  if (plan.wave_records && plan.wave_ints == (int64_t)64 * FT_PATH_WAVES(d) * nums.v[1]) {
    plan.prog_records = plan.wave_records;
    plan.narrow_in_programs = FT_WHOLE_PATHS;
  }
  if ((plan.prog_table || plan.narrow_table) && d >= 32) {
    Unlocked unlocked;
    // the launch was arranged as block programs (launch_schedule.block_programs)
    return ft_decode_programs(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), qr.s0, qr.s1, k.stride(0), k.stride(1), v.stride(0),
                              v.stride(1), orow.s0, orow.s1, i32(*index[0]), i32(*index[1]), i32(*index[2]), i32(*index[3]),
                              i32(*index[4]), i32(*index[5]), i32(*index[6]), i32(*index[7]), i32(*index[8]),
                              static_cast<float*>(mid_o.data_ptr()), mid_o.stride(0), mid_o.stride(1),
                              static_cast<float*>(mid_lse.data_ptr()), mid_lse.stride(0), nums.v, offs.v, plan.prog_table,
                              plan.num_programs, plan.narrow_in_programs, plan.narrow_table, plan.prog_records, plan.req_table,
                              (int)qr.n, (int)qr.heads, heads_kv, d, (float)scale, dtype, stream);
  }
  const Pair q_tiles = int32_pair(phase_q_tiles), kv_tiles = int32_pair(phase_kv_tiles);
  Unlocked unlocked;
  return ft_decode(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), qr.s0, qr.s1, k.stride(0), k.stride(1), v.stride(0),
                   v.stride(1), orow.s0, orow.s1, i32(*index[0]), i32(*index[1]), i32(*index[2]), i32(*index[3]), i32(*index[4]),
                   i32(*index[5]), i32(*index[6]), i32(*index[7]), i32(*index[8]), static_cast<float*>(mid_o.data_ptr()),
                   mid_o.stride(0), mid_o.stride(1), static_cast<float*>(mid_lse.data_ptr()), mid_lse.stride(0), nums.v, offs.v,
                   q_tiles.v, kv_tiles.v, (int)qr.n, (int)qr.heads, heads_kv, d, (float)scale, dtype, stream);
}

// decode(q, k_buffer, v_buffer, o, the nine index tensors, mid_o, mid_lse, phase_node_nums,
//        phase_node_offsets, phase_q_tile_sizes, phase_kv_tile_sizes, sm_scale) -> code
PyObject* decode(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 20) {
    PyErr_SetString(PyExc_TypeError, "decode takes 20 arguments");
    return nullptr;
  }
  try {
    const at::Tensor &q = tensor(args[0]), &k = tensor(args[1]), &v = tensor(args[2]), &o = tensor(args[3]);
    const at::Tensor* index[9];
    for (int i = 0; i < 9; ++i) index[i] = &tensor(args[4 + i]);
    return PyLong_FromLong(decode_call(q, rows_of(q), k, v, o, rows_of(o), index, tensor(args[13]), tensor(args[14]), args[15], args[16],
                                       args[17], args[18], args[19]));
  } catch (const PyFailure&) {
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}

int store_call(const at::Tensor& kn, const at::Tensor& vn, const at::Tensor& loc, const at::Tensor& kb, const at::Tensor& vb) {
  for (const at::Tensor* t : {&kn, &vn, &loc, &kb, &vb}) need_gpu(*t);
  const int64_t hkv = kb.size(1), d = kb.size(2);
  if (vb.dim() != 3 || vb.size(1) != hkv || vb.size(2) != d || vb.scalar_type() != kb.scalar_type())
    refuse("k_buffer and v_buffer must have the same heads, head size and dtype");
  if (kn.scalar_type() != kb.scalar_type() || vn.scalar_type() != kb.scalar_type()) refuse("the new rows must have the pools' dtype");
  for (const at::Tensor* t : {&kn, &vn, &kb, &vb}) need_inner_contiguous(*t);
  const Rows k = rows_as(kn, hkv, d), v = rows_as(vn, hkv, d);
  if (v.n != k.n || loc.numel() != k.n) refuse("cache_k, cache_v and out_cache_loc must name the same number of tokens");
  if ((loc.scalar_type() != at::kInt && loc.scalar_type() != at::kLong) || !loc.is_contiguous())
    refuse("out_cache_loc must be a contiguous int32 or int64 tensor");
  const int dtype = dtype_code(kb);
  const ft_stream_t stream = stream_of(kb);
  Unlocked unlocked;
  return ft_store_kv(kn.data_ptr(), vn.data_ptr(), k.s0, k.s1, v.s0, v.s1, loc.data_ptr(), loc.scalar_type() == at::kLong, (int)k.n,
                     kb.data_ptr(), vb.data_ptr(), kb.stride(0), kb.stride(1), vb.stride(0), vb.stride(1),
                     std::min(kb.size(0), vb.size(0)), (int)hkv, (int)d, dtype, stream);
}

// store_kv(cache_k, cache_v, out_cache_loc, k_buffer, v_buffer) -> code
PyObject* store_kv(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 5) {
    PyErr_SetString(PyExc_TypeError, "store_kv takes 5 arguments");
    return nullptr;
  }
  try {
    return PyLong_FromLong(store_call(tensor(args[0]), tensor(args[1]), tensor(args[2]), tensor(args[3]), tensor(args[4])));
  } catch (const PyFailure&) {
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}

// decode_layer(q, o, k_buffer, v_buffer, req_to_token, metadata, heads, qk_dim, v_dim, sm_scale): the
// serving hook's decode on flat q [tokens, heads * qk_dim] and o, with the index tensors, scratch and
// phase lists of a FastTreeMetadata -> code
PyObject* decode_layer(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 10) {
    PyErr_SetString(PyExc_TypeError, "decode_layer takes 10 arguments");
    return nullptr;
  }
  try {
    const at::Tensor &q = tensor(args[0]), &o = tensor(args[1]);
    const int64_t heads = integer(args[6]), qk_dim = integer(args[7]), v_dim = integer(args[8]);
    PyObject* held[kMetaAttributes] = {};
    struct Release {
      PyObject** p;
      ~Release() { for (int i = 0; i < kMetaAttributes; ++i) Py_XDECREF(p[i]); }
    } release{held};
    for (int i = 0; i < kMetaAttributes; ++i)
      if (!(held[i] = PyObject_GetAttr(args[5], g_meta_attributes[i]))) throw PyFailure{};
    const at::Tensor* index[9] = {&tensor(args[4])};
    for (int i = 0; i < 8; ++i) index[1 + i] = &tensor(held[i]);
    return PyLong_FromLong(decode_call(q, rows_as(q, heads, qk_dim), tensor(args[2]), tensor(args[3]), o, rows_as(o, heads, v_dim), index,
                                       tensor(held[8]), tensor(held[9]), held[10], held[11], held[12], held[13], args[9]));
  } catch (const PyFailure&) {
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"decode", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(decode)), METH_FASTCALL, "One decode call; returns the C ABI's code."},
    {"decode_layer", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(decode_layer)), METH_FASTCALL,
     "The serving hook's decode call; returns the C ABI's code."},
    {"store_kv", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(store_kv)), METH_FASTCALL,
     "The step's new K and V rows into the pools; returns the C ABI's code."},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_torch_binding", "Per-layer calls on torch tensors.", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__torch_binding(void) {
  PyObject* lib = PyImport_ImportModule("fasttree_hip._lib");
  if (!lib) return nullptr;
  g_library_error = PyObject_GetAttrString(lib, "FastTreeLibraryError");
  Py_DECREF(lib);
  if (!g_library_error) return nullptr;
  struct { PyObject** at; const char* name; } names[] = {
      {&g_prog_table, "prog_table"}, {&g_narrow_table, "narrow_table"}, {&g_prog_records, "prog_records"},
      {&g_req_table, "req_table"}, {&g_num_programs, "num_programs"}, {&g_narrow_in_programs, "narrow_in_programs"},
      {&g_wave_records, "wave_records"}, {&g_records_version, "records_version"}};
  for (auto& n : names)
    if (!(*n.at = PyUnicode_InternFromString(n.name))) return nullptr;
  for (int i = 0; i < kMetaAttributes; ++i)
    if (!(g_meta_attributes[i] = PyUnicode_InternFromString(kMetaNames[i]))) return nullptr;
  return PyModule_Create(&module);
}
