// Host path of inference calls and training steps in C++ (CPython module dkernel_amd._host): what ops.py does for a
// forward that needs no gradient - checks, outputs, scratch, the argument block of dk_fwd - without
// the interpreter.  A single-token step or a short prompt keeps the GPU busy for 8 - 15 us; the
// Python launcher took 15 us of host time per call around the launch itself (2.5 us).  For the two halves of a training
// step (train_forward, train_backward) it is the launch alone: which tables, lengths and gradients, and all of autograd, stay
// in ops.py.
//
// The functions take the common case only: tensors as the kernels want them.  They return None,
// having done nothing, for anything else (tensors on the host, strides to be fixed, lengths of another
// type, gradients, tables in an order of their own, wrong arguments of any kind): the caller then takes
// the path in ops.py, which handles it or raises.  The C ABI is reached through the addresses that
// bind() gets from the library that ops.py has loaded.
//
// Everything that comes from Python objects is read first; allocations and the launch run without the
// interpreter lock (Unlocked), as they do through torch's own bindings and ctypes: threads that serve on
// several streams do not wait for each other's launches, nor a launch into a full queue for a host callback
// that needs the lock.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/core/grad_mode.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <cstdlib>
#include <cstring>
#include <optional>

#include "../../include/dkernel_hip.h"

namespace {

int (*fwd_fn)(const dk_fwd_args *) = nullptr;
size_t (*fwd_bytes_fn)(const dk_fwd_args *) = nullptr;
int (*fwd_paged_fn)(const dk_fwd_args *, const dk_paged_kv *) = nullptr;
int (*bwd_fn)(const dk_bwd_args *, const dk_row_lengths *) = nullptr;
size_t (*bwd_bytes_fn)(const dk_bwd_args *, const dk_row_lengths *) = nullptr;

PyObject *k_max_seqlen, *k_causal, *k_group, *k_max_row, *k_uneven, *k_unsorted, *k_fixed, *k_out, *k_inference;

struct Unsupported {};  // thrown by the helpers below, turned into None

struct Unlocked {  // the interpreter lock is released while this lives
  PyThreadState *state = PyEval_SaveThread();
  Unlocked() = default;
  Unlocked(const Unlocked &) = delete;
  ~Unlocked() { PyEval_RestoreThread(state); }
};

const at::Tensor &tensor(PyObject *o) {
  if (!THPVariable_CheckExact(o)) throw Unsupported{};
  return THPVariable_Unpack(o);
}
const at::Tensor *optional_tensor(PyObject *o) { return o == Py_None ? nullptr : &tensor(o); }

void need(bool ok) {
  if (!ok) throw Unsupported{};
}

int64_t integer(PyObject *o) {
  const long v = PyLong_AsLong(o);
  if (v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    throw Unsupported{};
  }
  return v;
}

bool truth(PyObject *o) { return o == Py_True || (o != Py_False && o && PyObject_IsTrue(o) == 1); }

PyObject *item(PyObject *dict, PyObject *key) {  // borrowed; nullptr when absent
  PyObject *v = PyDict_GetItemWithError(dict, key);
  if (!v) PyErr_Clear();
  return v;
}

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kBFloat16: return DK_BF16;
    case at::kHalf: return DK_F16;
    case at::kFloat: return DK_F32;
    default: throw Unsupported{};
  }
}

dk_tensor view(const at::Tensor &t, int b, int h, int s) {  // b < 0: packed, no batch dimension
  const auto st = t.strides();
  return dk_tensor{t.data_ptr(), b < 0 ? 0 : st[b], st[h], st[s]};
}

bool rows_aligned(const at::Tensor &t) {  // as ops._matrix_core_applies
  const auto st = t.strides();
  for (size_t i = 0; i + 1 < st.size(); ++i)
    if (st[i] % 8) return false;
  return (reinterpret_cast<uintptr_t>(t.data_ptr()) % 16) == 0;
}

const int32_t *lengths(const at::Tensor *t, int64_t n, int dev) {
  if (!t) return nullptr;
  need(t->is_cuda() && t->get_device() == dev && t->scalar_type() == at::kInt && t->dim() == 1 && t->size(0) == n &&
       (n <= 1 || t->stride(0) == 1));
  return static_cast<const int32_t *>(t->data_ptr());
}

void fill_lut(dk_lut &l, const at::Tensor &ptr, const at::Tensor &idx, int dev, int64_t rows, int64_t cols, int64_t sub,
              int64_t group, int64_t max_row, bool uneven, bool fixed_walk) {
  need(ptr.dim() == 2 && ptr.scalar_type() == at::kInt && idx.scalar_type() == at::kInt && ptr.is_cuda() &&
       idx.is_cuda() && ptr.get_device() == dev && idx.get_device() == dev && ptr.stride(1) == 1);
  l = dk_lut{};
  if (idx.dim() == 3) {
    need(idx.size(2) == 2 && idx.stride(2) == 1 && idx.stride(1) == 2);
    l.entry_width = 2;
  } else {
    need(idx.dim() == 2 && (idx.stride(1) == 1 || idx.size(1) <= 1));
    l.entry_width = 1;
  }
  l.ptr = static_cast<const int32_t *>(ptr.data_ptr());
  l.idx = static_cast<const int32_t *>(idx.data_ptr());
  l.ptr_stride_h = ptr.stride(0), l.idx_stride_h = idx.stride(0);
  l.num_heads = (int32_t)ptr.size(0), l.num_rows = (int32_t)ptr.size(1) - 1;
  l.block_rows = (int32_t)rows, l.block_cols = (int32_t)cols;
  l.group = (int32_t)group, l.max_row_entries = (int32_t)max_row, l.sub_block = (int32_t)sub;
  l.uneven_heads = uneven, l.fixed_walk = fixed_walk;
}

// A table's tensors, held across the launch: another thread may give the module other ones meanwhile.
struct Table {
  at::Tensor ptr, idx;
};

// The module's table for these tensors: tables = (crow name, col name, rows, cols, masked crow name or
// None, masked col name, tile, sub_block), names of entries of `buffers`.
Table choose_lut(dk_lut &l, PyObject *buffers, PyObject *tables, int64_t masked_max_row, bool masked_ok, int dev, int64_t group,
                int64_t max_row, bool uneven, bool fixed_walk) {
  need(PyDict_Check(buffers) && PyTuple_Check(tables) && PyTuple_GET_SIZE(tables) == 8);
  const bool masked = masked_ok && PyTuple_GET_ITEM(tables, 4) != Py_None;
  const int at = masked ? 4 : 0;
  PyObject *crow = item(buffers, PyTuple_GET_ITEM(tables, at)), *col = item(buffers, PyTuple_GET_ITEM(tables, at + 1));
  need(crow && col);
  const int64_t rows = integer(PyTuple_GET_ITEM(tables, at + 2)), last = integer(PyTuple_GET_ITEM(tables, at + 3));
  Table t{tensor(crow), tensor(col)};
  fill_lut(l, t.ptr, t.idx, dev, rows, masked ? rows : last, masked ? last : 0, group, masked ? masked_max_row : max_row, uneven,
           fixed_walk);
  return t;
}

// What the module's kwargs say
struct Options {
  int64_t max_seqlen, group, max_row;
  bool causal, uneven, unsorted, fixed_walk;
  explicit Options(PyObject *kw) {
    need(PyDict_Check(kw) && !item(kw, k_out) && !item(kw, k_inference));
    PyObject *len = item(kw, k_max_seqlen), *g = item(kw, k_group), *row = item(kw, k_max_row), *c = item(kw, k_causal);
    need(len && g && row && c);
    max_seqlen = integer(len), group = integer(g), max_row = integer(row);
    causal = truth(c);
    uneven = truth(item(kw, k_uneven));
    unsorted = truth(item(kw, k_unsorted));
    fixed_walk = truth(item(kw, k_fixed));
  }
};

double scale_of(PyObject *o, int64_t dim) {
  double s = 0;
  if (PyFloat_Check(o))
    s = PyFloat_AS_DOUBLE(o);
  else if (PyLong_Check(o))
    s = (double)integer(o);
  else
    need(o == Py_None);
  return s != 0 ? s : 1.0 / std::sqrt((double)dim);
}

void check_qkv(const at::Tensor &q, const at::Tensor &k, const at::Tensor &v) {
  need(q.is_cuda() && k.is_cuda() && v.is_cuda() && q.scalar_type() == k.scalar_type() && q.scalar_type() == v.scalar_type());
  need(q.get_device() == k.get_device() && q.get_device() == v.get_device() && q.get_device() == c10::hip::current_device());
  need(k.sizes() == v.sizes() && q.dim() == k.dim() && q.size(-1) == k.size(-1) && q.size(-1) > 0);
  need(q.stride(-1) == 1 && k.stride(-1) == 1 && v.stride(-1) == 1);
  need(!(at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad())));
}

void check_heads(const dk_lut &l, int64_t hq, int64_t hkv) {
  need(hkv > 0 && hq % hkv == 0 && (l.num_heads == 1 || l.num_heads == hkv || l.num_heads == hq));
}

void *current_stream() { return static_cast<void *>(c10::hip::getCurrentHIPStream().stream()); }

// Scratch, launch.  Returns the scratch's size, or throws when the library refuses (the Python path
// then repeats the call and raises the library's message).
size_t launch(dk_fwd_args &a, const at::Tensor &q, bool use_workspace) {
  a.stream = current_stream();
  const size_t bytes = use_workspace ? fwd_bytes_fn(&a) : 0;
  at::Tensor ws;
  if (bytes) {
    ws = at::empty({(int64_t)bytes}, q.options().dtype(at::kByte));
    a.workspace = ws.data_ptr(), a.workspace_bytes = bytes;
  }
  need(fwd_fn(&a) == DK_OK);
  return bytes;
}

PyObject *result(const at::Tensor &out, const at::Tensor &lse, size_t bytes) {
  PyObject *o = THPVariable_Wrap(out), *l = lse.defined() ? THPVariable_Wrap(lse) : Py_NewRef(Py_None), *n = PyLong_FromSize_t(bytes);
  PyObject *t = PyTuple_New(3);
  PyTuple_SET_ITEM(t, 0, o), PyTuple_SET_ITEM(t, 1, l), PyTuple_SET_ITEM(t, 2, n);
  return t;
}

// forward(q, k, v, sm_scale, buffers, tables, masked_max_row, kwargs, seq_dim, cu_seqlen_k, cu_seqlen_q,
//         left_paddings, seqlens, return_lse, impl, use_workspace) -> (out, lse or None, scratch bytes) or None
PyObject *forward_impl(PyObject *const *args) {
  const at::Tensor &q = tensor(args[0]), &k = tensor(args[1]), &v = tensor(args[2]);
  check_qkv(q, k, v);
  const Options opt(args[7]);
  const at::Tensor *cu_k = optional_tensor(args[9]), *cu_q = optional_tensor(args[10]);
  const at::Tensor *left = optional_tensor(args[11]), *right = optional_tensor(args[12]);
  const bool want_lse = truth(args[13]), use_workspace = truth(args[15]);
  const int64_t impl = integer(args[14]);
  const int dev = q.get_device();
  const int64_t D = q.size(-1);

  dk_fwd_args a{};
  a.dtype = dtype_code(q.scalar_type());
  a.causal = opt.causal, a.impl = (int32_t)impl, a.head_dim = (int32_t)D;
  const double scale = scale_of(args[3], D);
  a.sm_scale = (float)scale;
  const bool masked_ok = scale > 0 && impl != DK_IMPL_GENERIC && a.dtype != DK_F32 && D % 8 == 0 && D <= 256 &&
                         rows_aligned(q) && rows_aligned(k) && rows_aligned(v);
  at::Tensor out, lse;
  Table table;
  std::optional<Unlocked> unlocked;

  if (q.dim() == 4) {
    need(!cu_k && !cu_q);
    const int64_t seq_dim = args[8] == Py_None ? 1 : integer(args[8]);
    need(seq_dim == 1 || seq_dim == 2);
    const int s = (int)seq_dim, h = 3 - s;
    const int64_t B = q.size(0), Lq = q.size(s), Lk = k.size(s), Hq = q.size(h), Hkv = k.size(h);
    need(B > 0 && Lq > 0 && k.size(0) == B && Lk <= opt.max_seqlen && !(opt.unsorted && Lq > 1));
    const bool padded = left || right;
    table = choose_lut(a.csr, args[4], args[5], integer(args[6]), masked_ok, dev, opt.group, opt.max_row,
                       opt.uneven && !(padded && Lq == 1), opt.fixed_walk);
    check_heads(a.csr, Hq, Hkv);
    a.seqs.batch = (int32_t)B, a.seqs.max_q_len = (int32_t)Lq, a.seqs.max_k_len = (int32_t)Lk;
    if (padded) {
      need((Lq == 1 || Lq == Lk) && !(left && right));  // (both: the ends are sums, made by ops.py)
      a.seqs.k_starts = lengths(left, B, dev);
      a.seqs.k_ends = lengths(right, B, dev);
      if (Lq > 1) {
        a.seqs.q_starts = a.seqs.k_starts, a.seqs.q_ends = a.seqs.k_ends;
        a.seqs.packed = 4;  // the kernels clear the padding rows
      }
    }
    unlocked.emplace();
    out = at::empty(q.sizes(), q.options());
    if (want_lse) lse = at::empty({B, Hq, Lq}, q.options().dtype(at::kFloat));
    a.q = view(q, 0, h, s), a.k = view(k, 0, h, s), a.v = view(v, 0, h, s), a.o = view(out, 0, h, s);
    if (want_lse) a.lse = dk_rowvec{static_cast<float *>(lse.data_ptr()), Hq * Lq, Lq, 1};
    a.num_q_heads = (int32_t)Hq, a.num_kv_heads = (int32_t)Hkv;
  } else {
    need(q.dim() == 3 && cu_k && !left && !right);
    const int64_t B = cu_k->dim() == 1 ? cu_k->size(0) - 1 : 0, T = q.size(0), Hq = q.size(1), Hkv = k.size(1);
    need(B > 0 && T > 0);
    const int32_t *ck = lengths(cu_k, B + 1, dev), *cq = nullptr;
    bool single = false;
    if (cu_q)
      cq = lengths(cu_q, B + 1, dev);
    else if (T == B)
      single = true;  // one query token per sequence: lets the library take the split-KV decode kernel
    else {
      need(T == k.size(0));
      cq = ck;
    }
    table = choose_lut(a.csr, args[4], args[5], integer(args[6]), masked_ok, dev, opt.group, opt.max_row, opt.uneven && !single,
                       opt.fixed_walk);
    check_heads(a.csr, Hq, Hkv);
    a.seqs = dk_seqs{(int32_t)B, (int32_t)T, (int32_t)k.size(0), single ? 3 : want_lse ? 5 : 1, cq, cq ? cq + 1 : nullptr, ck, ck + 1};
    unlocked.emplace();
    out = at::empty(q.sizes(), q.options());
    if (want_lse) lse = at::empty({Hq, T}, q.options().dtype(at::kFloat));
    a.q = view(q, -1, 1, 0), a.k = view(k, -1, 1, 0), a.v = view(v, -1, 1, 0), a.o = view(out, -1, 1, 0);
    if (want_lse) a.lse = dk_rowvec{static_cast<float *>(lse.data_ptr()), 0, T, 1};
    a.num_q_heads = (int32_t)Hq, a.num_kv_heads = (int32_t)Hkv;
  }
  const size_t bytes = launch(a, q, use_workspace);
  unlocked.reset();
  return result(out, lse, bytes);
}

// paged(q, k_pool, v_pool, block_table, context_lens, sm_scale, buffers, tables, masked_max_row, max_row, group,
//       max_seqlen, return_lse, k_scale, v_scale, impl) -> (out, lse or None, scratch bytes) or None
PyObject *paged_impl(PyObject *const *args) {
  const at::Tensor &q = tensor(args[0]), &k = tensor(args[1]), &v = tensor(args[2]), &table = tensor(args[3]), &lens = tensor(args[4]);
  need(!std::getenv("DKERNEL_DEBUG"));
  need(q.is_cuda() && k.is_cuda() && v.is_cuda() && q.get_device() == k.get_device() && q.get_device() == v.get_device() &&
       q.get_device() == c10::hip::current_device());
  need((q.dim() == 3 || (q.dim() == 4 && q.size(1) == 1)) && k.dim() == 4 && k.sizes() == v.sizes() && k.scalar_type() == v.scalar_type());
  need(q.stride(-1) == 1 && k.stride(3) == 1 && v.stride(3) == 1);
  const int dev = q.get_device(), h = q.dim() - 2;
  const int64_t B = q.size(0), Hq = q.size(h), D = q.size(h + 1), page = k.size(1), Hkv = k.size(2);
  need(B > 0 && D > 0 && k.size(3) == D && Hkv > 0 && Hq % Hkv == 0);
  need(table.is_cuda() && table.get_device() == dev && table.scalar_type() == at::kInt && table.dim() == 2 && table.size(0) == B &&
       table.stride(1) == 1);
  dk_fwd_args a{};
  a.dtype = dtype_code(q.scalar_type());
  const bool fp8 = k.scalar_type() == at::kFloat8_e4m3fn;
  need(fp8 || k.scalar_type() == q.scalar_type());
  const double scale = scale_of(args[5], D);
  a.sm_scale = (float)scale;
  a.causal = 1, a.impl = (int32_t)integer(args[15]), a.head_dim = (int32_t)D;
  // (paged decode runs on the matrix-core kernels only: always the masked table of a module that has one)
  const Table lut_tensors = choose_lut(a.csr, args[6], args[7], integer(args[8]), true, dev, integer(args[10]), integer(args[9]),
                                       false, false);
  check_heads(a.csr, Hq, Hkv);
  a.seqs = dk_seqs{(int32_t)B, 1, (int32_t)std::min(table.size(1) * page, integer(args[11])), 0, nullptr, nullptr, nullptr,
                   lengths(&lens, B, dev)};
  const bool want_lse = truth(args[12]);
  const double ks = PyFloat_AsDouble(args[13]), vs = PyFloat_AsDouble(args[14]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    throw Unsupported{};
  }
  std::optional<Unlocked> unlocked;
  unlocked.emplace();
  at::Tensor out = at::empty(q.sizes(), q.options()), lse;
  if (want_lse) {
    lse = at::empty({B, Hq, 1}, q.options().dtype(at::kFloat));
    a.lse = dk_rowvec{static_cast<float *>(lse.data_ptr()), Hq, 1, 1};
  }
  a.q = dk_tensor{q.data_ptr(), q.stride(0), q.stride(h), 0}, a.o = dk_tensor{out.data_ptr(), out.stride(0), out.stride(h), 0};
  a.k = dk_tensor{k.data_ptr(), 0, k.stride(2), k.stride(1)}, a.v = dk_tensor{v.data_ptr(), 0, v.stride(2), v.stride(1)};
  a.num_q_heads = (int32_t)Hq, a.num_kv_heads = (int32_t)Hkv;
  a.stream = current_stream();
  const dk_paged_kv pg{static_cast<const int32_t *>(table.data_ptr()), table.stride(0), k.stride(0), v.stride(0), (int32_t)page,
                       fp8 ? DK_FP8_E4M3 : a.dtype, (float)ks, (float)vs};
  const size_t bytes = fwd_bytes_fn(&a);
  at::Tensor ws = at::empty({(int64_t)std::max<size_t>(bytes, 16)}, q.options().dtype(at::kByte));
  a.workspace = ws.data_ptr(), a.workspace_bytes = bytes;
  need(fwd_paged_fn(&a, &pg) == DK_OK);
  unlocked.reset();
  return result(out, lse, bytes);
}

// The bytes of a ctypes structure
template <typename T>
T structure(PyObject *o) {
  Py_buffer b;
  if (PyObject_GetBuffer(o, &b, PyBUF_SIMPLE) != 0) {
    PyErr_Clear();
    throw Unsupported{};
  }
  T t;
  const bool ok = b.len == (Py_ssize_t)sizeof(T);
  if (ok) std::memcpy(&t, b.buf, sizeof(T));
  PyBuffer_Release(&b);
  need(ok);
  return t;
}

// A tensor of a training step: on `dev`, of q's type, rows of consecutive elements
void check_row_tensor(const at::Tensor &t, const at::Tensor &q) {
  need(t.is_cuda() && t.get_device() == q.get_device() && t.scalar_type() == q.scalar_type() && t.dim() == 4 && t.stride(3) == 1);
}

// train_forward(q, k, v, csr, sm_scale, seq_dim, causal, impl, want_lse, use_workspace) -> (out, lse or None, scratch bytes) or None
PyObject *train_forward_impl(PyObject *const *args) {
  const at::Tensor &q = tensor(args[0]), &k = tensor(args[1]), &v = tensor(args[2]);
  check_row_tensor(q, q), check_row_tensor(k, q), check_row_tensor(v, q);
  need(q.get_device() == c10::hip::current_device());
  dk_fwd_args a{};
  a.csr = structure<dk_lut>(args[3]);
  const double scale = PyFloat_AsDouble(args[4]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    throw Unsupported{};
  }
  const int64_t seq_dim = integer(args[5]);
  need(seq_dim == 1 || seq_dim == 2);
  const int s = (int)seq_dim, h = 3 - s;
  const int64_t B = q.size(0), Lq = q.size(s), Lk = k.size(s), Hq = q.size(h), Hkv = k.size(h), D = q.size(3);
  need(B > 0 && Lq > 0 && Lk > 0 && D > 0 && k.sizes() == v.sizes() && k.size(0) == B && k.size(3) == D);
  check_heads(a.csr, Hq, Hkv);
  a.dtype = dtype_code(q.scalar_type());
  a.causal = truth(args[6]), a.impl = (int32_t)integer(args[7]), a.head_dim = (int32_t)D, a.sm_scale = (float)scale;
  const bool want_lse = truth(args[8]), use_workspace = truth(args[9]);
  a.seqs.batch = (int32_t)B, a.seqs.max_q_len = (int32_t)Lq, a.seqs.max_k_len = (int32_t)Lk;
  a.num_q_heads = (int32_t)Hq, a.num_kv_heads = (int32_t)Hkv;
  at::Tensor out, lse;
  std::optional<Unlocked> unlocked;
  unlocked.emplace();
  out = at::empty(q.sizes(), q.options());
  if (want_lse) {
    lse = at::empty({B, Hq, Lq}, q.options().dtype(at::kFloat));
    a.lse = dk_rowvec{static_cast<float *>(lse.data_ptr()), Hq * Lq, Lq, 1};
  }
  a.q = view(q, 0, h, s), a.k = view(k, 0, h, s), a.v = view(v, 0, h, s), a.o = view(out, 0, h, s);
  const size_t bytes = launch(a, q, use_workspace);
  unlocked.reset();
  return result(out, lse, bytes);
}

// train_backward(q, k, v, o, dout, lse, dlse or None, dq or None, dk or None, dv or None, csr, csc, lengths, sm_scale, seq_dim,
//                causal, impl, use_workspace) -> (dq, dk, dv) or None
PyObject *train_backward_impl(PyObject *const *args) {
  const at::Tensor &q = tensor(args[0]), &k = tensor(args[1]), &v = tensor(args[2]), &o = tensor(args[3]), &dout = tensor(args[4]);
  const at::Tensor &lse = tensor(args[5]), *dlse = optional_tensor(args[6]);
  need(bwd_fn);
  const at::Tensor *given[3] = {optional_tensor(args[7]), optional_tensor(args[8]), optional_tensor(args[9])}, *like[3] = {&q, &k, &v};
  for (const at::Tensor *t : {&q, &k, &v, &o, &dout}) check_row_tensor(*t, q);
  need(q.get_device() == c10::hip::current_device());
  need(k.sizes() == v.sizes() && o.sizes() == q.sizes() && dout.sizes() == q.sizes() && k.size(0) == q.size(0) && k.size(3) == q.size(3));
  for (int i = 0; i < 3; ++i)
    if (given[i]) {
      check_row_tensor(*given[i], q);
      need(given[i]->sizes() == like[i]->sizes());
    }
  dk_bwd_args a{};
  a.csr = structure<dk_lut>(args[10]), a.csc = structure<dk_lut>(args[11]);
  const dk_row_lengths lengths = structure<dk_row_lengths>(args[12]);
  const double scale = PyFloat_AsDouble(args[13]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    throw Unsupported{};
  }
  const int64_t seq_dim = integer(args[14]);
  need(seq_dim == 1 || seq_dim == 2);
  const int s = (int)seq_dim, h = 3 - s;
  const int64_t B = q.size(0), Lq = q.size(s), Lk = k.size(s), Hq = q.size(h), Hkv = k.size(h), D = q.size(3);
  need(B > 0 && Lq > 0 && Lk > 0 && D > 0);
  check_heads(a.csr, Hq, Hkv), check_heads(a.csc, Hq, Hkv);
  auto rows = [&](const at::Tensor &t) {
    need(t.is_cuda() && t.get_device() == q.get_device() && t.scalar_type() == at::kFloat && t.dim() == 3 && t.size(0) == B && t.size(1) == Hq &&
         t.size(2) == Lq);
    return dk_rowvec{static_cast<float *>(t.data_ptr()), t.stride(0), t.stride(1), t.stride(2)};
  };
  a.lse = rows(lse);
  if (dlse) a.dlse = rows(*dlse);
  a.dtype = dtype_code(q.scalar_type());
  a.causal = truth(args[15]), a.impl = (int32_t)integer(args[16]), a.head_dim = (int32_t)D, a.sm_scale = (float)scale;
  const bool use_workspace = truth(args[17]);
  a.seqs.batch = (int32_t)B, a.seqs.max_q_len = (int32_t)Lq, a.seqs.max_k_len = (int32_t)Lk;
  a.num_q_heads = (int32_t)Hq, a.num_kv_heads = (int32_t)Hkv;
  at::Tensor grads[3], delta, ws;
  std::optional<Unlocked> unlocked;
  unlocked.emplace();
  for (int i = 0; i < 3; ++i) grads[i] = given[i] ? *given[i] : at::empty(like[i]->sizes(), like[i]->options());
  delta = at::empty({B, Hq, Lq}, q.options().dtype(at::kFloat));
  a.q = view(q, 0, h, s), a.k = view(k, 0, h, s), a.v = view(v, 0, h, s), a.o = view(o, 0, h, s), a.dout = view(dout, 0, h, s);
  a.dq = view(grads[0], 0, h, s), a.dk = view(grads[1], 0, h, s), a.dv = view(grads[2], 0, h, s);
  a.delta = static_cast<float *>(delta.data_ptr());
  a.stream = current_stream();
  const size_t bytes = use_workspace ? bwd_bytes_fn(&a, &lengths) : 0;
  if (bytes) {
    ws = at::empty({(int64_t)bytes}, q.options().dtype(at::kByte));
    a.workspace = ws.data_ptr(), a.workspace_bytes = bytes;
  }
  need(bwd_fn(&a, &lengths) == DK_OK);
  unlocked.reset();
  PyObject *t = PyTuple_New(3);
  for (int i = 0; i < 3; ++i) PyTuple_SET_ITEM(t, i, THPVariable_Wrap(grads[i]));
  return t;
}

template <PyObject *(*Impl)(PyObject *const *), int N>
PyObject *entry(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != N || !fwd_fn) {
    PyErr_SetString(PyExc_TypeError, "wrong number of arguments, or bind() was not called");
    return nullptr;
  }
  // Nothing done here is recorded for gradients.  autograd calls both halves of a training step with gradient mode off, unless
  // the backward is to be differentiated itself; with it on, an input that asks for gradients leaves the call to ops.py: told
  // without the cost of an exception.
  if (at::GradMode::is_enabled())
    for (int i = 0; i < 3; ++i)
      if (THPVariable_Check(args[i]) && THPVariable_Unpack(args[i]).requires_grad()) Py_RETURN_NONE;
  try {
    return Impl(args);
  } catch (const Unsupported &) {
    Py_RETURN_NONE;
  } catch (const c10::OutOfMemoryError &e) {  // (torch's own exception, raised by the path in ops.py again)
    Py_RETURN_NONE;
  } catch (const std::exception &e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

// bind(address of dk_fwd, of dk_fwd_workspace_bytes, of dk_fwd_paged[, of dk_bwd_balanced, of dk_bwd_balanced_workspace_bytes])
PyObject *bind(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != 3 && n != 5) {
    PyErr_SetString(PyExc_TypeError, "bind takes three or five addresses");
    return nullptr;
  }
  void *p[5] = {};
  for (int i = 0; i < n; ++i) {
    p[i] = PyLong_AsVoidPtr(args[i]);
    if (PyErr_Occurred()) return nullptr;
  }
  fwd_bytes_fn = reinterpret_cast<decltype(fwd_bytes_fn)>(p[1]);
  fwd_paged_fn = reinterpret_cast<decltype(fwd_paged_fn)>(p[2]);
  if (n == 5) {
    bwd_bytes_fn = reinterpret_cast<decltype(bwd_bytes_fn)>(p[4]);
    bwd_fn = reinterpret_cast<decltype(bwd_fn)>(p[3]);
  }
  fwd_fn = reinterpret_cast<decltype(fwd_fn)>(p[0]);
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", (PyCFunction)(void (*)(void))bind, METH_FASTCALL, "Addresses of the C ABI's forward functions."},
    {"forward", (PyCFunction)(void (*)(void))entry<forward_impl, 16>, METH_FASTCALL, "Forward without gradients, or None."},
    {"paged", (PyCFunction)(void (*)(void))entry<paged_impl, 16>, METH_FASTCALL, "Paged decode step, or None."},
    {"train_forward", (PyCFunction)(void (*)(void))entry<train_forward_impl, 10>, METH_FASTCALL, "Forward of a training step, or None."},
    {"train_backward", (PyCFunction)(void (*)(void))entry<train_backward_impl, 18>, METH_FASTCALL, "Backward of a training step, or None."},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
  k_max_seqlen = PyUnicode_InternFromString("max_seqlen"), k_causal = PyUnicode_InternFromString("causal");
  k_group = PyUnicode_InternFromString("lut_group"), k_max_row = PyUnicode_InternFromString("lut_max_row");
  k_uneven = PyUnicode_InternFromString("uneven_heads"), k_unsorted = PyUnicode_InternFromString("unsorted_rows");
  k_fixed = PyUnicode_InternFromString("fixed_walk");
  k_out = PyUnicode_InternFromString("out"), k_inference = PyUnicode_InternFromString("inference");
  return PyModule_Create(&module);
}
