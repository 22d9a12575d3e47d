// Python face of the hot-path entry points of libquail_hip.so: the argument
// checks, the output allocations and the launch of quail_amd/kernels.py in one
// native call each. A chunk of a few tokens is bound by this work and not by
// the GPU: through ctypes a call cost 11-14 us of host time (torch.empty 1.8-2.5
// us an output, the current stream 2.8, the conversion of 12-30 arguments and
// the launch 4-5), against 5-12 us on the GPU; here it costs 4-5 us,
// and the one-row MLP block went from 40 to 29 us, the one-row attention block
// from 59 to 39, four layers of one row from 472 to 352.
// Host code only; the kernels are reached through the C ABI.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include <ATen/ops/empty.h>
#include <ATen/ops/empty_strided.h>
#include <c10/hip/HIPStream.h>

#include <string>

#include "../../include/quail_hip.h"

namespace {

constexpr int64_t kGroup = 128;   // fp8 quant group (kernels.GROUP)
constexpr int kPageTokens = 16;   // tokens per arena page (kernels.PAGE_TOKENS)
constexpr auto kE4m3 = at::kFloat8_e4m3fn;

[[noreturn]] void bad_value(const std::string& message) {
  PyErr_SetString(PyExc_ValueError, message.c_str());
  throw python_error();
}

const char* dtype_name(at::ScalarType t) {
  switch (t) {
    case at::kBFloat16: return "torch.bfloat16";
    case at::kFloat8_e4m3fn: return "torch.float8_e4m3fn";
    case at::kFloat: return "torch.float32";
    case at::kHalf: return "torch.float16";
    case at::kDouble: return "torch.float64";
    case at::kByte: return "torch.uint8";
    case at::kChar: return "torch.int8";
    case at::kInt: return "torch.int32";
    case at::kLong: return "torch.int64";
    default: return c10::toString(t);
  }
}

std::string shape_of(const at::Tensor& t) {
  std::string s = "(";
  for (int64_t i = 0; i < t.dim(); ++i)
    s += (i ? ", " : "") + std::to_string(t.size(i));
  return s + (t.dim() == 1 ? ",)" : ")");
}

const at::Tensor& tensor(PyObject* o, const char* name) {
  if (!THPVariable_Check(o)) throw torch::TypeError(std::string(name) + " must be a tensor");
  return THPVariable_Unpack(o);
}
// None gives an undefined tensor, whose pointer is null: also for tensors that
// an entry point requires, which refuses the null (as a ValueError)
at::Tensor optional_tensor(PyObject* o, const char* name) {
  return o == Py_None ? at::Tensor() : tensor(o, name);
}
int64_t integer(PyObject* o) {
  const int64_t v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) throw python_error();
  return v;
}
// int(o): a count that may come as a float or a 0-d tensor
int64_t to_int(PyObject* o) {
  THPObjectPtr n(PyNumber_Long(o));
  if (!n) throw python_error();
  return integer(n.get());
}
// float(o)
double real(PyObject* o) {
  double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) {
    PyErr_Clear();
    THPObjectPtr f(PyNumber_Float(o));
    if (!f) throw python_error();
    v = PyFloat_AS_DOUBLE(f.get());
  }
  return v;
}
bool truth(PyObject* o) {
  const int v = PyObject_IsTrue(o);
  if (v < 0) throw python_error();
  return v != 0;
}
void arity(Py_ssize_t got, Py_ssize_t want, const char* what) {
  if (got != want) throw torch::TypeError(std::string(what) + " takes " + std::to_string(want) +
                                          " arguments, got " + std::to_string(got));
}

// kernels._check
void check(const at::Tensor& t, at::ScalarType dtype, const char* name, int64_t dim) {
  if (!t.is_cuda()) bad_value(std::string(name) + " must be a GPU tensor");
  if (t.scalar_type() != dtype)
    bad_value(std::string(name) + " must be " + dtype_name(dtype) + ", got " +
              dtype_name(t.scalar_type()));
  if (t.dim() != dim)
    bad_value(std::string(name) + " must have " + std::to_string(dim) + " dims, got " + shape_of(t));
  if (t.stride(-1) != 1) bad_value(std::string(name) + " rows must be contiguous");
}

void* ptr(const at::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

// The current stream of the current device, as torch.cuda.current_stream().
qh_stream_t stream() { return c10::hip::getCurrentHIPStream().stream(); }

// An output or workspace, allocated without the GIL as torch.empty does: an
// allocation may wait for the device.
at::Tensor empty(at::IntArrayRef sizes, const at::TensorOptions& options) {
  pybind11::gil_scoped_release no_gil;
  return at::empty(sizes, options);
}
at::Tensor rows_like(const at::Tensor& x, int64_t n, int64_t width, at::ScalarType dtype) {
  return empty({n, width}, x.options().dtype(dtype));
}
// fp32 scales stored (width / 128, n), viewed (n, width / 128)
at::Tensor col_major(const at::Tensor& x, int64_t n, int64_t width) {
  const at::TensorOptions options = x.options().dtype(at::kFloat);
  pybind11::gil_scoped_release no_gil;
  return at::empty_strided({n, width / kGroup}, {1, n > 1 ? n : 1}, options);
}

// Runs one C entry point without the GIL and turns its status into the
// exception _hip.call raises.
template <typename... P, typename... A>
void call(const char* name, int (*entry)(P...), A... args) {
  int status;
  {
    pybind11::gil_scoped_release no_gil;
    status = entry((P)args...);
  }
  if (status == QH_OK) return;
  const std::string message = std::string(name) + ": " + qh_last_error();
  if (status == QH_E_ARGUMENT || status == QH_E_UNSUPPORTED || status == QH_E_WORKSPACE)
    bad_value(message);
  throw std::runtime_error(message);
}
#define QH_CALL(entry, ...) call(#entry, entry, __VA_ARGS__)

PyObject* wrap(const at::Tensor& t) { return THPVariable_Wrap(t); }
PyObject* pack(std::initializer_list<at::Tensor> ts) {
  PyObject* out = PyTuple_New((Py_ssize_t)ts.size());
  if (!out) throw python_error();
  Py_ssize_t i = 0;
  for (const at::Tensor& t : ts) {
    PyObject* o;
    if (t.defined()) {
      o = wrap(t);
    } else {
      Py_INCREF(Py_None);
      o = Py_None;
    }
    PyTuple_SET_ITEM(out, i++, o);
  }
  return out;
}

// ---- norm ---------------------------------------------------------------------

PyObject* add_rmsnorm_quant(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 5, "add_rmsnorm_quant");
  const at::Tensor& x = tensor(v[0], "x");
  const at::Tensor& weight = tensor(v[1], "weight");
  const at::Tensor residual = optional_tensor(v[3], "residual");
  check(x, at::kBFloat16, "x", 2);
  check(weight, at::kBFloat16, "weight", 1);
  const int64_t T = x.size(0), H = x.size(1);
  if (residual.defined()) {
    check(residual, at::kBFloat16, "residual", 2);
    if (residual.sizes() != x.sizes()) bad_value("residual shape differs from x");
  }
  at::Tensor q = rows_like(x, T, H, kE4m3);
  at::Tensor scales = col_major(x, T, H);
  QH_CALL(qh_add_rmsnorm_quant, ptr(x), x.stride(0), ptr(residual),
          residual.defined() ? residual.stride(0) : 0, ptr(weight), (float)real(v[2]), T, H, ptr(q),
          (float*)ptr(scales), (int)truth(v[4]), stream());
  return pack({q, scales});
  END_HANDLE_TH_ERRORS
}

PyObject* final_norm(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 5, "final_norm");
  const at::Tensor& hidden = tensor(v[0], "hidden");
  const at::Tensor& residual = tensor(v[1], "residual");
  const at::Tensor& idx = tensor(v[2], "final_idx");
  check(hidden, at::kBFloat16, "hidden", 2);
  check(residual, at::kBFloat16, "residual", 2);
  if (!hidden.is_contiguous() || !residual.is_contiguous())
    bad_value("hidden and residual must be contiguous");
  const int64_t R = idx.numel(), H = hidden.size(1);
  at::Tensor out = rows_like(hidden, R, H, at::kBFloat16);
  QH_CALL(qh_final_norm, ptr(hidden), ptr(residual), (const int64_t*)ptr(idx), R, H,
          ptr(optional_tensor(v[3], "weight")), (float)real(v[4]), ptr(out), stream());
  return wrap(out);
  END_HANDLE_TH_ERRORS
}

PyObject* fused_add_rms_norm(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 4, "fused_add_rms_norm");
  const at::Tensor& hidden = tensor(v[0], "hidden");
  const at::Tensor& residual = tensor(v[1], "residual");
  check(hidden, at::kBFloat16, "hidden", 2);
  check(residual, at::kBFloat16, "residual", 2);
  if (!hidden.is_contiguous() || !residual.is_contiguous())
    bad_value("hidden and residual must be contiguous");
  if (hidden.sizes() != residual.sizes()) bad_value("hidden and residual shapes differ");
  QH_CALL(qh_fused_add_rms_norm, ptr(hidden), ptr(residual), hidden.size(0), hidden.size(1),
          ptr(optional_tensor(v[2], "weight")), (float)real(v[3]), stream());
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// ---- GEMMs ----------------------------------------------------------------------

struct Gemm {
  const at::Tensor &a, &sa, &w, &sw;
  int64_t M, N, K;
};

// kernels._check_gemm
Gemm gemm_operands(PyObject* const* v) {
  Gemm g{tensor(v[0], "a"), tensor(v[1], "a_scales"), tensor(v[2], "w"), tensor(v[3], "w_scales"),
         0, 0, 0};
  check(g.a, kE4m3, "a", 2);
  check(g.w, kE4m3, "w", 2);
  g.M = g.a.size(0);
  g.K = g.a.size(1);
  g.N = g.w.size(0);
  if (g.w.size(1) != g.K) bad_value("K mismatch: a " + shape_of(g.a) + " w " + shape_of(g.w));
  const int64_t nk = g.K / kGroup;
  if (g.sa.scalar_type() != at::kFloat || g.sa.dim() != 2 || g.sa.size(0) != g.M ||
      g.sa.size(1) != nk || (g.M > 1 && g.sa.stride(0) != 1) || (g.M > 0 && g.sa.stride(1) != g.M))
    bad_value("a_scales must be a (M, K/128) view of column-major fp32");
  if (g.sw.scalar_type() != at::kFloat || g.sw.dim() != 2 || g.sw.size(0) != g.N / kGroup ||
      g.sw.size(1) != nk || !g.sw.is_contiguous())
    bad_value("w_scales must be contiguous fp32 (N/128, K/128)");
  return g;
}

PyObject* fp8_gemm_nt(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 6, "fp8_gemm_nt");
  const Gemm g = gemm_operands(v);
  at::Tensor out = optional_tensor(v[4], "out");
  if (!out.defined()) out = rows_like(g.a, g.M, g.N, at::kBFloat16);
  const bool hw = truth(v[5]);
  call(hw ? "qh_fp8_gemm_nt_ue8m0" : "qh_fp8_gemm_nt", hw ? qh_fp8_gemm_nt_ue8m0 : qh_fp8_gemm_nt,
       ptr(g.a), g.a.stride(0), (const float*)ptr(g.sa), ptr(g.w), g.w.stride(0),
       (const float*)ptr(g.sw), ptr(out), out.stride(0), g.M, g.N, g.K, stream());
  return wrap(out);
  END_HANDLE_TH_ERRORS
}

PyObject* fp8_gemm_silu_quant(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 6, "fp8_gemm_silu_quant");
  const Gemm g = gemm_operands(v);
  const bool ue8m0 = truth(v[4]), hw = truth(v[5]);
  if (g.N % (2 * kGroup)) bad_value("gate_up rows " + std::to_string(g.N) + " must be a multiple of 256");
  if (hw && !ue8m0) bad_value("ue8m0_scales=True writes UE8M0 output scales: pass ue8m0=True");
  const int64_t inter = g.N / 2;
  at::Tensor q = rows_like(g.a, g.M, inter, kE4m3);
  at::Tensor scales = col_major(g.a, g.M, inter);
  if (hw)
    QH_CALL(qh_fp8_gemm_silu_quant_ue8m0, ptr(g.a), g.a.stride(0), (const float*)ptr(g.sa), ptr(g.w),
            g.w.stride(0), (const float*)ptr(g.sw), g.M, inter, g.K, ptr(q), q.stride(0),
            (float*)ptr(scales), stream());
  else
    QH_CALL(qh_fp8_gemm_silu_quant, ptr(g.a), g.a.stride(0), (const float*)ptr(g.sa), ptr(g.w),
            g.w.stride(0), (const float*)ptr(g.sw), g.M, inter, g.K, ptr(q), q.stride(0),
            (float*)ptr(scales), (int)ue8m0, stream());
  return pack({q, scales});
  END_HANDLE_TH_ERRORS
}

// a, a_scales, w, w_scales, positions, cos_sin, q_weight, k_weight, eps, n_q,
// n_kv, k_pool, v_pool, row_dst, ue8m0_scales
PyObject* fp8_gemm_qkv_rope(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 15, "fp8_gemm_qkv_rope");
  const Gemm g = gemm_operands(v);
  const at::Tensor& positions = tensor(v[4], "positions");
  const at::Tensor& cos_sin = tensor(v[5], "cos_sin");
  const at::Tensor qw = optional_tensor(v[6], "q_weight"), kw = optional_tensor(v[7], "k_weight");
  const float eps = (float)real(v[8]);
  const int64_t n_q = integer(v[9]), n_kv = integer(v[10]);
  const at::Tensor k_pool = optional_tensor(v[11], "k_pool"), v_pool = optional_tensor(v[12], "v_pool");
  const at::Tensor row_dst = optional_tensor(v[13], "row_dst");
  const int hw = (int)truth(v[14]);
  check(cos_sin, at::kBFloat16, "cos_sin", 2);
  if (g.N != (n_q + 2 * n_kv) * 128 || cos_sin.size(1) != 128)
    bad_value("qkv weight rows must be (n_q + 2 n_kv) * 128 with head_dim 128");
  if (positions.scalar_type() != at::kLong || positions.numel() != g.M || !positions.is_contiguous())
    bad_value("positions must be contiguous int64, one per row");
  at::Tensor q = rows_like(g.a, g.M, n_q * 128, at::kBFloat16);
  if (!row_dst.defined()) {
    at::Tensor k = rows_like(g.a, g.M, n_kv * 128, at::kBFloat16);
    at::Tensor vv = rows_like(g.a, g.M, n_kv * 128, at::kBFloat16);
    QH_CALL(qh_fp8_gemm_qkv_rope, ptr(g.a), g.a.stride(0), (const float*)ptr(g.sa), ptr(g.w),
            g.w.stride(0), (const float*)ptr(g.sw), g.M, g.K, n_q, n_kv,
            (const int64_t*)ptr(positions), ptr(cos_sin), cos_sin.size(0), ptr(qw), ptr(kw), eps,
            ptr(q), q.stride(0), ptr(k), ptr(vv), k.stride(0), hw, stream());
    return pack({q, k, vv});
  }
  if (row_dst.scalar_type() != at::kLong || row_dst.numel() != g.M || !row_dst.is_contiguous())
    bad_value("row_dst must be contiguous int64, one arena row per row");
  QH_CALL(qh_fp8_gemm_qkv_rope_kv, ptr(g.a), g.a.stride(0), (const float*)ptr(g.sa), ptr(g.w),
          g.w.stride(0), (const float*)ptr(g.sw), g.M, g.K, n_q, n_kv,
          (const int64_t*)ptr(positions), ptr(cos_sin), cos_sin.size(0), ptr(qw), ptr(kw), eps,
          ptr(q), q.stride(0), ptr(k_pool), ptr(v_pool), (const int64_t*)ptr(row_dst), kPageTokens,
          hw, stream());
  return wrap(q);
  END_HANDLE_TH_ERRORS
}

// ---- attention --------------------------------------------------------------------

// q3, cu_q, kv_len, n_queries, max_q, softmax_scale, causal, k_pool, v_pool,
// table, n_kv, q_rows, ue8m0
PyObject* attention_fp8(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 13, "attention_fp8");
  const at::Tensor& q3 = tensor(v[0], "q");
  const at::Tensor& cu_q = tensor(v[1], "cu_q");
  const at::Tensor kv_len = optional_tensor(v[2], "kv_len");
  const int64_t n_queries = integer(v[3]), max_q = to_int(v[4]);
  const at::Tensor& k_pool = tensor(v[7], "k_pool");
  const at::Tensor v_pool = optional_tensor(v[8], "v_pool");
  const at::Tensor& table = tensor(v[9], "table");
  const at::Tensor q_rows = optional_tensor(v[11], "q_rows");
  check(q3, at::kBFloat16, "q", 3);
  const int64_t n_q = q3.size(1), d = q3.size(2), n_seqs = cu_q.numel() - 1;
  if (d != kGroup) bad_value("one quant group per head needs head_dim 128");
  at::Tensor q = rows_like(q3, n_queries, n_q * d, kE4m3);
  at::Tensor scales = col_major(q3, n_queries, n_q * d);
  at::Tensor ws = empty({(int64_t)qh_attention_workspace_bytes((int)n_seqs)},
                            q3.options().dtype(at::kByte));
  QH_CALL(qh_attention_fp8, ptr(q3), q3.stride(0), q3.size(0), (const int64_t*)ptr(q_rows),
          ptr(k_pool), ptr(v_pool), k_pool.size(0), (const int32_t*)ptr(table), table.size(1),
          kPageTokens, (const int32_t*)ptr(cu_q), (const int32_t*)ptr(kv_len), n_seqs, n_queries,
          max_q, n_q, integer(v[10]), d, (float)real(v[5]), (int)truth(v[6]), ptr(q), q.stride(0),
          (float*)ptr(scales), (int)truth(v[12]), ptr(ws), ws.numel(), stream());
  return pack({q, scales});
  END_HANDLE_TH_ERRORS
}

// q3, k_rows, v_rows, cu_a, seg_read, softmax_scale, k_pool, v_pool, table,
// used, fp8, ue8m0, resident
PyObject* tree_attention(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 13, "tree_attention");
  const at::Tensor& q3 = tensor(v[0], "q");
  const at::Tensor &k_rows = tensor(v[1], "k_rows"), &v_rows = tensor(v[2], "v_rows");
  const at::Tensor &cu_a = tensor(v[3], "cu_a"), &seg_read = tensor(v[4], "seg_read");
  const at::Tensor k_pool = optional_tensor(v[6], "k_pool"), v_pool = optional_tensor(v[7], "v_pool");
  const at::Tensor table = optional_tensor(v[8], "table"), used = optional_tensor(v[9], "used");
  const bool fp8 = truth(v[10]);
  check(q3, at::kBFloat16, "q", 3);
  check(k_rows, at::kBFloat16, "k_rows", 3);
  check(v_rows, at::kBFloat16, "v_rows", 3);
  const int64_t T = q3.size(0), n_q = q3.size(1), d = q3.size(2), n_kv = k_rows.size(1);
  if (k_rows.size(0) != T || v_rows.sizes() != k_rows.sizes() || k_rows.stride(0) != v_rows.stride(0))
    bad_value("k_rows / v_rows must be [T, n_kv, d] with one row stride");
  if (k_rows.stride(1) != d || q3.stride(1) != d)
    bad_value("heads of q / k_rows / v_rows must be contiguous");
  const int64_t n_seg = cu_a.numel() - 1;
  if (seg_read.scalar_type() != at::kInt || seg_read.numel() != n_seg)
    bad_value("seg_read must be int32 with one entry per segment");
  const int64_t n_reads = table.defined() ? table.size(0) : 0;
  if (n_reads && (!used.defined() || used.numel() != n_reads))
    bad_value("used must have one entry per page-table row");
  at::Tensor ws = empty({(int64_t)qh_attention_workspace_bytes((int)n_seg)},
                            q3.options().dtype(at::kByte));
  at::Tensor out, q, scales;
  if (fp8) {
    if (d != kGroup) bad_value("one quant group per head needs head_dim 128");
    q = rows_like(q3, T, n_q * d, kE4m3);
    scales = col_major(q3, T, n_q * d);
  } else {
    out = empty({T, n_q, d}, q3.options());
  }
  const bool resident = truth(v[12]);
  call(resident ? "qh_tree_attention_resident" : "qh_tree_attention",
       resident ? qh_tree_attention_resident : qh_tree_attention, ptr(q3), q3.stride(0), T, ptr(k_rows),
       ptr(v_rows), k_rows.stride(0), (const int32_t*)ptr(cu_a), (const int32_t*)ptr(seg_read), n_seg,
       ptr(k_pool), ptr(v_pool), k_pool.defined() ? k_pool.size(0) : 0, (const int32_t*)ptr(table),
       table.defined() ? table.size(1) : 0, (const int32_t*)ptr(used), n_reads, kPageTokens, n_q, n_kv,
       d, (float)real(v[5]), ptr(out), out.defined() ? out.stride(0) : 0, ptr(q),
       q.defined() ? q.stride(0) : 0, (float*)ptr(scales), (int)truth(v[11]), ptr(ws), ws.numel(),
       stream());
  return fp8 ? pack({q, scales}) : wrap(out);
  END_HANDLE_TH_ERRORS
}

// ---- rows -------------------------------------------------------------------------

PyObject* gather_rows(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 3, "gather_rows");
  const at::Tensor &table = tensor(v[0], "table"), &idx = tensor(v[1], "idx");
  at::Tensor out = optional_tensor(v[2], "out");
  check(table, at::kBFloat16, "table", 2);
  if (idx.scalar_type() != at::kLong || !idx.is_contiguous()) bad_value("idx must be contiguous int64");
  const int64_t rows = idx.numel(), W = table.size(1);
  if (!out.defined()) out = rows_like(table, rows, W, at::kBFloat16);
  QH_CALL(qh_gather_rows, ptr(table), table.stride(0), (const int64_t*)ptr(idx), rows, W, ptr(out),
          stream());
  return wrap(out);
  END_HANDLE_TH_ERRORS
}

PyObject* gather_quant_rows(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 3, "gather_quant_rows");
  const at::Tensor &q = tensor(v[0], "q"), &scales = tensor(v[1], "scales"), &idx = tensor(v[2], "idx");
  check(q, kE4m3, "q", 2);
  const int64_t T = q.size(0), W = q.size(1);
  if (scales.scalar_type() != at::kFloat || scales.dim() != 2 || scales.size(0) != T ||
      scales.size(1) != W / kGroup || (T > 0 && (scales.stride(0) != 1 || scales.stride(1) != T)))
    bad_value("scales must be the column-major (T, W/128) fp32 view");
  if (idx.scalar_type() != at::kLong || idx.dim() != 1 || !idx.is_contiguous())
    bad_value("idx must be a contiguous 1-d int64 tensor");
  const int64_t rows = idx.numel();
  at::Tensor out = rows_like(q, rows, W, kE4m3);
  at::Tensor out_scales = col_major(q, rows, W);
  QH_CALL(qh_gather_quant_rows, ptr(q), q.stride(0), (const float*)ptr(scales), T,
          (const int64_t*)ptr(idx), rows, W, ptr(out), out.stride(0), (float*)ptr(out_scales), stream());
  return pack({out, out_scales});
  END_HANDLE_TH_ERRORS
}

// ---- readout ------------------------------------------------------------------------

PyObject* answer_bits(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 4, "answer_bits");
  const at::Tensor &normed = tensor(v[0], "normed"), &w = tensor(v[1], "w_ans");
  check(normed, at::kBFloat16, "normed", 2);
  const int64_t R = normed.size(0), H = normed.size(1);
  at::Tensor bits = empty({R}, normed.options().dtype(at::kByte)), margin;
  if (truth(v[3])) margin = empty({R}, normed.options().dtype(at::kFloat));
  QH_CALL(qh_answer_bits, ptr(normed), R, H, ptr(w), w.size(0),
          (const uint8_t*)ptr(optional_tensor(v[2], "is_true")), (uint8_t*)ptr(bits), (float*)ptr(margin),
          stream());
  return pack({bits, margin});
  END_HANDLE_TH_ERRORS
}

PyObject* answer_logits(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 3, "answer_logits");
  const at::Tensor &normed = tensor(v[0], "normed"), &w = tensor(v[1], "w_ans");
  check(normed, at::kBFloat16, "normed", 2);
  const int64_t R = normed.size(0), H = normed.size(1);
  at::Tensor best_t = empty({R}, normed.options()), best_f = empty({R}, normed.options());
  QH_CALL(qh_answer_logits, ptr(normed), R, H, ptr(w), w.size(0),
          (const uint8_t*)ptr(optional_tensor(v[2], "is_true")), ptr(best_t), ptr(best_f), stream());
  return pack({best_t, best_f});
  END_HANDLE_TH_ERRORS
}

#define OP(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {OP(add_rmsnorm_quant), OP(final_norm), OP(fused_add_rms_norm),
                          OP(fp8_gemm_nt), OP(fp8_gemm_silu_quant), OP(fp8_gemm_qkv_rope),
                          OP(attention_fp8), OP(tree_attention), OP(gather_rows),
                          OP(gather_quant_rows), OP(answer_bits), OP(answer_logits),
                          {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_ops", nullptr, -1, kMethods};

}  // namespace

PyMODINIT_FUNC PyInit__ops() { return PyModule_Create(&kModule); }
