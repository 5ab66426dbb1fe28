// Host side of the hip backend: the calls a layer makes many times per step, from Python objects to the C
// ABI without the interpreter in between.
//
// A training step of one layer is 25-30 launches (80 with four nanobatches), and in Python each of them cost
// 10-20 us of argument checks, stride queries, allocation and ctypes conversion around a 3 us launch: short
// sequences and thin tensor-parallel shards were bound by it.  Here one call checks the operands, allocates
// the outputs from PyTorch's caching allocator and launches on the caller's current stream.
//
// Every function takes the case it was written for — bf16 tensors on the device, operands the kernels
// address in place, shapes that fit together — and answers None to anything else; the caller then goes
// through the backend's general Python path, which copies what has to be copied and words the errors.  A
// code other than KR_OK from the library raises.  From the first allocation to the launch the interpreter is
// free for other threads.  Nothing is kept between calls except how much workspace a GEMM shape asks for,
// which is a pure function of its sizes.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <cstdint>
#include <mutex>
#include <string>
#include <unordered_map>

#include "../../include/kareus_hip.h"

namespace {

using at::Tensor;

// ---- Python arguments -----------------------------------------------------------------------------
bool is_tensor(PyObject* o) { return THPVariable_Check(o); }
const Tensor& tensor(PyObject* o) { return THPVariable_Unpack(o); }
bool on_device(const Tensor& t, at::ScalarType type) { return t.is_cuda() && t.scalar_type() == type; }
bool bf16_arg(PyObject* o) { return is_tensor(o) && on_device(tensor(o), at::kBFloat16); }
bool f32_arg(PyObject* o) { return is_tensor(o) && on_device(tensor(o), at::kFloat); }
bool absent(PyObject* o) { return o == Py_None; }

// sizes that a tracer keeps as symbols: the Python side's views carry them on
bool symbolic(const Tensor& t) { return t.unsafeGetTensorImpl()->has_symbolic_sizes_strides(); }

PyObject* none() { Py_RETURN_NONE; }
PyObject* wrap(Tensor t) { return THPVariable_Wrap(std::move(t)); }
void* ptr(const Tensor& t) { return t.data_ptr(); }
void* ptr_or_null(PyObject* o) { return absent(o) ? nullptr : tensor(o).data_ptr(); }
void* stream() { return (void*)c10::hip::getCurrentHIPStream().stream(); }

PyObject* failed(const std::string& what, int rc) {
  PyErr_Format(PyExc_RuntimeError, "%s failed: %s (code %d)", what.c_str(), kr_error_string(rc), rc);
  return nullptr;
}

// numbers: what Python cannot convert ends the call with Python's error, before anything is launched
struct PythonError : std::exception {};
int64_t integer(PyObject* o) {
  const int64_t v = PyLong_AsLong(o);
  if (v == -1 && PyErr_Occurred()) throw PythonError();
  return v;
}
double real(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw PythonError();
  return v;
}
uint64_t seed_value(PyObject* o) {
  const uint64_t v = PyLong_AsUnsignedLongLong(o);
  if (v == (uint64_t)-1 && PyErr_Occurred()) throw PythonError();
  return v;
}
bool truth(PyObject* o) {
  const int v = PyObject_IsTrue(o);
  if (v < 0) throw PythonError();
  return v == 1;
}

// From the first allocation to the launch the interpreter is free for other threads: an allocation may have to
// wait for the device to give cached blocks back, and a launch for room in a full queue.
struct WithoutInterpreter {
  PyThreadState* const state = PyEval_SaveThread();
  ~WithoutInterpreter() { PyEval_RestoreThread(state); }
};

// exceptions leave as PyTorch's own bindings let them out: out of memory as torch.OutOfMemoryError
template <typename F>
PyObject* guarded(F&& f) {
  try {
    return f();
  } catch (const PythonError&) {
    return nullptr;
  } catch (...) {
    torch::translate_exception_to_python(std::current_exception());
    return nullptr;
  }
}

// ---- operands the kernels address in place ------------------------------------------------------------
// A matrix [rows, cols] with one row stride, or the [s, r, cols] slice of a [s, b, cols] tensor whose rows
// come in runs of r (see "Row runs" in kareus_hip.h); tensors of more dimensions count when their leading
// ones merge, which is for the callers that would otherwise copy them: the others take max_dims.
struct Operand {
  int64_t rows = 0, cols = 0, ld = 0;
  int run_rows = 1;
  int64_t run_ld = 0;
  bool ok = false;
};
constexpr int64_t kMaxRunRows = 16;

Operand operand(const Tensor& t, int64_t max_run_rows = kMaxRunRows, int64_t max_dims = 64) {
  Operand o;
  const int64_t d = t.dim();
  if (d < 2 || d > max_dims || t.stride(d - 1) != 1 || t.numel() == 0) return o;
  o.cols = t.size(d - 1);
  // merge the leading dimensions from the inside out
  int64_t rows = 1, ld = 0;
  bool merged = true;
  for (int64_t i = d - 2; i >= 0; --i) {
    if (t.size(i) == 1) continue;
    if (rows == 1) {
      ld = t.stride(i);
    } else if (t.stride(i) != rows * ld) {
      merged = false;
      break;
    }
    rows *= t.size(i);
  }
  if (merged) {
    // (the stride of one row says nothing; a caller that is strict about dimensions passes a matrix's on as it is)
    if (rows == 1) ld = max_dims <= 3 && d == 2 ? t.stride(0) : (o.cols + 7) / 8 * 8;
    if (ld % 8 || ld < o.cols) return o;
    o.rows = rows;
    o.ld = ld;
    o.ok = true;
    return o;
  }
  if (d != 3) return o;
  const int64_t r = t.size(1), outer = t.stride(0), inner = t.stride(1);
  if (inner % 8 || inner < o.cols || outer % 8 || (r & (r - 1)) || r > max_run_rows || outer < r * inner) return o;
  o.rows = t.size(0) * r;
  o.ld = inner;
  o.run_rows = (int)r;
  o.run_ld = outer;
  o.ok = true;
  return o;
}

// the operand of a call that refuses what is neither a matrix nor a [s, r, cols] tensor / not a matrix
Operand operand3(const Tensor& t) { return operand(t, kMaxRunRows, 3); }
Operand operand2(const Tensor& t) { return operand(t, 1, 2); }

Tensor matrix(int64_t rows, int64_t cols, const Tensor& like) { return at::empty({rows, cols}, like.options()); }
Tensor bytes(size_t n, const Tensor& like) { return at::empty({(int64_t)n}, like.options().dtype(at::kByte)); }

// rows_view(t, max_run_rows): ``t`` as the kernels address it in place — [rows, cols] when one row stride does,
// t itself when its rows come in runs — or None
PyObject* py_rows_view(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  return guarded([&]() -> PyObject* {
    if (n_args != 2 || !is_tensor(a[0]) || symbolic(tensor(a[0]))) return none();
    PyObject* t = a[0];
    const Tensor& x = tensor(t);
    const Operand o = operand(x, integer(a[1]));
    if (!o.ok) return none();
    if (x.dim() == 2 || o.run_rows > 1) return Py_NewRef(t);
    return wrap(x.view({o.rows, o.cols}));  // (relative to x: as_strided would bind a trace to x's place in its storage)
  });
}

// ---- GEMM ----------------------------------------------------------------------------------------------
// workspace bytes of a shape: pure in its sizes, remembered because planning costs as much as a launch
size_t gemm_workspace(int layout, int m, int n, int k, bool alone) {
  struct Hash {
    size_t operator()(const std::array<int, 5>& a) const {
      size_t h = 1469598103934665603ull;
      for (int v : a) h = (h ^ (size_t)(unsigned)v) * 1099511628211ull;
      return h;
    }
  };
  static std::mutex guard;
  static std::unordered_map<std::array<int, 5>, size_t, Hash> known;
  const std::array<int, 5> key{layout, m, n, k, alone ? 1 : 0};
  std::lock_guard<std::mutex> lock(guard);
  auto it = known.find(key);
  if (it != known.end()) return it->second;
  if (known.size() > 4096) known.clear();
  // 0.1: the weight the dispatcher gives a launch's own latency beside other streams
  const size_t n_bytes =
      alone ? kr_gemm_workspace_bytes(layout, m, n, k) : kr_gemm_workspace_bytes_shared(layout, m, n, k, 0.1f);
  known.emplace(key, n_bytes);
  return n_bytes;
}

bool fits_int(int64_t v) { return v > 0 && v < ((int64_t)1 << 31); }

// What a product's epilogue takes along: the residual, or the activation's input (operand and address), or the
// activation's output.
struct Epilogue {
  int kind = KR_GEMM_EPI_NONE;
  const void* aux = nullptr;
  Operand ox;
  void* out2 = nullptr;
  int64_t ld_out2 = 0;
};

// allocates the workspace and launches; the operands have been checked, ``out`` is there
int run_gemm(int layout, int64_t m, int64_t n, int64_t k, const Tensor& a, const Operand& oa, const Tensor& b,
             const Operand& ob, const Tensor& out, const Operand& oc, bool accumulate, int split, const Epilogue& e,
             int max_cus) {
  const int epilogue = e.kind | (split == 2 ? KR_GEMM_BESIDE_OTHER_STREAMS : 0);
  Tensor ws;
  size_t ws_bytes = 0;
  if (e.kind == KR_GEMM_EPI_NONE && split != 0 && oc.run_rows == 1) {
    ws_bytes = gemm_workspace(layout, (int)m, (int)n, (int)k, split == 1);
    if (ws_bytes) ws = bytes(ws_bytes, a);
  }
  void* ws_ptr = ws_bytes ? ptr(ws) : nullptr;
  if (oa.run_rows > 1 || oc.run_rows > 1 || e.ox.run_rows > 1)
    return kr_gemm_bf16_runs(layout, (int)m, (int)n, (int)k, ptr(a), oa.ld, oa.run_rows, oa.run_ld, ptr(b), ob.ld,
                             ptr(out), oc.ld, oc.run_rows, oc.run_ld, accumulate, epilogue, e.aux, e.ox.ld, e.ox.run_rows,
                             e.ox.run_ld, e.out2, e.ld_out2, max_cus, ws_ptr, ws_bytes, stream());
  return kr_gemm_bf16_fused(layout, (int)m, (int)n, (int)k, ptr(a), oa.ld, ptr(b), ob.ld, ptr(out), oc.ld, accumulate,
                            epilogue, e.aux, e.ox.ld, e.out2, e.ld_out2, max_cus, ws_ptr, ws_bytes, stream());
}
PyObject* gemm_failed(int layout, int64_t m, int64_t n, int64_t k, int epi, int rc) {
  return failed("kr_gemm_bf16(layout=" + std::to_string(layout) + ", M=" + std::to_string(m) + ", N=" + std::to_string(n) +
                    ", K=" + std::to_string(k) + ", epilogue=" + std::to_string(epi) + ")",
                rc);
}

// gemm(layout, a, b, m, n, k, out, accumulate, split, residual, swiglu_out, swiglu_bwd_x, max_cus); split: 0 never,
// 1 the GEMM has the device to itself, 2 beside other streams
PyObject* py_gemm(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  return guarded([&]() -> PyObject* {
    if (n_args != 13) return none();
    const int layout = (int)integer(a[0]);
    const int64_t m = integer(a[3]), n = integer(a[4]), k = integer(a[5]);
    const bool accumulate = truth(a[7]);
    const int split = (int)integer(a[8]);
    const int max_cus = (int)integer(a[12]);
    PyObject *p_out = a[6], *p_res = a[9], *p_act = a[10], *p_pre = a[11];
    if (!bf16_arg(a[1]) || !bf16_arg(a[2])) return none();
    for (PyObject* p : {p_out, p_res, p_act, p_pre})
      if (!absent(p) && !bf16_arg(p)) return none();
    if (!absent(p_res) + !absent(p_act) + !absent(p_pre) > 1) return none();
    const Tensor &ta = tensor(a[1]), &tb = tensor(a[2]);
    const Operand oa = operand3(ta);
    const Operand ob = operand2(tb);
    if (!oa.ok || !ob.ok) return none();
    const bool a_t = layout == KR_GEMM_NT, b_t = layout != KR_GEMM_TN;
    if (layout < KR_GEMM_TN || layout > KR_GEMM_NT || oa.rows != (a_t ? k : m) || oa.cols != (a_t ? m : k) ||
        ob.rows != (b_t ? k : n) || ob.cols != (b_t ? n : k) || !fits_int(m) || !fits_int(n) || !fits_int(k))
      return none();
    Epilogue e;
    int64_t out_cols = n;
    if (!absent(p_res)) {
      e.ox = operand3(tensor(p_res));
      if (!e.ox.ok || e.ox.rows != m || e.ox.cols != n) return none();
      e.kind = KR_GEMM_EPI_ADD;
      e.aux = ptr(tensor(p_res));
    } else if (!absent(p_act)) {
      const Tensor& act = tensor(p_act);
      if (act.dim() != 2 || act.size(0) != m || act.size(1) * 2 != n || act.stride(1) != 1) return none();
      e.kind = KR_GEMM_EPI_SWIGLU;
      e.out2 = ptr(act);
      e.ld_out2 = act.stride(0);
    } else if (!absent(p_pre)) {
      const Tensor& pre = tensor(p_pre);
      if (accumulate || pre.dim() != 2 || pre.size(0) != m || pre.size(1) != 2 * n || pre.stride(1) != 1) return none();
      e.kind = KR_GEMM_EPI_SWIGLU_BWD;
      e.ox.ld = pre.stride(0);
      e.aux = ptr(pre);
      out_cols = 2 * n;
    }
    if (accumulate && absent(p_out)) return none();
    Tensor out;
    Operand oc;
    if (absent(p_out)) {
      if (out_cols % 8) return none();
      oc.rows = m, oc.cols = oc.ld = out_cols;
    } else {
      out = tensor(p_out);
      oc = operand3(out);
      if (!oc.ok || oc.rows != m || oc.cols != out_cols) return none();
    }
    int rc;
    {
      WithoutInterpreter free;
      if (!out.defined()) out = matrix(m, out_cols, ta);
      rc = run_gemm(layout, m, n, k, ta, oa, tb, ob, out, oc, accumulate, split, e, max_cus);
    }
    if (rc != KR_OK) return gemm_failed(layout, m, n, k, e.kind, rc);
    return absent(p_out) ? wrap(std::move(out)) : Py_NewRef(p_out);
  });
}

// operand pairs of a weight gradient over several nanobatches: matrices of one shape and one row stride in every pair (those of
// ``dys`` may be in row runs, all alike), a multiple of 64 rows each
struct Pieces {
  Py_ssize_t n = 0;
  Tensor held[2 * KR_GEMM_MAX_SEGMENTS];  // the lists may change while the interpreter is free
  Operand a, b;
};
bool pieces(PyObject* dys, PyObject* xs, Pieces& p) {
  if (!PyList_Check(dys) || !PyList_Check(xs)) return false;
  p.n = PyList_GET_SIZE(dys);
  if (p.n < 1 || p.n > KR_GEMM_MAX_SEGMENTS || PyList_GET_SIZE(xs) != p.n) return false;
  for (Py_ssize_t i = 0; i < p.n; ++i) {
    PyObject *dy = PyList_GET_ITEM(dys, i), *x = PyList_GET_ITEM(xs, i);
    if (!bf16_arg(dy) || !bf16_arg(x)) return false;
    const Operand oa = operand3(tensor(dy)), ob = operand3(tensor(x));
    if (!oa.ok || !ob.ok || ob.run_rows > 1 || oa.rows != ob.rows || oa.rows % 64 || tensor(x).device() != tensor(dy).device())
      return false;
    if (i == 0) {
      p.a = oa, p.b = ob;
    } else if (oa.rows != p.a.rows || oa.ld != p.a.ld || oa.run_rows != p.a.run_rows || oa.run_ld != p.a.run_ld ||
               ob.ld != p.b.ld || oa.cols != p.a.cols || ob.cols != p.b.cols) {
      return false;
    }
    p.held[2 * i] = tensor(dy);
    p.held[2 * i + 1] = tensor(x);
  }
  return true;
}

// wgrad_segments_ok(dys, xs) -> True, or None where the Python side has to look
PyObject* py_wgrad_segments_ok(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  return guarded([&]() -> PyObject* {
    Pieces p;
    if (n_args != 2 || !pieces(a[0], a[1], p)) return none();
    Py_RETURN_TRUE;
  });
}

// wgrad_segments(dys, xs, out, accumulate, split, max_cus): sum of dys[i]^T . xs[i] in one launch, None when the pairs
// are not pieces the kernel takes
PyObject* py_wgrad_segments(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  return guarded([&]() -> PyObject* {
    Pieces p;
    if (n_args != 6 || !pieces(a[0], a[1], p)) return none();
    const Py_ssize_t nseg = p.n;
    const void *pa[KR_GEMM_MAX_SEGMENTS], *pb[KR_GEMM_MAX_SEGMENTS];
    const Operand &fa = p.a, &fb = p.b;
    Tensor* const held = p.held;
    const int64_t m = fa.cols, n = fb.cols, k = fa.rows * nseg;
    if (!fits_int(m) || !fits_int(n) || !fits_int(k)) return none();
    const bool accumulate = truth(a[3]);
    const int split = (int)integer(a[4]), max_cus = (int)integer(a[5]);
    if (absent(a[2]) ? accumulate : !bf16_arg(a[2])) return none();
    Tensor out;
    Operand oc;
    if (absent(a[2])) {
      if (n % 8) return none();
      oc.ld = n;
    } else {
      out = tensor(a[2]);
      oc = operand2(out);
      if (!oc.ok || oc.rows != m || oc.cols != n) return none();
    }
    int rc;
    {
      WithoutInterpreter free;
      if (!out.defined()) out = matrix(m, n, held[0]);
      const size_t ws_bytes = split ? gemm_workspace(KR_GEMM_NT, (int)m, (int)n, (int)k, split == 1) : 0;
      Tensor ws;
      if (ws_bytes) ws = bytes(ws_bytes, held[0]);
      for (Py_ssize_t i = 0; i < nseg; ++i) pa[i] = ptr(held[2 * i]), pb[i] = ptr(held[2 * i + 1]);
      rc = kr_gemm_bf16_nt_segments((int)m, (int)n, (int)fa.rows, (int)nseg, pa, fa.ld, fa.run_rows, fa.run_ld, pb, fb.ld,
                                    ptr(out), oc.ld, accumulate, split == 2 ? KR_GEMM_BESIDE_OTHER_STREAMS : 0, max_cus,
                                    ws_bytes ? ptr(ws) : nullptr, ws_bytes, stream());
    }
    if (rc != KR_OK)
      return failed("kr_gemm_bf16_nt_segments(M=" + std::to_string(m) + ", N=" + std::to_string(n) + ", k_seg=" +
                        std::to_string(fa.rows) + ", nseg=" + std::to_string(nseg) + ")",
                    rc);
    return absent(a[2]) ? wrap(std::move(out)) : Py_NewRef(a[2]);
  });
}

// ---- RMSNorm -----------------------------------------------------------------------------------------------
bool is_gamma(PyObject* o, int64_t cols) {
  return bf16_arg(o) && tensor(o).dim() == 1 && tensor(o).size(0) == cols && tensor(o).is_contiguous();
}

// rmsnorm_fwd(x, gamma, eps) -> (y [rows, cols], rstd [rows])
PyObject* py_rmsnorm_fwd(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  return guarded([&]() -> PyObject* {
    if (n_args != 3 || !bf16_arg(a[0])) return none();
    const Tensor& x = tensor(a[0]);
    const Operand o = operand(x);
    if (!o.ok || !is_gamma(a[1], o.cols) || !fits_int(o.rows)) return none();
    const float eps = (float)real(a[2]);
    const Tensor& gamma = tensor(a[1]);
    Tensor y, rstd;
    int rc;
    {
      WithoutInterpreter free;
      y = matrix(o.rows, o.cols, x);
      rstd = at::empty({o.rows}, x.options().dtype(at::kFloat));
      rc = o.run_rows > 1 ? kr_rmsnorm_fwd_runs(ptr(x), ptr(gamma), ptr(y), (float*)ptr(rstd), (int)o.rows, (int)o.cols, o.ld,
                                                o.run_rows, o.run_ld, eps, stream())
                          : kr_rmsnorm_fwd(ptr(x), ptr(gamma), ptr(y), (float*)ptr(rstd), (int)o.rows, (int)o.cols, o.ld, eps,
                                           stream());
    }
    if (rc != KR_OK) return failed("kr_rmsnorm_fwd", rc);
    PyObject *py = wrap(std::move(y)), *pr = wrap(std::move(rstd));
    return Py_BuildValue("(NN)", py, pr);
  });
}

// rmsnorm_bwd(dy, x, rstd, gamma, residual_grad, out, partials) -> (dx, dgamma or None)
PyObject* py_rmsnorm_bwd(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  return guarded([&]() -> PyObject* {
    if (n_args != 7 || !bf16_arg(a[0]) || !bf16_arg(a[1]) || !f32_arg(a[2])) return none();
    const Tensor &dy = tensor(a[0]), &x = tensor(a[1]), &rstd = tensor(a[2]);
    const Operand od = operand2(dy), ox = operand(x);
    if (!od.ok || !ox.ok || od.rows != ox.rows || od.cols != ox.cols || !fits_int(ox.rows) ||
        !is_gamma(a[3], ox.cols) || !rstd.is_contiguous() || rstd.numel() != ox.rows)
      return none();
    Operand orr, oc;
    if (!absent(a[4])) {
      if (!bf16_arg(a[4])) return none();
      orr = operand(tensor(a[4]));
      if (!orr.ok || orr.rows != ox.rows || orr.cols != ox.cols) return none();
    }
    if (!absent(a[5]) && !bf16_arg(a[5])) return none();
    const int rows = (int)ox.rows, cols = (int)ox.cols;
    Tensor dx, dgamma, partials;
    if (absent(a[5])) {
      if (cols % 8) return none();
      oc.ld = cols;
    } else {
      dx = tensor(a[5]);
      oc = operand3(dx);
      if (!oc.ok || oc.rows != ox.rows || oc.cols != ox.cols) return none();
    }
    if (!absent(a[6])) {
      if (!f32_arg(a[6])) return none();
      partials = tensor(a[6]);
      if (partials.dim() != 2 || !partials.is_contiguous() || partials.size(1) != cols ||
          partials.size(0) != kr_rmsnorm_bwd_partial_rows(rows, cols))
        return none();
    }
    const Tensor& gamma = tensor(a[3]);
    int rc;
    {
      WithoutInterpreter free;
      if (!dx.defined()) dx = matrix(rows, cols, x);
      Tensor ws = partials;
      if (!partials.defined()) {
        dgamma = at::empty({ox.cols}, x.options());
        ws = bytes(kr_rmsnorm_bwd_workspace_bytes(rows, cols), x);
      }
      void* dg = dgamma.defined() ? ptr(dgamma) : nullptr;
      const void* res = ptr_or_null(a[4]);
      rc = (ox.run_rows > 1 || orr.run_rows > 1 || oc.run_rows > 1)
               ? kr_rmsnorm_bwd_add_runs(ptr(dy), ptr(x), (const float*)ptr(rstd), ptr(gamma), res, ptr(dx), dg, ptr(ws), rows,
                                         cols, od.ld, ox.ld, ox.run_rows, ox.run_ld, orr.ld, orr.run_rows, orr.run_ld, oc.ld,
                                         oc.run_rows, oc.run_ld, stream())
               : kr_rmsnorm_bwd_add(ptr(dy), ptr(x), (const float*)ptr(rstd), ptr(gamma), res, ptr(dx), dg, ptr(ws), rows, cols,
                                    od.ld, ox.ld, orr.ld, oc.ld, stream());
    }
    if (rc != KR_OK) return failed("kr_rmsnorm_bwd_add", rc);
    PyObject* pdx = absent(a[5]) ? wrap(std::move(dx)) : Py_NewRef(a[5]);
    PyObject* pdg = dgamma.defined() ? wrap(std::move(dgamma)) : Py_NewRef(Py_None);
    return Py_BuildValue("(NN)", pdx, pdg);
  });
}

// ---- rotary embedding on a fused QKV buffer, in place ------------------------------------------------------
// (the table is one row per position: a dimension between the rows and the channels has to be a 1)
bool is_rotary_table(const Tensor& fr, int64_t s, int64_t hd) {
  return fr.dim() >= 2 && fr.is_contiguous() && fr.size(-1) == hd && fr.numel() == fr.size(0) * hd && fr.size(0) >= s;
}
int run_rope(const Tensor& f, const Tensor& fr, bool backward) {
  const int64_t s = f.size(0), b = f.size(1), slots = f.size(3), heads = f.size(2) * slots, hd = f.size(4);
  return kr_rope(ptr(f), ptr(f), (const float*)ptr(fr), (int)s, (int)b, (int)heads, (int)hd, b * heads * hd, heads * hd, hd,
                 b * heads * hd, heads * hd, hd, backward, (int)slots, (int)slots - 1, stream());
}

// rope_fused(fused [s, b, ng, per + 2, hd], per, freqs [rows >= s, 1.., hd] fp32, backward) -> True
PyObject* py_rope_fused(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  return guarded([&]() -> PyObject* {
    if (n_args != 4 || !bf16_arg(a[0]) || !f32_arg(a[2])) return none();
    const Tensor &f = tensor(a[0]), &fr = tensor(a[2]);
    const int64_t per = integer(a[1]);
    const bool backward = truth(a[3]);
    if (f.dim() != 5 || !f.is_contiguous() || f.size(3) != per + 2 || !is_rotary_table(fr, f.size(0), f.size(4))) return none();
    if (!fits_int(f.size(0)) || !fits_int(f.size(1)) || !fits_int(f.size(2) * f.size(3))) return none();
    int rc;
    {
      WithoutInterpreter free;
      rc = run_rope(f, fr, backward);
    }
    if (rc != KR_OK) return failed("kr_rope", rc);
    Py_RETURN_TRUE;
  });
}

// split_qkv(mixed [.., ng * (per + 2) * hd] dense, ng, per, hd) -> (q [.., ng, per, hd], k [.., ng, hd], v, fused [.., ng,
// per + 2, hd]): views
PyObject* py_split_qkv(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  return guarded([&]() -> PyObject* {
    if (n_args != 4 || !is_tensor(a[0]) || symbolic(tensor(a[0]))) return none();
    const Tensor& m = tensor(a[0]);
    const int64_t ng = integer(a[1]), per = integer(a[2]), hd = integer(a[3]);
    if (m.dim() != 3 || !m.is_contiguous() || m.size(2) != ng * (per + 2) * hd) return none();
    const Tensor fused = m.view({m.size(0), m.size(1), ng, per + 2, hd});
    PyObject *q = wrap(fused.narrow(3, 0, per)), *k = wrap(fused.select(3, per)), *v = wrap(fused.select(3, per + 1));
    return Py_BuildValue("(NNNN)", q, k, v, wrap(fused));
  });
}

// ---- attention ------------------------------------------------------------------------------------------------
struct QStrides {
  int64_t s, b, g, h;
};
// (seq, batch, group, head-in-group) strides of a dense [s, b, nq, hd] or a grouped [s, b, ng, per, hd] tensor
QStrides q_strides(const Tensor& t, int64_t per) {
  if (t.dim() == 5) return {t.stride(0), t.stride(1), t.stride(2), t.stride(3)};
  return {t.stride(0), t.stride(1), per * t.stride(2), t.stride(2)};
}
struct AttnShape {
  int s, b, nq, nkv, hd;
  int64_t per;
  bool ok;
};
AttnShape attn_shape(const Tensor& q, const Tensor& k, const Tensor& v) {
  AttnShape r{};
  if ((q.dim() != 4 && q.dim() != 5) || k.dim() != 4 || v.dim() != 4 || k.sizes() != v.sizes()) return r;
  const int64_t nq = q.dim() == 5 ? q.size(2) * q.size(3) : q.size(2), nkv = k.size(2), hd = k.size(3);
  if (q.size(0) != k.size(0) || q.size(1) != k.size(1) || q.size(-1) != hd || nkv == 0 || nq % nkv ||
      (q.dim() == 5 && q.size(2) != nkv) || q.stride(-1) != 1 || k.stride(-1) != 1 || v.stride(-1) != 1)
    return r;
  if (!fits_int(q.size(0)) || !fits_int(q.size(1)) || !fits_int(nq)) return r;
  r = {(int)q.size(0), (int)q.size(1), (int)nq, (int)nkv, (int)hd, nq / nkv, true};
  return r;
}
std::string attn_name(const char* what, const AttnShape& c) {
  return std::string(what) + "(s=" + std::to_string(c.s) + ", b=" + std::to_string(c.b) + ", nq=" + std::to_string(c.nq) +
         ", nkv=" + std::to_string(c.nkv) + ", hd=" + std::to_string(c.hd) + ")";
}

int run_attn_fwd(const AttnShape& c, const Tensor& q, const Tensor& k, const Tensor& v, float scale, int flags, Tensor& o,
                 Tensor& lse) {
  o = at::empty({c.s, c.b, c.nq, c.hd}, q.options());
  lse = at::empty({c.b, c.nq, c.s}, q.options().dtype(at::kFloat));
  Tensor ws;
  const QStrides sq = q_strides(q, c.per), so = q_strides(o, c.per);
  const size_t n = (flags & KR_ATTN_GENERAL_KERNELS)
                       ? 0
                       : kr_attn_fwd_workspace_bytes_strided(c.s, c.b, c.nq, c.nkv, c.hd,
                                                             std::max({sq.s, so.s, k.stride(0), v.stride(0)}));
  if (n) ws = bytes(n, q);
  return kr_attn_fwd_ws(ptr(q), ptr(k), ptr(v), ptr(o), (float*)ptr(lse), c.s, c.b, c.nq, c.nkv, c.hd, scale, sq.s, sq.b, sq.g,
                        sq.h, k.stride(0), k.stride(1), k.stride(2), v.stride(0), v.stride(1), v.stride(2), so.s, so.b, so.g,
                        so.h, flags | KR_ATTN_IN_PLACE, n ? ptr(ws) : nullptr, n, stream());
}

// attn_fwd(q, k, v, scale, flags) -> (o [s, b, nq, hd], lse [b, nq, s])
PyObject* py_attn_fwd(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  return guarded([&]() -> PyObject* {
    if (n_args != 5 || !bf16_arg(a[0]) || !bf16_arg(a[1]) || !bf16_arg(a[2])) return none();
    const Tensor &q = tensor(a[0]), &k = tensor(a[1]), &v = tensor(a[2]);
    const AttnShape c = attn_shape(q, k, v);
    if (!c.ok) return none();
    const float scale = (float)real(a[3]);
    const int flags = (int)integer(a[4]);
    Tensor o, lse;
    int rc;
    {
      WithoutInterpreter free;
      rc = run_attn_fwd(c, q, k, v, scale, flags, o, lse);
    }
    if (rc != KR_OK) return failed(attn_name("kr_attn_fwd", c), rc);
    PyObject *po = wrap(std::move(o)), *pl = wrap(std::move(lse));
    return Py_BuildValue("(NN)", po, pl);
  });
}

// the gradients of a grouped q, k and v: views of one buffer [s, b, nkv, per + 2, hd]
struct AttnGrads {
  Tensor fused, mixed, dq, dk, dv;
};
bool attn_bwd_ok(const AttnShape& c, const Tensor& q, const Tensor& o, const Tensor& lse) {
  return c.ok && q.dim() == 5 && o.is_contiguous() && lse.is_contiguous() &&
         o.numel() == (int64_t)c.s * c.b * c.nq * c.hd && lse.numel() == (int64_t)c.b * c.nq * c.s;
}
int run_attn_bwd(const AttnShape& c, const Tensor& dout, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o,
                 const Tensor& lse, float scale, int flags, AttnGrads& g) {
  const int64_t s = c.s, b = c.b, ng = c.nkv, hd = c.hd, group = (c.per + 2) * hd, w = ng * group;
  g.fused = at::empty({s, b, ng, c.per + 2, hd}, q.options());
  g.mixed = g.fused.view({s, b, w});
  g.dq = g.fused.as_strided({s, b, ng, c.per, hd}, {b * w, w, group, hd, 1}, 0);
  g.dk = g.fused.as_strided({s, b, ng, hd}, {b * w, w, group, 1}, c.per * hd);
  g.dv = g.fused.as_strided({s, b, ng, hd}, {b * w, w, group, 1}, (c.per + 1) * hd);
  const QStrides sq = q_strides(q, c.per);
  const int64_t os = b * c.nq * hd, ob = c.nq * hd, og = c.per * hd;
  const size_t n = kr_attn_bwd_workspace_bytes_strided(c.s, c.b, c.nq, c.nkv, c.hd,
                                                       std::max({sq.s, k.stride(0), v.stride(0), os, b * w}));
  const Tensor ws = bytes(n < 16 ? 16 : n, q);
  return kr_attn_bwd_flags(ptr(dout), ptr(q), ptr(k), ptr(v), ptr(o), (const float*)ptr(lse), ptr(g.dq), ptr(g.dk), ptr(g.dv),
                           ptr(ws), c.s, c.b, c.nq, c.nkv, c.hd, scale, sq.s, sq.b, sq.g, sq.h, k.stride(0), k.stride(1),
                           k.stride(2), v.stride(0), v.stride(1), v.stride(2), os, ob, og, hd, os, ob, og, hd, b * w, w, group,
                           hd, b * w, w, group, b * w, w, group, flags, stream());
}

// attn_bwd(do, q, k, v, o, lse, scale, flags) -> (dq, dk, dv, mixed, fused) for a grouped q: views of one buffer
// [s, b, nkv, per + 2, hd] (``fused``; ``mixed`` is the same memory as [s, b, features])
PyObject* py_attn_bwd(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  return guarded([&]() -> PyObject* {
    if (n_args != 8) return none();
    for (int i = 0; i < 5; ++i)
      if (!bf16_arg(a[i])) return none();
    if (!f32_arg(a[5])) return none();
    const Tensor &dout = tensor(a[0]), &q = tensor(a[1]), &k = tensor(a[2]), &v = tensor(a[3]), &o = tensor(a[4]),
                 &lse = tensor(a[5]);
    const AttnShape c = attn_shape(q, k, v);
    if (!attn_bwd_ok(c, q, o, lse) || !dout.is_contiguous() || dout.numel() != o.numel()) return none();
    const float scale = (float)real(a[6]);
    const int flags = (int)integer(a[7]);
    AttnGrads g;
    int rc;
    {
      WithoutInterpreter free;
      rc = run_attn_bwd(c, dout, q, k, v, o, lse, scale, flags, g);
    }
    if (rc != KR_OK) return failed(attn_name("kr_attn_bwd", c), rc);
    PyObject *pq = wrap(std::move(g.dq)), *pk = wrap(std::move(g.dk)), *pv = wrap(std::move(g.dv));
    PyObject* pm = wrap(std::move(g.mixed));
    PyObject* pf = wrap(std::move(g.fused));
    return Py_BuildValue("(NNNNN)", pq, pk, pv, pm, pf);
  });
}

// ---- hidden dropout ---------------------------------------------------------------------------------------------
// dropout_add(x, residual, p, out, seed) -> (out, mask); without a seed it is drawn from PyTorch's CPU generator, as
// torch.randint draws it, once the operands have been found to fit
PyObject* py_dropout_add(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  return guarded([&]() -> PyObject* {
    if (n_args != 5 || !bf16_arg(a[0]) || !bf16_arg(a[1])) return none();
    const Tensor &x = tensor(a[0]), &r = tensor(a[1]);
    if (x.sizes() != r.sizes()) return none();
    const Operand ox = operand(x), orr = operand(r);
    if (!ox.ok || ox.run_rows > 1 || !orr.ok || orr.run_rows > 1) return none();
    if (!absent(a[3]) && (!bf16_arg(a[3]) || tensor(a[3]).sizes() != x.sizes())) return none();
    const double p = real(a[2]);
    if (!(p >= 0.0 && p < 1.0)) return none();
    if (absent(a[4]) && !absent(a[3])) {
      // (the caller has not looked at ``out`` yet: one row per entry of the first dimension, as it takes them)
      const Tensor& t = tensor(a[3]);
      int64_t inner = 1;
      for (int64_t i = t.dim() - 1; i >= 1; --i) {
        if (t.size(i) != 1 && t.stride(i) != inner) return none();
        inner *= t.size(i);
      }
      if (t.dim() < 2 || t.stride(0) % 8 || t.stride(0) < inner || t.device() != x.device()) return none();
    }
    uint64_t seed = absent(a[4]) ? 0 : seed_value(a[4]);
    Tensor out, mask;
    Operand oc;
    if (absent(a[3])) {
      oc.ld = ox.cols;
      if (oc.ld % 8) return none();
    } else {
      out = tensor(a[3]);
      oc = operand(out);
      if (!oc.ok || oc.run_rows > 1) return none();
    }
    if (absent(a[4])) seed = (uint64_t)at::randint(0, (int64_t)1 << 62, {1}, at::TensorOptions().dtype(at::kLong)).item<int64_t>();
    int rc;
    {
      WithoutInterpreter free;
      if (!out.defined()) out = at::empty(x.sizes(), x.options());
      mask = at::empty(x.sizes(), x.options().dtype(at::kByte));
      rc = kr_dropout_add(ptr(x), ox.ld, ptr(r), orr.ld, ptr(out), oc.ld, ptr(mask), ox.rows, (int)ox.cols, (float)p, seed, 0,
                          stream());
    }
    if (rc != KR_OK) return failed("kr_dropout_add", rc);
    PyObject* po = absent(a[3]) ? wrap(std::move(out)) : Py_NewRef(a[3]);
    PyObject* pm = wrap(std::move(mask));
    return Py_BuildValue("(NN)", po, pm);
  });
}

// dropout_bwd(dy, mask, scale) -> dx
PyObject* py_dropout_bwd(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  return guarded([&]() -> PyObject* {
    if (n_args != 3 || !bf16_arg(a[0]) || !is_tensor(a[1]) || !on_device(tensor(a[1]), at::kByte)) return none();
    const Tensor &dy = tensor(a[0]), &mask = tensor(a[1]);
    const Operand o = operand(dy);
    if (!o.ok || o.run_rows > 1 || mask.sizes() != dy.sizes() || !mask.is_contiguous()) return none();
    const float scale = (float)real(a[2]);
    Tensor dx;
    int rc;
    {
      WithoutInterpreter free;
      dx = at::empty(dy.sizes(), dy.options());
      rc = kr_dropout_bwd(ptr(dy), o.ld, ptr(mask), ptr(dx), o.cols, o.rows, (int)o.cols, scale, stream());
    }
    if (rc != KR_OK) return failed("kr_dropout_bwd", rc);
    return wrap(std::move(dx));
  });
}

// ---- the operators of a partition in one call ----------------------------------------------------------------------
// What stands between two schedule points of a decoder layer is a fixed chain of operators: norm, QKV projection, split,
// rotary embedding, attention, out-projection; or norm, fc1, activation, fc2.  The chains below run the launches of such an
// operator sequence in the same order, with the same plans and results as one call per operator, and hand back what each of
// them saves; between the launches the interpreter had spent several times what the launches cost.  Whatever a chain does not
// take is answered with None before anything is launched.

// The call that a chain is at, for the error that its operator's own call would raise.
struct Step {
  const char* name = "";
  AttnShape attention{};   // (ok: one of the attention's calls)
  bool product = false;
  int layout = 0, epi = 0;
  int64_t m = 0, n = 0, k = 0;
  void call(const char* what, const AttnShape& c = AttnShape{}) { name = what, attention = c, product = false; }
};
PyObject* failed(const Step& at, int rc) {
  if (at.product) return gemm_failed(at.layout, at.m, at.n, at.k, at.epi, rc);
  return failed(at.attention.ok ? attn_name(at.name, at.attention) : at.name, rc);
}
int run_gemm(Step& at, int layout, int64_t m, int64_t n, int64_t k, const Tensor& a, const Operand& oa, const Tensor& b, const Operand& ob,
             const Tensor& out, const Operand& oc, int split, const Epilogue& e, int max_cus) {
  at.product = true;
  at.layout = layout, at.epi = e.kind, at.m = m, at.n = n, at.k = k;
  return run_gemm(layout, m, n, k, a, oa, b, ob, out, oc, false, split, e, max_cus);
}

// (no references of a failed chain's tensors are left behind)
PyObject* pack(std::initializer_list<Tensor*> items) {
  PyObject* t = PyTuple_New((Py_ssize_t)items.size());
  if (!t) return nullptr;
  Py_ssize_t i = 0;
  for (Tensor* v : items) PyTuple_SET_ITEM(t, i++, v && v->defined() ? wrap(std::move(*v)) : Py_NewRef(Py_None));
  return t;
}
bool is_weight(PyObject* o, int64_t rows, int64_t cols) {
  if (!bf16_arg(o) || symbolic(tensor(o))) return false;
  const Operand w = operand2(tensor(o));
  return w.ok && w.rows == rows && w.cols == cols;
}
Operand dense(int64_t rows, int64_t cols) {
  Operand o;
  o.rows = rows, o.cols = o.ld = cols, o.ok = true;
  return o;
}
// the output of a product: the caller's tensor, or a new dense one (``given`` stays undefined)
struct Output {
  Tensor t;
  Operand o;
  bool ok = false;
};
Output output(PyObject* given, int64_t rows, int64_t cols) {
  Output r;
  if (absent(given)) {
    r.o = dense(rows, cols);
    r.ok = cols % 8 == 0;
  } else if (bf16_arg(given)) {
    r.t = tensor(given);
    r.o = operand3(r.t);
    r.ok = r.o.ok && r.o.rows == rows && r.o.cols == cols;
  }
  return r;
}
bool residual(PyObject* o, int64_t rows, int64_t cols, Epilogue& e) {
  if (absent(o)) return true;
  if (!bf16_arg(o)) return false;
  e.ox = operand3(tensor(o));
  e.kind = KR_GEMM_EPI_ADD;
  e.aux = ptr(tensor(o));
  return e.ox.ok && e.ox.rows == rows && e.ox.cols == cols;
}
// x [s, b, h] of a norm and what it makes: the rows as the kernels address them, y and rstd
struct Norm {
  Operand o;
  Tensor rows, y, rstd;
};
int run_norm(const Tensor& x, const Tensor& gamma, float eps, Norm& n) {
  n.rows = n.o.run_rows > 1 ? x : x.view({n.o.rows, n.o.cols});
  n.y = matrix(n.o.rows, n.o.cols, x);
  n.rstd = at::empty({n.o.rows}, x.options().dtype(at::kFloat));
  return n.o.run_rows > 1 ? kr_rmsnorm_fwd_runs(ptr(x), ptr(gamma), ptr(n.y), (float*)ptr(n.rstd), (int)n.o.rows, (int)n.o.cols,
                                                n.o.ld, n.o.run_rows, n.o.run_ld, eps, stream())
                          : kr_rmsnorm_fwd(ptr(x), ptr(gamma), ptr(n.y), (float*)ptr(n.rstd), (int)n.o.rows, (int)n.o.cols,
                                           n.o.ld, eps, stream());
}
bool norm_input(PyObject* x, PyObject* gamma, Norm& n) {
  if (!bf16_arg(x) || symbolic(tensor(x)) || tensor(x).dim() != 3) return false;
  n.o = operand(tensor(x));
  return n.o.ok && is_gamma(gamma, n.o.cols) && fits_int(n.o.rows) && n.o.cols % 8 == 0;
}
// what a chain saved is dropped as the engine does it op by op: the tensor object loses its memory
void release(std::initializer_list<PyObject*> items) {
  for (PyObject* o : items)
    if (!absent(o)) tensor(o).set_data(at::empty({0}, tensor(o).options()));
}

// release(list of tensors): the same from Python
PyObject* py_release(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  return guarded([&]() -> PyObject* {
    if (n_args != 1 || !PyList_Check(a[0])) return none();
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(a[0]); ++i)
      if (is_tensor(PyList_GET_ITEM(a[0], i))) release({PyList_GET_ITEM(a[0], i)});
    return none();
  });
}

// attn_chain_fwd(x, gamma, eps, w_qkv, gamma_q, gamma_k, qk_eps, freqs, ng, per, hd, scale, beside other streams, split_qkv, w_proj, split_proj,
// residual, out, max_cus) -> (y, x rows, rstd, normed, q, k, v, o, lse, o rows, mixed, qk rstd); the last two are None without
// the per-head norms.  y [s, b, h] has the residual added where one is given, and is None where ``out`` takes it.
PyObject* py_attn_chain_fwd(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  return guarded([&]() -> PyObject* {
    if (n_args != 19) return none();
    Norm n;
    if (!norm_input(a[0], a[1], n) || !f32_arg(a[7])) return none();
    const Tensor &x = tensor(a[0]), &freqs = tensor(a[7]);
    const float eps = (float)real(a[2]);
    const int64_t s = x.size(0), b = x.size(1), t = n.o.rows, h = n.o.cols;
    const int64_t ng = integer(a[8]), per = integer(a[9]), hd = integer(a[10]);
    const float scale = (float)real(a[11]);
    const int flags = truth(a[12]) ? KR_ATTN_BESIDE_OTHER_STREAMS : 0;
    const int split_qkv = (int)integer(a[13]), split_proj = (int)integer(a[15]), max_cus = (int)integer(a[18]);
    if (ng <= 0 || per <= 0 || hd <= 0) return none();
    const int64_t w = ng * (per + 2) * hd, wo = ng * per * hd;
    if (!is_weight(a[3], w, h) || w % 8 || !is_rotary_table(freqs, s, hd) || !fits_int(s) || !fits_int(b) || !fits_int(w))
      return none();
    const bool qk = !absent(a[4]);
    float qk_eps = 0.f;
    if (qk) {
      if (!is_gamma(a[4], hd) || !is_gamma(a[5], hd)) return none();
      qk_eps = (float)real(a[6]);
    }
    if (!bf16_arg(a[14]) || symbolic(tensor(a[14])) || tensor(a[14]).dim() != 2) return none();
    const int64_t out_cols = tensor(a[14]).size(0);
    Epilogue e;
    Output y = output(a[17], t, out_cols);
    if (!is_weight(a[14], out_cols, wo) || !fits_int(out_cols) || wo % 8 || !y.ok || !residual(a[16], t, out_cols, e)) return none();
    const Tensor &gamma = tensor(a[1]), &wq = tensor(a[3]), &wp = tensor(a[14]);
    const Operand o_wq = operand2(wq), o_wp = operand2(wp);
    Tensor mixed, fused, qk_rstd, q, k, v, o, lse, o2d;
    int rc;
    Step at;
    at.call("kr_rmsnorm_fwd");
    {
      WithoutInterpreter free;
      rc = run_norm(x, gamma, eps, n);
      if (rc == KR_OK) {
        mixed = matrix(t, w, x);
        rc = run_gemm(at, KR_GEMM_TN, t, w, h, n.y, dense(t, h), wq, o_wq, mixed, dense(t, w), split_qkv, Epilogue{}, max_cus);
        mixed = mixed.view({s, b, w});
        fused = mixed.view({s, b, ng, per + 2, hd});
      }
      if (rc == KR_OK && qk) {
        at.call("kr_qk_norm_fwd");
        fused = at::empty({s, b, ng, per + 2, hd}, x.options());
        qk_rstd = at::empty({t, 1, ng, per + 1}, x.options().dtype(at::kFloat));
        rc = kr_qk_norm_fwd(ptr(mixed), ptr(tensor(a[4])), ptr(tensor(a[5])), ptr(fused), (float*)ptr(qk_rstd), t, (int)ng,
                            (int)per, (int)hd, qk_eps, stream());
      }
      if (rc == KR_OK) {
        at.call("kr_rope");
        rc = run_rope(fused, freqs, false);
      }
      if (rc == KR_OK) {
        q = fused.narrow(3, 0, per), k = fused.select(3, per), v = fused.select(3, per + 1);
        const AttnShape c = attn_shape(q, k, v);
        at.call("kr_attn_fwd", c);
        rc = run_attn_fwd(c, q, k, v, scale, flags, o, lse);
      }
      if (rc == KR_OK) {
        o2d = o.view({t, wo});
        if (absent(a[17])) y.t = matrix(t, out_cols, x);
        rc = run_gemm(at, KR_GEMM_TN, t, out_cols, wo, o2d, dense(t, wo), wp, o_wp, y.t, y.o, split_proj, e, max_cus);
        if (absent(a[17])) y.t = y.t.view({s, b, out_cols});
      }
    }
    if (rc != KR_OK) return failed(at, rc);
    if (!qk) mixed = Tensor();
    if (!absent(a[17])) y.t = Tensor();
    return pack({&y.t, &n.rows, &n.rstd, &n.y, &q, &k, &v, &o, &lse, &o2d, &mixed, &qk_rstd});
  });
}

// mlp_chain_fwd(x, gamma, eps, w1, split1, fuse_activation, w2, split2, residual, out, max_cus) -> (y, x rows, rstd, normed,
// fc1's output, the activation); y as above
PyObject* py_mlp_chain_fwd(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  return guarded([&]() -> PyObject* {
    if (n_args != 11) return none();
    Norm n;
    if (!norm_input(a[0], a[1], n)) return none();
    const Tensor& x = tensor(a[0]);
    const float eps = (float)real(a[2]);
    const int split1 = (int)integer(a[4]), split2 = (int)integer(a[7]), max_cus = (int)integer(a[10]);
    const bool fuse = truth(a[5]);
    const int64_t s = x.size(0), b = x.size(1), t = n.o.rows, h = n.o.cols;
    for (int i : {3, 6})
      if (!bf16_arg(a[i]) || symbolic(tensor(a[i])) || tensor(a[i]).dim() != 2) return none();
    const Tensor &w1 = tensor(a[3]), &w2 = tensor(a[6]), &gamma = tensor(a[1]);
    const int64_t two_f = w1.size(0), f = two_f / 2, out_cols = w2.size(0);
    Epilogue e;
    Output y = output(a[9], t, out_cols);
    if (!is_weight(a[3], two_f, h) || two_f % 16 || !fits_int(two_f) || !is_weight(a[6], out_cols, f) || !fits_int(out_cols) ||
        !y.ok || !residual(a[8], t, out_cols, e))
      return none();
    const Operand o1 = operand2(w1), o2 = operand2(w2);
    Tensor pre, act;
    int rc;
    Step at;
    at.call("kr_rmsnorm_fwd");
    {
      WithoutInterpreter free;
      rc = run_norm(x, gamma, eps, n);
      if (rc == KR_OK) {
        act = matrix(t, f, x);
        pre = matrix(t, two_f, x);
        Epilogue swiglu;
        if (fuse) {
          swiglu.kind = KR_GEMM_EPI_SWIGLU;
          swiglu.out2 = ptr(act);
          swiglu.ld_out2 = f;
        }
        rc = run_gemm(at, KR_GEMM_TN, t, two_f, h, n.y, dense(t, h), w1, o1, pre, dense(t, two_f), split1, swiglu, max_cus);
      }
      if (rc == KR_OK && !fuse) {
        at.call("kr_swiglu_fwd");
        rc = kr_swiglu_fwd(ptr(pre), ptr(act), t, (int)f, stream());
      }
      if (rc == KR_OK) {
        if (absent(a[9])) y.t = matrix(t, out_cols, x);
        rc = run_gemm(at, KR_GEMM_TN, t, out_cols, f, act, dense(t, f), w2, o2, y.t, y.o, split2, e, max_cus);
        if (absent(a[9])) y.t = y.t.view({s, b, out_cols});
      }
    }
    if (rc != KR_OK) return failed(at, rc);
    if (!absent(a[9])) y.t = Tensor();
    return pack({&y.t, &n.rows, &n.rstd, &n.y, &pre, &act});
  });
}

// dy [.., cols] of a chain's last projection
bool grad_input(PyObject* o, int64_t rows, int64_t cols, Operand& od) {
  if (!bf16_arg(o) || symbolic(tensor(o))) return false;
  od = operand3(tensor(o));
  return od.ok && od.rows == rows && od.cols == cols;
}
bool is_saved(PyObject* o, int64_t rows, int64_t cols) {
  return bf16_arg(o) && tensor(o).dim() == 2 && tensor(o).is_contiguous() && tensor(o).size(0) == rows && tensor(o).size(1) == cols;
}

// Calls the caller's function between two steps of a chain, if there is one; false: it raised.
bool called(PyObject* function) {
  if (absent(function)) return true;
  PyObject* got = PyObject_CallNoArgs(function);
  Py_XDECREF(got);
  return got != nullptr;
}

// mlp_chain_bwd(dy, w2, fc1's output, activation, w1, normed, split2, split1, weight gradients, max_cus, between) -> (dx [rows, h],
// gradient of fc1's output, dw2, dw1).  With ``weight gradients`` the saved tensors lose their memory once they are used; without,
// the caller takes the two weight gradients and the last two results are None.  ``between`` (None or a function without arguments) is
// called where fc2's weight gradient may be taken: behind fc2's input gradient.
PyObject* py_mlp_chain_bwd(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  return guarded([&]() -> PyObject* {
    if (n_args != 11) return none();
    for (int i : {1, 4})
      if (!bf16_arg(a[i]) || tensor(a[i]).dim() != 2) return none();
    const Tensor &w2 = tensor(a[1]), &w1 = tensor(a[4]);
    const int64_t cols = w2.size(0), f = w2.size(1), h = w1.size(1);
    if (!bf16_arg(a[3]) || tensor(a[3]).dim() != 2) return none();
    const int64_t t = tensor(a[3]).size(0);
    Operand od;
    if (!fits_int(t) || !fits_int(cols) || f % 8 || h % 8 || cols % 8 || !is_weight(a[1], cols, f) || !is_weight(a[4], 2 * f, h) ||
        !is_saved(a[2], t, 2 * f) || !is_saved(a[3], t, f) || !is_saved(a[5], t, h) || !grad_input(a[0], t, cols, od))
      return none();
    const int split2 = (int)integer(a[6]), split1 = (int)integer(a[7]), max_cus = (int)integer(a[9]);
    const bool wgrad = truth(a[8]);
    const Tensor &dy = tensor(a[0]), &pre = tensor(a[2]), &act = tensor(a[3]), &normed = tensor(a[5]);
    const Operand o1 = operand2(w1), o2 = operand2(w2);
    Tensor dpre, dx, dw2, dw1;
    int rc;
    Step at;
    {
      WithoutInterpreter free;
      dpre = matrix(t, 2 * f, dy);
      Epilogue e;
      e.kind = KR_GEMM_EPI_SWIGLU_BWD;
      e.ox.ld = 2 * f;
      e.aux = ptr(pre);
      rc = run_gemm(at, KR_GEMM_NN, t, f, cols, dy, od, w2, o2, dpre, dense(t, 2 * f), split2, e, max_cus);
      if (rc == KR_OK && wgrad) {
        dw2 = matrix(cols, f, dy);
        rc = run_gemm(at, KR_GEMM_NT, cols, f, t, dy, od, act, dense(t, f), dw2, dense(cols, f), split2, Epilogue{}, max_cus);
      }
    }
    if (rc != KR_OK) return failed(at, rc);
    if (!called(a[10])) return nullptr;
    if (wgrad) release({a[2], a[3]});
    {
      WithoutInterpreter free;
      dx = matrix(t, h, dy);
      rc = run_gemm(at, KR_GEMM_NN, t, h, 2 * f, dpre, dense(t, 2 * f), w1, o1, dx, dense(t, h), split1, Epilogue{}, max_cus);
      if (rc == KR_OK && wgrad) {
        dw1 = matrix(2 * f, h, dy);
        rc = run_gemm(at, KR_GEMM_NT, 2 * f, h, t, dpre, dense(t, 2 * f), normed, dense(t, h), dw1, dense(2 * f, h), split1,
                      Epilogue{}, max_cus);
      }
    }
    if (rc != KR_OK) return failed(at, rc);
    if (wgrad) release({a[5]});
    return pack({&dx, &dpre, &dw2, &dw1});
  });
}

// attn_chain_bwd(dy, w_proj, q, k, v, o, lse, o rows, freqs, scale, beside other streams, mixed, qk rstd, gamma_q, gamma_k, w_qkv, normed,
// split_proj, split_qkv, weight gradients, max_cus, between) -> (dx [rows, h], gradient of the QKV projection's output [rows, w],
// dw_proj, dw_qkv, dgamma_q, dgamma_k).  Saved tensors, weight gradients and ``between`` as in mlp_chain_bwd.
PyObject* py_attn_chain_bwd(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  return guarded([&]() -> PyObject* {
    if (n_args != 22) return none();
    for (int i : {2, 3, 4, 5})
      if (!bf16_arg(a[i])) return none();
    if (!f32_arg(a[6]) || !f32_arg(a[8])) return none();
    for (int i : {1, 15})
      if (!bf16_arg(a[i]) || tensor(a[i]).dim() != 2) return none();
    const Tensor &q = tensor(a[2]), &k = tensor(a[3]), &v = tensor(a[4]), &o = tensor(a[5]), &lse = tensor(a[6]),
                 &freqs = tensor(a[8]), &wp = tensor(a[1]), &wq = tensor(a[15]);
    const AttnShape c = attn_shape(q, k, v);
    if (!attn_bwd_ok(c, q, o, lse)) return none();
    const int64_t t = (int64_t)c.s * c.b, wo = (int64_t)c.nq * c.hd, w = (int64_t)c.nkv * (c.per + 2) * c.hd, cols = wp.size(0),
                  h = wq.size(1);
    Operand od;
    if (!fits_int(t) || !fits_int(cols) || wo % 8 || w % 8 || h % 8 || cols % 8 || !is_weight(a[1], cols, wo) ||
        !is_weight(a[15], w, h) || !is_saved(a[7], t, wo) || !is_saved(a[16], t, h) || !is_rotary_table(freqs, c.s, c.hd) ||
        !grad_input(a[0], t, cols, od))
      return none();
    const bool qk = !absent(a[13]);
    if (qk) {
      if (!bf16_arg(a[11]) || !f32_arg(a[12]) || !is_gamma(a[13], c.hd) || !is_gamma(a[14], c.hd)) return none();
      const Tensor &m = tensor(a[11]), &r = tensor(a[12]);
      if (!m.is_contiguous() || m.numel() != t * w || !r.is_contiguous() || r.numel() != t * c.nkv * (c.per + 1)) return none();
    }
    const float scale = (float)real(a[9]);
    const int flags = truth(a[10]) ? KR_ATTN_BESIDE_OTHER_STREAMS : 0;
    const int split_proj = (int)integer(a[17]), split_qkv = (int)integer(a[18]), max_cus = (int)integer(a[20]);
    const bool wgrad = truth(a[19]);
    const Tensor &dy = tensor(a[0]), &o2d = tensor(a[7]), &normed = tensor(a[16]);
    const Operand o_wp = operand2(wp), o_wq = operand2(wq);
    Tensor dout, dwp, dwq, dx, dgq, dgk, dmixed;
    AttnGrads g;
    int rc;
    Step at;
    {
      WithoutInterpreter free;
      dout = matrix(t, wo, dy);
      rc = run_gemm(at, KR_GEMM_NN, t, wo, cols, dy, od, wp, o_wp, dout, dense(t, wo), split_proj, Epilogue{}, max_cus);
      if (rc == KR_OK && wgrad) {
        dwp = matrix(cols, wo, dy);
        rc = run_gemm(at, KR_GEMM_NT, cols, wo, t, dy, od, o2d, dense(t, wo), dwp, dense(cols, wo), split_proj, Epilogue{},
                      max_cus);
      }
    }
    if (rc != KR_OK) return failed(at, rc);
    if (!called(a[21])) return nullptr;
    if (wgrad) release({a[7]});
    at.call("kr_attn_bwd", c);
    {
      WithoutInterpreter free;
      rc = run_attn_bwd(c, dout, q, k, v, o, lse, scale, flags, g);
      dout = Tensor();
      if (rc == KR_OK) {
        at.call("kr_rope");
        rc = run_rope(g.fused, freqs, true);
      }
    }
    if (rc != KR_OK) return failed(at, rc);
    if (wgrad) release({a[2], a[3], a[4], a[5], a[6]});
    at.call("kr_qk_norm_bwd");
    {
      WithoutInterpreter free;
      if (qk) {
        const Tensor &gq = tensor(a[13]), &gk = tensor(a[14]);
        dgq = at::empty({c.hd}, gq.options());
        dgk = at::empty({c.hd}, gk.options());
        const size_t n = kr_qk_norm_bwd_workspace_bytes(t, c.nkv, (int)c.per, c.hd);
        const Tensor ws = bytes(n < 16 ? 16 : n, g.fused);
        rc = kr_qk_norm_bwd(ptr(g.fused), ptr(tensor(a[11])), (const float*)ptr(tensor(a[12])), ptr(gq), ptr(gk), ptr(dgq), ptr(dgk),
                            ptr(ws), t, c.nkv, (int)c.per, c.hd, stream());
      }
    }
    if (rc != KR_OK) return failed(at, rc);
    if (wgrad && qk) release({a[11], a[12]});
    {
      WithoutInterpreter free;
      dmixed = g.mixed.view({t, w});
      dx = matrix(t, h, dmixed);
      rc = run_gemm(at, KR_GEMM_NN, t, h, w, dmixed, dense(t, w), wq, o_wq, dx, dense(t, h), split_qkv, Epilogue{}, max_cus);
      if (rc == KR_OK && wgrad) {
        dwq = matrix(w, h, dmixed);
        rc = run_gemm(at, KR_GEMM_NT, w, h, t, dmixed, dense(t, w), normed, dense(t, h), dwq, dense(w, h), split_qkv, Epilogue{},
                      max_cus);
      }
    }
    if (rc != KR_OK) return failed(at, rc);
    if (wgrad) release({a[16]});
    return pack({&dx, &dmixed, &dwp, &dwq, &dgq, &dgk});
  });
}

// rmsnorm_dgamma(partials [n, cols] fp32, gamma) -> the weight gradient
PyObject* py_rmsnorm_dgamma(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  return guarded([&]() -> PyObject* {
    if (n_args != 2 || !f32_arg(a[0]) || tensor(a[0]).dim() != 2 || !tensor(a[0]).is_contiguous() ||
        !is_gamma(a[1], tensor(a[0]).size(1)) || !fits_int(tensor(a[0]).size(0)) || !fits_int(tensor(a[0]).size(1)))
      return none();
    const Tensor &p = tensor(a[0]), &gamma = tensor(a[1]);
    Tensor dgamma;
    int rc;
    {
      WithoutInterpreter free;
      dgamma = at::empty({p.size(1)}, gamma.options());
      rc = kr_rmsnorm_dgamma((const float*)ptr(p), (int)p.size(0), (int)p.size(1), ptr(dgamma), stream());
    }
    if (rc != KR_OK) return failed("kr_rmsnorm_dgamma", rc);
    return wrap(std::move(dgamma));
  });
}

PyMethodDef kMethods[] = {
    {"rows_view", (PyCFunction)(void*)py_rows_view, METH_FASTCALL, nullptr},
    {"gemm", (PyCFunction)(void*)py_gemm, METH_FASTCALL, nullptr},
    {"wgrad_segments_ok", (PyCFunction)(void*)py_wgrad_segments_ok, METH_FASTCALL, nullptr},
    {"wgrad_segments", (PyCFunction)(void*)py_wgrad_segments, METH_FASTCALL, nullptr},
    {"rmsnorm_fwd", (PyCFunction)(void*)py_rmsnorm_fwd, METH_FASTCALL, nullptr},
    {"rmsnorm_bwd", (PyCFunction)(void*)py_rmsnorm_bwd, METH_FASTCALL, nullptr},
    {"rope_fused", (PyCFunction)(void*)py_rope_fused, METH_FASTCALL, nullptr},
    {"split_qkv", (PyCFunction)(void*)py_split_qkv, METH_FASTCALL, nullptr},
    {"attn_fwd", (PyCFunction)(void*)py_attn_fwd, METH_FASTCALL, nullptr},
    {"attn_bwd", (PyCFunction)(void*)py_attn_bwd, METH_FASTCALL, nullptr},
    {"dropout_add", (PyCFunction)(void*)py_dropout_add, METH_FASTCALL, nullptr},
    {"dropout_bwd", (PyCFunction)(void*)py_dropout_bwd, METH_FASTCALL, nullptr},
    {"release", (PyCFunction)(void*)py_release, METH_FASTCALL, nullptr},
    {"attn_chain_fwd", (PyCFunction)(void*)py_attn_chain_fwd, METH_FASTCALL, nullptr},
    {"mlp_chain_fwd", (PyCFunction)(void*)py_mlp_chain_fwd, METH_FASTCALL, nullptr},
    {"mlp_chain_bwd", (PyCFunction)(void*)py_mlp_chain_bwd, METH_FASTCALL, nullptr},
    {"attn_chain_bwd", (PyCFunction)(void*)py_attn_chain_bwd, METH_FASTCALL, nullptr},
    {"rmsnorm_dgamma", (PyCFunction)(void*)py_rmsnorm_dgamma, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_native", "Host side of the hip backend.", -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&kModule); }
