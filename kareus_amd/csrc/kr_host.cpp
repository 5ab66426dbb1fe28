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
    int epi = KR_GEMM_EPI_NONE;
    const void* aux = nullptr;
    Operand ox;
    void* out2 = nullptr;
    int64_t ld_out2 = 0;
    int64_t out_cols = n;
    if (!absent(p_res)) {
      ox = operand3(tensor(p_res));
      if (!ox.ok || ox.rows != m || ox.cols != n) return none();
      epi = KR_GEMM_EPI_ADD;
      aux = ptr(tensor(p_res));
    } else if (!absent(p_act)) {
      const Tensor& act = tensor(p_act);
      if (act.dim() != 2 || act.size(0) != m || act.size(1) * 2 != n || act.stride(1) != 1) return none();
      epi = KR_GEMM_EPI_SWIGLU;
      out2 = ptr(act);
      ld_out2 = act.stride(0);
    } else if (!absent(p_pre)) {
      const Tensor& pre = tensor(p_pre);
      if (accumulate || pre.dim() != 2 || pre.size(0) != m || pre.size(1) != 2 * n || pre.stride(1) != 1) return none();
      epi = KR_GEMM_EPI_SWIGLU_BWD;
      ox.ld = pre.stride(0);
      aux = ptr(pre);
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
    const int epilogue = epi | (split == 2 ? KR_GEMM_BESIDE_OTHER_STREAMS : 0);
    int rc;
    {
      WithoutInterpreter free;
      if (!out.defined()) out = matrix(m, out_cols, ta);
      Tensor ws;
      size_t ws_bytes = 0;
      if (epi == KR_GEMM_EPI_NONE && split != 0 && oc.run_rows == 1) {
        ws_bytes = gemm_workspace(layout, (int)m, (int)n, (int)k, split == 1);
        if (ws_bytes) ws = bytes(ws_bytes, ta);
      }
      void* ws_ptr = ws_bytes ? ptr(ws) : nullptr;
      if (oa.run_rows > 1 || oc.run_rows > 1 || ox.run_rows > 1) {
        rc = kr_gemm_bf16_runs(layout, (int)m, (int)n, (int)k, ptr(ta), oa.ld, oa.run_rows, oa.run_ld, ptr(tb), ob.ld,
                               ptr(out), oc.ld, oc.run_rows, oc.run_ld, accumulate, epilogue, aux, ox.ld, ox.run_rows,
                               ox.run_ld, out2, ld_out2, max_cus, ws_ptr, ws_bytes, stream());
      } else {
        rc = kr_gemm_bf16_fused(layout, (int)m, (int)n, (int)k, ptr(ta), oa.ld, ptr(tb), ob.ld, ptr(out), oc.ld,
                                accumulate, epilogue, aux, ox.ld, out2, ld_out2, max_cus, ws_ptr, ws_bytes, stream());
      }
    }
    if (rc != KR_OK)
      return failed("kr_gemm_bf16(layout=" + std::to_string(layout) + ", M=" + std::to_string(m) + ", N=" +
                        std::to_string(n) + ", K=" + std::to_string(k) + ", epilogue=" + std::to_string(epi) + ")",
                    rc);
    return absent(p_out) ? wrap(std::move(out)) : Py_NewRef(p_out);
  });
}

// wgrad_segments(dys, xs, out, accumulate, split, max_cus): sum of dys[i]^T . xs[i] in one launch, None when the pairs
// are not pieces the kernel takes
PyObject* py_wgrad_segments(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  return guarded([&]() -> PyObject* {
    if (n_args != 6 || !PyList_Check(a[0]) || !PyList_Check(a[1])) return none();
    const Py_ssize_t nseg = PyList_GET_SIZE(a[0]);
    if (nseg < 1 || nseg > KR_GEMM_MAX_SEGMENTS || PyList_GET_SIZE(a[1]) != nseg) return none();
    const void *pa[KR_GEMM_MAX_SEGMENTS], *pb[KR_GEMM_MAX_SEGMENTS];
    Tensor held[2 * KR_GEMM_MAX_SEGMENTS];  // the lists may change while the interpreter is free
    Operand fa, fb;
    for (Py_ssize_t i = 0; i < nseg; ++i) {
      PyObject *dy = PyList_GET_ITEM(a[0], i), *x = PyList_GET_ITEM(a[1], i);
      if (!bf16_arg(dy) || !bf16_arg(x)) return none();
      const Operand oa = operand3(tensor(dy)), ob = operand3(tensor(x));
      if (!oa.ok || !ob.ok || ob.run_rows > 1 || oa.rows != ob.rows || oa.rows % 64 ||
          tensor(x).device() != tensor(dy).device())
        return none();
      if (i == 0) {
        fa = oa, fb = ob;
      } else if (oa.rows != fa.rows || oa.ld != fa.ld || oa.run_rows != fa.run_rows || oa.run_ld != fa.run_ld ||
                 ob.ld != fb.ld || oa.cols != fa.cols || ob.cols != fb.cols) {
        return none();
      }
      held[2 * i] = tensor(dy);
      held[2 * i + 1] = tensor(x);
    }
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
// rope_fused(fused [s, b, ng, per + 2, hd], per, freqs [rows >= s, 1.., hd] fp32, backward) -> True
PyObject* py_rope_fused(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  return guarded([&]() -> PyObject* {
    if (n_args != 4 || !bf16_arg(a[0]) || !f32_arg(a[2])) return none();
    const Tensor &f = tensor(a[0]), &fr = tensor(a[2]);
    const int64_t per = integer(a[1]);
    const bool backward = truth(a[3]);
    // (the table is one row per position: a dimension between the rows and the channels has to be a 1)
    if (f.dim() != 5 || !f.is_contiguous() || f.size(3) != per + 2 || fr.dim() < 2 || !fr.is_contiguous() ||
        fr.size(-1) != f.size(4) || fr.numel() != fr.size(0) * f.size(4) || fr.size(0) < f.size(0))
      return none();
    const int64_t s = f.size(0), b = f.size(1), slots = f.size(3), heads = f.size(2) * slots, hd = f.size(4);
    if (!fits_int(s) || !fits_int(b) || !fits_int(heads)) return none();
    int rc;
    {
      WithoutInterpreter free;
      rc = kr_rope(ptr(f), ptr(f), (const float*)ptr(fr), (int)s, (int)b, (int)heads, (int)hd, b * heads * hd, heads * hd, hd,
                   b * heads * hd, heads * hd, hd, backward, (int)slots, (int)slots - 1, stream());
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
      o = at::empty({c.s, c.b, c.nq, c.hd}, q.options());
      lse = at::empty({c.b, c.nq, c.s}, q.options().dtype(at::kFloat));
      Tensor ws;
      const QStrides sq = q_strides(q, c.per), so = q_strides(o, c.per);
      const size_t n = (flags & KR_ATTN_GENERAL_KERNELS)
                           ? 0
                           : kr_attn_fwd_workspace_bytes_strided(c.s, c.b, c.nq, c.nkv, c.hd,
                                                                 std::max({sq.s, so.s, k.stride(0), v.stride(0)}));
      if (n) ws = bytes(n, q);
      rc = kr_attn_fwd_ws(ptr(q), ptr(k), ptr(v), ptr(o), (float*)ptr(lse), c.s, c.b, c.nq, c.nkv, c.hd, scale, sq.s, sq.b,
                          sq.g, sq.h, k.stride(0), k.stride(1), k.stride(2), v.stride(0), v.stride(1), v.stride(2), so.s,
                          so.b, so.g, so.h, flags | KR_ATTN_IN_PLACE, n ? ptr(ws) : nullptr, n, stream());
    }
    if (rc != KR_OK) return failed(attn_name("kr_attn_fwd", c), rc);
    PyObject *po = wrap(std::move(o)), *pl = wrap(std::move(lse));
    return Py_BuildValue("(NN)", po, pl);
  });
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
    if (!c.ok || q.dim() != 5 || !dout.is_contiguous() || !o.is_contiguous() || !lse.is_contiguous() ||
        dout.numel() != (int64_t)c.s * c.b * c.nq * c.hd || o.numel() != dout.numel() ||
        lse.numel() != (int64_t)c.b * c.nq * c.s)
      return none();
    const float scale = (float)real(a[6]);
    const int flags = (int)integer(a[7]);
    const int64_t s = c.s, b = c.b, ng = c.nkv, hd = c.hd, g = (c.per + 2) * hd, w = ng * g;
    Tensor fused, mixed, dq, dk, dv;
    int rc;
    {
      WithoutInterpreter free;
      fused = at::empty({s, b, ng, c.per + 2, hd}, q.options());
      mixed = fused.view({s, b, w});
      dq = fused.as_strided({s, b, ng, c.per, hd}, {b * w, w, g, hd, 1}, 0);
      dk = fused.as_strided({s, b, ng, hd}, {b * w, w, g, 1}, c.per * hd);
      dv = fused.as_strided({s, b, ng, hd}, {b * w, w, g, 1}, (c.per + 1) * hd);
      const QStrides sq = q_strides(q, c.per);
      const int64_t os = b * c.nq * hd, ob = c.nq * hd, og = c.per * hd;
      const size_t n = kr_attn_bwd_workspace_bytes_strided(c.s, c.b, c.nq, c.nkv, c.hd,
                                                           std::max({sq.s, k.stride(0), v.stride(0), os, b * w}));
      Tensor ws = bytes(n < 16 ? 16 : n, q);
      rc = kr_attn_bwd_flags(ptr(dout), ptr(q), ptr(k), ptr(v), ptr(o), (const float*)ptr(lse), ptr(dq), ptr(dk), ptr(dv),
                             ptr(ws), c.s, c.b, c.nq, c.nkv, c.hd, scale, sq.s, sq.b, sq.g, sq.h, k.stride(0), k.stride(1),
                             k.stride(2), v.stride(0), v.stride(1), v.stride(2), os, ob, og, hd, os, ob, og, hd, b * w, w, g, hd,
                             b * w, w, g, b * w, w, g, flags, stream());
    }
    if (rc != KR_OK) return failed(attn_name("kr_attn_bwd", c), rc);
    PyObject *pq = wrap(std::move(dq)), *pk = wrap(std::move(dk)), *pv = wrap(std::move(dv));
    PyObject* pm = wrap(std::move(mixed));
    PyObject* pf = wrap(std::move(fused));
    return Py_BuildValue("(NNNNN)", pq, pk, pv, pm, pf);
  });
}

// ---- hidden dropout ---------------------------------------------------------------------------------------------
// dropout_add(x, residual, p, out, seed) -> (out, mask)
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
    const uint64_t seed = seed_value(a[4]);
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

PyMethodDef kMethods[] = {
    {"rows_view", (PyCFunction)(void*)py_rows_view, METH_FASTCALL, nullptr},
    {"gemm", (PyCFunction)(void*)py_gemm, METH_FASTCALL, nullptr},
    {"wgrad_segments", (PyCFunction)(void*)py_wgrad_segments, METH_FASTCALL, nullptr},
    {"rmsnorm_fwd", (PyCFunction)(void*)py_rmsnorm_fwd, METH_FASTCALL, nullptr},
    {"rmsnorm_bwd", (PyCFunction)(void*)py_rmsnorm_bwd, METH_FASTCALL, nullptr},
    {"rope_fused", (PyCFunction)(void*)py_rope_fused, METH_FASTCALL, nullptr},
    {"split_qkv", (PyCFunction)(void*)py_split_qkv, METH_FASTCALL, nullptr},
    {"attn_fwd", (PyCFunction)(void*)py_attn_fwd, METH_FASTCALL, nullptr},
    {"attn_bwd", (PyCFunction)(void*)py_attn_bwd, METH_FASTCALL, nullptr},
    {"dropout_add", (PyCFunction)(void*)py_dropout_add, METH_FASTCALL, nullptr},
    {"dropout_bwd", (PyCFunction)(void*)py_dropout_bwd, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_native", "Host side of the hip backend.", -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&kModule); }
