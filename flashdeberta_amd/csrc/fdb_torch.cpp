// Host path of the operators in native code: what stands between a Python call and the launches of libfdb_hip.so.
//
// A short sequence's attention takes the GPU about ten microseconds, so the time of such a call is what the host spends
// on it.  Building the argument block through ctypes, attribute by attribute, and the views and allocations around it took
// 22 us per forward call (57 us for a module layer with its remembered projections); the same work here -- tensor
// metadata read in place, one scratch allocation for everything that does not leave the call -- takes a fifth of that.
//
// This file is glue on torch's C++ interface (ATen tensors, the caching allocator, the current stream); everything that
// runs on the GPU is behind include/fdb.h.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/HIPContextLight.h>
#include <c10/hip/HIPGuard.h>
#include <c10/hip/HIPStream.h>
#include <hipblaslt/hipblaslt.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <map>
#include <memory>
#include <mutex>
#include <optional>
#include <tuple>
#include <utility>
#include <vector>

#include "../../include/fdb.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

// ---- Python arguments -------------------------------------------------------------------------------------------
// What an entry uses after it has let go of the interpreter's lock it holds by a reference of its own: another thread may put
// another tensor into the Python object meanwhile.
const Tensor& tensor_arg(PyObject* o, const char* name) {
  TORCH_CHECK_TYPE(THPVariable_Check(o), name, " must be a tensor");
  return THPVariable_Unpack(o);
}
OptTensor opt_tensor_arg(PyObject* o, const char* name) {
  if (o == Py_None) return std::nullopt;
  return tensor_arg(o, name);
}
int64_t int_arg(PyObject* o) {
  if (!PyLong_CheckExact(o)) {  // numpy integers, bools, zero-dimensional tensors
    PyObject* n = PyNumber_Long(o);
    if (!n) throw python_error();
    const int64_t v = PyLong_AsLongLong(n);
    Py_DECREF(n);
    if (v == -1 && PyErr_Occurred()) throw python_error();
    return v;
  }
  const int64_t v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) throw python_error();
  return v;
}
double float_arg(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw python_error();
  return v;
}
bool bool_arg(PyObject* o) {
  const int v = PyObject_IsTrue(o);
  if (v < 0) throw python_error();
  return v != 0;
}

// What an entry does once its arguments are read -- allocations, searches for a kernel, launches that wait for a place in a queue --
// is done without the interpreter's lock, so that the threads of a program do not wait for one another.
using NoGil = pybind11::gil_scoped_release;

[[noreturn]] void throw_python() {  // the pending Python error, carried out of the scope that holds the lock
  python_error e;
  e.persist();
  throw e;
}

// Negative codes are argument errors (ValueError), positive ones HIP errors (RuntimeError).
void check(int code, const char* what) {
  if (code == 0) return;
  TORCH_CHECK_VALUE(code > 0, what, " failed: ", fdb_strerror(code), " (code ", code, ")");
  TORCH_CHECK(false, what, " failed: ", fdb_strerror(code), " (code ", code, ")");
}

int fdb_dtype_of(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return FDB_F32;
    case at::kBFloat16: return FDB_BF16;
    case at::kHalf: return FDB_F16;
    default: return -1;
  }
}

// Memory that can be read through data_ptr(): not a wrapper around other tensors (quantised or distributed parameters, functorch's).
bool plain_memory(const Tensor& t) {
  constexpr c10::DispatchKeySet wrapped({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                         c10::DispatchKey::Conjugate, c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor});
  return t.layout() == at::kStrided && !t.key_set().has_any(wrapped);
}

void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

int64_t att_span(int64_t buckets, int64_t max_relative) { return buckets > 0 ? buckets : max_relative; }

// ---- matrix products -----------------------------------------------------------------------------------------------
// The projections around the attention are plain products, which hipBLASLt does; torch's own call of it costs the host
// 17 us (it builds descriptors and asks for the heuristic's choice each time), more than the GPU needs for the product of a
// short batch.  Here both are kept per (shape, strides, type, epilogue) and the call is the launch alone.
//   D [M, N] (row stride ldd) = op(A) op(B) (+ bias over N) (+ D): row-major matrices, A [M, K] or its transpose, B [K, N] or its transpose.
struct GemmKey {
  hipblasLtHandle_t handle;
  int64_t m, n, k, lda, ldb, ldd;
  int32_t type, flags;  // flags: 1 A transposed, 2 B transposed, 4 bias, 8 accumulate onto D
  bool operator<(const GemmKey& o) const {
    return std::tie(handle, m, n, k, lda, ldb, ldd, type, flags) < std::tie(o.handle, o.m, o.n, o.k, o.lda, o.ldb, o.ldd, o.type, o.flags);
  }
};
struct GemmPlan {
  hipblasLtMatmulDesc_t desc = nullptr;
  hipblasLtMatrixLayout_t a = nullptr, b = nullptr, d = nullptr;
  hipblasLtMatmulAlgo_t algo;
  int64_t workspace = 0;
  bool usable = false;   // the library has a kernel for this product
  GemmPlan() = default;
  GemmPlan(const GemmPlan&) = delete;
  GemmPlan& operator=(const GemmPlan&) = delete;
  ~GemmPlan() {
    if (a) hipblasLtMatrixLayoutDestroy(a);
    if (b) hipblasLtMatrixLayoutDestroy(b);
    if (d) hipblasLtMatrixLayoutDestroy(d);
    if (desc) hipblasLtMatmulDescDestroy(desc);
  }
};
constexpr size_t kMostPlans = 512;  // a plan is a few hundred bytes; a program with more shapes than this starts over

void blas(hipblasStatus_t s, const char* what) { TORCH_CHECK(s == HIPBLAS_STATUS_SUCCESS, what, " failed: hipBLASLt status ", (int)s); }

hipDataType blas_type(at::ScalarType t) { return t == at::kBFloat16 ? HIP_R_16BF : HIP_R_16F; }  // the callers refuse other types

// The library is column-major: D^T [N, M] = op(B)^T op(A)^T, so B's memory is its first operand and A's the second.
// A plan belongs to a handle of torch's, and torch lends a handle of a device to one thread at a time: the bias pointer that a plan
// carries into its launch, and the launch, need no lock.  The mutex is held for a look into the map alone.
std::mutex g_plans_mutex;
std::map<GemmKey, std::shared_ptr<GemmPlan>> g_plans;
std::shared_ptr<GemmPlan> gemm_plan(const GemmKey& key) {
  {
    const std::lock_guard<std::mutex> lock(g_plans_mutex);
    const auto hit = g_plans.find(key);
    if (hit != g_plans.end()) return hit->second;
  }
  const auto plan = std::make_shared<GemmPlan>();
  GemmPlan& p = *plan;
  blas(hipblasLtMatmulDescCreate(&p.desc, HIPBLAS_COMPUTE_32F, HIP_R_32F), "hipblasLtMatmulDescCreate");
  const auto set = [&](hipblasLtMatmulDescAttributes_t what, const void* v, size_t n) { blas(hipblasLtMatmulDescSetAttribute(p.desc, what, v, n), "hipblasLtMatmulDescSetAttribute"); };
  const hipblasOperation_t op_first = key.flags & 2 ? HIPBLAS_OP_T : HIPBLAS_OP_N, op_second = key.flags & 1 ? HIPBLAS_OP_T : HIPBLAS_OP_N;
  set(HIPBLASLT_MATMUL_DESC_TRANSA, &op_first, sizeof(op_first));
  set(HIPBLASLT_MATMUL_DESC_TRANSB, &op_second, sizeof(op_second));
  const auto type = (hipDataType)key.type;
  if (key.flags & 4) {
    const hipblasLtEpilogue_t e = HIPBLASLT_EPILOGUE_BIAS;
    set(HIPBLASLT_MATMUL_DESC_EPILOGUE, &e, sizeof(e));
    set(HIPBLASLT_MATMUL_DESC_BIAS_DATA_TYPE, &type, sizeof(type));
  }
  // row-major [M, K] with row stride lda is column-major [K, M]
  blas(hipblasLtMatrixLayoutCreate(&p.a, type, key.flags & 2 ? key.k : key.n, key.flags & 2 ? key.n : key.k, key.ldb), "hipblasLtMatrixLayoutCreate");
  blas(hipblasLtMatrixLayoutCreate(&p.b, type, key.flags & 1 ? key.m : key.k, key.flags & 1 ? key.k : key.m, key.lda), "hipblasLtMatrixLayoutCreate");
  blas(hipblasLtMatrixLayoutCreate(&p.d, type, key.n, key.m, key.ldd), "hipblasLtMatrixLayoutCreate");
  hipblasLtMatmulPreference_t pref = nullptr;
  blas(hipblasLtMatmulPreferenceCreate(&pref), "hipblasLtMatmulPreferenceCreate");
  const size_t most = at::cuda::getCUDABlasLtWorkspaceSize();  // torch's own bound, so that the choice is torch's own
  hipblasLtMatmulHeuristicResult_t found = {};
  int n = 0;
  hipblasLtMatmulPreferenceSetAttribute(pref, HIPBLASLT_MATMUL_PREF_MAX_WORKSPACE_BYTES, &most, sizeof(most));
  const hipblasStatus_t rc = hipblasLtMatmulAlgoGetHeuristic(key.handle, p.desc, p.a, p.b, p.d, p.d, pref, 1, &found, &n);
  hipblasLtMatmulPreferenceDestroy(pref);
  p.usable = rc == HIPBLAS_STATUS_SUCCESS && n > 0;   // a plan without a kernel is kept, too: the next call need not ask again
  p.algo = found.algo;
  p.workspace = (int64_t)found.workspaceSize;
  const std::lock_guard<std::mutex> lock(g_plans_mutex);
  if (g_plans.size() >= kMostPlans) g_plans.clear();   // one that another thread is using lives until it is done
  g_plans.emplace(key, plan);
  return plan;
}

struct Mat {  // the first `rows` rows of a row-major matrix; one of more dimensions is contiguous, its leading ones taken together
  const Tensor& t;
  int64_t rows;
  int64_t cols() const { return t.size(-1); }
  int64_t ld() const { return t.dim() == 2 ? t.stride(0) : cols(); }   // a dimension of one may have any stride
  Tensor view() const { return t.dim() == 2 ? t.narrow(0, 0, rows) : t.view({-1, cols()}).narrow(0, 0, rows); }
};
// The product by hipBLASLt; false where that has no kernel for it or does not start the one it named.
bool library_product(Mat a, bool trans_a, Mat b, bool trans_b, Mat d, const Tensor* bias = nullptr, bool accumulate = false) {
  const Tensor& on = d.t;
  const hipblasLtHandle_t handle = at::cuda::getCurrentCUDABlasLtHandle();   // the callers have made d's device the current one
  const auto plan = gemm_plan(GemmKey{handle, trans_a ? a.cols() : a.rows, trans_b ? b.rows : b.cols(), trans_a ? a.rows : a.cols(), a.ld(), b.ld(), d.ld(),
                                      (int32_t)blas_type(on.scalar_type()),
                                      (trans_a ? 1 : 0) | (trans_b ? 2 : 0) | (bias ? 4 : 0) | (accumulate ? 8 : 0)});
  GemmPlan& p = *plan;
  if (!p.usable) return false;
  Tensor ws;
  if (p.workspace > 0) ws = at::empty({p.workspace}, on.options().dtype(at::kByte));
  const float one = 1.f, beta = accumulate ? 1.f : 0.f;
  const void* bias_at = bias ? bias->data_ptr() : nullptr;
  if (bias) blas(hipblasLtMatmulDescSetAttribute(p.desc, HIPBLASLT_MATMUL_DESC_BIAS_POINTER, &bias_at, sizeof(bias_at)), "hipblasLtMatmulDescSetAttribute");
  return hipblasLtMatmul(handle, p.desc, &one, b.t.data_ptr(), p.a, a.t.data_ptr(), p.b, &beta, d.t.data_ptr(), p.d, d.t.data_ptr(), p.d, &p.algo,
                         p.workspace > 0 ? ws.data_ptr() : nullptr, p.workspace, (hipStream_t)stream_of(on)) == HIPBLAS_STATUS_SUCCESS;
}
// The same product by torch, whose own route does not end at hipBLASLt.
void torch_product(Mat a, bool trans_a, Mat b, bool trans_b, Mat d, const Tensor* bias = nullptr, bool accumulate = false) {
  const Tensor x = trans_a ? a.view().t() : a.view(), y = trans_b ? b.view().t() : b.view();
  Tensor out = d.view();
  if (bias) at::addmm_out(out, bias->narrow(0, 0, y.size(1)), x, y);
  else if (accumulate) out.addmm_(x, y);
  else at::mm_out(out, x, y);
}
void product(Mat a, bool trans_a, Mat b, bool trans_b, Mat d, const Tensor* bias = nullptr, bool accumulate = false) {
  if (!library_product(a, trans_a, b, trans_b, d, bias, accumulate)) torch_product(a, trans_a, b, trans_b, d, bias, accumulate);
}

// The projections of a padded batch's real rows, x [batch * length, k]: the attention reads no other row of them.  Whether it was done.
struct Lengths {
  const OptTensor &start, &len;
};
// `cleared`: with zeros in the rows of padding, which are not written otherwise.
bool project_real(const Tensor& x, const Tensor& w, const Tensor& b, int64_t cols, const Tensor& out, int64_t batch, int64_t length, const Lengths& real, bool cleared) {
  const OptTensor &start = real.start, &len = real.len;
  const int64_t k = x.size(-1);
  if (!len || !fdb_gemm_real_serves(batch, length, cols, k, k)) return false;
  for (const OptTensor* t : {&start, &len})
    if (*t && ((*t)->scalar_type() != at::kInt || !(*t)->is_contiguous() || (*t)->numel() != batch || (*t)->device() != x.device() || !plain_memory(**t))) return false;
  const auto entry = cleared ? fdb_gemm_real_cleared : fdb_gemm_real;
  const int rc = entry(x.data_ptr(), w.data_ptr(), b.data_ptr(), out.data_ptr(), start ? (const int32_t*)start->data_ptr() : nullptr, (const int32_t*)len->data_ptr(),
                       (int32_t)batch, (int32_t)length, (int32_t)cols, (int32_t)k, k, w.stride(0), cols, fdb_dtype_of(x.scalar_type()), stream_of(x));
  if (rc > 0) check(rc, "fdb_gemm_real");
  return rc == 0;   // a negative code: a size or an alignment it is not built for
}

// x [..., K] . w [N, K]^T + bias -> [..., N], followed by GELU or an addition of `residual` [..., N] where asked for, as torch computes
// them one after the other: bit for bit (the library's choice is torch's, and fdb_gemm adds up as it does).  With `own`, a product of at
// most 32 rows takes the library's streaming kernel, whose waves share the contraction.
enum class Then { nothing, gelu, add };
// With `real`, only the rows that a padded batch's lengths name have to be there.
Tensor project(const Tensor& x_in, const Tensor& w, const OptTensor& bias, bool own, Then then = Then::nothing, const Tensor* residual = nullptr, const Lengths* real = nullptr) {
  const auto type = x_in.scalar_type();
  const bool half = type == at::kBFloat16 || type == at::kHalf;
  const int64_t k = x_in.size(-1), m = k > 0 ? x_in.numel() / k : 0;
  const auto rest = [&](Tensor y) {
    if (then == Then::add) y.add_(*residual);
    else if (then == Then::gelu) at::gelu_(y);
    return y;
  };
  if (!x_in.is_cuda() || !half || !plain_memory(x_in) || !plain_memory(w) || (bias && !plain_memory(*bias)) || w.scalar_type() != type ||
      (bias && bias->scalar_type() != type) || m < 2 || w.dim() != 2 || w.stride(1) != 1 || w.stride(0) < k || k != w.size(1) ||
      w.device() != x_in.device() || !bias || bias->device() != x_in.device() || bias->dim() != 1 || bias->size(0) != w.size(0) || !bias->is_contiguous())
    return rest(at::linear(x_in, w, bias));
  const c10::hip::HIPGuard guard(x_in.get_device());
  const Tensor x = x_in.contiguous();
  const int64_t n = w.size(0);
  auto size = x.sizes().vec();
  size.back() = n;
  const Tensor out = at::empty(size, x.options());
  if (m <= 32 && own) {
    const int rc = fdb_linear(x.data_ptr(), w.data_ptr(), bias->data_ptr(), out.data_ptr(), (int32_t)m, (int32_t)n, (int32_t)k, k, w.stride(0), n, fdb_dtype_of(type), stream_of(x));
    if (rc == 0) return rest(out);
    if (rc > 0) check(rc, "fdb_linear");  // a negative code: a size or alignment it is not built for
  }
  if (real && then == Then::nothing && x.dim() == 3 && project_real(x, w, *bias, n, out, x.size(0), x.size(1), *real, false)) return out;
  const int epilogue = then == Then::gelu ? FDB_GEMM_GELU : then == Then::add ? FDB_GEMM_RESIDUAL : FDB_GEMM_PLAIN;
  if (fdb_gemm_serves(m, n, k, epilogue)) {
    Tensor r;
    if (then == Then::add && residual->scalar_type() == type && residual->sizes() == out.sizes() && residual->device() == x.device() && plain_memory(*residual))
      r = residual->contiguous();
    if (then != Then::add || r.defined()) {
      const int rc = fdb_gemm(x.data_ptr(), w.data_ptr(), bias->data_ptr(), r.defined() ? r.data_ptr() : nullptr, out.data_ptr(), (int32_t)m, (int32_t)n,
                              (int32_t)k, k, w.stride(0), n, n, epilogue, fdb_dtype_of(type), stream_of(x));
      if (rc == 0) return out;
      if (rc > 0) check(rc, "fdb_gemm");
    }
  }
  return rest(library_product({x, m}, false, {w, n}, true, {out, m}, &*bias) ? out : at::linear(x_in, w, bias));
}

// product(a, rows_a, trans_a, b, rows_b, trans_b, d, rows_d, bias or None, accumulate, library): into d, by hipBLASLt (whether it has
// done it) or by torch
PyObject* py_product(PyObject*, PyObject* const* x, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 11, "product takes 11 arguments");
  const Tensor ta = tensor_arg(x[0], "a"), tb = tensor_arg(x[3], "b"), td = tensor_arg(x[6], "d");
  const Mat a{ta, int_arg(x[1])}, b{tb, int_arg(x[4])}, d{td, int_arg(x[7])};
  const OptTensor bias = opt_tensor_arg(x[8], "bias");
  const bool trans_a = bool_arg(x[2]), trans_b = bool_arg(x[5]), accumulate = bool_arg(x[9]), library = bool_arg(x[10]);
  bool done = true;
  {
    const NoGil released;
    const c10::OptionalDeviceGuard guard(d.t.device());
    if (library) done = library_product(a, trans_a, b, trans_b, d, bias ? &*bias : nullptr, accumulate);
    else torch_product(a, trans_a, b, trans_b, d, bias ? &*bias : nullptr, accumulate);
  }
  return PyBool_FromLong(done);
  END_HANDLE_TH_ERRORS
}

// linear(x, weight, bias, own) -> x . weight^T + bias
PyObject* py_linear(PyObject*, PyObject* const* x, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 4, "linear takes 4 arguments");
  const Tensor in = tensor_arg(x[0], "x"), weight = tensor_arg(x[1], "weight");
  const OptTensor bias = opt_tensor_arg(x[2], "bias");
  const bool own = bool_arg(x[3]);
  Tensor out;
  {
    const NoGil released;
    out = project(in, weight, bias, own);
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// ---- the delta table on the device ---------------------------------------------------------------------------------
// One per (buckets, positions, device), built by the Python callable registered below and kept for the life of the
// process like the host table it comes from.  Threads of a program share them, autograd's among them, which do not hold the GIL.
struct Lut {
  Tensor table;
  int32_t radius = 0;
};
PyObject* g_lut_source = nullptr;
std::mutex g_lut_mutex;
std::map<std::tuple<int64_t, int64_t, int>, Lut> g_luts;  // entries are never erased: references to them stay valid

const Lut& lut_for(int64_t buckets, int64_t max_relative, const Tensor& on) {
  const auto key = std::make_tuple(buckets, max_relative, (int)on.get_device());
  {
    const std::lock_guard<std::mutex> lock(g_lut_mutex);
    const auto hit = g_luts.find(key);
    if (hit != g_luts.end()) return hit->second;
  }
  Lut lut;
  {
    const pybind11::gil_scoped_acquire gil;  // taken without the mutex: another thread may hold the GIL and wait for the mutex
    PyObject* dev = THPDevice_New(on.device());
    if (!dev) throw_python();
    PyObject* r = PyObject_CallFunction(g_lut_source, "LLN", (long long)buckets, (long long)max_relative, dev);
    if (!r) throw_python();
    lut = {THPVariable_Unpack(PyTuple_GET_ITEM(r, 0)), (int32_t)PyLong_AsLong(PyTuple_GET_ITEM(r, 1))};
    Py_DECREF(r);
  }
  const std::lock_guard<std::mutex> lock(g_lut_mutex);
  return g_luts.emplace(key, std::move(lut)).first->second;
}

// ---- forward -----------------------------------------------------------------------------------------------------
// K_r / Q_r as [H, 2S, D] with a unit last stride (a leading singleton batch dimension, as the module produces it, is dropped).
Tensor pos_arg(const Tensor& x, int64_t H, int64_t D, int64_t span, const char* name) {
  Tensor t = x.dim() == 4 && x.size(0) == 1 ? x.select(0, 0) : x;
  TORCH_CHECK_VALUE(t.dim() == 3 && t.size(0) == H && t.size(2) == D && t.size(1) >= 2 * span, name,
                    " must be the projected relative embeddings [H=", H, ", >=2S=", 2 * span, ", D=", D, "], got ", x.sizes(),
                    ". (The pre-multiplied [B,H,L,2S] bias tensors of the reference op are not an input here: the product is fused "
                    "into the kernel.)");
  return t.stride(2) == 1 ? t : t.contiguous();
}

Tensor unit_last(const Tensor& x) { return x.stride(-1) == 1 ? x : x.contiguous(); }

// Per-row bounds of a padded batch / per-head scales: a contiguous GPU vector of n entries, kept alive by the caller's `keep`.
const void* vector_arg(const Tensor& x, at::ScalarType type, int64_t n, const char* name, const char* what, std::vector<Tensor>& keep) {
  TORCH_CHECK_VALUE(x.scalar_type() == type && x.is_cuda() && x.numel() == n, name, " must be ", what);
  keep.push_back(x.contiguous());
  return keep.back().data_ptr();
}

struct Fwd {
  OptTensor pos_key, pos_query, cu, seq_start, seq_len, q_scale, k_scale, pk_scale, pq_scale, out, workspace;
  int64_t max_seqlen = -1, buckets = 0, max_relative = 0, far_splits = 0, near_splits = 0, part = 0;
  double sm_scale = NAN;  // NaN: 1 / sqrt(D * terms)
  bool causal = false, return_lse = false, single_kernel = false, no_alloc = false;
  PyObject* ask = nullptr;  // packed calls: asks the library for the workspace size (address of the argument block -> bytes)
};

constexpr int64_t up256(int64_t n) { return (n + 255) & ~(int64_t)255; }

// The scratch of a call (log-sum-exp hand-over, work-list, partial results) is one allocation, cut up here; the caching
// allocator hands it to the next call on this stream, whose launches queue up behind this call's.
void launch_forward(fdb_attn_args& a, const Tensor& on, bool need_lse, const Fwd& o) {
  void* stream = stream_of(on);
  const int64_t lse_bytes = need_lse && !a.lse ? up256((int64_t)a.total_tokens * a.heads * 4) : 0;
  const int64_t wl_bytes = a.cu_seqlens && fdb_needs_worklist(a.total_tokens, a.batch, a.heads) ? up256(fdb_worklist_ints(a.total_tokens, a.batch) * 4) : 0;
  // the size depends on whether these buffers are there, not on where
  if (lse_bytes) a.lse = (float*)16;
  if (a.cu_seqlens) a.worklist = (int32_t*)16;   // (where there is none, this stands for it: nobody reads it)
  int64_t ws_bytes = 0;
  if (o.workspace) {
    const Tensor& w = *o.workspace;
    TORCH_CHECK_VALUE(w.scalar_type() == at::kByte && w.is_cuda() && w.is_contiguous(), "workspace must be a contiguous uint8 GPU tensor");
    if (w.numel() > 0) {
      a.workspace = w.data_ptr();
      a.workspace_bytes = w.numel();
    }
  } else if (o.ask && a.cu_seqlens) {
    const pybind11::gil_scoped_acquire gil;
    PyObject* r = PyObject_CallFunction(o.ask, "K", (unsigned long long)(uintptr_t)&a);
    if (!r) throw_python();
    ws_bytes = PyLong_AsLongLong(r);
    Py_DECREF(r);
    if (ws_bytes == -1 && PyErr_Occurred()) throw_python();
  } else {
    ws_bytes = fdb_attn_workspace_bytes(&a);
  }
  Tensor scratch;
  if (lse_bytes + wl_bytes + ws_bytes > 0) {
    scratch = at::empty({lse_bytes + wl_bytes + ws_bytes}, on.options().dtype(at::kByte));
    char* p = (char*)scratch.data_ptr();
    if (lse_bytes) a.lse = (float*)p;
    if (wl_bytes) a.worklist = (int32_t*)(p + lse_bytes);
    if (ws_bytes) {
      a.workspace = p + lse_bytes + wl_bytes;
      a.workspace_bytes = ws_bytes;
    }
  }
  if (wl_bytes) check(fdb_build_worklist(a.cu_seqlens, a.batch, a.total_tokens, a.worklist, stream), "fdb_build_worklist");
  if (o.part) check(fdb_attn_fwd_part(&a, (int32_t)o.part, stream), "fdb_attn_fwd_part");
  else check(fdb_attn_fwd(&a, stream), "fdb_attn_fwd");
}

// The rest of a call whose q, k, v, out, sizes and dtype are in `a`: position tensors, row bounds, scales, scratch, launches.
// `on`: a tensor of the device; returns the log-sum-exp tensor where the caller asked for it.
Tensor run_forward(fdb_attn_args& a, const Tensor& on, at::ScalarType qt, const Fwd& o) {
  const int64_t B = a.batch, H = a.heads, D = a.head_dim, span = att_span(o.buckets, o.max_relative);
  Tensor pk, pq;
  if (o.pos_key) pk = pos_arg(*o.pos_key, H, D, span, "pos_key");
  if (o.pos_query) pq = pos_arg(*o.pos_query, H, D, span, "pos_query");
  TORCH_CHECK_VALUE(!pk.defined() || pk.scalar_type() == qt, "pos_key dtype ", pk.scalar_type(), " does not match q dtype ", qt);
  TORCH_CHECK_VALUE(!pq.defined() || pq.scalar_type() == qt, "pos_query dtype ", pq.scalar_type(), " does not match q dtype ", qt);
  for (const Tensor* t : {&pk, &pq})
    TORCH_CHECK_VALUE(!t->defined() || t->device() == on.device(), "pos_key and pos_query must be on q's device ", on.device(), ", got ", t->device());
  const bool has_pos = pk.defined() || pq.defined();
  const int terms = 1 + (pk.defined() ? 1 : 0) + (pq.defined() ? 1 : 0);
  if (has_pos) {
    const Lut& lut = lut_for(o.buckets, o.max_relative, on);
    a.delta_lut = (const int16_t*)lut.table.data_ptr();
    a.lut_radius = lut.radius;
    a.att_span = (int32_t)span;
  }
  TORCH_CHECK_VALUE(!o.no_alloc || (!o.single_kernel && !o.workspace), "no_alloc excludes single_kernel and a caller-owned workspace");
  // The log-sum-exp buffer is also the hand-over between the far-tile and near-tile launches, so it is always provided
  // when a position term is present (T*H floats), unless the caller wants one kernel.
  Tensor lse;
  if (o.return_lse) {
    lse = at::empty({a.total_tokens, H}, on.options().dtype(at::kFloat));
    a.lse = (float*)lse.data_ptr();
  }
  std::vector<Tensor> keep;
  if (o.cu) {
    a.cu_seqlens = (const int32_t*)o.cu->data_ptr();
  } else {
    const char* what = "an int32 GPU tensor with one entry per batch row";
    if (o.seq_start) a.seq_start = (const int32_t*)vector_arg(*o.seq_start, at::kInt, B, "seq_start", what, keep);
    if (o.seq_len) a.seq_len = (const int32_t*)vector_arg(*o.seq_len, at::kInt, B, "seq_len", what, keep);
  }
  if (pk.defined()) a.pos_key = pk.data_ptr(), a.pk_stride_h = pk.stride(0), a.pk_stride_r = pk.stride(1);
  if (pq.defined()) a.pos_query = pq.data_ptr(), a.pq_stride_h = pq.stride(0), a.pq_stride_r = pq.stride(1);
  if (a.dtype == FDB_FP8_E4M3) {
    const char* what = "a float32 GPU tensor with one entry per head";
    if (o.q_scale) a.q_scale = (const float*)vector_arg(*o.q_scale, at::kFloat, H, "q_scale", what, keep);
    if (o.k_scale) a.k_scale = (const float*)vector_arg(*o.k_scale, at::kFloat, H, "k_scale", what, keep);
    if (o.pk_scale) a.pk_scale = (const float*)vector_arg(*o.pk_scale, at::kFloat, H, "pk_scale", what, keep);
    if (o.pq_scale) a.pq_scale = (const float*)vector_arg(*o.pq_scale, at::kFloat, H, "pq_scale", what, keep);
  }
  a.causal = o.causal ? 1 : 0;
  a.sm_scale = (float)(std::isnan(o.sm_scale) ? 1.0 / std::sqrt((double)(D * terms)) : o.sm_scale);
  a.far_splits = (int32_t)o.far_splits, a.near_splits = (int32_t)o.near_splits;
  if (o.no_alloc) check(fdb_attn_fwd_noalloc(&a, stream_of(on)), "fdb_attn_fwd_noalloc");
  else launch_forward(a, on, has_pos && !o.single_kernel, o);
  return lse;
}

std::pair<Tensor, Tensor> forward(const Tensor& q_in, const Tensor& k_in, const Tensor& v_in, const Fwd& o) {
  TORCH_CHECK(q_in.is_cuda(), "disentangled_attention_fwd runs on the GPU only; got device ", q_in.device());
  const bool varlen = o.cu.has_value();
  int64_t B, L, H, D, T;
  if (varlen) {
    TORCH_CHECK_VALUE(q_in.dim() == 3, "with cu_seqlens, q/k/v must be [T, H, D]");
    T = q_in.size(0), H = q_in.size(1), D = q_in.size(2);
    B = o.cu->numel() - 1;
    L = o.max_seqlen >= 0 ? o.max_seqlen : T;
    TORCH_CHECK_VALUE(o.cu->scalar_type() == at::kInt && o.cu->is_cuda(), "cu_seqlens must be an int32 tensor on the GPU");
  } else {
    TORCH_CHECK_VALUE(q_in.dim() == 4, "q/k/v must be [B, L, H, D] (or [T, H, D] with cu_seqlens)");
    B = q_in.size(0), L = q_in.size(1), H = q_in.size(2), D = q_in.size(3);
    T = B * L;
  }
  TORCH_CHECK_VALUE(k_in.sizes() == q_in.sizes() && v_in.sizes() == q_in.sizes(), "q, k, v must have the same shape (self-attention): ",
                    q_in.sizes(), " ", k_in.sizes(), " ", v_in.sizes());
  TORCH_CHECK_VALUE(k_in.device() == q_in.device() && v_in.device() == q_in.device() && (!o.out || o.out->device() == q_in.device()),
                    "q, k, v (and out) must be on one device");
  const auto qt = q_in.scalar_type();
  const bool fp8 = qt == at::kFloat8_e4m3fn;
  fdb_attn_args a = {};
  if (fp8) {
    TORCH_CHECK_VALUE(k_in.scalar_type() == qt && v_in.scalar_type() == at::kBFloat16, "fp8 path: q and k float8_e4m3fn, v bfloat16");
    TORCH_CHECK_VALUE(o.q_scale && o.k_scale && (!o.pos_key || o.pk_scale) && (!o.pos_query || o.pq_scale),
                      "fp8 path: q_scale, k_scale and a scale for each position tensor are required");
    a.dtype = FDB_FP8_E4M3;
  } else {
    TORCH_CHECK_VALUE(fdb_dtype_of(qt) >= 0 && k_in.scalar_type() == qt && v_in.scalar_type() == qt, "unsupported dtypes ", qt, " ",
                      k_in.scalar_type(), " ", v_in.scalar_type());
    a.dtype = fdb_dtype_of(qt);
  }
  const Tensor q = unit_last(q_in), k = unit_last(k_in), v = unit_last(v_in);
  const c10::hip::HIPGuard guard(q.get_device());
  Tensor out;
  if (o.out) {
    out = *o.out;
    TORCH_CHECK_VALUE(out.sizes() == q.sizes() && out.scalar_type() == v.scalar_type() && out.stride(-1) == 1,
                      "out must have q's shape, v's dtype and a unit stride on D");
  } else {
    out = at::empty(q.sizes(), v.options());
  }
  a.q = q.data_ptr(), a.k = k.data_ptr(), a.v = v.data_ptr(), a.out = out.data_ptr();
  const int64_t t_ax = varlen ? 0 : 1;
  a.q_stride_b = varlen ? 0 : q.stride(0), a.q_stride_t = q.stride(t_ax), a.q_stride_h = q.stride(t_ax + 1);
  a.k_stride_b = varlen ? 0 : k.stride(0), a.k_stride_t = k.stride(t_ax), a.k_stride_h = k.stride(t_ax + 1);
  a.v_stride_b = varlen ? 0 : v.stride(0), a.v_stride_t = v.stride(t_ax), a.v_stride_h = v.stride(t_ax + 1);
  a.o_stride_b = varlen ? 0 : out.stride(0), a.o_stride_t = out.stride(t_ax), a.o_stride_h = out.stride(t_ax + 1);
  a.batch = (int32_t)B, a.heads = (int32_t)H, a.head_dim = (int32_t)D, a.max_seqlen = (int32_t)L, a.total_tokens = (int32_t)T;
  const Tensor lse = run_forward(a, q, qt, o);
  return {out, lse};
}

// attention_fwd(q, k, v, pos_key, pos_query, cu_seqlens, max_seqlen, sm_scale, position_buckets, max_relative_positions, causal,
//               return_lse, seq_start, seq_len, q_scale, k_scale, pos_key_scale, pos_query_scale, out, single_kernel, far_splits,
//               near_splits, workspace, no_alloc, part, ask) -> out or (out, lse)
PyObject* py_attention_fwd(PyObject*, PyObject* const* x, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 26, "attention_fwd takes 26 arguments");
  Fwd o;
  o.pos_key = opt_tensor_arg(x[3], "pos_key");
  o.pos_query = opt_tensor_arg(x[4], "pos_query");
  o.cu = opt_tensor_arg(x[5], "cu_seqlens");
  if (x[6] != Py_None) o.max_seqlen = int_arg(x[6]);
  if (x[7] != Py_None) o.sm_scale = float_arg(x[7]);
  o.buckets = int_arg(x[8]);
  o.max_relative = int_arg(x[9]);
  o.causal = bool_arg(x[10]);
  o.return_lse = bool_arg(x[11]);
  o.seq_start = opt_tensor_arg(x[12], "seq_start");
  o.seq_len = opt_tensor_arg(x[13], "seq_len");
  o.q_scale = opt_tensor_arg(x[14], "q_scale");
  o.k_scale = opt_tensor_arg(x[15], "k_scale");
  o.pk_scale = opt_tensor_arg(x[16], "pos_key_scale");
  o.pq_scale = opt_tensor_arg(x[17], "pos_query_scale");
  o.out = opt_tensor_arg(x[18], "out");
  o.single_kernel = bool_arg(x[19]);
  o.far_splits = int_arg(x[20]);
  o.near_splits = int_arg(x[21]);
  o.workspace = opt_tensor_arg(x[22], "workspace");
  o.no_alloc = bool_arg(x[23]);
  o.part = int_arg(x[24]);
  o.ask = x[25];
  const Tensor q = tensor_arg(x[0], "q"), k = tensor_arg(x[1], "k"), v = tensor_arg(x[2], "v");
  std::pair<Tensor, Tensor> r;
  {
    const NoGil released;
    r = forward(q, k, v, o);
  }
  PyObject* out = nullptr;
  if (x[18] != Py_None) {
    out = x[18];
    Py_INCREF(out);
  } else {
    out = THPVariable_Wrap(std::move(r.first));
  }
  if (!o.return_lse) return out;
  return Py_BuildValue("NN", out, THPVariable_Wrap(std::move(r.second)));
  END_HANDLE_TH_ERRORS
}

// ---- backward with the tables in the kernel -----------------------------------------------------------------------------
// A tensor of t's sizes whose memory runs like t's where t is dense (so that the gradient of a transposed view is contiguous where the
// view's base is), else contiguous.
Tensor empty_as(const Tensor& t) {
  const bool ok = t.is_non_overlapping_and_dense() && t.stride(-1) == 1;
  return ok ? at::empty_strided(t.sizes(), t.strides(), t.options()) : at::empty(t.sizes(), t.options());
}

bool backward_in_tables(const Tensor& q, const OptTensor& pk, const OptTensor& pq) {
  return (q.scalar_type() == at::kBFloat16 || q.scalar_type() == at::kHalf) && q.dim() == 4 && q.size(3) == 64 && pk && pq && q.is_cuda();
}

struct Strided {  // [B, L, H, 64] somewhere in memory
  const void* p;
  int64_t b, t, h;
};
Strided strided(const Tensor& x) { return {x.data_ptr(), x.stride(0), x.stride(1), x.stride(2)}; }

struct BwdSettings {
  double sm_scale;
  int64_t buckets, max_relative;
  bool causal;
  OptTensor seq_start, seq_len;
};

struct Table {  // [H, rows, 64] somewhere in memory
  const void* p;
  int64_t h, r;
};
Table table_of(const Tensor& x) { return {x.data_ptr(), x.stride(0), x.stride(1)}; }

// dq, dk, dv and the tables' gradients (one set of strides for both) into the given memory
void backward(const Tensor& on, int64_t B, int64_t L, int64_t H, Strided q, Strided k, Strided v, Strided out, Strided dout, const Tensor& lse,
              Table pk, Table pq, Strided dq, Strided dk, Strided dv, Table dpk, Table dpq, const BwdSettings& o) {
  fdb_attn_bwd_tables_args a = {};
  const auto set = [](const Strided& s, int64_t& b, int64_t& t, int64_t& h) {
    b = s.b, t = s.t, h = s.h;
    return s.p;
  };
  a.q = set(q, a.q_stride_b, a.q_stride_t, a.q_stride_h);
  a.k = set(k, a.k_stride_b, a.k_stride_t, a.k_stride_h);
  a.v = set(v, a.v_stride_b, a.v_stride_t, a.v_stride_h);
  a.out = set(out, a.out_stride_b, a.out_stride_t, a.out_stride_h);
  a.dout = set(dout, a.do_stride_b, a.do_stride_t, a.do_stride_h);
  a.dq = const_cast<void*>(set(dq, a.dq_stride_b, a.dq_stride_t, a.dq_stride_h));
  a.dk = const_cast<void*>(set(dk, a.dk_stride_b, a.dk_stride_t, a.dk_stride_h));
  a.dv = const_cast<void*>(set(dv, a.dv_stride_b, a.dv_stride_t, a.dv_stride_h));
  a.pos_key = pk.p, a.pk_stride_h = pk.h, a.pk_stride_r = pk.r;
  a.pos_query = pq.p, a.pq_stride_h = pq.h, a.pq_stride_r = pq.r;
  a.d_pos_key = const_cast<void*>(dpk.p), a.d_pos_query = const_cast<void*>(dpq.p);
  a.dp_stride_h = dpk.h, a.dp_stride_r = dpk.r;
  a.lse = (const float*)lse.data_ptr();
  std::vector<Tensor> keep;
  const char* what = "an int32 GPU tensor with one entry per batch row";
  if (o.seq_start) a.seq_start = (const int32_t*)vector_arg(*o.seq_start, at::kInt, B, "seq_start", what, keep);
  if (o.seq_len) a.seq_len = (const int32_t*)vector_arg(*o.seq_len, at::kInt, B, "seq_len", what, keep);
  const Lut& lut = lut_for(o.buckets, o.max_relative, on);
  a.delta_lut = (const int16_t*)lut.table.data_ptr();
  a.lut_radius = lut.radius;
  a.att_span = (int32_t)att_span(o.buckets, o.max_relative);
  a.batch = (int32_t)B, a.heads = (int32_t)H, a.head_dim = 64, a.seqlen = (int32_t)L;
  a.dtype = fdb_dtype_of(on.scalar_type());
  a.causal = o.causal ? 1 : 0;
  a.sm_scale = (float)o.sm_scale;
  const int64_t bytes = fdb_attn_bwd_tables_workspace_bytes(&a);
  if (bytes < 0) check((int)bytes, "fdb_attn_bwd_tables");
  const Tensor ws = at::empty({bytes}, on.options().dtype(at::kByte));
  a.workspace = ws.data_ptr();
  check(fdb_attn_bwd_tables(&a, stream_of(on)), "fdb_attn_bwd_tables");
}

// dq, dk, dv, d pos_key, d pos_query of the operator
std::array<Tensor, 5> backward_of(const Tensor& q_in, const Tensor& k_in, const Tensor& v_in, const Tensor& out_in, const Tensor& lse, const Tensor& dout_in,
                                  const Tensor& pk_in, const Tensor& pq_in, const BwdSettings& o) {
  for (const Tensor* t : {&k_in, &v_in, &out_in, &dout_in})
    TORCH_CHECK_VALUE(t->sizes() == q_in.sizes() && t->scalar_type() == q_in.scalar_type() && t->device() == q_in.device(),
                      "k, v, out and dout must have q's shape, dtype and device");
  TORCH_CHECK_VALUE(lse.scalar_type() == at::kFloat && lse.device() == q_in.device() && lse.numel() == q_in.size(0) * q_in.size(1) * q_in.size(2),
                    "lse must be the forward's float32 [B*L, H]");
  for (const Tensor* t : {&pk_in, &pq_in})
    TORCH_CHECK_VALUE(t->scalar_type() == q_in.scalar_type() && t->device() == q_in.device(), "pos_key and pos_query must have q's dtype and device");
  const Tensor q = unit_last(q_in), k = unit_last(k_in), v = unit_last(v_in), out = unit_last(out_in), dout = unit_last(dout_in);
  const int64_t B = q.size(0), L = q.size(1), H = q.size(2), D = q.size(3), span = att_span(o.buckets, o.max_relative);
  const c10::hip::HIPGuard guard(q.get_device());
  const Tensor pk = pos_arg(pk_in, H, D, span, "pos_key"), pq = pos_arg(pq_in, H, D, span, "pos_query");
  const Tensor dq = empty_as(q_in), dk = empty_as(k_in), dv = empty_as(v_in);
  const int64_t rows = std::max(pk.size(1), pq.size(1));   // one layout for both; rows past 2S take no part
  const Tensor dpos = rows > 2 * span ? at::zeros({2, H, rows, D}, pk.options()) : at::empty({2, H, rows, D}, pk.options());
  Tensor dpk = dpos.select(0, 0), dpq = dpos.select(0, 1);
  backward(q, B, L, H, strided(q), strided(k), strided(v), strided(out), strided(dout), lse, table_of(pk), table_of(pq), strided(dq), strided(dk),
           strided(dv), table_of(dpk), table_of(dpq), o);
  if (pk.size(1) != rows) dpk = dpk.narrow(1, 0, pk.size(1));
  if (pq.size(1) != rows) dpq = dpq.narrow(1, 0, pq.size(1));
  return {dq, dk, dv, dpk.reshape(pk_in.sizes()), dpq.reshape(pq_in.sizes())};
}

// The fused forward and the backward above as one autograd node.
struct AttentionNode : public torch::autograd::Function<AttentionNode> {
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& pk, const Tensor& pq,
                        const Fwd* o) {
    at::AutoDispatchBelowADInplaceOrView below;
    Fwd with = *o;
    with.pos_key = pk, with.pos_query = pq;
    with.return_lse = true;
    auto r = ::forward(q, k, v, with);
    ctx->save_for_backward({q, k, v, r.first, r.second, pk, pq, o->seq_start.value_or(Tensor()), o->seq_len.value_or(Tensor())});
    const int terms = 3;
    ctx->saved_data["sm_scale"] = std::isnan(o->sm_scale) ? 1.0 / std::sqrt((double)(q.size(3) * terms)) : o->sm_scale;
    ctx->saved_data["buckets"] = o->buckets;
    ctx->saved_data["max_relative"] = o->max_relative;
    ctx->saved_data["causal"] = o->causal;
    return r.first;
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
    const auto s = ctx->get_saved_variables();
    const auto opt = [](const Tensor& t) { return t.defined() ? OptTensor(t) : std::nullopt; };
    const BwdSettings o{ctx->saved_data["sm_scale"].toDouble(), ctx->saved_data["buckets"].toInt(), ctx->saved_data["max_relative"].toInt(),
                        ctx->saved_data["causal"].toBool(), opt(s[7]), opt(s[8])};
    at::AutoDispatchBelowADInplaceOrView below;
    auto r = backward_of(s[0], s[1], s[2], s[3], s[4], grads[0], s[5], s[6], o);
    return {r[0], r[1], r[2], r[3], r[4], Tensor()};
  }
};

// attention_node(q, k, v, pos_key, pos_query, sm_scale, position_buckets, max_relative_positions, causal, seq_start, seq_len, out, far_splits,
//                near_splits, workspace) -> out, differentiable; None where backward_in_tables does not serve
PyObject* py_attention_node(PyObject*, PyObject* const* x, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 15, "attention_node takes 15 arguments");
  const Tensor q = tensor_arg(x[0], "q"), k = tensor_arg(x[1], "k"), v = tensor_arg(x[2], "v");
  const OptTensor pk = opt_tensor_arg(x[3], "pos_key"), pq = opt_tensor_arg(x[4], "pos_query");
  if (!backward_in_tables(q, pk, pq)) Py_RETURN_NONE;
  Fwd o;
  if (x[5] != Py_None) o.sm_scale = float_arg(x[5]);
  o.buckets = int_arg(x[6]);
  o.max_relative = int_arg(x[7]);
  o.causal = bool_arg(x[8]);
  o.seq_start = opt_tensor_arg(x[9], "seq_start");
  o.seq_len = opt_tensor_arg(x[10], "seq_len");
  o.out = opt_tensor_arg(x[11], "out");
  o.far_splits = int_arg(x[12]);
  o.near_splits = int_arg(x[13]);
  o.workspace = opt_tensor_arg(x[14], "workspace");
  Tensor out;
  {
    const NoGil released;
    out = AttentionNode::apply(q, k, v, *pk, *pq, (const Fwd*)&o);
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// attention_bwd(q, k, v, out, lse, dout, pos_key, pos_query, sm_scale, position_buckets, max_relative_positions, causal, seq_start, seq_len)
//   -> (dq, dk, dv, d pos_key, d pos_query)
PyObject* py_attention_bwd(PyObject*, PyObject* const* x, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 14, "attention_bwd takes 14 arguments");
  const BwdSettings o{float_arg(x[8]), int_arg(x[9]), int_arg(x[10]), bool_arg(x[11]), opt_tensor_arg(x[12], "seq_start"), opt_tensor_arg(x[13], "seq_len")};
  const Tensor q = tensor_arg(x[0], "q"), k = tensor_arg(x[1], "k"), v = tensor_arg(x[2], "v"), out = tensor_arg(x[3], "out"), lse = tensor_arg(x[4], "lse"),
               dout = tensor_arg(x[5], "dout"), pk = tensor_arg(x[6], "pos_key"), pq = tensor_arg(x[7], "pos_query");
  std::array<Tensor, 5> r;
  {
    const NoGil released;
    r = backward_of(q, k, v, out, lse, dout, pk, pq, o);
  }
  PyObject* t = PyTuple_New(5);
  for (int i = 0; i < 5; ++i) PyTuple_SET_ITEM(t, i, THPVariable_Wrap(r[i]));
  return t;
  END_HANDLE_TH_ERRORS
}

// x: pos_key, pos_query, heads, sm_scale, position_buckets, max_relative_positions, seq_start, seq_len
struct LayerCall {
  Fwd o;
  int64_t heads;
  explicit LayerCall(PyObject* const* x) : heads(int_arg(x[2])) {
    o.pos_key = opt_tensor_arg(x[0], "pos_key");
    o.pos_query = opt_tensor_arg(x[1], "pos_query");
    o.sm_scale = float_arg(x[3]);
    o.buckets = int_arg(x[4]);
    o.max_relative = int_arg(x[5]);
    o.seq_start = opt_tensor_arg(x[6], "seq_start");
    o.seq_len = opt_tensor_arg(x[7], "seq_len");
  }
};

// The whole layer in one launch where it is that small (fdb_layer_small); undefined where it is not, or where the tensors are not what that takes.
Tensor layer_small(const Tensor& hidden, const Tensor& w, const OptTensor& bias, const LayerCall& call) {
  const auto type = hidden.scalar_type();
  const Fwd& o = call.o;
  if (hidden.dim() != 3 || (type != at::kBFloat16 && type != at::kHalf) || !hidden.is_cuda() || !o.pos_key || !o.pos_query) return {};
  const int64_t B = hidden.size(0), L = hidden.size(1), C = hidden.size(2), H = call.heads, span = att_span(o.buckets, o.max_relative);
  if (!fdb_layer_small_serves(B, L, H, C) || w.dim() != 2 || w.size(0) != 3 * 64 * H || w.size(1) != C || w.stride(1) != 1 || span < 1 ||
      (bias && (bias->dim() != 1 || bias->size(0) != w.size(0) || !bias->is_contiguous())))
    return {};
  const Tensor* const all[] = {&hidden, &w, bias ? &*bias : &w, &*o.pos_key, &*o.pos_query};
  for (const Tensor* t : all)
    if (t->scalar_type() != type || t->device() != hidden.device() || !plain_memory(*t)) return {};
  const Tensor pk = pos_arg(*o.pos_key, H, 64, span, "pos_key"), pq = pos_arg(*o.pos_query, H, 64, span, "pos_query");
  const c10::hip::HIPGuard guard(hidden.get_device());
  const Tensor x = hidden.contiguous(), out = at::empty({B, L, H * 64}, x.options());
  const Lut& lut = lut_for(o.buckets, o.max_relative, x);
  std::vector<Tensor> keep;
  const char* what = "an int32 GPU tensor with one entry per batch row";
  const int32_t* const start = o.seq_start ? (const int32_t*)vector_arg(*o.seq_start, at::kInt, B, "seq_start", what, keep) : nullptr;
  const int32_t* const len = o.seq_len ? (const int32_t*)vector_arg(*o.seq_len, at::kInt, B, "seq_len", what, keep) : nullptr;
  const float scale = (float)(std::isnan(o.sm_scale) ? 1.0 / std::sqrt(64.0 * 3) : o.sm_scale);
  const int rc = fdb_layer_small(x.data_ptr(), w.data_ptr(), bias ? bias->data_ptr() : nullptr, pk.data_ptr(), pq.data_ptr(), out.data_ptr(), start, len,
                                 (const int16_t*)lut.table.data_ptr(), (int32_t)B, (int32_t)L, (int32_t)H, (int32_t)C, C, w.stride(0), pk.stride(0), pk.stride(1), pq.stride(0),
                                 pq.stride(1), (int32_t)span, lut.radius, scale, fdb_dtype_of(type), stream_of(x));
  if (rc > 0) check(rc, "fdb_layer_small");
  return rc == 0 ? out : Tensor();   // a negative code: an alignment or a stride it is not built for
}

// The three input projections as one product over the concatenated weights, and the attention on its columns where they lie.
Tensor layer_attention(const Tensor& hidden, const Tensor& weight, const OptTensor& bias, const LayerCall& call, bool own) {
  TORCH_CHECK_VALUE(hidden.dim() == 3, "hidden_states must be [B, L, hidden]");
  if (own) {   // (adds up in another order than the library, like the streamed products)
    const Tensor done = layer_small(hidden, weight, bias, call);
    if (done.defined()) return done;
  }
  const Lengths real{call.o.seq_start, call.o.seq_len};
  const Tensor qkv = project(hidden, weight, bias, own, Then::nothing, nullptr, &real);
  TORCH_CHECK(qkv.is_cuda(), "disentangled_attention_fwd runs on the GPU only; got device ", qkv.device());
  const auto type = qkv.scalar_type();
  TORCH_CHECK_VALUE(fdb_dtype_of(type) >= 0, "unsupported dtype ", type);
  const int64_t B = qkv.size(0), L = qkv.size(1), H = call.heads, D = qkv.size(2) / (3 * H), width = H * D;
  const c10::hip::HIPGuard guard(qkv.get_device());
  const Tensor out = at::empty({B, L, width}, qkv.options());
  fdb_attn_args a = {};
  const char* p = (const char*)qkv.data_ptr();
  const int64_t bytes = width * qkv.element_size();
  a.dtype = fdb_dtype_of(type);
  a.q = p, a.k = p + bytes, a.v = p + 2 * bytes, a.out = out.data_ptr();
  a.q_stride_b = a.k_stride_b = a.v_stride_b = L * 3 * width;
  a.q_stride_t = a.k_stride_t = a.v_stride_t = 3 * width;
  a.q_stride_h = a.k_stride_h = a.v_stride_h = a.o_stride_h = D;
  a.o_stride_b = L * width, a.o_stride_t = width;
  a.batch = (int32_t)B, a.heads = (int32_t)H, a.head_dim = (int32_t)D, a.max_seqlen = (int32_t)L, a.total_tokens = (int32_t)(B * L);
  run_forward(a, qkv, type, call.o);
  return out;
}

// One layer's attention in training, from the hidden states and the relative embeddings through the three projections (shared
// by the tables): a node of its own.  What autograd would run as one product per projection and tensor, a reduction per bias and
// an addition per shared tensor is here
//   forward   q | k | v = hidden . W^T + b (of a long padded batch the real rows) and Q_r | K_r = rel . W[q, k]^T + b[q, k], W the three weights on top of each other;
//   backward  d hidden = d qkv . W,  d W = d qkv^T . hidden (+ d pos^T . rel onto the rows of q and k),  d rel = d pos . W[q, k],
//             d b = the column sums of d qkv and d pos.
struct LayerArgs {
  int64_t heads = 0;
  BwdSettings o;
};
// The three weights and the three biases under one another.
std::pair<Tensor, Tensor> joined(const Tensor& qw, const Tensor& qb, const Tensor& kw, const Tensor& kb, const Tensor& vw, const Tensor& vb, at::ScalarType type, void* stream) {
  bool plain = true;
  for (const Tensor* t : {&qw, &kw, &vw, &qb, &kb, &vb}) plain = plain && t->is_contiguous();
  if (plain) {
    const Tensor w = at::empty({3 * qw.size(0), qw.size(1)}, qw.options()), b = at::empty({3 * qb.size(0)}, qb.options());
    const void* const ws[3] = {qw.data_ptr(), kw.data_ptr(), vw.data_ptr()};
    const void* const bs[3] = {qb.data_ptr(), kb.data_ptr(), vb.data_ptr()};
    const int rc = fdb_join(ws, bs, w.data_ptr(), b.data_ptr(), qw.numel() * 2, qb.numel() * 2, stream);
    if (rc == 0) return {w, b};
    if (rc > 0) check(rc, "fdb_join");
  }
  return {at::cat({qw, kw, vw}), at::cat({qb, kb, vb})};
}
// out [rows, cols] = the first rows of x . the first cols rows of w^T + b
void projected(const Tensor& x, int64_t rows, const Tensor& w, const Tensor& b, int64_t cols, const Tensor& out) {
  const int64_t k = x.size(-1);
  if (fdb_gemm_serves(rows, cols, k, FDB_GEMM_PLAIN)) {
    const int rc = fdb_gemm(x.data_ptr(), w.data_ptr(), b.data_ptr(), nullptr, out.data_ptr(), (int32_t)rows, (int32_t)cols, (int32_t)k, k, k, cols, 0, FDB_GEMM_PLAIN,
                            fdb_dtype_of(x.scalar_type()), stream_of(x));
    if (rc == 0) return;
    if (rc > 0) check(rc, "fdb_gemm");
  }
  product({x, rows}, false, {w, cols}, true, {out, rows}, &b);
}

struct LayerNode : public torch::autograd::Function<LayerNode> {
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& hidden_in, const Tensor& rel_in, const Tensor& qw, const Tensor& qb,
                        const Tensor& kw, const Tensor& kb, const Tensor& vw, const Tensor& vb, const LayerArgs* args) {
    at::AutoDispatchBelowADInplaceOrView below;
    const Tensor hidden = hidden_in.contiguous(), rel = rel_in.contiguous();
    const c10::hip::HIPGuard guard(hidden.get_device());
    const int64_t B = hidden.size(0), L = hidden.size(1), C = hidden.size(2), H = args->heads, D = qw.size(0) / H, W = H * D;
    const int64_t span = att_span(args->o.buckets, args->o.max_relative), rows = 2 * span, esz = hidden.element_size();
    const auto type = hidden.scalar_type();
    Tensor w, b;
    std::tie(w, b) = joined(qw, qb, kw, kb, vw, vb, type, stream_of(hidden));
    const Tensor qkv = at::empty({B * L, 3 * W}, hidden.options()), pos = at::empty({rows, 2 * W}, hidden.options());
    // rows of padding: nothing of the node reads them, but hooks on its saved tensors do
    if (!project_real(hidden, w, b, 3 * W, qkv, B, L, {args->o.seq_start, args->o.seq_len}, true)) projected(hidden, B * L, w, b, 3 * W, qkv);
    projected(rel, rows, w, b, 2 * W, pos);
    const Tensor out = at::empty({B, L, W}, hidden.options());
    fdb_attn_args a = {};
    const char* p = (const char*)qkv.data_ptr();
    a.dtype = fdb_dtype_of(type);
    a.q = p, a.k = p + W * esz, a.v = p + 2 * W * esz, a.out = out.data_ptr();
    a.q_stride_b = a.k_stride_b = a.v_stride_b = L * 3 * W;
    a.q_stride_t = a.k_stride_t = a.v_stride_t = 3 * W;
    a.q_stride_h = a.k_stride_h = a.v_stride_h = a.o_stride_h = D;
    a.o_stride_b = L * W, a.o_stride_t = W;
    a.batch = (int32_t)B, a.heads = (int32_t)H, a.head_dim = (int32_t)D, a.max_seqlen = (int32_t)L, a.total_tokens = (int32_t)(B * L);
    Fwd f;
    f.sm_scale = args->o.sm_scale, f.buckets = args->o.buckets, f.max_relative = args->o.max_relative;
    f.seq_start = args->o.seq_start, f.seq_len = args->o.seq_len;
    f.return_lse = true;
    const std::array<int64_t, 3> size{H, rows, D}, stride{D, 2 * W, 1};
    f.pos_query = pos.as_strided(size, stride, 0);
    f.pos_key = pos.as_strided(size, stride, W);
    const Tensor lse = run_forward(a, qkv, type, f);
    ctx->save_for_backward({hidden, rel, w, qkv, pos, out, lse, args->o.seq_start.value_or(Tensor()), args->o.seq_len.value_or(Tensor())});
    ctx->saved_data["heads"] = H;
    ctx->saved_data["sm_scale"] = args->o.sm_scale;
    ctx->saved_data["buckets"] = args->o.buckets;
    ctx->saved_data["max_relative"] = args->o.max_relative;
    ctx->saved_data["rel_rows"] = rel_in.size(0);
    return out;
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
    const auto s = ctx->get_saved_variables();
    const Tensor &hidden = s[0], &rel = s[1], &w = s[2], &qkv = s[3], &pos = s[4], &out = s[5], &lse = s[6];
    at::AutoDispatchBelowADInplaceOrView below;
    const auto opt = [](const Tensor& t) { return t.defined() ? OptTensor(t) : std::nullopt; };
    const BwdSettings o{ctx->saved_data["sm_scale"].toDouble(), ctx->saved_data["buckets"].toInt(), ctx->saved_data["max_relative"].toInt(), false, opt(s[7]), opt(s[8])};
    const c10::hip::HIPGuard guard(hidden.get_device());
    const int64_t B = hidden.size(0), L = hidden.size(1), C = hidden.size(2), H = ctx->saved_data["heads"].toInt(), W = w.size(0) / 3, D = W / H;
    const int64_t rows = pos.size(0), n = B * L, esz = hidden.element_size(), rel_rows = ctx->saved_data["rel_rows"].toInt();
    const auto type = hidden.scalar_type();
    const Tensor dout = grads[0].contiguous();
    const Tensor dqkv = at::empty({n, 3 * W}, hidden.options()), dpos = at::empty({rows, 2 * W}, hidden.options());
    const auto at_col = [&](const Tensor& t, int64_t col) { return (const void*)((const char*)t.data_ptr() + col * W * esz); };
    const auto part = [&](const Tensor& t, int64_t col) { return Strided{at_col(t, col), L * 3 * W, 3 * W, D}; };
    const auto whole = [&](const Tensor& t) { return Strided{t.data_ptr(), L * W, W, D}; };
    const auto table = [&](const Tensor& t, int64_t col) { return Table{at_col(t, col), D, 2 * W}; };
    ::backward(hidden, B, L, H, part(qkv, 0), part(qkv, 1), part(qkv, 2), whole(out), whole(dout), lse, table(pos, 1), table(pos, 0), part(dqkv, 0),
               part(dqkv, 1), part(dqkv, 2), table(dpos, 1), table(dpos, 0), o);
    Tensor dhidden, drel, dw, db;
    const bool for_hidden = ctx->needs_input_grad(0), for_rel = ctx->needs_input_grad(1);
    const bool for_weights = ctx->needs_input_grad(2) || ctx->needs_input_grad(4) || ctx->needs_input_grad(6);
    const bool for_biases = ctx->needs_input_grad(3) || ctx->needs_input_grad(5) || ctx->needs_input_grad(7);
    const int code = fdb_dtype_of(type);
    // tokens and tables in one launch; a negative code is a size or an alignment these kernels are not built for: two products then
    if (for_hidden) dhidden = at::empty(hidden.sizes(), hidden.options());
    if (for_rel) drel = rel_rows > rows ? at::zeros({rel_rows, C}, hidden.options()) : at::empty({rel_rows, C}, hidden.options());
    if (for_hidden || for_rel) {
      int rc = FDB_ERR_SHAPE;
      if (n <= INT32_MAX && C <= INT32_MAX && fdb_dgrad_serves(for_hidden ? n : 0, for_rel ? rows : 0, C))
        rc = fdb_dgrad(dqkv.data_ptr(), for_hidden ? (int32_t)n : 0, (int32_t)(3 * W), dpos.data_ptr(), for_rel ? (int32_t)rows : 0, (int32_t)(2 * W),
                       w.data_ptr(), (int32_t)C, for_hidden ? dhidden.data_ptr() : nullptr, for_rel ? drel.data_ptr() : nullptr, code, stream_of(hidden));
      if (rc > 0) check(rc, "fdb_dgrad");
      if (rc < 0 && for_hidden) product({dqkv, n}, false, {w, 3 * W}, false, {dhidden, n});
      if (rc < 0 && for_rel) product({dpos, rows}, false, {w, 2 * W}, false, {drel, rows});
    }
    bool sums_done = false;
    if (for_weights) {
      dw = at::empty({3 * W, C}, hidden.options());
      db = at::empty({3 * W}, hidden.options());
      int rc = FDB_ERR_SHAPE;
      if (n <= INT32_MAX && C % 64 == 0) {
        const Tensor ws = at::empty({fdb_wgrad_workspace_bytes((int32_t)n, (int32_t)rows, (int32_t)(3 * W), (int32_t)C)}, hidden.options().dtype(at::kByte));
        rc = fdb_wgrad(dqkv.data_ptr(), hidden.data_ptr(), (int32_t)n, (int32_t)(3 * W), dpos.data_ptr(), rel.data_ptr(), (int32_t)rows, (int32_t)(2 * W), (int32_t)C, dw.data_ptr(),
                       db.data_ptr(), ws.data_ptr(), code, stream_of(hidden));
        if (rc > 0) check(rc, "fdb_wgrad");
      }
      sums_done = rc == 0;
      if (rc < 0) {
        product({dqkv, n}, true, {hidden, n}, false, {dw, 3 * W});
        product({dpos, rows}, true, {rel, rows}, false, {dw, 2 * W}, nullptr, true);
      }
    }
    if (for_biases && !sums_done) {
      db = at::empty({3 * W}, hidden.options());
      const Tensor ws = at::empty({fdb_column_sums_workspace_bytes(n, 3 * W, rows)}, hidden.options().dtype(at::kByte));
      check(fdb_column_sums(dqkv.data_ptr(), n, 3 * W, dpos.data_ptr(), rows, 2 * W, db.data_ptr(), ws.data_ptr(), code, stream_of(hidden)), "fdb_column_sums");
    }
    if (!for_biases) db = Tensor();
    const auto rows_of = [&](const Tensor& t, int64_t i) { return t.defined() ? t.narrow(0, i * W, W) : Tensor(); };
    return {dhidden, drel, rows_of(dw, 0), rows_of(db, 0), rows_of(dw, 1), rows_of(db, 1), rows_of(dw, 2), rows_of(db, 2), Tensor()};
  }
};

// layer_node(hidden, rel, q_weight, q_bias, k_weight, k_bias, v_weight, v_bias, heads, sm_scale, position_buckets, max_relative_positions,
//            seq_start, seq_len) -> context [B, L, H*D], differentiable; None for tensors it is not built for
PyObject* py_layer_node(PyObject*, PyObject* const* x, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 14, "layer_node takes 14 arguments");
  const Tensor hidden = tensor_arg(x[0], "hidden");
  LayerArgs a;
  a.heads = int_arg(x[8]);
  a.o = BwdSettings{float_arg(x[9]), int_arg(x[10]), int_arg(x[11]), false, opt_tensor_arg(x[12], "seq_start"), opt_tensor_arg(x[13], "seq_len")};
  const auto type = hidden.scalar_type();
  if (!hidden.is_cuda() || !plain_memory(hidden) || (type != at::kBFloat16 && type != at::kHalf) || hidden.dim() != 3 || hidden.numel() == 0 || a.heads < 1) Py_RETURN_NONE;
  Tensor t[7];
  for (int i = 0; i < 7; ++i) {
    if (x[i + 1] == Py_None) Py_RETURN_NONE;
    t[i] = tensor_arg(x[i + 1], "parameters");
    if (t[i].scalar_type() != type || t[i].device() != hidden.device() || !plain_memory(t[i])) Py_RETURN_NONE;
  }
  const int64_t C = hidden.size(2), W = t[1].size(0), span = att_span(a.o.buckets, a.o.max_relative);
  if (t[0].dim() != 2 || t[0].size(0) < 2 * span || t[0].size(1) != C || W != 64 * a.heads || C % 8) Py_RETURN_NONE;
  for (int i = 1; i < 7; i += 2)
    if (t[i].dim() != 2 || t[i].size(0) != W || t[i].size(1) != C || t[i + 1].dim() != 1 || t[i + 1].size(0) != W) Py_RETURN_NONE;
  Tensor out;
  {
    const NoGil released;
    out = LayerNode::apply(hidden, t[0], t[1], t[2], t[3], t[4], t[5], t[6], (const LayerArgs*)&a);
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// layer_attention(hidden, weight, bias, pos_key, pos_query, heads, sm_scale, position_buckets, max_relative_positions, seq_start,
//                 seq_len, own) -> context [B, L, H*D]
PyObject* py_layer_attention(PyObject*, PyObject* const* x, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 12, "layer_attention takes 12 arguments");
  const Tensor hidden = tensor_arg(x[0], "hidden"), weight = tensor_arg(x[1], "weight");
  const OptTensor bias = opt_tensor_arg(x[2], "bias");
  const LayerCall call(x + 3);
  const bool own = bool_arg(x[11]);
  Tensor out;
  {
    const NoGil released;
    out = layer_attention(hidden, weight, bias, call, own);
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// encoder_layer(hidden, weight, bias, pos_key, ..., seq_len [as layer_attention], out_weight, out_bias, norm1_weight, norm1_bias, eps1,
//               up_weight, up_bias, down_weight, down_bias, norm2_weight, norm2_bias, eps2) -> hidden states of the next layer
// A whole post-norm encoder layer with GELU; the caller has checked that the layer is one.  Products, sums, norms and GELU round where its
// modules' would, and the products add up in the same order, so the result has the same bits: in a 16-bit type twelve layers turn one
// differing rounding into a percent.
PyObject* py_encoder_layer(PyObject*, PyObject* const* x, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 23, "encoder_layer takes 23 arguments");
  const Tensor hidden = tensor_arg(x[0], "hidden");
  struct Norm {
    const Tensor weight, bias;
    double eps;
    explicit Norm(PyObject* const* p) : weight(tensor_arg(p[0], "norm_weight")), bias(tensor_arg(p[1], "norm_bias")), eps(float_arg(p[2])) {}
    Tensor operator()(const Tensor& y) const { return at::layer_norm(y, {y.size(-1)}, weight, bias, eps); }
  };
  struct Linear {
    const Tensor weight;
    OptTensor bias;
    explicit Linear(PyObject* const* p) : weight(tensor_arg(p[0], "weight")), bias(opt_tensor_arg(p[1], "bias")) {}
    Tensor operator()(const Tensor& y, Then then, const Tensor* residual = nullptr) const { return project(y, weight, bias, false, then, residual); }
  };
  const Linear in(x + 1), out(x + 11), up(x + 16), down(x + 18);
  const LayerCall call(x + 3);
  const Norm norm1(x + 13), norm2(x + 20);
  Tensor next;
  {
    const NoGil released;
    const Tensor context = layer_attention(hidden, in.weight, in.bias, call, false);
    const c10::hip::HIPGuard guard(hidden.get_device());
    const Tensor attended = norm1(out(context, Then::add, &hidden));
    next = norm2(down(up(attended, Then::gelu), Then::add, &attended));
  }
  return THPVariable_Wrap(std::move(next));
  END_HANDLE_TH_ERRORS
}

// ---- e4m3 quantisation ---------------------------------------------------------------------------------------------
// quantize_e4m3(x0, x1 or None) -> (y0, scale0[, y1, scale1]); shapes and layouts are checked by the callers' contract below
PyObject* py_quantize(PyObject*, PyObject* const* x, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 2, "quantize_e4m3 takes 2 arguments");
  const bool pair = x[1] != Py_None;
  const Tensor a0 = tensor_arg(x[0], "x0");
  const Tensor a1 = pair ? tensor_arg(x[1], "x1") : a0;
  const char* name = pair ? "quantize_e4m3_per_head_pair" : "quantize_e4m3_per_head";
  for (const Tensor* t : {&a0, &a1})
    TORCH_CHECK_VALUE(t->is_cuda() && t->scalar_type() == at::kBFloat16, name, pair ? " expects bfloat16 GPU tensors" : " expects a bfloat16 GPU tensor");
  TORCH_CHECK_VALUE(a0.sizes() == a1.sizes(), name, ": shapes differ: ", a0.sizes(), " ", a1.sizes());
  const int64_t H = a0.size(-2), D = a0.size(-1);
  Tensor y0, y1, s0, s1;
  {
    const NoGil released;
    Tensor r0 = a0.reshape({-1, H, D}), r1 = pair ? a1.reshape({-1, H, D}) : r0;
    if (r0.strides() != r1.strides() || r0.stride(2) != 1) r0 = r0.contiguous(), r1 = r1.contiguous();
    const c10::hip::HIPGuard guard(r0.get_device());
    const int64_t tokens = r0.size(0), count = pair ? 2 : 1;
    const Tensor y = at::empty({count, tokens, H, D}, r0.options().dtype(at::kFloat8_e4m3fn));
    const Tensor scale = at::empty({count, H}, r0.options().dtype(at::kFloat));
    const Tensor ws = at::empty({count * H}, r0.options().dtype(at::kInt));
    char* y_at = (char*)y.data_ptr();
    float* s_at = (float*)scale.data_ptr();
    if (pair)
      check(fdb_quant_e4m3_per_head_pair(r0.data_ptr(), r1.data_ptr(), r0.stride(0), r0.stride(1), y_at, y_at + tokens * H * D, H * D, D, s_at, s_at + H,
                                         (uint32_t*)ws.data_ptr(), (int32_t)tokens, (int32_t)H, (int32_t)D, stream_of(r0)),
            "fdb_quant_e4m3_per_head_pair");
    else
      check(fdb_quant_e4m3_per_head(r0.data_ptr(), r0.stride(0), r0.stride(1), y_at, H * D, D, s_at, (uint32_t*)ws.data_ptr(), (int32_t)tokens,
                                    (int32_t)H, (int32_t)D, stream_of(r0)),
            "fdb_quant_e4m3_per_head");
    y0 = y.select(0, 0).reshape(a0.sizes()), s0 = scale.select(0, 0);
    if (pair) y1 = y.select(0, 1).reshape(a1.sizes()), s1 = scale.select(0, 1);
  }
  if (!pair) return Py_BuildValue("NN", THPVariable_Wrap(std::move(y0)), THPVariable_Wrap(std::move(s0)));
  return Py_BuildValue("NNNN", THPVariable_Wrap(std::move(y0)), THPVariable_Wrap(std::move(s0)), THPVariable_Wrap(std::move(y1)),
                       THPVariable_Wrap(std::move(s1)));
  END_HANDLE_TH_ERRORS
}

// ---- bounds of a padding mask -----------------------------------------------------------------------------------------
// mask_bounds(mask [B, L], [B, L, L] or [B, 1, L, L] on the GPU) -> (seq_start, seq_len) int32 [B]; None for an element type it
// does not read.
PyObject* py_mask_bounds(PyObject*, PyObject* const* x, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 1, "mask_bounds takes 1 argument");
  const Tensor m = tensor_arg(x[0], "mask");
  const bool real = m.is_floating_point();
  if (!m.is_cuda() || m.is_complex() || m.dim() < 2 || m.dim() > 4 || (real && m.element_size() == 1)) Py_RETURN_NONE;
  const int64_t B = m.size(0), L = m.size(-1);
  if (B < 1 || L < 1 || (m.dim() > 2 && m.size(-2) != L)) Py_RETURN_NONE;
  const int64_t step = m.stride(-1) + (m.dim() > 2 ? m.stride(-2) : 0);  // a square mask's diagonal says which tokens are real
  Tensor start, length;
  {
    const NoGil released;
    const c10::hip::HIPGuard guard(m.get_device());
    const Tensor out = at::empty({2, B}, m.options().dtype(at::kInt));
    int32_t* p = (int32_t*)out.data_ptr();
    check(fdb_mask_bounds(m.data_ptr(), (int32_t)m.element_size(), real ? 1 : 0, m.stride(0), step, (int32_t)B, (int32_t)L, p, p + B, stream_of(m)),
          "fdb_mask_bounds");
    start = out.select(0, 0), length = out.select(0, 1);
  }
  return Py_BuildValue("NN", THPVariable_Wrap(std::move(start)), THPVariable_Wrap(std::move(length)));
  END_HANDLE_TH_ERRORS
}

PyObject* py_register_lut_source(PyObject*, PyObject* fn) {
  Py_INCREF(fn);
  Py_XDECREF(g_lut_source);
  g_lut_source = fn;
  Py_RETURN_NONE;
}

// ---- modules whose calls a fused path takes the place of --------------------------------------------------------------
// untouched(modules, kinds) -> whether every module does what its kind (class, the class's own forward) does, unseen: exactly of
// that class, which nobody has given another forward, no hooks on it, no `forward` of its own, not compiled by itself.  A layer
// asks this of some twenty modules per call; in Python the look-ups took longer than the launch of a short product.
PyObject* py_untouched(PyObject*, PyObject* const* x, Py_ssize_t n) {
  static PyObject* const forward = PyUnicode_InternFromString("forward");
  static PyObject* const compiled = PyUnicode_InternFromString("_compiled_call_impl");
  static PyObject* const hooks[] = {PyUnicode_InternFromString("_forward_hooks"), PyUnicode_InternFromString("_forward_pre_hooks"),
                                    PyUnicode_InternFromString("_backward_hooks"), PyUnicode_InternFromString("_backward_pre_hooks")};
  if (n != 2 || !PyTuple_Check(x[0]) || !PyTuple_Check(x[1]) || PyTuple_GET_SIZE(x[0]) != PyTuple_GET_SIZE(x[1])) {
    PyErr_SetString(PyExc_TypeError, "untouched(modules, kinds) takes two tuples of one length");
    return nullptr;
  }
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(x[0]); ++i) {
    PyObject *m = PyTuple_GET_ITEM(x[0], i), *kind = PyTuple_GET_ITEM(x[1], i);
    if (!PyTuple_Check(kind) || PyTuple_GET_SIZE(kind) != 2) {
      PyErr_SetString(PyExc_TypeError, "untouched: a kind is a pair (class, its forward)");
      return nullptr;
    }
    if ((PyObject*)Py_TYPE(m) != PyTuple_GET_ITEM(kind, 0)) Py_RETURN_FALSE;
    PyObject* f = PyObject_GetAttr((PyObject*)Py_TYPE(m), forward);
    if (!f) return nullptr;
    Py_DECREF(f);   // the class keeps it
    if (f != PyTuple_GET_ITEM(kind, 1)) Py_RETURN_FALSE;
    PyObject* d = PyObject_GenericGetDict(m, nullptr);
    if (!d) return nullptr;
    bool plain = !PyDict_GetItemWithError(d, forward) && !PyDict_GetItemWithError(d, compiled);
    for (PyObject* name : hooks) {
      PyObject* h = PyDict_GetItemWithError(d, name);
      plain = plain && (!h || PyObject_IsTrue(h) == 0);
    }
    Py_DECREF(d);
    if (PyErr_Occurred()) return nullptr;
    if (!plain) Py_RETURN_FALSE;
  }
  Py_RETURN_TRUE;
}

// ---- Memo ---------------------------------------------------------------------------------------------------------
// One remembered value, valid while the tensors it was computed from are the same objects, have not been written in place
// (version counter), still sit in the same storage with the same dtype on the same device (`p.data = x` and `module.to(dtype)`
// swap those under an unchanged object), and `extra` compares equal.  The tensors are held weakly.
// A value belongs to the stream it was computed on, where whatever uses it, and whatever its memory is given to afterwards, comes
// after it; each stream has its own, for the last few streams.  One that is recorded into a graph belongs to that capture: outside
// it nothing has computed it yet, and a graph that took one from outside would keep, replay after replay, what followed from a mask
// or a weight then, in memory that is given back once the program has changed either.
struct Stamp {
  c10::weak_intrusive_ptr<c10::TensorImpl> impl;
  const void* data;
  int64_t version;
  at::ScalarType dtype;
  at::Device device;
};
struct Place {
  int64_t device = -1, stream = 0;
  unsigned long long capture = 0;
  bool operator==(const Place& o) const { return device == o.device && stream == o.stream && capture == o.capture; }
};
struct Remembered {
  Place place;
  std::vector<Stamp> stamps;
  PyObject* extra = nullptr;
  PyObject* value = nullptr;
  Remembered() = default;
  Remembered(const Remembered&) = delete;
  Remembered& operator=(const Remembered&) = delete;
  ~Remembered() {
    Py_XDECREF(extra);
    Py_XDECREF(value);
  }
};
typedef std::vector<std::shared_ptr<Remembered>> MemoState;   // the latest first
constexpr size_t kMostStreams = 4;
struct MemoObject {
  PyObject_HEAD
  MemoState* state;
};

bool tracked(const Tensor& t) { return t.defined() && !t.is_inference(); }  // inference tensors count no versions
bool plain(const Tensor& t) { return t.has_storage(); }
const void* address(const Tensor& t) { return plain(t) ? t.data_ptr() : nullptr; }

Place place_of(PyObject* tensors) {
  Place p;
  if (PyTuple_GET_SIZE(tensors) == 0) return p;
  const Tensor& t = tensor_arg(PyTuple_GET_ITEM(tensors, 0), "tensors");
  if (!t.is_cuda()) return p;
  const auto stream = c10::hip::getCurrentHIPStream(t.get_device());
  p.device = t.get_device();
  p.stream = stream.id();
  if (p.stream != 0) {  // the default stream cannot be captured
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    unsigned long long id = 0;
    const hipError_t e = hipStreamGetCaptureInfo(stream.stream(), &status, &id);
    TORCH_CHECK(e == hipSuccess, "hipStreamGetCaptureInfo failed: ", hipGetErrorString(e));
    if (status != hipStreamCaptureStatusNone) p.capture = id;
  }
  return p;
}

// values whose capture is over, or another one: moved out, to be given back when nothing here is being walked over
MemoState drop_captures(MemoState& all, const Place& now) {
  MemoState gone;
  for (size_t i = all.size(); i-- > 0;)
    if (all[i]->place.capture != 0 && all[i]->place.capture != now.capture) {
      gone.push_back(std::move(all[i]));
      all.erase(all.begin() + i);
    }
  return gone;
}
PyObject* memo_get(PyObject* self, PyObject* const* x, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  MemoState& all = *((MemoObject*)self)->state;
  TORCH_CHECK_TYPE(n >= 1 && n <= 2 && PyTuple_Check(x[0]), "get(tensors, extra=None) takes a tuple of tensors");
  if (all.empty()) Py_RETURN_NONE;
  const Place now = place_of(x[0]);
  const MemoState gone = drop_captures(all, now);
  std::shared_ptr<Remembered> s;
  for (const auto& r : all)
    if (r->place == now) {
      s = r;
      break;
    }
  const Py_ssize_t count = PyTuple_GET_SIZE(x[0]);
  if (!s || (size_t)count != s->stamps.size()) Py_RETURN_NONE;
  PyObject* extra = n > 1 ? x[1] : Py_None;
  if (extra != s->extra) {
    const int same = PyObject_RichCompareBool(extra, s->extra, Py_EQ);
    if (same < 0) throw python_error();
    if (!same) Py_RETURN_NONE;
  }
  for (Py_ssize_t i = 0; i < count; ++i) {
    const Tensor& t = tensor_arg(PyTuple_GET_ITEM(x[0], i), "tensors");
    const Stamp& st = s->stamps[i];
    if (st.impl._unsafe_get_target() != t.unsafeGetTensorImpl() || !tracked(t) || (int64_t)t._version() != st.version || address(t) != st.data ||
        t.scalar_type() != st.dtype || t.device() != st.device)
      Py_RETURN_NONE;
  }
  Py_INCREF(s->value);
  return s->value;
  END_HANDLE_TH_ERRORS
}
PyObject* memo_put(PyObject* self, PyObject* const* x, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n >= 2 && n <= 3 && PyTuple_Check(x[0]), "put(tensors, value, extra=None) takes a tuple of tensors");
  const Py_ssize_t count = PyTuple_GET_SIZE(x[0]);
  const auto fresh = std::make_shared<Remembered>();
  fresh->place = place_of(x[0]);
  bool all_tracked = true;
  for (Py_ssize_t i = 0; i < count && all_tracked; ++i) {
    const Tensor& t = tensor_arg(PyTuple_GET_ITEM(x[0], i), "tensors");
    all_tracked = tracked(t);
    if (all_tracked) fresh->stamps.push_back(Stamp{c10::weak_intrusive_ptr<c10::TensorImpl>(t.getIntrusivePtr()), address(t), (int64_t)t._version(), t.scalar_type(), t.device()});
  }
  MemoState& all = *((MemoObject*)self)->state;
  MemoState gone = drop_captures(all, fresh->place);
  for (size_t i = all.size(); i-- > 0;)
    if (all[i]->place == fresh->place) {
      gone.push_back(std::move(all[i]));
      all.erase(all.begin() + i);
    }
  if (all_tracked) {
    Py_INCREF(fresh->extra = n > 2 ? x[2] : Py_None);
    Py_INCREF(fresh->value = x[1]);
    all.insert(all.begin(), fresh);
    if (all.size() > kMostStreams) {
      gone.push_back(std::move(all.back()));
      all.pop_back();
    }
  }
  Py_INCREF(x[1]);
  return x[1];
  END_HANDLE_TH_ERRORS
}
PyObject* memo_reduce(PyObject* self, PyObject*) {  // copies and pickles of a module start with nothing remembered
  return Py_BuildValue("O()", (PyObject*)Py_TYPE(self));
}
PyObject* memo_new(PyTypeObject* type, PyObject*, PyObject*) {
  MemoObject* m = (MemoObject*)type->tp_alloc(type, 0);
  if (m) m->state = new MemoState();
  return (PyObject*)m;
}
int memo_traverse(PyObject* self, visitproc visit, void* arg) {
  const MemoState* all = ((MemoObject*)self)->state;
  if (all)
    for (const auto& r : *all) {
      if (r.use_count() > 1) continue;   // a call that is running holds it, too
      Py_VISIT(r->extra);
      Py_VISIT(r->value);
    }
  return 0;
}
int memo_gc_clear(PyObject* self) {
  MemoState gone;
  if (MemoState* all = ((MemoObject*)self)->state) gone.swap(*all);
  return 0;
}
void memo_dealloc(PyObject* self) {
  PyObject_GC_UnTrack(self);
  memo_gc_clear(self);
  delete ((MemoObject*)self)->state;
  Py_TYPE(self)->tp_free(self);
}
PyMethodDef memo_methods[] = {
    {"get", (PyCFunction)(void*)memo_get, METH_FASTCALL, "get(tensors, extra=None): the value remembered for these tensors, or None"},
    {"put", (PyCFunction)(void*)memo_put, METH_FASTCALL, "put(tensors, value, extra=None): remembers the value and returns it"},
    {"__reduce__", memo_reduce, METH_NOARGS, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyTypeObject MemoType = {PyVarObject_HEAD_INIT(nullptr, 0)};

PyMethodDef module_methods[] = {
    {"attention_fwd", (PyCFunction)(void*)py_attention_fwd, METH_FASTCALL, nullptr},
    {"attention_node", (PyCFunction)(void*)py_attention_node, METH_FASTCALL, nullptr},
    {"layer_node", (PyCFunction)(void*)py_layer_node, METH_FASTCALL, nullptr},
    {"attention_bwd", (PyCFunction)(void*)py_attention_bwd, METH_FASTCALL, nullptr},
    {"layer_attention", (PyCFunction)(void*)py_layer_attention, METH_FASTCALL, nullptr},
    {"product", (PyCFunction)(void*)py_product, METH_FASTCALL, nullptr},
    {"linear", (PyCFunction)(void*)py_linear, METH_FASTCALL, nullptr},
    {"encoder_layer", (PyCFunction)(void*)py_encoder_layer, METH_FASTCALL, nullptr},
    {"quantize_e4m3", (PyCFunction)(void*)py_quantize, METH_FASTCALL, nullptr},
    {"mask_bounds", (PyCFunction)(void*)py_mask_bounds, METH_FASTCALL, nullptr},
    {"untouched", (PyCFunction)(void*)py_untouched, METH_FASTCALL, nullptr},
    {"register_lut_source", py_register_lut_source, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_native", "Native host path of the operators.", -1, module_methods};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) {
  MemoType.tp_name = "flashdeberta_amd._native.Memo";
  MemoType.tp_basicsize = sizeof(MemoObject);
  MemoType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_GC;
  MemoType.tp_doc = "One remembered value, valid while the tensors it was computed from are unchanged, on the stream it was computed on.";
  MemoType.tp_new = memo_new;
  MemoType.tp_traverse = memo_traverse;
  MemoType.tp_clear = memo_gc_clear;
  MemoType.tp_dealloc = memo_dealloc;
  MemoType.tp_methods = memo_methods;
  if (PyType_Ready(&MemoType) < 0) return nullptr;
  PyObject* m = PyModule_Create(&module_def);
  if (!m) return nullptr;
  Py_INCREF(&MemoType);
  PyModule_AddObject(m, "Memo", (PyObject*)&MemoType);
  return m;
}
