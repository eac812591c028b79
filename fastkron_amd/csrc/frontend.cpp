// The PyTorch front end's host path in native code: from tensors to one library call (fastkron_amd/torch_frontend.py has
// the entry points, the autograd functions and the messages of refused operands).
//
// A product of small operands costs what the host spends on it: in Python the shape rules, three allocations, a dozen
// ctypes objects and the stream look-up took 27 of the 34.5 us of a vector against 8x8 (x) 8x8 (x) 8x8 (now 7 to 7.5 us with
// its kernel of 5 us).  Everything between the Python call and the C API happens here instead; nothing is kept between calls.
// A function returns None for operands that it does not take (the Python side then says why), a fastKronError as a
// whole number where the library refuses the call, and otherwise its tensors; product returns False for a call that is
// to be recorded for gradients.
//
// Rules (reference pyfastkron/fastkronbase.py:104-518): leading dimensions are batches, broadcast between X, the factors
// and Y; neighbouring ones that all operands have alike are one; one dimension is a strided-batched call (stride 0 = shared
// operand), two of which the factors have one a call with both, otherwise the largest is the call's and the others a loop; a
// batch of X against shared factors is more rows of one problem (MKM); transposed views are passed as their buffer.
#include <Python.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>
#include <c10/core/GradMode.h>

#include <cstdint>
#include <mutex>

#include "../../include/fastkron.h"
#include "../../include/fastkron_ext.h"

namespace {

using at::Tensor;
using Dims = c10::SmallVector<int64_t, 8>;

constexpr int kMaxFactors = 64;
constexpr int64_t kMaxCount = UINT32_MAX;                      // rows, batch entries and factor extents are 32-bit numbers in the C API

// Entry points of the library that Python has loaded.
struct Api {
  decltype(&sgemkm) sgemkm_; decltype(&dgemkm) dgemkm_; decltype(&sgekmm) sgekmm_; decltype(&dgekmm) dgekmm_;
  decltype(&sgemkmStridedBatched) sgemkmB; decltype(&dgemkmStridedBatched) dgemkmB;
  decltype(&sgekmmStridedBatched) sgekmmB; decltype(&dgekmmStridedBatched) dgekmmB;
  decltype(&gekmmSizes) sizes; decltype(&fastKronSetStream) setStream;
  decltype(&fastKronProductOuter) productOuter;
  decltype(&fastKronGradSizes) gradSizes; decltype(&fastKronGradForward) gradForward; decltype(&fastKronGradBackwardSteps) gradSteps;
} api;

int64_t prod(at::IntArrayRef d) { int64_t n = 1; for (int64_t v : d) n *= v; return n; }
Dims batchOf(const Tensor& t) { return t.dim() > 2 ? Dims(t.sizes().begin(), t.sizes().end() - 2) : Dims(); }

bool broadcast(const Dims& a, const Dims& b, Dims* out) {
  const size_t n = std::max(a.size(), b.size());
  out->assign(n, 1);
  for (size_t i = 0; i < n; i++) {
    const int64_t x = i < n - a.size() ? 1 : a[i - (n - a.size())], y = i < n - b.size() ? 1 : b[i - (n - b.size())];
    if (x != y && x != 1 && y != 1) return false;
    (*out)[i] = x == 1 ? y : x;
  }
  return true;
}

// X and factors as the library takes them: row-major buffers (the swapped one of a transposed view, op T).
struct Operands {
  bool mkm, vec;                              // vec: X has one dimension
  fastKronOp opX, opF;
  Tensor x, f[kMaxFactors];
  uint32_t N, Ps[kMaxFactors], Qs[kMaxFactors];
  int64_t M, K, L;
  Dims xb, fb, zb, zshape;                    // batch dimensions of X, of the factors and of the result

  void setZShape() {
    zshape = zb;
    zshape.push_back(mkm ? M : L); zshape.push_back(mkm ? L : M);
  }
  bool f64() const { return x.scalar_type() == at::kDouble; }
  // batch of X against shared factors: more rows of the same problem (MKM, X stored row-major)
  bool folds() const {
    return mkm && !zb.empty() && fb.empty() && opX == fastKronOp_N && prod(zb) <= kMaxCount / std::max<int64_t>(M, 1);
  }
  // no entry along an outer batch dimension: a loop of no calls (an innermost dimension of no entries is refused by the call)
  bool noCalls() const { return zb.size() > 1 && prod(at::IntArrayRef(zb.data(), zb.size() - 1)) == 0 && !folds(); }
};

bool usable(const Tensor& t) { return t.defined() && t.is_cuda() && t.layout() == at::kStrided; }

bool swapped(const Tensor& t) { return !t.is_contiguous() && t.dim() >= 2 && t.mT().is_contiguous(); }
Tensor buffer(const Tensor& t, fastKronOp op) { return (op == fastKronOp_T ? t.mT() : t).contiguous(); }

// Shapes and storage only, nothing is copied before all of a call's rules have been looked at (a call that is recorded for
// gradients comes back through the autograd function); ops: the storage to use (0: as the tensors are stored).
bool describe(bool mkm, PyObject* px, PyObject* pfs, int opX, int opF, Operands* o) {
  if (!THPVariable_Check(px) || !(PyList_Check(pfs) || PyTuple_Check(pfs))) return false;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(pfs);
  if (n == 0 || n > kMaxFactors) return false;
  Tensor x = THPVariable_Unpack(px);
  if (!usable(x) || (x.scalar_type() != at::kFloat && x.scalar_type() != at::kDouble) || x.dim() == 0) return false;
  o->mkm = mkm; o->N = (uint32_t)n; o->vec = x.dim() == 1;
  if (o->vec) x = mkm ? x.reshape({1, -1}) : x.reshape({-1, 1});
  bool anyT = false, anyN = false;
  for (Py_ssize_t i = 0; i < n; i++) {
    PyObject* pf = PySequence_Fast_GET_ITEM(pfs, i);
    if (!THPVariable_Check(pf)) return false;
    const Tensor& f = THPVariable_Unpack(pf);
    if (!usable(f) || f.dim() < 2 || f.scalar_type() != x.scalar_type() || f.device() != x.device()) return false;
    if (i && f.sizes().slice(0, f.dim() - 2) != o->f[0].sizes().slice(0, o->f[0].dim() - 2)) return false;
    o->f[i] = f;
    (swapped(f) ? anyT : anyN) = true;
    const int64_t a = f.size(-2), b = f.size(-1);
    if (a == 0 || b == 0 || a > kMaxCount || b > kMaxCount) return false;
    o->Ps[i] = (uint32_t)(mkm ? a : b); o->Qs[i] = (uint32_t)(mkm ? b : a);
  }
  o->fb = batchOf(o->f[0]);
  o->xb = batchOf(x);
  o->M = mkm ? x.size(-2) : x.size(-1); o->K = mkm ? x.size(-1) : x.size(-2);
  if (o->M > kMaxCount) return false;
  int64_t k = 1;
  o->L = 1;
  for (Py_ssize_t i = 0; i < n; i++) { k *= o->Ps[i]; o->L *= o->Qs[i]; }
  if (k != o->K || !broadcast(o->xb, o->fb, &o->zb)) return false;
  o->setZShape();
  o->opX = opX ? (fastKronOp)opX : swapped(x) ? fastKronOp_T : fastKronOp_N;
  o->opF = opF ? (fastKronOp)opF : anyT && !anyN ? fastKronOp_T : fastKronOp_N;      // one op is passed for all factors
  o->x = x;
  return true;
}
// ... and the buffers
void makeBuffers(Operands* o) {
  o->x = buffer(o->x, o->opX);
  for (uint32_t i = 0; i < o->N; i++) o->f[i] = buffer(o->f[i], o->opF);
}

struct Call { fastKronHandle handle; void* stream; };

// handle, stream, mkm: the first arguments of every function
bool callOf(PyObject* const* args, Call* c, bool* mkm) {
  c->handle = (fastKronHandle)PyLong_AsVoidPtr(args[0]);
  c->stream = PyLong_AsVoidPtr(args[1]);
  *mkm = PyObject_IsTrue(args[2]) == 1;
  return !PyErr_Occurred();
}

// While the library runs, without the interpreter's lock: other Python threads go on while it tunes or waits for room in the
// launch queue (they stood still through the 18 ms in which a first call was tuned).  Threads share the default handle and
// each call sets its stream, so one call at a time.  No Python object is touched in its scope.
class LibraryCall {
 public:
  LibraryCall() : thread_(PyEval_SaveThread()) { one().lock(); }
  ~LibraryCall() { one().unlock(); PyEval_RestoreThread(thread_); }
  LibraryCall(const LibraryCall&) = delete;
 private:
  static std::mutex& one() { static std::mutex m; return m; }
  PyThreadState* thread_;
};

PyObject* failed(fastKronError e) { return PyLong_FromLong((long)e); }

fastKronError call(const Call& c, const Operands& o, uint32_t M, const void* x, const void* const* f, void* z, double alpha,
                   double beta, const void* y, void* t1, void* t2) {
  const fastKronBackend B = fastKronBackend_HIP;
  if (o.f64()) {
    if (o.mkm) return api.dgemkm_(c.handle, B, M, o.N, (uint32_t*)o.Ps, (uint32_t*)o.Qs, (double*)x, o.opX, (const double**)f, o.opF, (double*)z,
                                  alpha, beta, (const double*)y, (double*)t1, (double*)t2);
    return api.dgekmm_(c.handle, B, o.N, (uint32_t*)o.Qs, (uint32_t*)o.Ps, M, (const double**)f, o.opF, (double*)x, o.opX, (double*)z, alpha, beta,
                       (const double*)y, (double*)t1, (double*)t2);
  }
  if (o.mkm) return api.sgemkm_(c.handle, B, M, o.N, (uint32_t*)o.Ps, (uint32_t*)o.Qs, (float*)x, o.opX, (const float**)f, o.opF, (float*)z,
                                (float)alpha, (float)beta, (const float*)y, (float*)t1, (float*)t2);
  return api.sgekmm_(c.handle, B, o.N, (uint32_t*)o.Qs, (uint32_t*)o.Ps, M, (const float**)f, o.opF, (float*)x, o.opX, (float*)z, (float)alpha,
                     (float)beta, (const float*)y, (float*)t1, (float*)t2);
}

fastKronError callBatched(const Call& c, const Operands& o, const void* x, uint64_t sx, const void* const* f, uint64_t* sf, void* z,
                          uint64_t sz, double alpha, double beta, uint32_t batch, const void* y, uint64_t sy, void* t1, void* t2) {
  const fastKronBackend B = fastKronBackend_HIP;
  const uint32_t M = (uint32_t)o.M;
  if (o.f64()) {
    if (o.mkm) return api.dgemkmB(c.handle, B, M, o.N, (uint32_t*)o.Ps, (uint32_t*)o.Qs, (double*)x, o.opX, sx, (const double**)f, o.opF, sf,
                                  (double*)z, sz, alpha, beta, batch, (const double*)y, sy, (double*)t1, (double*)t2);
    return api.dgekmmB(c.handle, B, o.N, (uint32_t*)o.Qs, (uint32_t*)o.Ps, M, (const double**)f, o.opF, sf, (double*)x, o.opX, sx, (double*)z, sz,
                       alpha, beta, batch, (const double*)y, sy, (double*)t1, (double*)t2);
  }
  if (o.mkm) return api.sgemkmB(c.handle, B, M, o.N, (uint32_t*)o.Ps, (uint32_t*)o.Qs, (float*)x, o.opX, sx, (const float**)f, o.opF, sf,
                                (float*)z, sz, (float)alpha, (float)beta, batch, (const float*)y, sy, (float*)t1, (float*)t2);
  return api.sgekmmB(c.handle, B, o.N, (uint32_t*)o.Qs, (uint32_t*)o.Ps, M, (const float**)f, o.opF, sf, (float*)x, o.opX, sx, (float*)z, sz,
                     (float)alpha, (float)beta, batch, (const float*)y, sy, (float*)t1, (float*)t2);
}

// product(handle, stream, mkm, x, fs, alpha, beta, y) -> z, or False
PyObject* product(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  Call c; bool mkm;
  if (nargs != 8 || !callOf(args, &c, &mkm)) { if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "product: 8 arguments"); return nullptr; }
  const double alpha = PyFloat_AsDouble(args[5]), beta = PyFloat_AsDouble(args[6]);
  if (PyErr_Occurred()) return nullptr;
  Operands o;
  if (!describe(mkm, args[3], args[4], 0, 0, &o)) Py_RETURN_NONE;
  if (c10::GradMode::is_enabled()) {
    bool wanted = THPVariable_Unpack(args[3]).requires_grad();
    for (uint32_t i = 0; i < o.N; i++) wanted = wanted || THPVariable_Unpack(PySequence_Fast_GET_ITEM(args[4], i)).requires_grad();
    if (wanted) Py_RETURN_FALSE;
  }
  Tensor y;
  Dims yb;
  if (args[7] != Py_None) {
    if (!THPVariable_Check(args[7])) Py_RETURN_NONE;
    y = THPVariable_Unpack(args[7]);
    if (!usable(y) || y.scalar_type() != o.x.scalar_type() || y.device() != o.x.device()) Py_RETURN_NONE;
    if (o.vec && y.dim() == 1) y = mkm ? y.reshape({1, -1}) : y.reshape({-1, 1});
    if (y.dim() < 2 || y.size(-2) != o.zshape[o.zshape.size() - 2] || y.size(-1) != o.zshape.back()) Py_RETURN_NONE;
    yb = batchOf(y);
    Dims both;
    if (!broadcast(yb, o.zb, &both) || both != o.zb) Py_RETURN_NONE;
    y = y.contiguous();
  } else if (beta != 0.0) Py_RETURN_NONE;
  makeBuffers(&o);

  Tensor z = at::empty(o.zshape, o.x.options());
  const size_t es = z.element_size();
  const bool fold = o.folds() && (!y.defined() || yb == o.zb);
  const int64_t M = fold ? o.M * prod(o.zb) : o.M;
  const bool one = fold || o.zb.empty();
  if (!one && o.zb.back() > kMaxCount) return failed(fastKronInvalidKMMProblem);
  size_t ye = 0, te = 0;
  fastKronError e = api.sizes(c.handle, (uint32_t)M, o.N, o.Ps, o.Qs, &ye, &te);
  if (e != fastKronSuccess) return failed(e);
  // more entries in a call than the innermost dimension has only while the temporaries stay small beside the operands (X of
  // (64, 1) entries and factors of (2): two temporaries of 64 entries would be as much as Z again)
  auto room = [&](int64_t entries) { return entries <= o.zb.back() || te * (size_t)entries * es <= (size_t)256 << 20; };
  // batch dimensions as steps of every operand in entries, neighbours merged where all operands go on in one
  struct Dim { int64_t n, x, f, y, z; };
  c10::SmallVector<Dim, 8> dims;
  if (!one) {
    int64_t x = 1, f = 1, s = 1, zz = 1;
    auto step = [](const Dims& b, size_t fromBack, int64_t* run) {
      if (fromBack >= b.size() || b[b.size() - 1 - fromBack] == 1) return (int64_t)0;
      const int64_t r = *run;
      *run *= b[b.size() - 1 - fromBack];
      return r;
    };
    for (size_t i = 0; i < o.zb.size(); i++) {
      const int64_t n = o.zb[o.zb.size() - 1 - i];
      Dim d{n, step(o.xb, i, &x), step(o.fb, i, &f), step(yb, i, &s), zz};
      zz *= n;
      if (!dims.empty() && prod(o.zb) > 0) {
        Dim& in = dims.back();
        if (n == 1) continue;
        if (in.n == 1 && room(n)) { in = d; continue; }
        if (d.x == in.x * in.n && d.f == in.f * in.n && d.y == in.y * in.n && in.n * n <= kMaxCount && room(in.n * n)) { in.n *= n; continue; }
      }
      dims.push_back(d);
    }
  }
  size_t largest = 0;
  for (size_t i = 1; i < dims.size(); i++) if (dims[i].n > dims[largest].n && prod(o.zb) > 0 && dims[i].n <= kMaxCount && room(dims[i].n)) largest = i;
  const int64_t inner = one ? 1 : dims[largest].n;
  // both temporaries in one allocation, each on a 256-byte boundary
  const size_t withF = dims.size() == 2 ? (dims[0].f != 0) + (dims[1].f != 0) : 0;
  const bool both = withF == 1 && prod(o.zb) > 0 && prod(o.zb) <= 65535 && room(prod(o.zb));
  const size_t tn = te * (size_t)(both ? prod(o.zb) : inner), off = (tn * es + 255) / 256 * 256 / es;
  Tensor temp = at::empty({(int64_t)(off + tn)}, o.x.options());
  char* t1 = (char*)temp.data_ptr();
  char* t2 = t1 ? t1 + off * es : nullptr;
  auto run = [&]() -> fastKronError {
    LibraryCall unlocked;
    fastKronError e = api.setStream(c.handle, fastKronBackend_HIP, &c.stream);
    if (e != fastKronSuccess) return e;
    const void* f[kMaxFactors];
    if (one) {
      for (uint32_t i = 0; i < o.N; i++) f[i] = o.f[i].data_ptr();
      return call(c, o, (uint32_t)M, o.x.data_ptr(), f, z.data_ptr(), alpha, beta, y.defined() ? y.data_ptr() : nullptr, t1, t2);
    }
    const int64_t xblk = o.M * o.K, zblk = o.M * o.L;
    if (both) {
      const Dim& in = dims[dims[0].f != 0 ? 0 : 1], & out = dims[dims[0].f != 0 ? 1 : 0];
      const uint64_t sx[2] = {(uint64_t)(out.x * xblk), (uint64_t)(in.x * xblk)}, sz[2] = {(uint64_t)(out.z * zblk), (uint64_t)(in.z * zblk)};
      const uint64_t sy[2] = {(uint64_t)(out.y * zblk), (uint64_t)(in.y * zblk)};
      const uint32_t count[2] = {(uint32_t)out.n, (uint32_t)in.n};
      for (uint32_t i = 0; i < o.N; i++) f[i] = o.f[i].data_ptr();
      return api.productOuter(c.handle, mkm, o.f64(), (uint32_t)o.M, o.N, o.Ps, o.Qs, o.x.data_ptr(), o.opX, sx, f, o.opF, z.data_ptr(), sz, alpha,
                              beta, count, y.defined() ? y.data_ptr() : nullptr, sy, t1, t2);
    }
    const Dim in = dims[largest];
    uint64_t sf[kMaxFactors];
    for (uint32_t i = 0; i < o.N; i++) sf[i] = (uint64_t)in.f * o.Ps[i] * o.Qs[i];
    int64_t outer = 1;
    for (size_t i = 0; i < dims.size(); i++) if (i != largest) outer *= dims[i].n;
    for (int64_t lin = 0; lin < outer; lin++) {
      int64_t rem = lin, xo = 0, fo = 0, yo = 0, zo = 0;
      for (size_t i = 0; i < dims.size(); i++) {
        if (i == largest) continue;
        const int64_t k = rem % dims[i].n;
        rem /= dims[i].n;
        xo += k * dims[i].x; fo += k * dims[i].f; yo += k * dims[i].y; zo += k * dims[i].z;
      }
      for (uint32_t i = 0; i < o.N; i++) f[i] = (char*)o.f[i].data_ptr() + (size_t)fo * o.Ps[i] * o.Qs[i] * es;
      e = callBatched(c, o, (char*)o.x.data_ptr() + (size_t)(xo * xblk) * es, in.x * xblk, f, sf, (char*)z.data_ptr() + (size_t)(zo * zblk) * es,
                      in.z * zblk, alpha, beta, (uint32_t)inner, y.defined() ? (char*)y.data_ptr() + (size_t)(yo * zblk) * es : nullptr,
                      y.defined() ? in.y * zblk : 0, t1, t2);
      if (e != fastKronSuccess) return e;
    }
    return e;
  };
  e = run();
  if (e != fastKronSuccess) return failed(e);
  if (o.vec) {
    Dims s = o.zb;
    s.push_back(-1);
    z = z.reshape(s);
  }
  return THPVariable_Wrap(std::move(z));
  END_HANDLE_TH_ERRORS
}

// The operands of a differentiated call as the library's gradient functions take them: batches flattened to one dimension
// of nb entries; an operand that is broadcast over a part of it only is expanded first.
struct GradOperands {
  bool perBatch; int64_t nb; uint64_t strideX; const void* f[kMaxFactors];
};
bool gradOperands(Operands* o, GradOperands* g) {
  g->nb = prod(o->zb);
  if (g->nb > kMaxCount) return false;
  makeBuffers(o);
  const int64_t nx = prod(o->xb), nf = prod(o->fb);
  g->perBatch = nf > 1;
  g->strideX = nx > 1 ? (uint64_t)(o->M * o->K) : 0;
  auto expand = [&](Tensor& t) {
    Dims s = o->zb;
    s.push_back(t.size(-2)); s.push_back(t.size(-1));
    t = t.expand(s).contiguous();
  };
  if (nx != 1 && nx != g->nb) expand(o->x);
  if (nf != 1 && nf != g->nb) for (uint32_t i = 0; i < o->N; i++) expand(o->f[i]);
  for (uint32_t i = 0; i < o->N; i++) g->f[i] = o->f[i].data_ptr();
  return true;
}

// The kernels know a tensor by its address only: one that comes back from a saved-tensors hook, or as a gradient, of another
// type or on another device would be read beyond its end or not be there at all.
void requireLike(const Tensor& t, const Tensor& x, const char* what) {
  TORCH_CHECK(usable(t) && t.device() == x.device() && t.scalar_type() == x.scalar_type(), "Expected ", what, " to be ", x.scalar_type(),
              " on ", x.device(), " like the operands, but it is ", t.defined() ? t.toString() : std::string("undefined"));
}

// grad_forward(handle, stream, mkm, x, fs) -> (z, kept for the backward pass, storage of X, of the factors)
PyObject* gradForward(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  Call c; bool mkm;
  if (nargs != 5 || !callOf(args, &c, &mkm)) { if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "grad_forward: 5 arguments"); return nullptr; }
  Operands o; GradOperands g;
  if (!describe(mkm, args[3], args[4], 0, 0, &o)) Py_RETURN_NONE;
  if (o.noCalls() && !o.vec)
    return Py_BuildValue("NNii", THPVariable_Wrap(at::empty(o.zshape, o.x.options())), THPVariable_Wrap(at::empty({0}, o.x.options())), (int)o.opX, (int)o.opF);
  if (!gradOperands(&o, &g)) Py_RETURN_NONE;
  size_t save = 0, work = 0;
  fastKronError e = api.gradSizes(c.handle, mkm, o.f64(), (uint32_t)o.M, o.N, o.Ps, o.Qs, o.opX, g.strideX, g.perBatch, (uint32_t)g.nb, &save, &work);
  if (e != fastKronSuccess) return failed(e);
  Tensor z = at::empty(o.zshape, o.x.options()), kept = at::empty({(int64_t)save}, o.x.options());
  {
    LibraryCall unlocked;
    e = api.setStream(c.handle, fastKronBackend_HIP, &c.stream);
    if (e == fastKronSuccess)
      e = api.gradForward(c.handle, mkm, o.f64(), (uint32_t)o.M, o.N, o.Ps, o.Qs, o.x.data_ptr(), o.opX, g.strideX, g.f, o.opF, g.perBatch,
                          (uint32_t)g.nb, z.data_ptr(), kept.data_ptr());
  }
  if (e != fastKronSuccess) return failed(e);
  if (o.vec) {
    Dims s = o.zb;
    s.push_back(-1);
    z = z.reshape(s);
  }
  return Py_BuildValue("NNii", THPVariable_Wrap(std::move(z)), THPVariable_Wrap(std::move(kept)), (int)o.opX, (int)o.opF);
  END_HANDLE_TH_ERRORS
}

// Where the gradient of a step's input is PyTorch's product instead of the library's backward kernel, which takes 64 rows of
// the factor per workgroup with all of Q contracted in one chain of loads, reads the gradient again for every 64 rows, and has
// one workgroup per CU (or the factor in memory, from Q = 273 in fp64 on) for wide factors.  Measured, the launch alone
// against the product with its copies and its host time, of which some 10 us are the share of a call from here, in us:
//   Q > 384 (fp64 272): 64x4096, 15 rows fp32 485 / 26, 16x1024, 3906 columns 79 / 34, 1024x1024, 3906 rows fp32 555 / 64 and
//   244 rows fp64 203 / 34, 512x512, 122 columns fp32 37 / 32, 64x512, 122 rows 59 / 33 (the smallest measured);
//   otherwise P or Q above 128 from 2^27 multiply-adds on: 256x256, 15625 columns fp32 70 / 34, 224x224, 17857 rows fp32
//   94 / 28, 160x160, 12500 rows fp64 84 / 24; below, the kernel: 384x384, 162 columns fp32 16 / 31, 256x256, 1953 columns
//   fp32 11 / 34, 160x160, 3125 rows 26 / 25, 224x224, 1116 columns fp64 33 / 21.
// Up to 128 the kernel's launches for both gradients are never behind in all.  The gradient of the factor is the kernel's
// everywhere, also where the product is up to 1.5 times faster (512x512 and more, fp32 columns): its sums are 2 to 7 times
// closer to 64-bit ones.
bool wideStep(const Operands& o, uint32_t i, int64_t rows) {
  const int64_t P = o.Ps[i], Q = o.Qs[i];
  return std::max(P, Q) > 128 && (Q > (o.f64() ? 272 : 384) || (double)rows * P * Q >= 134217728.0);
}

// The gradient of the input of step i (S slices of P): g M x (Q, S) -> M x (S, P) for MKM, (Q, S) x M -> (S, P) x M for KMM.
Tensor wideInputGradient(const Operands& o, const GradOperands& gr, uint32_t i, int64_t S, const Tensor& g) {
  const int64_t P = o.Ps[i], Q = o.Qs[i], M = o.M, nb = gr.nb;
  const bool pMajor = o.mkm == (o.opF == fastKronOp_N);                  // stored P x Q, else Q x P
  const Tensor f = gr.perBatch ? (pMajor ? o.f[i].view({nb, P, Q}).mT() : o.f[i].view({nb, Q, P}))           // Q x P
                               : (pMajor ? o.f[i].view({P, Q}).t() : o.f[i].view({Q, P}));
  if (o.mkm || M == 1) {
    const Tensor a = g.view({nb, M, Q, S}).transpose(2, 3);
    return gr.perBatch ? at::bmm(a.reshape({nb, M * S, Q}), f) : at::mm(a.reshape({nb * M * S, Q}), f);
  }
  const Tensor a = g.view({nb, Q, S * M});
  const Tensor r = gr.perBatch || nb > 1 ? at::bmm(gr.perBatch ? f.mT() : f.t().expand({nb, P, Q}), a) : at::mm(f.t(), a[0]);
  return r.view({nb, P, S, M}).transpose(1, 2).contiguous();
}

// grad_backward(handle, stream, mkm, x, fs, opX, opF, grad of z, kept, need x, need fs) -> (grad of x, of every factor)
PyObject* gradBackward(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  Call c; bool mkm;
  if (nargs != 11 || !callOf(args, &c, &mkm)) { if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "grad_backward: 11 arguments"); return nullptr; }
  const long opX = PyLong_AsLong(args[5]), opF = PyLong_AsLong(args[6]);
  if (PyErr_Occurred()) return nullptr;
  Operands o; GradOperands g;
  // (the storage of the forward pass: what was kept depends on it, also if the operands come back stored another way)
  if (!THPVariable_Check(args[7]) || !THPVariable_Check(args[8]) || !PyTuple_Check(args[10]) ||
      !describe(mkm, args[3], args[4], (int)opX, (int)opF, &o) || PyTuple_GET_SIZE(args[10]) != (Py_ssize_t)o.N) Py_RETURN_NONE;
  const bool needX = PyObject_IsTrue(args[9]) == 1;
  auto needF = [&](uint32_t i) { return PyObject_IsTrue(PyTuple_GET_ITEM(args[10], i)) == 1; };
  if (o.noCalls()) {
    PyObject* out = PyTuple_New(1 + (Py_ssize_t)o.N);
    for (uint32_t i = 0; out && i <= o.N; i++) {
      const Tensor& t = THPVariable_Unpack(i ? PySequence_Fast_GET_ITEM(args[4], i - 1) : args[3]);
      if (i ? needF(i - 1) : needX) PyTuple_SET_ITEM(out, i, THPVariable_Wrap(at::zeros(t.sizes(), o.x.options())));
      else { Py_INCREF(Py_None); PyTuple_SET_ITEM(out, i, Py_None); }
    }
    return out;
  }
  if (!gradOperands(&o, &g)) Py_RETURN_NONE;
  requireLike(THPVariable_Unpack(args[7]), o.x, "the gradient");
  requireLike(THPVariable_Unpack(args[8]), o.x, "the buffer kept by the forward pass");
  const Tensor gz = THPVariable_Unpack(args[7]).contiguous(), kept = THPVariable_Unpack(args[8]).contiguous();
  size_t save = 0, work = 0;
  fastKronError e = api.gradSizes(c.handle, mkm, o.f64(), (uint32_t)o.M, o.N, o.Ps, o.Qs, o.opX, g.strideX, g.perBatch, (uint32_t)g.nb, &save, &work);
  if (e != fastKronSuccess) return failed(e);
  TORCH_CHECK(gz.numel() == prod(o.zshape), "Expected a gradient of ", prod(o.zshape), " elements, got ", gz.numel());
  TORCH_CHECK(kept.numel() == (int64_t)save, "Expected a buffer of ", save, " elements from the forward pass, got ", kept.numel());
  Tensor gx, gf[kMaxFactors];
  void* gfp[kMaxFactors];
  Dims xs = o.zb;
  xs.push_back(mkm ? o.M : o.K); xs.push_back(mkm ? o.K : o.M);
  for (uint32_t i = 0; i < o.N; i++) {
    gfp[i] = nullptr;
    if (!needF(i)) continue;
    Dims s = g.perBatch ? o.zb : Dims();
    s.push_back(mkm ? o.Ps[i] : o.Qs[i]); s.push_back(mkm ? o.Qs[i] : o.Ps[i]);
    gf[i] = at::empty(s, o.x.options());
    gfp[i] = gf[i].data_ptr();
  }
  const Tensor scratch = at::empty({(int64_t)work}, o.x.options());
  auto steps = [&](uint32_t first, uint32_t last, const Tensor& gOut, const Tensor& gIn) {
    LibraryCall unlocked;
    fastKronError r = api.setStream(c.handle, fastKronBackend_HIP, &c.stream);
    if (r == fastKronSuccess)
      r = api.gradSteps(c.handle, mkm, o.f64(), (uint32_t)o.M, o.N, o.Ps, o.Qs, o.x.data_ptr(), o.opX, g.strideX, g.f, o.opF, g.perBatch,
                        (uint32_t)g.nb, first, last, gOut.data_ptr(), kept.data_ptr(), gIn.defined() ? gIn.data_ptr() : nullptr, gfp, scratch.data_ptr());
    return r;
  };
  // columns behind step i, and whether the gradient of its input is needed
  int64_t cols = o.L;
  uint32_t lastWanted = 0;
  for (uint32_t i = 0; i < o.N; i++) if (gfp[i]) lastWanted = i;
  auto inputWanted = [&](uint32_t i) { return i + 1 == o.N ? needX : i < lastWanted || needX; };
  auto wide = [&](uint32_t i, int64_t k) { return inputWanted(i) && wideStep(o, i, g.nb * o.M * (k / o.Qs[i])); };
  Tensor gNow = gz;
  for (uint32_t i = 0; i < o.N && (i <= lastWanted || needX);) {
    uint32_t last = i;
    int64_t k = cols / o.Qs[i] * o.Ps[i];                                // columns of the input of step `last`
    const bool product = wide(i, cols);
    if (!product) for (; last + 1 < o.N && !wide(last + 1, k); last++) k = k / o.Qs[last + 1] * o.Ps[last + 1];
    Tensor gIn;
    if (!product && inputWanted(last)) {
      gIn = last + 1 == o.N ? at::empty(xs, o.x.options()) : at::empty({g.nb * o.M * k}, o.x.options());
    }
    e = steps(i, last, gNow, gIn);
    if (e != fastKronSuccess) return failed(e);
    if (product) gIn = wideInputGradient(o, g, i, cols / o.Qs[i], gNow);
    gNow = gIn; cols = k; i = last + 1;
  }
  if (needX) gx = gNow.sizes() == at::IntArrayRef(xs) ? gNow : gNow.view(xs);
  PyObject* out = PyTuple_New(1 + (Py_ssize_t)o.N);
  if (!out) return nullptr;
  auto put = [&](Py_ssize_t at, Tensor t) {
    if (!t.defined()) { Py_INCREF(Py_None); PyTuple_SET_ITEM(out, at, Py_None); }
    else PyTuple_SET_ITEM(out, at, THPVariable_Wrap(std::move(t)));
  };
  // gradients are summed over the dimensions that were broadcast
  if (needX) {
    const Tensor& x = THPVariable_Unpack(args[3]);
    gx = o.vec ? gx.sum_to_size({xs[xs.size() - 2], xs.back()}).reshape(x.sizes()) : gx.sizes() == x.sizes() ? gx : gx.sum_to_size(x.sizes());
  }
  put(0, needX ? gx : Tensor());
  for (uint32_t i = 0; i < o.N; i++) {
    const Tensor& f = THPVariable_Unpack(PySequence_Fast_GET_ITEM(args[4], i));
    if (gf[i].defined() && gf[i].sizes() != f.sizes()) gf[i] = g.perBatch ? gf[i].sum_to_size(f.sizes()) : gf[i].reshape(f.sizes());
    put(1 + i, gf[i]);
  }
  return out;
  END_HANDLE_TH_ERRORS
}

// batched(tensor): under vmap, old or new style, a tensor has no address to pass on
PyObject* batched(PyObject*, PyObject* t) {
  if (!THPVariable_Check(t)) Py_RETURN_FALSE;
  const c10::DispatchKeySet keys = THPVariable_Unpack(t).key_set();
  return PyBool_FromLong(keys.has(c10::DispatchKey::Batched) || keys.has(c10::DispatchKey::FuncTorchBatched));
}

// use(addresses of the entry points, in the order of Api)
PyObject* use(PyObject*, PyObject* addresses) {
  void* a[sizeof(Api) / sizeof(void*)];
  constexpr Py_ssize_t n = sizeof(Api) / sizeof(void*);
  if (!PyTuple_Check(addresses) || PyTuple_GET_SIZE(addresses) != n) { PyErr_SetString(PyExc_TypeError, "use: a tuple of addresses"); return nullptr; }
  for (Py_ssize_t i = 0; i < n; i++) a[i] = PyLong_AsVoidPtr(PyTuple_GET_ITEM(addresses, i));
  if (PyErr_Occurred()) return nullptr;
  memcpy((void*)&api, a, sizeof(api));
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"use", (PyCFunction)use, METH_O, nullptr},
    {"batched", (PyCFunction)batched, METH_O, nullptr},
    {"product", (PyCFunction)(void (*)(void))product, METH_FASTCALL, nullptr},
    {"grad_forward", (PyCFunction)(void (*)(void))gradForward, METH_FASTCALL, nullptr},
    {"grad_backward", (PyCFunction)(void (*)(void))gradBackward, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_frontend", nullptr, -1, methods};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject* PyInit__frontend(void) { return PyModule_Create(&module); }
