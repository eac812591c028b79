// Gradients of a GeMKM / GeKMM: a forward pass that keeps every step's input and a backward pass that goes through the
// steps in the opposite order, one launch per step for the gradients of the step's input and of its factor
// (kernels/gradient_mfma.hip), one launch that adds the partial sums of all factors.
//
// Adjacent small factors are replaced by their Kronecker product first (exact algebra), so that a chain of n small
// factors takes fewer passes over the data; the gradients of the product's sources follow from its own gradient
// (one small launch for all of them).
// The reference chains PyTorch matmuls through the intermediates of its forward family, one factor at a time
// (reference pyfastkron/fastkrontorch.py:160-217).
#include "handle.h"

#include <algorithm>
#include <cstring>

#include "kernels/gradient.h"
#include "kernels/launch.h"

namespace fk {

namespace {

constexpr uint64_t kMaxRows = (1ull << 31) - 16;       // rows per launch of the step kernel
constexpr uint32_t kMaxGridBatch = 65535;

size_t roundUp(size_t v) { return (v + 63) & ~(size_t)63; }       // elements: 256-byte (fp32) boundaries and better

// The chain as the two passes run it.
struct GradPlan {
  KronProblem q;                    // merged chain, MKM or KMM, op(X) = N; F, X, Z, inter not set
  uint32_t lo[kMaxFactors], hi[kMaxFactors];      // sources of factor g of q
  bool pMajor;                      // storage of the sources: element (p, q) at p*Q + q
  bool outTransposed;               // gradients of the factors are Q x P (KMM)
  bool copyX;                       // op(X) = T: X is copied transposed
  uint32_t xBatch;                  // entries of that copy
  // offsets into `save`, in elements
  size_t saveX, saveF[kMaxFactors], saveI[kMaxFactors], saveTotal;
  // offsets into `work`
  size_t workG[2], workP[kMaxFactors], workD[kMaxFactors], workTotal;
  uint32_t parts[kMaxFactors];      // partial sums of factor g per batch entry
};

// Row ranges of at most kMaxRows of a step: calls f(first o, count of o, first t, count of t).
template <typename F> void forRowChunks(uint64_t O, uint64_t Tn, F f) {
  if (Tn > kMaxRows) {
    for (uint64_t o = 0; o < O; o++)
      for (uint64_t t = 0; t < Tn; t += kMaxRows) f(o, (uint64_t)1, t, std::min(kMaxRows, Tn - t));
    return;
  }
  const uint64_t per = std::max<uint64_t>(1, kMaxRows / Tn);
  for (uint64_t o = 0; o < O; o += per) f(o, std::min(per, O - o), (uint64_t)0, Tn);
}

struct StepShape { uint64_t O, Tn; };               // rows u = o*Tn + t
StepShape stepShape(const KronProblem& q, uint32_t g) {
  const uint64_t S = q.colsBefore(g) / q.P[g];
  return q.mm == MMType::MKM ? StepShape{q.M, S} : StepShape{S, q.M};
}

// Estimated seconds of the forward and backward launches of one factor of P x Q on `rows` rows: bytes at 6 TB/s; the
// matrix instructions of both passes (4 + 8 per 16x16 block of the factor and 16 rows; 32 cycles each in fp32, about
// 100 measured for the fp64 form) on 1024 SIMDs at 2.4 GHz; and what the launches take however few rows there are, 10 us
// and the chain of one wave's tile (64x64: 5 us in fp32, 8 in fp64).  Measured, small chains of 8x8: 11 us per factor,
// as pairs of 64x64 17 us in fp32 and 21 to 30 in fp64, and 14 us for forming the products and splitting their gradients.
double stepCost(uint64_t rows, uint32_t P, uint32_t Q, DType dt) {
  const double bytes = (double)rows * (3.0 * P + 2.0 * Q) * (double)dtypeSize(dt);
  const uint32_t big = std::max(P, Q), zb = big <= 16 ? 1 : big <= 32 ? 2 : 4;      // the kernel's block of the factor
  const double blocks = (double)((P + 16 * zb - 1) / (16 * zb)) * (double)((Q + 16 * zb - 1) / (16 * zb)) * zb * zb;
  const double cycles = (double)rows / 16.0 * blocks * 12.0 * (dt == DType::F32 ? 32.0 : 100.0);
  return bytes / 6e12 + cycles / (1024.0 * 2.4e9) + 10e-6 + (dt == DType::F32 ? 5e-6 : 8e-6) * zb * zb / 16.0;
}

// Groups of adjacent factors with the least estimated time; a group of several factors becomes one of at most 64x64.
void groupFactors(const KronProblem& p, GradPlan* gp) {
  const uint32_t N = p.N;
  double best[kMaxFactors + 1];
  uint32_t from[kMaxFactors + 1];
  best[0] = 0;
  for (uint32_t end = 1; end <= N; end++) {
    best[end] = 1e300;
    uint64_t P = 1, Q = 1;
    const uint64_t cols = p.colsBefore(end - 1);
    for (uint32_t lo = end; lo-- > 0;) {
      P *= p.P[lo]; Q *= p.Q[lo];
      const uint32_t n = end - lo;
      if (n > 1 && (P > 64 || Q > 64 || n > kMaxMergeSources)) break;
      const double c = best[lo] + stepCost((uint64_t)p.M * p.batch * (cols / P), (uint32_t)P, (uint32_t)Q, p.dt);
      if (c < best[end]) { best[end] = c; from[end] = lo; }
    }
  }
  double plain = 0;
  for (uint32_t i = 0; i < N; i++) plain += stepCost((uint64_t)p.M * p.batch * (p.colsBefore(i) / p.P[i]), p.P[i], p.Q[i], p.dt);
  // Forming the products and splitting their gradients are two more launches, 14 us together.  A program that goes through
  // autograd spends about 75 us of host time on the two passes and 3.6 us per launch besides, on which short launches
  // wait: the longer of the two decides (dgekmm 8x8^5 x 16: plain, 11 launches, 70 us on the device, 130 us a pass;
  // merged, 9 launches, 80 and 123 us).
  uint32_t groups = 0;
  for (uint32_t end = N; end > 0; end = from[end]) groups++;
  auto pass = [](double device, uint32_t launches) { return std::max(device, 75e-6 + 3.6e-6 * launches); };
  const bool merge = groups < N && pass(best[N] + 14e-6, 2 * groups + 3) < pass(plain, 2 * N + 1);
  uint32_t n = 0;
  for (uint32_t end = N; end > 0; n++) {
    const uint32_t lo = merge ? from[end] : end - 1;
    gp->lo[n] = lo; gp->hi[n] = end - 1;
    end = lo;
  }
  std::reverse(gp->lo, gp->lo + n);
  std::reverse(gp->hi, gp->hi + n);
  KronProblem& q = gp->q;
  q.N = n;
  for (uint32_t g = 0; g < n; g++) {
    q.P[g] = q.Q[g] = 1;
    for (uint32_t i = gp->lo[g]; i <= gp->hi[g]; i++) { q.P[g] *= p.P[i]; q.Q[g] *= p.Q[i]; }
  }
}

fastKronError makePlan(const Handle::GradProblem& p, GradPlan* gp) {
  if (p.N == 0 || p.N > kMaxFactors || p.M == 0 || p.batch == 0 || !p.P || !p.Q) return fastKronInvalidKMMProblem;
  KronProblem& q = gp->q;
  q = KronProblem{};
  q.mm = p.mm; q.dt = p.dt; q.M = p.M; q.N = p.N; q.batch = p.batch;
  for (uint32_t i = 0; i < p.N; i++) {
    if (p.P[i] == 0 || p.Q[i] == 0) return fastKronInvalidKMMProblem;
    q.P[i] = p.P[i]; q.Q[i] = p.Q[i];
  }
  q.opX = fastKronOp_N; q.opF = p.opF;
  gp->pMajor = (p.mm == MMType::MKM) == (p.opF == fastKronOp_N);
  gp->outTransposed = p.mm == MMType::KMM;
  gp->copyX = p.opX == fastKronOp_T && p.M > 1;
  gp->xBatch = (p.batch > 1 && p.strideX != 0) ? p.batch : 1;
  if (q.mm == MMType::KMM && q.M == 1) {
    // a single column is the MKM of the same vector with transposed factors
    q.mm = MMType::MKM;
    q.opF = p.opF == fastKronOp_N ? fastKronOp_T : fastKronOp_N;
  }
  const uint64_t K = q.K();
  // batches against shared factors are more rows of one problem (MKM)
  if (q.mm == MMType::MKM && q.batch > 1 && !p.perBatchF && p.strideX != 0 && (p.strideX == q.M * K || gp->copyX) &&
      (uint64_t)q.M * q.batch < (1ull << 32)) {
    q.M *= q.batch; q.batch = 1;
  }
  const KronProblem single = q;
  groupFactors(single, gp);
  const size_t nb = q.batch;
  size_t off = 0;
  auto take = [&](size_t elems) { const size_t o = off; off += roundUp(elems); return o; };
  gp->saveX = gp->copyX ? take((size_t)gp->xBatch * p.M * K) : 0;
  for (uint32_t g = 0; g < q.N; g++)
    gp->saveF[g] = gp->lo[g] < gp->hi[g] ? take((p.perBatchF ? nb : 1) * (size_t)q.P[g] * q.Q[g]) : 0;
  for (uint32_t g = 1; g < q.N; g++) gp->saveI[g] = take(nb * q.M * q.colsAfter(g));      // output of step g
  gp->saveTotal = off;
  off = 0;
  size_t widest = 0;
  for (uint32_t g = 0; g + 1 < q.N; g++) widest = std::max<size_t>(widest, q.colsBefore(g));
  for (int i = 0; i < 2; i++) gp->workG[i] = q.N > 1u + i ? take(nb * q.M * widest) : 0;
  for (uint32_t g = 0; g < q.N; g++) {
    const StepShape s = stepShape(q, g);
    uint32_t parts = 0;
    forRowChunks(s.O, s.Tn, [&](uint64_t, uint64_t on, uint64_t, uint64_t tn) { parts += gradWorkgroups(q.P[g], q.Q[g], on * tn, q.batch); });
    gp->parts[g] = parts;
    gp->workP[g] = take(nb * parts * q.P[g] * q.Q[g]);
    gp->workD[g] = gp->lo[g] < gp->hi[g] ? take((p.perBatchF ? nb : 1) * (size_t)q.P[g] * q.Q[g]) : 0;
  }
  gp->workTotal = off;
  return fastKronSuccess;
}

// Sources of merged factor g, as the merging kernel reads them.
void mergeGroupOf(const Handle::GradProblem& p, const GradPlan& gp, uint32_t g, MergeGroup* mg) {
  mg->count = gp.hi[g] - gp.lo[g] + 1;
  for (uint32_t j = 0; j < mg->count; j++) {
    const uint32_t fi = gp.lo[g] + j;
    mg->src[j] = p.F[fi]; mg->p[j] = p.P[fi]; mg->q[j] = p.Q[fi];
    mg->sp[j] = gp.pMajor ? (int64_t)p.Q[fi] : 1;
    mg->sq[j] = gp.pMajor ? 1 : (int64_t)p.P[fi];
  }
}

}  // namespace

fastKronError Handle::gradSizes(const GradProblem& p, size_t* saveElems, size_t* workElems) const {
  if (!saveElems || !workElems) return fastKronInvalidArgument;
  GradPlan gp;
  fastKronError e = makePlan(p, &gp);
  if (e != fastKronSuccess) return e;
  *saveElems = gp.saveTotal; *workElems = gp.workTotal;
  return fastKronSuccess;
}

fastKronError Handle::gradForward(const GradProblem& p, void* Z, void* save) {
  if (!Z || !p.X || !p.F) return fastKronInvalidArgument;
  for (uint32_t i = 0; i < p.N; i++) if (!p.F[i]) return fastKronInvalidKMMProblem;
  GradPlan gp;
  fastKronError e = makePlan(p, &gp);
  if (e != fastKronSuccess) return e;
  if (gp.saveTotal && !save) return fastKronInvalidArgument;
  e = ensureDevice();
  if (e != fastKronSuccess) return e;
  launchLog_.clear();
  const size_t es = dtypeSize(p.dt);
  char* sv = (char*)save;
  KronProblem q = gp.q;
  q.X = p.X; q.strideX = q.batch > 1 ? p.strideX : 0;
  if (gp.copyX) {
    KronProblem t{};
    t.mm = p.mm; t.dt = p.dt; t.M = p.M; t.N = p.N; t.batch = p.batch; t.X = p.X; t.strideX = p.strideX;
    for (uint32_t i = 0; i < p.N; i++) { t.P[i] = p.P[i]; t.Q[i] = p.Q[i]; }
    void* xt = sv + gp.saveX * es;
    if (launchTransposeX(t, xt, (uint64_t)p.M * t.K()) != hipSuccess) return fastKronInvalidArgument;
    q.X = xt; q.strideX = q.batch > 1 && gp.xBatch > 1 ? (uint64_t)p.M * t.K() : 0;
    q.xJustWritten = true;
  }
  MergeArgs ma{};
  ma.batch = p.perBatchF ? q.batch : 1;
  auto flush = [&]() { const hipError_t he = ma.groups ? launchMergeFactors(ma, p.dt, stream_) : hipSuccess; ma.groups = 0; return he; };
  for (uint32_t g = 0; g < q.N; g++) {
    const size_t pq = (size_t)q.P[g] * q.Q[g];
    q.strideF[g] = p.perBatchF && q.batch > 1 ? pq : 0;
    q.F[g] = p.F[gp.lo[g]];
    if (gp.lo[g] == gp.hi[g]) continue;
    MergeGroup& mg = ma.g[ma.groups++];
    mergeGroupOf(p, gp, g, &mg);
    mg.dst = sv + gp.saveF[g] * es;
    mg.dsp = gp.pMajor ? (int64_t)q.Q[g] : 1;
    mg.dsq = gp.pMajor ? 1 : (int64_t)q.P[g];
    q.F[g] = mg.dst;
    if (ma.groups == kMaxMergeGroups && flush() != hipSuccess) return fastKronInvalidArgument;
  }
  if (flush() != hipSuccess) return fastKronInvalidArgument;
  q.forward = true; q.strided = q.batch > 1; q.haveStrideInter = true;
  for (uint32_t g = 1; g < q.N; g++) {
    q.inter[g - 1] = sv + gp.saveI[g] * es;
    q.strideInter[g - 1] = (uint64_t)q.M * q.colsAfter(g);
  }
  q.Z = Z; q.strideZ = q.batch > 1 ? (uint64_t)q.M * q.L() : 0;
  q.alpha = 1.0; q.beta = 0.0;
  callWs_ = false;
  return runOnline(q, nullptr, nullptr, nullptr);
}

fastKronError Handle::gradBackward(const GradProblem& p, const void* gZ, void* save, void* gX, void* const* gF, void* work) {
  if (!gZ || !p.X || !p.F || !gF) return fastKronInvalidArgument;
  for (uint32_t i = 0; i < p.N; i++) if (!p.F[i]) return fastKronInvalidKMMProblem;
  GradPlan gp;
  fastKronError e = makePlan(p, &gp);
  if (e != fastKronSuccess) return e;
  if ((gp.saveTotal && !save) || (gp.workTotal && !work)) return fastKronInvalidArgument;
  e = ensureDevice();
  if (e != fastKronSuccess) return e;
  const KronProblem& q = gp.q;
  const size_t es = dtypeSize(p.dt);
  const uint32_t ve = (uint32_t)(16 / es);
  char* sv = (char*)save;
  char* wk = (char*)work;
  const bool mkm = q.mm == MMType::MKM;
  // the last factor (in chain order) whose gradient is wanted: nothing behind it is computed unless gX is
  int lastWanted = -1;
  bool wanted[kMaxFactors];
  for (uint32_t g = 0; g < q.N; g++) {
    wanted[g] = false;
    for (uint32_t i = gp.lo[g]; i <= gp.hi[g]; i++) wanted[g] = wanted[g] || gF[i];
    if (wanted[g]) lastWanted = (int)g;
  }
  if (gX) lastWanted = (int)q.N - 1;

  const void* g = gZ;
  uint64_t gBatch = q.batch > 1 ? (uint64_t)q.M * q.L() : 0;
  for (int i = 0; i <= lastWanted; i++) {
    const uint64_t Kin = q.colsBefore(i), S = Kin / q.P[i];
    const bool lastStep = i + 1 == (int)q.N;
    GradStepArgs a{};
    a.P = q.P[i]; a.Q = q.Q[i];
    const bool merged = gp.lo[i] < gp.hi[i];
    const char* F = merged ? sv + gp.saveF[i] * es : (const char*)p.F[gp.lo[i]];
    a.f_sp = gp.pMajor ? (int64_t)a.Q : 1;
    a.f_sq = gp.pMajor ? 1 : (int64_t)a.P;
    a.f_batch = p.perBatchF && q.batch > 1 ? (uint64_t)a.P * a.Q : 0;
    const char* in; uint64_t inBatch;
    if (lastStep) {
      in = gp.copyX ? sv + gp.saveX * es : (const char*)p.X;
      inBatch = q.batch > 1 ? (gp.copyX ? (gp.xBatch > 1 ? (uint64_t)q.M * Kin : 0) : p.strideX) : 0;
    } else {
      in = sv + gp.saveI[i + 1] * es;
      inBatch = (uint64_t)q.M * Kin;
    }
    void* gin = nullptr;
    if (lastStep) gin = gX;
    else if (i < lastWanted) gin = wk + gp.workG[i & 1] * es;
    const uint64_t ginBatch = (uint64_t)q.M * Kin;
    if (mkm) {
      a.in_o = (int64_t)Kin; a.in_t = a.P; a.in_p = 1;
      a.g_o = (int64_t)(S * a.Q); a.g_t = 1; a.g_q = (int64_t)S;
    } else {
      a.in_o = (int64_t)a.P * q.M; a.in_t = 1; a.in_p = q.M;
      a.g_o = q.M; a.g_t = 1; a.g_q = (int64_t)(S * q.M);
    }
    a.in_batch = inBatch; a.g_batch = gBatch; a.gin_batch = ginBatch;
    if (!wanted[i] && !gin) { g = gin; gBatch = ginBatch; continue; }
    const StepShape sh = stepShape(q, i);
    uint32_t partFirst = 0;
    hipError_t he = hipSuccess;
    forRowChunks(sh.O, sh.Tn, [&](uint64_t o0, uint64_t on, uint64_t t0, uint64_t tn) {
      GradStepArgs c = a;
      const int64_t inOff = (int64_t)o0 * a.in_o + (int64_t)t0 * a.in_t, gOff = (int64_t)o0 * a.g_o + (int64_t)t0 * a.g_t;
      c.Tn = (uint32_t)tn; c.U = (uint32_t)(on * tn);
      if (tn > 1) {
        uint32_t s = 0;
        while ((1ull << s) < tn) s++;
        c.tnShift = 31 + s;
        c.tnMagic = ((1ull << c.tnShift) / tn) + 1;
      }
      c.gridX = gradWorkgroups(c.P, c.Q, c.U, q.batch);
      c.partStride = gp.parts[i]; c.partFirst = partFirst;
      partFirst += c.gridX;
      for (uint32_t b0 = 0; b0 < q.batch && he == hipSuccess; b0 += kMaxGridBatch) {
        c.batch = std::min(q.batch - b0, kMaxGridBatch);
        c.in = in + ((size_t)b0 * inBatch + inOff) * es;
        c.g = (const char*)g + ((size_t)b0 * gBatch + gOff) * es;
        c.gin = gin ? (char*)gin + ((size_t)b0 * ginBatch + inOff) * es : nullptr;
        c.f = F + (size_t)b0 * a.f_batch * es;
        c.partial = wanted[i] ? wk + (gp.workP[i] + (size_t)b0 * gp.parts[i] * c.P * c.Q) * es : nullptr;
        auto aligned = [&](const void* ptr, int64_t s1, int64_t s2, uint64_t sb) {
          return (uintptr_t)ptr % 16 == 0 && s1 % ve == 0 && s2 % ve == 0 && sb % ve == 0;
        };
        const bool t4 = tn % 4 == 0;
        c.vecG = t4 && aligned(c.g, c.g_o, c.g_q, gBatch);
        c.vecIn = t4 && c.in_t == 1 && aligned(c.in, c.in_o, c.in_p, inBatch);
        c.vecOut = c.gin && c.in_p == 1 && c.P % 4 == 0 && aligned(c.gin, c.in_o, c.in_t, ginBatch);
        he = launchGradStep(c, p.dt, stream_);
      }
    });
    if (he != hipSuccess) return fastKronInvalidArgument;
    g = gin; gBatch = ginBatch;
  }

  // sum the partial sums of all factors, then split the gradients of merged factors
  GradReduceArgs ra{};
  GradUnmergeArgs ua{};
  ua.perBatch = p.perBatchF; ua.outTransposed = gp.outTransposed;
  const uint32_t fBatch = p.perBatchF ? q.batch : 1;
  auto reduceNow = [&]() -> hipError_t {
    for (uint32_t b0 = 0; b0 < fBatch && ra.count; b0 += kMaxGridBatch) {
      GradReduceArgs c = ra;
      for (uint32_t i = 0; i < c.count; i++) {
        const size_t pq = (size_t)c.r[i].P * c.r[i].Q;
        c.r[i].partial = (const char*)c.r[i].partial + (size_t)b0 * c.r[i].count * pq * es;
        c.r[i].out = (char*)c.r[i].out + (size_t)b0 * pq * es;
      }
      const hipError_t he = launchGradReduce(c, std::min(fBatch - b0, kMaxGridBatch), p.dt, stream_);
      if (he != hipSuccess) return he;
    }
    ra.count = 0;
    return hipSuccess;
  };
  for (int i = 0; i <= lastWanted; i++) {
    if (!wanted[i]) continue;
    GradReduce& r = ra.r[ra.count++];
    r.P = q.P[i]; r.Q = q.Q[i];
    r.count = gp.parts[i] * (p.perBatchF ? 1 : q.batch);
    r.partial = wk + gp.workP[i] * es;
    const bool merged = gp.lo[i] < gp.hi[i];
    r.out = merged ? (void*)(wk + gp.workD[i] * es) : gF[gp.lo[i]];
    const bool tr = !merged && gp.outTransposed;
    r.osp = tr ? 1 : r.Q; r.osq = tr ? r.P : 1;
    if (ra.count == kMaxGradReduce && reduceNow() != hipSuccess) return fastKronInvalidArgument;
  }
  if (reduceNow() != hipSuccess) return fastKronInvalidArgument;
  auto unmergeNow = [&]() -> hipError_t {
    for (uint32_t b0 = 0; b0 < fBatch && ua.groups; b0 += kMaxGridBatch) {
      GradUnmergeArgs c = ua;
      for (uint32_t k = 0; k < c.groups; k++) {
        uint64_t pq = 1;
        for (uint32_t j = 0; j < c.g[k].count; j++) {
          const uint64_t n = (uint64_t)c.g[k].p[j] * c.g[k].q[j];
          pq *= n;
          c.g[k].src[j] = (const char*)c.g[k].src[j] + (p.perBatchF ? (size_t)b0 * n * es : 0);
          if (c.out[k][j]) c.out[k][j] = (char*)c.out[k][j] + (size_t)b0 * n * es;
        }
        c.g[k].dst = (char*)c.g[k].dst + (size_t)b0 * pq * es;
      }
      const hipError_t he = launchGradUnmerge(c, std::min(fBatch - b0, kMaxGridBatch), p.dt, stream_);
      if (he != hipSuccess) return he;
    }
    ua.groups = 0;
    return hipSuccess;
  };
  for (int i = 0; i <= lastWanted; i++) {
    if (!wanted[i] || gp.lo[i] == gp.hi[i]) continue;
    const uint32_t k = ua.groups++;
    mergeGroupOf(p, gp, i, &ua.g[k]);
    ua.g[k].dst = wk + gp.workD[i] * es;
    for (uint32_t j = 0; j < kMaxMergeSources; j++) ua.out[k][j] = j < ua.g[k].count ? gF[gp.lo[i] + j] : nullptr;
    if (ua.groups == kMaxUnmergeGroups && unmergeNow() != hipSuccess) return fastKronInvalidArgument;
  }
  if (unmergeNow() != hipSuccess) return fastKronInvalidArgument;
  return fastKronSuccess;
}

}  // namespace fk
