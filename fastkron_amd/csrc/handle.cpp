#include "handle.h"
#include "kernels/launch.h"

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>

namespace fk {

static int logLevel() {
  static int lvl = -1;
  if (lvl < 0) {
    const char* e = getenv("FASTKRON_LOG");          // reference src/env/env.cpp:57-65
    lvl = 0;
    if (e && (!strcmp(e, "INFO") || !strcmp(e, "info"))) lvl = 1;
    if (e && (!strcmp(e, "DEBUG") || !strcmp(e, "debug"))) lvl = 2;
  }
  return lvl;
}

Handle::Handle(uint32_t backends) : backends_(backends) {
  // the plans that ship with the library first, then the user's own file on top of them
  const std::string shipped = KernelDB::shippedPath();
  if (!shipped.empty()) db_.loadFile(shipped, true);
  if (const char* e = getenv("FASTKRON_CHUNK_MB")) chunkMB_ = atol(e);          // read when the handle is created
  dbPath_ = KernelDB::defaultPath();
  if (!dbPath_.empty()) db_.loadFile(dbPath_);
}

Handle::~Handle() {
  if (mergeWs_ && mergeWsOwned_) (void)hipFree(mergeWs_);
  if (mergeWsEvent_) (void)hipEventDestroy(mergeWsEvent_);
}

void Handle::setPlanOnly(bool on) {
  planOnly_ = on;
  if (!on && mergeWs_ && !mergeWsOwned_) {
    // the stand-in address of plan-only mode must never reach a launch: without it initHIP allocates the real one
    mergeWs_ = nullptr; mergeWsBytes_ = 0;
  }
  if (on && !dev_.valid) {
    // the device the library is written for: 256 compute units, 160 KB of LDS per workgroup
    selectCache_.clear();
    dev_.cus = 256; dev_.ldsPerBlock = 160 * 1024; dev_.waveSize = 64; dev_.xcdRoundRobin = true;
  }
  if (on && !mergeWs_) {
    // never dereferenced: in this mode no launch is made
    mergeWs_ = (void*)(uintptr_t)0x7f0000000000ull;
    mergeWsBytes_ = (size_t)kMaxMergeGroups * 64 * 64 * sizeof(double);
    mergeWsOwned_ = false;
  }
}

void Handle::setTunedDB(const char* path) {
  dbPath_ = path ? path : "";
  if (!dbPath_.empty()) db_.loadFile(dbPath_);
}

fastKronError Handle::ensureDevice() {
  if (dev_.valid) return fastKronSuccess;
  int d = 0;
  if (hipGetDevice(&d) != hipSuccess) return fastKronBackendNotAvailable;
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, d) != hipSuccess) return fastKronBackendNotAvailable;
  dev_.device = d;
  dev_.cus = prop.multiProcessorCount;
  dev_.ldsPerBlock = (int)prop.sharedMemPerBlock;
  dev_.waveSize = prop.warpSize;
  dev_.clockKHz = prop.clockRate;
  strncpy(dev_.arch, prop.gcnArchName, sizeof(dev_.arch) - 1);
  dev_.valid = true;
  selectCache_.clear();
  if (logLevel() >= 1)
    printf("[fastkron] device %d %s: %d CUs, %d B LDS per workgroup, wave %d, %d kHz\n", d, dev_.arch,
           dev_.cus, dev_.ldsPerBlock, dev_.waveSize, dev_.clockKHz);
  return fastKronSuccess;
}

fastKronError Handle::initHIP(void* ptrToStream) {
  if (!hasBackend(fastKronBackend_HIP)) return fastKronBackendNotAvailable;
  stream_ = ptrToStream ? *(hipStream_t*)ptrToStream : nullptr;
  hipInit_ = true;
  fastKronError e = ensureDevice();
  if (e != fastKronSuccess) return e;
  // the static scratch array of the calls that must not allocate: its address on this GPU is looked up here, once
  { void* p = nullptr; (void)staticScratchForCurrentDevice(&p); }
  // workspace for merged factors (kMaxMergeGroups products of at most 64x64 doubles); allocated here so that
  // the gemkm / gekmm calls themselves never allocate
  if (mergeWs_ && !mergeWsOwned_) { mergeWs_ = nullptr; mergeWsBytes_ = 0; }       // plan-only stand-in
  if (!mergeWs_) {
    mergeWsBytes_ = (size_t)kMaxMergeGroups * 64 * 64 * sizeof(double);
    // (behind the merged factors: the counter area of the kernels that synchronise their workgroups, zero once and
    // left zero by every launch that uses it)
    if (hipMalloc(&mergeWs_, mergeWsBytes_ + kSyncAreaBytes) != hipSuccess ||
        hipMemset((char*)mergeWs_ + mergeWsBytes_, 0, kSyncAreaBytes) != hipSuccess) {
      if (mergeWs_) (void)hipFree(mergeWs_);
      mergeWs_ = nullptr; mergeWsBytes_ = 0;
    }
    mergeWsOwned_ = mergeWs_ != nullptr;
    // how the device places workgroups on its XCDs, recorded once (the counter area serves as the 1 KB this needs
    // and is zeroed again afterwards)
    if (mergeWs_) {
      uint32_t* area = (uint32_t*)((char*)mergeWs_ + mergeWsBytes_);
      dev_.xcdRoundRobin = kmm4x6TwoPhasePlacementHolds(area, stream_);
      if (hipMemsetAsync(area, 0, kSyncAreaBytes, stream_) != hipSuccess || hipStreamSynchronize(stream_) != hipSuccess)
        dev_.xcdRoundRobin = false;
    }
    if (mergeWs_ && hipEventCreateWithFlags(&mergeWsEvent_, hipEventDisableTiming) != hipSuccess) mergeWsEvent_ = nullptr;
  }
  return fastKronSuccess;
}

fastKronError Handle::syncError(uint32_t* word) {
  *word = 0;
  if (planOnly_ || !mergeWs_ || !mergeWsOwned_) return fastKronSuccess;
  uint32_t* dev = (uint32_t*)syncArea() + 1;
  if (hipMemcpyAsync(word, dev, sizeof(uint32_t), hipMemcpyDeviceToHost, stream_) != hipSuccess ||
      hipMemsetAsync(dev, 0, sizeof(uint32_t), stream_) != hipSuccess || hipStreamSynchronize(stream_) != hipSuccess)
    return fastKronOtherError;
  return fastKronSuccess;
}

// The merged-factor workspace is the one piece of device state the handle owns.  A call on a new stream may
// overwrite it while launches of an earlier call on another stream still read it; the new stream is therefore made
// to wait for everything the old stream has been given so far.  (Nothing is recorded while either stream is being
// captured into a graph: a handle that is used under capture stays on one stream.)
void Handle::orderWorkspaceBehind(hipStream_t next) {
  if (!mergeWsUsed_ || !mergeWsEvent_ || next == mergeWsStream_) return;
  hipStreamCaptureStatus c0 = hipStreamCaptureStatusNone, c1 = hipStreamCaptureStatusNone;
  (void)hipStreamIsCapturing(mergeWsStream_, &c0);
  (void)hipStreamIsCapturing(next, &c1);
  if (c0 == hipStreamCaptureStatusNone && c1 == hipStreamCaptureStatusNone &&
      hipEventRecord(mergeWsEvent_, mergeWsStream_) == hipSuccess)
    (void)hipStreamWaitEvent(next, mergeWsEvent_, 0);
  mergeWsUsed_ = false;
}

fastKronError Handle::setStream(fastKronBackend backend, void* ptrToStream) {
  if (!ptrToStream) return fastKronInvalidArgument;                    // reference handle.cpp:94
  if (!hasBackend(backend)) return fastKronBackendNotAvailable;        // reference handle.cpp:95
  if (backend != fastKronBackend_HIP) return fastKronBackendNotAvailable;
  hipStream_t next = *(hipStream_t*)ptrToStream;
  if (next != stream_ && !planOnly_) orderWorkspaceBehind(next);
  stream_ = next;
  return fastKronSuccess;
}

// Columns of every step's output, widths[i] for the step of factor i.
static void stepWidths(uint32_t N, const uint32_t* Ps, const uint32_t* Qs, uint64_t* widths) {
  uint64_t w = 1;
  for (uint32_t i = 0; i < N; i++) w *= Ps[i];
  for (int i = (int)N - 1; i >= 0; i--) { w = (w / Ps[i]) * Qs[i]; widths[i] = w; }
}

// reference src/handle/handle.cpp:305-342,375-388: the temporary holds the widest step output
// (X itself is not counted), except for N == 1 where it is max(K, L) columns.
fastKronError Handle::sizes(uint32_t M, uint32_t N, const uint32_t* Ps, const uint32_t* Qs,
                            size_t* yElems, size_t* tmpElems) {
  if (!yElems || !tmpElems) return fastKronInvalidArgument;
  if (N == 0 || N > kMaxFactors || !Ps || !Qs) return fastKronInvalidKMMProblem;
  uint64_t K = 1, L = 1;
  for (uint32_t i = 0; i < N; i++) { K *= Ps[i]; L *= Qs[i]; }
  *yElems = (size_t)M * L;
  if (N == 1) { *tmpElems = (size_t)M * std::max(K, L); return fastKronSuccess; }
  uint64_t w[kMaxFactors];
  stepWidths(N, Ps, Qs, w);
  *tmpElems = (size_t)M * *std::max_element(w, w + N);
  return fastKronSuccess;
}

// reference src/handle/handle.cpp:390-408
fastKronError Handle::sizesForward(uint32_t M, uint32_t N, const uint32_t* Ps, const uint32_t* Qs,
                                   size_t* yElems, size_t* interElems) {
  if (!yElems || !interElems) return fastKronInvalidArgument;
  if (N == 0 || N > kMaxFactors || !Ps || !Qs) return fastKronInvalidKMMProblem;
  uint64_t w[kMaxFactors];
  stepWidths(N, Ps, Qs, w);
  for (uint32_t i = 1; i < N; i++) interElems[i - 1] = (size_t)M * w[i];
  *yElems = (size_t)M * w[0];
  return fastKronSuccess;
}

fastKronError Handle::xgemm(KronProblem p, fastKronBackend backend, void* temp1, void* temp2, const CallWorkspace* ws) {
  callWs_ = ws != nullptr;
  // argument checks in the order of reference src/handle/handle.cpp:116-122
  if (!p.forward) {
    if (p.Z == nullptr || temp1 == nullptr || !hasBackend(backend)) return fastKronInvalidArgument;
    if (p.Z == p.Y && temp2 == nullptr) return fastKronInvalidArgument;
  } else {
    if (p.Z == nullptr || !hasBackend(backend)) return fastKronInvalidArgument;
  }
  if (backend != fastKronBackend_HIP) return fastKronInvalidArgument;
  if (p.N == 0 || p.N > kMaxFactors || p.M == 0 || p.batch == 0) return fastKronInvalidKMMProblem;
  for (uint32_t i = 0; i < p.N; i++)
    if (p.P[i] == 0 || p.Q[i] == 0 || p.F[i] == nullptr) return fastKronInvalidKMMProblem;
  if (p.X == nullptr) return fastKronInvalidArgument;
  if (p.forward && p.N > 1)
    for (uint32_t i = 0; i + 1 < p.N; i++) if (!p.inter[i]) return fastKronInvalidArgument;
  // A call with a single batch entry never uses its strides: they are cleared here, for every entry point, so that no
  // plan that re-views the rows of one problem as batch entries of another (the two-part plan and the digits of a GeKMM
  // in place do) can carry a caller's stride into a batch index of its own.
  if (p.batch == 1) {
    p.strideX = p.strideZ = p.strideY = 0;
    for (uint32_t i = 0; i < p.N; i++) p.strideF[i] = p.strideInter[i] = 0;
    p.haveStrideInter = false;
  }

  // A KMM with a single column is the MKM of the same vector with transposed factors
  // (reference src/handle/handle.cpp:134-138).
  if (p.mm == MMType::KMM && p.M == 1) {
    p.mm = MMType::MKM;
    p.opF = (p.opF == fastKronOp_N) ? fastKronOp_T : fastKronOp_N;
    p.opX = fastKronOp_N;
  }

  fastKronError e = planOnly_ ? fastKronSuccess : ensureDevice();
  if (e != fastKronSuccess) return e;
  launchLog_.clear();

  // 1. A tuned record under the call's own problem string says everything: whether small factors are merged,
  //    whether the chain runs as a two-part plan, and which kernel runs which factors.  With tuning switched on a
  //    problem without a record is tuned here, once.  A record that does not fit the call's buffers falls through
  //    to the online selection.
  if (!p.forward) {
    Choice c;
    bool have = lookupChoice(p, &c);
    // (a GeKMM that runs as a GeMKM is tuned as that GeMKM, below)
    const bool asMKM = p.mm == MMType::KMM && useFusion() && temp2 && viaMKMOnline(p);
    if (!have && canTune() && !planOnly_ && !ws && !asMKM) {
      // a tuner that cannot run (no memory for its operand sets, no events) leaves the problem without a record:
      // the call then runs on the online selection, as it would untuned
      have = tune(p, temp2 != nullptr, &c) == fastKronSuccess;
    }
    if (have) {
      e = runChoice(p, c, temp1, temp2, ws);
      if (e != fastKronKernelNotFound) return e;
    }
  }

  // 2. Online selection.  A GeKMM whose X is stored transposed is the GeMKM of that buffer with a transposed result:
  //    the whole-row GeMKM kernels then apply, and one transposition at the end writes Z.
  //    With few columns that pays even when X has to be transposed first.
  if (p.mm == MMType::KMM && !p.forward && useFusion() && temp2 && viaMKMOnline(p)) {
    e = runViaMKM(p, backend, temp1, temp2, ws);
    if (e != fastKronKernelNotFound) return e;
  }
  //    With op(X) = T otherwise the question whether to transpose X ahead of the launches.
  if (p.opX == fastKronOp_T && !p.forward && useFusion()) {
    KronProblem pn;
    void* xt = nullptr;
    if (transposedProblem(p, temp1, temp2, &pn, &xt) && transposeFirstOnline(p, pn, temp1, temp2, ws)) {
      if (p.mm == MMType::MKM && p.M == 1) {
        // one row is stored the same either way (dgemkm 57x57^4: 299 us with the copy)
        KronProblem q = p;
        q.opX = fastKronOp_N;
        return runOnline(q, temp1, temp2, ws);
      }
      if (!planOnly_) {
        hipError_t he = launchTransposeX(p, xt, pn.strideX);
        if (he != hipSuccess) return fastKronInvalidArgument;
      }
      e = runOnline(pn, temp1, temp2, ws);
      if (e == fastKronSuccess) noteTranspose(p);
      return e;
    }
  }
  return runOnline(p, temp1, temp2, ws);
}

// How many launches the last planned call makes (entries of lastPlan_).
static size_t countLaunches(const std::string& plan) {
  size_t n = 0;
  for (char ch : plan) if (ch == ';') n++;
  return n;
}

fastKronError Handle::xgemmOuter(const KronProblem& p, uint32_t outer, uint64_t outerX, uint64_t outerZ, uint64_t outerY,
                                 fastKronBackend backend, void* temp1, void* temp2) {
  if (outer == 0 || p.batch == 0) return fastKronInvalidKMMProblem;
  if (outer > 1 && p.batch > 1) {              // (one entry of factors: they are shared, a strided batch of X)
    const fastKronError e = runOuter(p, outer, outerX, outerZ, outerY, temp1, temp2);
    if (e != fastKronKernelNotFound) return e;
  }
  const bool perFactors = outer > p.batch;
  for (uint32_t i = 0; i < (perFactors ? p.batch : outer); i++) {
    const KronProblem q = outerCall(p, outer, outerX, outerZ, outerY, i);
    if (const fastKronError e = xgemm(q, backend, temp1, temp2); e != fastKronSuccess) return e;
  }
  return fastKronSuccess;
}

// Call i of the loop: with fewer factors than outer entries one for each of them, the outer dimension as its batch; otherwise
// one for each outer entry.
KronProblem Handle::outerCall(const KronProblem& p, uint32_t outer, uint64_t outerX, uint64_t outerZ, uint64_t outerY, uint32_t i) {
  const size_t es = dtypeSize(p.dt);
  const bool perFactors = outer > p.batch;
  KronProblem q = p;
  q.X = (const char*)p.X + (size_t)i * (perFactors ? p.strideX : outerX) * es;
  q.Z = (char*)p.Z + (size_t)i * (perFactors ? p.strideZ : outerZ) * es;
  if (p.Y) q.Y = (const char*)p.Y + (size_t)i * (perFactors ? p.strideY : outerY) * es;
  if (perFactors) {
    q.batch = outer; q.strideX = outerX; q.strideZ = outerZ; q.strideY = outerY;
    for (uint32_t j = 0; j < p.N && j < kMaxFactors; j++) {
      if (p.F[j]) q.F[j] = (const char*)p.F[j] + (size_t)i * p.strideF[j] * es;
      q.strideF[j] = 0;
    }
  }
  return q;
}

// One series of `launches` against the loop's calls, whose plan is another one: merged factors, parts of rows and groups of columns
// are only there.  Passes over the operands decide, and what a launch costs beside them.  Of 1600 products (2 to 40 by 2 to 16
// entries, 0.1 to 240 MB, either type and layout) the series is faster in half, in 4 % the loop; 7 of those are left, by 1.1 to 1.3.
bool Handle::outerSeriesAhead(const KronProblem& p, uint32_t outer, uint64_t outerX, uint64_t outerZ, uint64_t outerY, size_t launches, void* temp1,
                              void* temp2) {
  // (whether the loop's operands have gaps decides on its plan)
  std::string ck = p.str() + "_outer" + std::to_string(outer);
  for (const uint64_t stride : {p.strideX, p.strideZ, p.strideY, outerX, outerZ, outerY}) ck += "_" + std::to_string(stride);
  if (auto it = outerCache_.find(ck); it != outerCache_.end()) return it->second;
  const KronProblem q = outerCall(p, outer, outerX, outerZ, outerY, 0);
  const bool wasPlanOnly = planOnly_;
  const std::string savedPlan = lastPlan_, savedLog = launchLog_;
  planOnly_ = true;
  const bool ok = xgemm(q, fastKronBackend_HIP, temp1, temp2) == fastKronSuccess;
  const size_t loop = countLaunches(lastPlan_);
  planOnly_ = wasPlanOnly;
  lastPlan_ = savedPlan; launchLog_ = savedLog;
  const double calls = std::min(outer, p.batch);
  const double mb = (double)(p.K() + p.L()) * p.M * outer * p.batch * dtypeSize(p.dt) * 1e-6;
  bool yes = true;
  if (ok && launches > loop) {
    // more passes, for fewer launches: a launch costs as much as 40 MB of a pass, 10 of the plain steps on columns in fp32 (us, series / loop:
    // sgemkm 460 x 14^3, 10 by 4 374 / 143, sgekmm 50 x 7^5, 9 by 7 505 / 257, 2 x 8^6, 8 by 3 179 / 101; sgemkm 32 x 13^3, 19 by 3
    // 41 / 54, dgemkm 20 x 11^3, 25 by 9 85 / 164)
    yes = (double)(launches - loop) * mb < calls * (double)loop * (p.mm == MMType::MKM || p.dt == DType::F64 ? 40 : 10);
  } else if (ok && launches >= 3 && mb > 256 && mb > 120 * calls) {
    // as many passes, and one of the loop's calls keeps what it writes in the 256 MB memory-side cache for its next launch without
    // being short of work (sgemkm 17 x 12^5, 4 by 3 575 / 471; with 30 to 100 MB a call 0.6 to 0.9)
    yes = false;
  }
  return outerCache_[ck] = yes;
}

// fastKronKernelNotFound: not in this form (nothing has been launched).
fastKronError Handle::runOuter(const KronProblem& p0, uint32_t outer, uint64_t outerX, uint64_t outerZ, uint64_t outerY, void* temp1, void* temp2) {
  trimCaches();
  KronProblem p = p0;
  if (!p.X || !p.Z || !temp1 || !temp2 || p.N == 0 || p.N > kMaxFactors || p.M == 0 || p.batch == 0 || p.forward || !useFusion() || canTune())
    return fastKronKernelNotFound;
  if ((uint64_t)outer * p.batch > 65535) return fastKronKernelNotFound;
  for (uint32_t i = 0; i < p.N; i++) if (p.P[i] == 0 || p.Q[i] == 0 || !p.F[i] || p.strideF[i] == 0) return fastKronKernelNotFound;
  if (p.mm == MMType::KMM && (p.M == 1 || p.opX == fastKronOp_T || viaMKMOnline(p))) return fastKronKernelNotFound;
  // (records say what a call of the loop runs)
  Choice tuned;
  if (db_.openRecords() || lookupChoice(p, &tuned) || lookupChoice(outerCall(p, outer, outerX, outerZ, outerY, 0), &tuned)) return fastKronKernelNotFound;
  if (const fastKronError e = planOnly_ ? fastKronSuccess : ensureDevice(); e != fastKronSuccess) return e;
  callWs_ = false;
  const uint32_t inner = p.batch;
  const KronProblem call = p;
  const uint64_t callX = outerX;
  KronProblem x = p;                       // the transposed copy: X's own entries only
  bool copy = false;
  if (p.opX == fastKronOp_T) {
    KronProblem pn;
    void* xt = nullptr;
    if (!transposedProblem(p, temp1, temp2, &pn, &xt)) return fastKronKernelNotFound;
    if (transposeFirstOnline(p, pn, temp1, temp2, nullptr)) {
      if (p.mm == MMType::MKM && p.M == 1) p.opX = fastKronOp_N;         // (one row is stored the same either way)
      else if (p.strideX != 0 && outerX != inner * p.strideX) return fastKronKernelNotFound;
      else {
        copy = true;
        // an X that both dimensions share is copied once and read by all of them
        x.batch = p.strideX != 0 ? outer * inner : outerX != 0 ? outer : 1;
        x.strideX = p.strideX != 0 ? p.strideX : outerX;
        p = pn;
        outerX = x.batch > 1 ? (uint64_t)p.M * p.K() * (x.batch / outer) : 0;
      }
    }
  }
  p.inner = inner; p.batch = outer * inner; p.strided = true;
  p.outerX = outerX; p.outerZ = outerZ; p.outerY = outerY;
  KronProblem flat = p;
  const Plan plan = select(flat);          // (a copy: the loop's plan is laid out before it runs)
  if (execute(p, plan, temp1, temp2, true) != fastKronSuccess) return fastKronKernelNotFound;
  if (!outerSeriesAhead(call, outer, callX, outerZ, outerY, plan.size() + (copy ? 1 : 0), temp1, temp2)) return fastKronKernelNotFound;
  lastPlan_ = p.str();
  for (auto& s : plan) lastPlan_ += ";" + std::to_string(s.lo) + "-" + std::to_string(s.hi) + ":" + db_.kernels()[s.kernel].name;
  launchLog_.clear();
  if (copy && !planOnly_ && launchTransposeX(x, const_cast<void*>(p.X), (uint64_t)p.M * p.K()) != hipSuccess) return fastKronInvalidArgument;
  const fastKronError e = execute(p, plan, temp1, temp2, planOnly_);
  if (e == fastKronSuccess && copy) noteTranspose(x);
  return e;
}

// Online rule for a GeKMM with op(X) = T: as the GeMKM of the same buffer plus a transposition of the result.
// FASTKRON_KMM_VIA_MKM=0 / 1 forces the answer.
bool Handle::viaMKMOnline(const KronProblem& p) const {
  static const int forced = [] { const char* e = getenv("FASTKRON_KMM_VIA_MKM"); return e ? atoi(e) : -1; }();
  if (p.L() >= (1ull << 32) || p.M < 2) return false;
  if (forced >= 0) return forced != 0;
  if (p.opX != fastKronOp_T) {
    // X has to be transposed as well, two more passes over the data: fp32 with fewer than 64 columns, square factors up
    // to 32x32 and at least 64 MB of X (sgekmm 16 x 8^8 2.91 -> 1.55 ms, 16 x 16^6 1.86 -> 1.55, 16 x 32^5 5.67 -> 4.36;
    // 32 x 8^6, 33 MB: no difference, 48 x 16^4, 13 MB: 23 -> 37 us; fp64 loses 1.1 to 1.6 times)
    if (p.dt != DType::F32 || p.M >= 64 || (uint64_t)p.M * p.K() * 4 < (64ull << 20)) return false;
    // (groups of small factors whose digits stay in place need no transposition: sgekmm 30 x 7^7 239 -> 159 us, 40 x 5^9
    // 1014 -> 562, 50 x 4^10 419 -> 285; chains with 8x8 factors keep this plan, which is fixed for them, 16 x 8^8 1532 / 1130)
    bool small = true;
    for (uint32_t i = 0; i < p.N; i++) {
      if (p.P[i] != p.Q[i] || p.P[i] > 32) return false;
      small = small && p.P[i] < 8;
    }
    if (!small) return true;
    // Without such groups (no equal neighbours, factors or gaps of every entry's own) chains of many launches gain (53 columns of
    // 7x7x6x7x5x7x6x3 1264 -> 869, 54 of 7x7x2x3x7x6x4x3x5 629 -> 535, six launches 0.98 to 1.06), and those of 8 to 23 columns (17 of
    // 5x3x6x5x4x5x6x6x5 499 -> 401); others lose (63 columns in three launches 725 / 1069, 4 columns of 7^8, 4 entries, 1302 / 1900).
    return p.M >= 8 && columnsPlan(p).empty() && (p.M < 24 || select(p).size() >= 6);
  }
  // Measured on the reference's published shapes with both operands transposed.  Square factors up to 32x32 gain 1.3
  // to 2.8 times in fp32 (sgekmm 1024 x 8^5 171 -> 112 us, 16 x 8^8 3.34 -> 1.20 ms) and up to 1.2 times in fp64.  With
  // fewer than 64 columns the GeKMM kernels move short pieces and larger factors gain as well (sgekmm 16 x 64^4 and
  // 16 x 128^3 1.27 times, fp64 up to 1.12 times); from 64 columns on, 64x64 and 128x128 factors are within 3 % in
  // fp32 or lose up to 10 % (320 x 128^3), fp64 chains of three 64x64 factors gain 1.1 times.
  uint32_t maxP = 0;
  for (uint32_t i = 0; i < p.N; i++) {
    if (p.P[i] != p.Q[i]) return false;
    if (p.P[i] > maxP) maxP = p.P[i];
  }
  return maxP <= 32 || p.M < 64 || (p.dt == DType::F64 && maxP == 64 && p.N >= 3);
}

// Z (L x M) = transpose(R) + beta * Y with R (M x L) = alpha * X^T (F_1 (x) ... (x) F_N) computed by the GeMKM path
// into temp1; the GeMKM uses temp2 and, when Z is free to be overwritten and large enough, Z as its temporaries.
fastKronError Handle::runViaMKM(const KronProblem& p, fastKronBackend backend, void* temp1, void* temp2, const CallWorkspace* ws) {
  size_t yElems = 0, tmpElems = 0;
  if (sizes(p.M, p.N, p.P, p.Q, &yElems, &tmpElems) != fastKronSuccess) return fastKronKernelNotFound;
  const uint64_t ML = (uint64_t)p.M * p.L();
  KronProblem q = p;
  q.mm = MMType::MKM;
  q.opF = (p.opF == fastKronOp_N) ? fastKronOp_T : fastKronOp_N;      // KMM factors are stored Q x P
  q.opX = fastKronOp_N;
  q.Z = temp1; q.strideZ = p.batch > 1 ? ML : 0;
  q.Y = nullptr; q.strideY = 0; q.beta = 0.0;
  q.zReadNext = true;
  const bool zFree = !(p.Y == p.Z && p.beta != 0.0);
  // (the entries of a temporary lie side by side: what lies between those of Z is not this call's)
  void* zTemp = (zFree && tmpElems <= ML && (p.batch == 1 || p.strideZ == ML)) ? p.Z : nullptr;
  fastKronError e;
  const bool copyX = p.opX != fastKronOp_T;
  if (copyX) {
    // X (K x M) goes to temp2 as M x K first; the GeMKM then has Z and, once its first launch has read it, temp2
    const uint64_t MK = (uint64_t)p.M * p.K();
    if (!zTemp || MK > tmpElems || p.K() >= (1ull << 32)) return fastKronKernelNotFound;
    const uint32_t nb = (p.batch > 1 && p.strideX != 0) ? p.batch : 1;         // a shared X is transposed once
    q.X = temp2; q.strideX = nb > 1 ? MK : 0; q.xJustWritten = true;
    if (!planOnly_) {
      constexpr uint32_t kMaxGridBatch = 65535;
      const size_t es = dtypeSize(p.dt);
      for (uint32_t b0 = 0; b0 < nb; b0 += kMaxGridBatch) {
        const uint32_t n = nb - b0 < kMaxGridBatch ? nb - b0 : kMaxGridBatch;
        if (launchTranspose((const char*)p.X + (size_t)b0 * p.strideX * es, (char*)temp2 + (size_t)b0 * MK * es, (uint32_t)p.K(), p.M, n,
                            p.strideX, MK, p.dt, stream_) != hipSuccess) return fastKronInvalidArgument;
      }
    }
    e = xgemm(q, backend, zTemp, temp2, ws);
  } else {
    e = xgemm(q, backend, temp2, zTemp, ws);
  }
  if (e != fastKronSuccess) return e;
  const size_t semi = lastPlan_.find(';');
  const std::string ty = p.dt == DType::F32 ? "f" : "d";
  lastPlan_ = p.str() + (copyX ? ";" + std::to_string(p.N - 1) + "-" + std::to_string(p.N - 1) + ":transpose_hip_gfx950_256_" + ty + "_x" : "") +
              (semi == std::string::npos ? "" : lastPlan_.substr(semi)) + ";0-0:transpose_hip_gfx950_256_" + ty + "_z";
  if (planOnly_) return fastKronSuccess;
  constexpr uint32_t kMaxGridBatch = 65535;
  const size_t es = dtypeSize(p.dt);
  const void* y = (p.beta != 0.0) ? p.Y : nullptr;
  // Z goes to the caller: streamed from the size on at which the kernels stream their results (Handle::execute)
  const bool streamZ = !p.zReadNext && (uint64_t)(y ? 3 : 2) * ML * p.batch * es >= (96ull << 20);
  for (uint32_t b0 = 0; b0 < p.batch; b0 += kMaxGridBatch) {
    const uint32_t n = p.batch - b0 < kMaxGridBatch ? p.batch - b0 : kMaxGridBatch;
    hipError_t he = launchTransposeAdd((const char*)temp1 + (size_t)b0 * ML * es, (char*)p.Z + (size_t)b0 * p.strideZ * es, p.M,
                                       (uint32_t)p.L(), n, ML, p.strideZ, y ? (const char*)y + (size_t)b0 * p.strideY * es : nullptr,
                                       p.strideY, p.beta, p.dt, stream_, streamZ);
    if (he != hipSuccess) return fastKronInvalidArgument;
  }
  return fastKronSuccess;
}

// The problem with X already transposed into `xt` (temp2, or temp1 when there is no temp2): false when X does not
// fit there.  The transposed copy has the compact layout, batch entries one after the other.
bool Handle::transposedProblem(const KronProblem& p, void* temp1, void* temp2, KronProblem* pn, void** xt) const {
  if (p.opX != fastKronOp_T) return false;
  size_t yElems = 0, tmpElems = 0;
  if (sizes(p.M, p.N, p.P, p.Q, &yElems, &tmpElems) != fastKronSuccess) return false;
  if ((size_t)p.M * p.K() > tmpElems) return false;                  // shrinking chains: X is larger than a temporary
  *xt = temp2 ? temp2 : temp1;
  if (!*xt) return false;
  *pn = p;
  pn->opX = fastKronOp_N;
  pn->X = *xt;
  pn->xJustWritten = true;
  pn->strideX = (p.batch > 1 && p.strideX != 0) ? (uint64_t)p.M * p.K() : 0;
  return true;
}

hipError_t Handle::launchTransposeX(const KronProblem& p, void* xt, uint64_t xtStride) {
  // MKM: op(X) = T means the buffer holds K x M; KMM: it holds M x K (reference tests/testBase.h:272-273,303-304)
  const uint32_t R = p.mm == MMType::MKM ? (uint32_t)p.K() : p.M;
  const uint32_t C = p.mm == MMType::MKM ? p.M : (uint32_t)p.K();
  const uint32_t nb = (p.batch > 1 && p.strideX != 0) ? p.batch : 1;       // a shared X is transposed once
  constexpr uint32_t kMaxGridBatch = 65535;
  for (uint32_t b0 = 0; b0 < nb; b0 += kMaxGridBatch) {
    const uint32_t n = nb - b0 < kMaxGridBatch ? nb - b0 : kMaxGridBatch;
    const size_t es = dtypeSize(p.dt);
    hipError_t he = launchTranspose((const char*)p.X + (size_t)b0 * p.strideX * es, (char*)xt + (size_t)b0 * xtStride * es, R, C, n,
                                    p.strideX, xtStride, p.dt, stream_);
    if (he != hipSuccess) return he;
  }
  return hipSuccess;
}

// lastPlan_ of a call that transposed X first: the call's own problem string, the transposition as a launch ahead
// of the last factor, then the launches of the untransposed problem.
void Handle::noteTranspose(const KronProblem& p) {
  const size_t semi = lastPlan_.find(';');
  const std::string rest = semi == std::string::npos ? "" : lastPlan_.substr(semi);
  lastPlan_ = p.str() + ";" + std::to_string(p.N - 1) + "-" + std::to_string(p.N - 1) + ":transpose_hip_gfx950_256_" +
              (p.dt == DType::F32 ? "f" : "d") + "_x" + rest;
}

// Online rule for op(X) = T: transpose first when that plus the launches of the untransposed problem are no more
// launches (passes over the data) than the kernels that read a transposed X need.  Both plans are laid out in
// plan-only mode on the call's own buffers; the answer is kept per problem.
bool Handle::transposeFirstOnline(const KronProblem& p, const KronProblem& pn, void* temp1, void* temp2,
                                  const CallWorkspace* ws) {
  // Lays a problem out in plan-only mode on the call's own buffers and counts its launches.
  auto plannedLaunches = [&](const KronProblem& q, bool* ok) {
    const bool wasPlanOnly = planOnly_;
    const std::string savedPlan = lastPlan_, savedLog = launchLog_;
    planOnly_ = true;
    *ok = runOnline(q, temp1, temp2, ws) == fastKronSuccess;
    const size_t n = countLaunches(lastPlan_);
    const std::string plan = lastPlan_;
    planOnly_ = wasPlanOnly;
    lastPlan_ = savedPlan; launchLog_ = savedLog;
    return std::make_pair(n, plan);
  };
  const std::string ck = p.str() + (temp2 ? "_t2" : "_t1");
  auto it = transposeCache_.find(ck);
  bool yes;
  if (it != transposeCache_.end()) yes = it->second;
  else {
    bool okT = false, okN = false;
    auto planT = plannedLaunches(p, &okT);
    size_t nT = planT.first;
    // a first launch that reads a transposed X through the padded step with a large factor counts twice: in the MKM layout
    // always (tuned plans: 128x128 chains run 1.3 to 3.3 times faster behind a transposed copy, pairs of single 64x64
    // steps 1.3 to 1.4 times); in the KMM layout, where that step reads the transposed X along its rows, only while X
    // stays in the caches (up to 64 MB the copy is ahead by 8 to 14 %, beyond that behind by 5 to 30 %)
    const uint64_t xBytes = p.M * p.K() * (p.dt == DType::F32 ? 4 : 8) * (uint64_t)(p.batch ? p.batch : 1);
    if (okT && p.P[p.N - 1] >= 64 && (p.mm == MMType::MKM || xBytes <= (64ull << 20))) {
      const std::string& pl = planT.second;
      const size_t s0 = pl.find(':');
      if (s0 != std::string::npos && pl.compare(s0 + 1, 6, "gekmm_") == 0 && pl.find("anyxany", s0) < pl.find(';', s0)) nT++;
    }
    const auto planN = plannedLaunches(pn, &okN);
    const size_t nN = planN.first;
    // with equal counts the copy goes first, except in the KMM layout with fewer than 64 columns, where the copy cannot
    // run on whole 64-wide tiles with 16-byte accesses (sgekmm 16x16^4 with 256 and 1024 columns: 1.26 times faster
    // behind the copy; 16 columns, 16x16^6: 1.16 times slower; factors below 16x16 read a transposed X too slowly in any
    // case)
    const bool copyOnTie = p.mm == MMType::MKM || p.M >= 64 || p.P[p.N - 1] < 16;
    yes = okN && (!okT || (copyOnTie ? 1 + nN <= nT : 1 + nN < nT));
    // where the copy makes the last two factors a launch of the pair of any sizes, that one's rule decides (opX = T, us: sgemkm
    // 284 rows of 33x33 13.9 without the copy / 15.5, dgemkm 6685 rows of 2x1, 32x40 18.9 / 33.2)
    const size_t n0 = planN.second.find(':');
    if (yes && okT && 1 + nN == nT && p.N >= 2 && n0 != std::string::npos && planN.second.find("_anyxany_64x64_2_", n0) < planN.second.find(';', n0)) {
      // (of the chain as it is merged: sgemkm 1673 rows of 2x2^5 10.7 without the copy / 14.8, dgemkm 213 rows of 4x4^4 10.7 / 13.8)
      KronProblem m;
      MergeArgs unused;
      if (!mergedProblem(pn, &m, &unused, ws)) m = pn;
      const uint32_t ps[2] = {m.P[m.N - 1], m.P[m.N - 2]}, qs[2] = {m.Q[m.N - 1], m.Q[m.N - 2]};
      yes = m.N < 2 || pairAnyAhead(ps, qs, (uint64_t)m.M * (m.K() / ((uint64_t)ps[0] * ps[1])), m.batch, m.dt, dev_, true);
    }
    transposeCache_[ck] = yes;           // the preference of the shape; the buffers of each call are checked below
  }
  if (!yes) return false;
  // Without a second temporary the transposed copy sits in temp1, which a plan of several launches writes while its
  // first launch still reads the copy.  How many launches the untransposed problem takes depends on the call's own
  // buffers (a misaligned operand moves it off the whole-row kernels), so this is asked on every call.
  if (!temp2) {
    bool okN = false;
    if (plannedLaunches(pn, &okN).first != 1 || !okN) return false;
  }
  return true;
}

// (Called where nothing refers to an entry.)
void Handle::trimCaches() {
  if (planCache_.size() > kMaxCached) planCache_.clear();
  if (selectCache_.size() > kMaxCached) selectCache_.clear();
  if (transposeCache_.size() > kMaxCached) transposeCache_.clear();
  if (outerCache_.size() > kMaxCached) outerCache_.clear();
}

// What the kernels' rules look at, as bytes.
static std::string selectionKey(const KronProblem& p, uint32_t more = 0) {
  uint32_t key[8 + 2 * kMaxFactors];
  uint64_t own = 0;
  for (uint32_t i = 0; i < p.N; i++) {
    key[8 + 2 * i] = p.P[i]; key[9 + 2 * i] = p.Q[i];
    if (p.batch > 1 && p.strideF[i] != 0) own |= 1ull << i;
  }
  key[0] = (uint32_t)p.mm; key[1] = (uint32_t)p.dt | more << 8; key[2] = (uint32_t)p.opX | (p.forward ? 256u : 0u) | (p.xJustWritten ? 512u : 0u);
  key[3] = p.M; key[4] = p.N; key[5] = p.batch; key[6] = (uint32_t)own; key[7] = (uint32_t)(own >> 32);
  return std::string((const char*)key, sizeof(uint32_t) * (8 + 2 * p.N));
}

fastKronError Handle::runOnline(KronProblem p, void* temp1, void* temp2, const CallWorkspace* ws) {
  trimCaches();
  fastKronError e;
  // (records without the merge / split fields are keyed by the chain as the online rules rewrite it, and are asked before them)
  auto recorded = [&](const KronProblem& q, Plan* plan) {
    int merge = -1;
    return !q.forward && db_.openRecords() && db_.lookupTuned(q.str(), plan, &merge) && merge < 0 && db_.validPlan(q, *plan, dev_);
  };
  auto recordedMerged = [&]() {
    KronProblem q;
    MergeArgs unused;
    Plan plan;
    return db_.openRecords() && recorded(mergedProblem(p, &q, &unused, ws) ? q : p, &plan);
  };
  if (useFusion() && p.mm == MMType::KMM && !p.forward && p.N >= 2 && p.M > 1 && !recordedMerged()) {
    bool pairs = false;                  // (neighbours that a group could hold)
    for (uint32_t i = 1; i < p.N; i++) pairs = pairs || (p.P[i] <= 8 && p.P[i] == p.P[i - 1] && p.P[i] == p.Q[i] && p.P[i] == p.Q[i - 1]);
    if (pairs) {
      const std::string ck = selectionKey(p, p.strideX == (uint64_t)p.M * p.K() ? 1 : 2);
      auto it = selectCache_.find(ck);
      if (it == selectCache_.end()) it = selectCache_.emplace(ck, columnsPlan(p)).first;
      if (!it->second.empty()) {
        e = runColumns(p, it->second, temp1, temp2);
        if (e != fastKronKernelNotFound) return e;
      }
    }
  }
  {
    KronProblem merged;
    if (useFusion() && mergeSmallFactors(p, &merged, ws)) p = merged;
  }

  Plan plan;
  const std::string key = p.str();
  const bool have = recorded(p, &plan);
  // chains longer than one whole-block kernel: the two-part plan, when the problem and the buffers allow it
  if (!have && useFusion()) {
    e = trySplitLeadingTrailing(p, temp1, temp2);
    if (e != fastKronKernelNotFound) return e;
  }
  if (!have) {
    const std::string ck = key + (p.forward ? "_fwd" : "") + (p.xJustWritten ? "_copy" : "") + (useFusion() ? "" : "_nofuse");
    auto it = planCache_.find(ck);
    if (it != planCache_.end()) plan = it->second;
    else {
      plan = db_.selectOnline(p, dev_, useFusion());
      planCache_[ck] = plan;
      if (logLevel() >= 1) {
        printf("[fastkron] %s ->", key.c_str());
        for (auto& s : plan) printf(" [%u,%u] %s", s.lo, s.hi, db_.kernels()[s.kernel].name.c_str());
        printf("\n");
      }
    }
  }
  // Kernel-specific requirements on the actual buffers (alignment, strides): a kernel that refuses them is left out
  // and the selection repeated (the 16-byte accesses of the whole-row and wide kernels need aligned operands, the
  // streaming kernels behind them in the list do not); one generic launch per factor is the last resort.
  std::vector<int> refusedKernels;
  for (int attempt = 0;; attempt++) {
    int refused = -1;
    e = execute(p, plan, temp1, temp2, true, &refused);
    if (e != fastKronKernelNotFound) break;
    if (refused < 0 || attempt >= 8 || db_.kernels()[refused].P == 0) {
      plan.clear();
      for (int i = (int)p.N - 1; i >= 0; i--) plan.push_back(PlanStep{(uint32_t)i, (uint32_t)i, db_.genericKernel(p.dt)});
      e = fastKronSuccess;
      break;
    }
    refusedKernels.push_back(refused);
    // (cached like the first selection, under the problem and the kernels left out)
    std::string rk = key + (p.forward ? "_fwd" : "") + (p.xJustWritten ? "_copy" : "") + (useFusion() ? "" : "_nofuse") + "|without";
    for (int k : refusedKernels) rk += ":" + std::to_string(k);
    auto it = planCache_.find(rk);
    if (it != planCache_.end()) plan = it->second;
    else { plan = db_.selectOnline(p, dev_, useFusion(), &refusedKernels); planCache_[rk] = plan; }
  }
  if (e != fastKronSuccess) return e;
  lastPlan_ = key;
  for (auto& s : plan)
    lastPlan_ += ";" + std::to_string(s.lo) + "-" + std::to_string(s.hi) + ":" + db_.kernels()[s.kernel].name;
  if (planOnly_) { launchLog_.clear(); return execute(p, plan, temp1, temp2, true); }
  return execute(p, plan, temp1, temp2);
}

const Plan& Handle::select(const KronProblem& p) const {
  const std::string key = selectionKey(p);
  auto it = selectCache_.find(key);
  if (it == selectCache_.end()) it = selectCache_.emplace(key, db_.selectOnline(p, dev_, true)).first;
  return it->second;
}

static bool isPow2(uint32_t v) { return v && !(v & (v - 1)); }

bool Handle::mergedProblem(const KronProblem& p, KronProblem* out, MergeArgs* args, const CallWorkspace* ws) const {
  void* const wsBase = ws ? ws->merge : mergeWs_;
  const size_t wsBytes = ws ? ws->mergeBytes : mergeWsBytes_;
  if (!wsBase || p.forward || p.N < 2) return false;
  // fp32 GeKMM already fuses small factors in registers; everything else gains from merging
  if (p.mm == MMType::KMM && p.dt == DType::F32) return false;
  if (p.batch > 1) for (uint32_t i = 0; i < p.N; i++) if (p.strideF[i] != 0) return false;
  // fp32: 16x16 products.  fp64: 64x64 products when the chain holds 8x8 (or 32x32) factors, which do not pack into
  // 16x16 ones; chains of 2x2 and 4x4 factors alone run faster as 16x16 products (a quarter of the multiplications,
  // and the wave-per-block kernel for three 16x16 factors: dgemkm 1024x4^8 0.57 -> 0.47 ms, 1024x4^6 60 -> 20 us).
  uint32_t target = 16;
  // fp64 rows of five 8x8 factors have a whole-row kernel of their own (one launch, one pass, an eighth of the
  // multiplications of 64x64 products): the chain stays as it is where that kernel is the online choice
  if (p.dt == DType::F64 && p.mm == MMType::MKM && p.N == 5) {
    bool all8 = true;
    for (uint32_t i = 0; i < p.N; i++) all8 = all8 && p.P[i] == 8 && p.Q[i] == 8;
    if (all8) {
      const Plan& whole = select(p);
      if (whole.size() == 1 && whole[0].lo == 0 && whole[0].hi == 4) return false;
    }
  }
  if (p.dt == DType::F64) {
    for (uint32_t i = 0; i < p.N; i++)
      if (p.P[i] == p.Q[i] && (p.P[i] == 8 || p.P[i] == 32)) target = 64;
  }
  // groups of adjacent square power-of-two factors, formed from the last factor towards the first, each as
  // large as fits the target size
  // fp64 chains of six or seven 8x8 factors: the trailing five stay as they are, for the whole-row kernel on the
  // blocks of 32768 columns (a two-part plan), and only the leading ones are merged (tuned: dgemkm 1024 x 8^6 1.95 ->
  // 1.79 ms, 256 x 8^6 0.52 -> 0.45 ms; with eight factors the merged chain takes as many launches and stays)
  int keepFrom = (int)p.N;
  if (p.dt == DType::F64 && p.mm == MMType::MKM && (p.N == 6 || p.N == 7) && p.opX == fastKronOp_N && dev_.rulesOfThumb) {
    bool all8 = true;
    for (uint32_t i = 0; i < p.N; i++) all8 = all8 && p.P[i] == 8 && p.Q[i] == 8;
    // (from 32 blocks on, as the kernel's own rule has it)
    const uint64_t blocks = (uint64_t)p.M * (p.N == 6 ? 8 : 64) * p.batch;
    if (all8 && blocks >= 32) keepFrom = (int)p.N - 5;
  }
  struct Grp { uint32_t lo, hi, size; };
  Grp grp[kMaxFactors];
  uint32_t ng = 0, mergedGroups = 0;
  for (int hi = (int)p.N - 1; hi >= 0;) {
    uint32_t size = p.P[hi];
    int lo = hi;
    const bool small = p.P[hi] == p.Q[hi] && isPow2(p.P[hi]) && p.P[hi] < target && hi < keepFrom;
    if (small)
      while (lo > 0 && p.P[lo - 1] == p.Q[lo - 1] && isPow2(p.P[lo - 1]) && size * p.P[lo - 1] <= target &&
             (uint32_t)(hi - lo + 1) < kMaxMergeSources) {
        lo--; size *= p.P[lo];
      }
    // a product smaller than 8 is not worth a kernel of its own size class: leave such factors alone
    if (lo < hi && size < 8) lo = hi, size = p.P[hi];
    grp[ng++] = Grp{(uint32_t)lo, (uint32_t)hi, size};
    if (lo < hi) mergedGroups++;
    hi = lo - 1;
  }
  if (mergedGroups == 0 || mergedGroups > kMaxMergeGroups) return false;

  const bool pMajor = (p.mm == MMType::MKM) == (p.opF == fastKronOp_N);   // as in makeStepArgs
  MergeArgs& ma = *args = MergeArgs{};
  KronProblem q = p;
  q.N = ng;
  size_t wsOff = 0;
  for (uint32_t g = 0; g < ng; g++) {
    const Grp& G = grp[ng - 1 - g];                    // groups were collected last to first
    q.strideF[g] = 0;
    if (G.lo == G.hi) {
      q.P[g] = p.P[G.lo]; q.Q[g] = p.Q[G.lo]; q.F[g] = p.F[G.lo]; q.strideF[g] = p.strideF[G.lo];
      continue;
    }
    MergeGroup& mg = ma.g[ma.groups++];
    mg.count = G.hi - G.lo + 1;
    for (uint32_t j = 0; j < mg.count; j++) {
      const uint32_t fi = G.lo + j;
      mg.src[j] = p.F[fi]; mg.p[j] = p.P[fi]; mg.q[j] = p.Q[fi];
      mg.sp[j] = pMajor ? (int64_t)p.Q[fi] : 1;
      mg.sq[j] = pMajor ? 1 : (int64_t)p.P[fi];
    }
    const size_t bytes = (size_t)G.size * G.size * dtypeSize(p.dt);
    if (wsOff + bytes > wsBytes) return false;
    mg.dst = (char*)wsBase + wsOff;
    mg.dsp = pMajor ? (int64_t)G.size : 1;
    mg.dsq = pMajor ? 1 : (int64_t)G.size;
    wsOff += (bytes + 255) & ~(size_t)255;
    q.P[g] = G.size; q.Q[g] = G.size; q.F[g] = mg.dst;
  }
  *out = q;
  return true;
}

bool Handle::mergeSmallFactors(const KronProblem& p, KronProblem* out, const CallWorkspace* ws) {
  MergeArgs ma;
  KronProblem q;
  if (!mergedProblem(p, &q, &ma, ws)) return false;
  if (!planOnly_) {
    if (!ws && mergeWsUsed_ && mergeWsStream_ != stream_) orderWorkspaceBehind(stream_);
    if (launchMergeFactors(ma, p.dt, stream_) != hipSuccess) return false;
    if (!ws) { mergeWsStream_ = stream_; mergeWsUsed_ = true; }
  }
  *out = q;
  return true;
}

// X (F_0 x ... x F_{N-1}) = first apply the trailing factors B = F_g x ... x F_{N-1} to every contiguous
// block of prod(P_g..) columns (an MKM problem on M * K_A "virtual rows", K_A = prod of the leading P), then
// apply the leading factors A = F_0 x ... x F_{g-1} across the blocks: for every row that is a KMM problem
// on a K_A x T matrix whose T columns are contiguous.  Two or three launches instead of N.  The layout
// between the two parts is [row][k_A][q_B] (digits in place), which only these two sub-problems see.
//
// buildSplit sets up the two sub-problems for g leading factors (q1: trailing factors, X -> temp1; q2: leading
// factors, temp1 -> Z with the call's epilogue) and returns false when the problem does not have that form.
bool Handle::buildSplit(const KronProblem& p, uint32_t g, void* temp1, void* temp2, KronProblem* q1out,
                        KronProblem* q2out) const {
  if (p.mm != MMType::MKM || p.forward || p.opX != fastKronOp_N) return false;
  if (!temp1 || !temp2 || p.N < 3 || g == 0 || g >= p.N) return false;
  const uint32_t nT = p.N - g;
  // KA x Tin columns come in; the trailing factors make Tout of every Tin, the leading ones LA of the KA blocks
  uint64_t KA = 1, LA = 1, Tin = 1, Tout = 1;
  for (uint32_t i = 0; i < g; i++) { KA *= p.P[i]; LA *= p.Q[i]; }
  for (uint32_t i = g; i < p.N; i++) { Tin *= p.P[i]; Tout *= p.Q[i]; }
  const uint64_t K = KA * Tin, L = LA * Tout, mid = KA * Tout;
  if (Tin >= (1ull << 32) || Tout >= (1ull << 32)) return false;
  {
    // the intermediate (M x KA x Tout) is one of the step outputs the temporaries are sized for; the second part uses
    // temp2 for the outputs of all but its last launch, each at most as wide as the widest step of the call
    size_t yElems = 0, tmpElems = 0;
    if (const_cast<Handle*>(this)->sizes(p.M, p.N, p.P, p.Q, &yElems, &tmpElems) != fastKronSuccess) return false;
    if ((uint64_t)p.M * mid > tmpElems) return false;
  }
  if (p.batch > 1) {
    if (p.strideX != (uint64_t)p.M * K || p.strideZ != (uint64_t)p.M * L) return false;
    if (p.Y && p.beta != 0.0 && p.strideY != (uint64_t)p.M * L) return false;
  }
  // the leading factors are read by a problem whose batch entries are the rows of this one: shared factors only
  for (uint32_t i = 0; i < g; i++) if (p.strideF[i] != 0) return false;
  if ((uint64_t)p.M * p.batch > 65535 || (uint64_t)p.M * KA >= (1ull << 31)) return false;

  // part 1: trailing factors, X -> temp1, no epilogue
  KronProblem q1 = p;
  q1.M = (uint32_t)(p.M * KA); q1.N = nT;
  for (uint32_t i = 0; i < nT; i++) {
    q1.P[i] = p.P[g + i]; q1.Q[i] = p.Q[g + i]; q1.F[i] = p.F[g + i]; q1.strideF[i] = p.strideF[g + i];
  }
  q1.Z = temp1; q1.strideZ = (uint64_t)p.M * mid;
  q1.Y = nullptr; q1.strideY = 0; q1.alpha = 1.0; q1.beta = 0.0;
  q1.zReadNext = true;

  // part 2: leading factors as a KMM over every row block; P x Q storage is the transpose of KMM's Q x P
  KronProblem q2 = p;
  q2.mm = MMType::KMM; q2.M = (uint32_t)Tout; q2.N = g;
  q2.opF = (p.opF == fastKronOp_N) ? fastKronOp_T : fastKronOp_N;
  q2.opX = fastKronOp_N;
  q2.X = temp1; q2.strideX = mid;
  q2.xJustWritten = true;
  q2.strideZ = L; q2.strideY = L;
  q2.batch = p.batch * p.M; q2.strided = true;
  for (uint32_t i = 0; i < g; i++) q2.strideF[i] = 0;
  *q1out = q1; *q2out = q2;
  return true;
}

// Validates (on the concrete buffers) and runs a two-part plan: plan1 on q1, plan2 on q2 with temp2 as its scratch.
fastKronError Handle::runSplit(const KronProblem& p, uint32_t g, const KronProblem& q1, const Plan& plan1,
                               const KronProblem& q2, const Plan& plan2, void* temp2) {
  if (plan1.size() != 1) return fastKronKernelNotFound;                    // q1 has no scratch of its own
  // more than two leading launches ping-pong between temp2 and Z, which must then not be Y
  if (plan2.size() > 2 && p.Y == p.Z && p.beta != 0.0) return fastKronKernelNotFound;
  if (execute(q1, plan1, nullptr, nullptr, true) != fastKronSuccess) return fastKronKernelNotFound;
  if (execute(q2, plan2, temp2, nullptr, true) != fastKronSuccess) return fastKronKernelNotFound;
  lastPlan_ = p.str();
  for (auto& s : plan1)
    lastPlan_ += ";" + std::to_string(g + s.lo) + "-" + std::to_string(g + s.hi) + ":" + db_.kernels()[s.kernel].name;
  for (auto& s : plan2)
    lastPlan_ += ";" + std::to_string(s.lo) + "-" + std::to_string(s.hi) + ":" + db_.kernels()[s.kernel].name;
  // Rows are independent, and the intermediate between the two parts is written once and read once.  With
  // FASTKRON_CHUNK_MB set, the rows go through the two parts in chunks whose intermediate has that size, every chunk
  // through the same stretch of temp1, so that the second part reads what the first wrote from the 256 MB memory-side
  // cache and the stretch is overwritten before most of it has to go out to HBM.  Off by default: measured on an
  // MI355X it loses (dgemkm 256 x 64^3: 496 us unchunked, 548 / 569 / 601 us with chunks of 192 / 128 / 64 MB; sgemkm
  // 1024 x 16^5: 2.98 ms against 3.33 ms at 128 MB; 1024 x 8^6, 1024 x 32^4, dgemkm 1024 x 16^4, sgemkm 16 x 16^6 likewise):
  // each chunk's launches start and drain on their own, which costs more than the cache returns.
  // (reference src/kmm/kmmalgo.cpp:72-115 plans whole-problem intermediates.)
  const uint32_t chunkRows = chunkRowsForCache(p, q2);
  auto forChunks = [&](bool dry) -> fastKronError {
    const size_t es = dtypeSize(p.dt);
    const uint64_t K = q2.strideX;                              // elements of one row of the problem
    const uint64_t KA = q1.M / p.M;                             // blocks of a row
    for (uint32_t m0 = 0; m0 < p.M; m0 += chunkRows) {
      const uint32_t rows = p.M - m0 < chunkRows ? p.M - m0 : chunkRows;
      KronProblem c1 = q1, c2 = q2;
      c1.M = (uint32_t)(rows * KA);
      c1.X = (const char*)q1.X + (size_t)m0 * K * es;
      c2.batch = rows;
      c2.Z = (char*)q2.Z + (size_t)m0 * K * es;
      if (q2.Y) c2.Y = (const char*)q2.Y + (size_t)m0 * K * es;
      fastKronError e = execute(c1, plan1, nullptr, nullptr, dry);
      if (e != fastKronSuccess) return e;
      e = execute(c2, plan2, temp2, nullptr, dry);
      if (e != fastKronSuccess) return e;
    }
    return fastKronSuccess;
  };
  if (chunkRows < p.M) {
    if (planOnly_) { launchLog_.clear(); return forChunks(true); }
    if (forChunks(true) != fastKronSuccess) return fastKronKernelNotFound;      // every chunk's buffers checked first
    return forChunks(false);
  }
  if (planOnly_) {
    launchLog_.clear();
    (void)execute(q1, plan1, nullptr, nullptr, true);
    return execute(q2, plan2, temp2, nullptr, true);
  }
  fastKronError e = execute(q1, plan1, nullptr, nullptr);
  if (e != fastKronSuccess) return e;
  return execute(q2, plan2, temp2, nullptr);
}

// Rows per chunk of a two-part plan (p.M: no chunking, the default).  FASTKRON_CHUNK_MB=<n> sets the size of a
// chunk's intermediate.
uint32_t Handle::chunkRowsForCache(const KronProblem& p, const KronProblem& q2) const {
  const long forcedMB = chunkMB_;
  if (forcedMB <= 0 || p.batch != 1 || p.M < 2 || p.forward || p.K() != p.L()) return p.M;
  const uint64_t rowBytes = q2.strideX * dtypeSize(p.dt);
  uint64_t rows = ((uint64_t)forcedMB << 20) / rowBytes;
  if (rows < 1) rows = 1;
  return rows >= p.M ? p.M : (uint32_t)rows;
}

// A Kronecker product acts on every digit of the row index by itself, so that a GeKMM may leave the digits where they are:
// with the factors behind `hi` applied already, the rows are H x K x (Q of those factors), and the factors lo .. hi are a
// problem of H entries (batch) with K rows and M * Q.. columns.  Nothing moves, the columns are many even when M is not.
bool Handle::columnsPart(const KronProblem& p, uint32_t lo, uint32_t hi, KronProblem* out) const {
  uint64_t H = 1, Kg = 1, Lg = 1, C = p.M;
  for (uint32_t i = 0; i < lo; i++) H *= p.P[i];
  for (uint32_t i = lo; i <= hi; i++) { Kg *= p.P[i]; Lg *= p.Q[i]; }
  for (uint32_t i = hi + 1; i < p.N; i++) C *= p.Q[i];
  if (C >= (1ull << 32) || H * p.batch >= (1ull << 32)) return false;
  // entries of the problem become H entries each: shared factors, and the caller's operands without gaps
  if (p.batch > 1 && H > 1) {
    for (uint32_t i = lo; i <= hi; i++) if (p.strideF[i] != 0) return false;
    if (hi == p.N - 1 && p.strideX != H * Kg * C) return false;
  }
  KronProblem q = p;
  q.N = hi - lo + 1;
  for (uint32_t i = 0; i < q.N; i++) { q.P[i] = p.P[lo + i]; q.Q[i] = p.Q[lo + i]; q.F[i] = p.F[lo + i]; q.strideF[i] = p.strideF[lo + i]; }
  q.M = (uint32_t)C; q.batch = (uint32_t)(H * p.batch); q.strided = q.batch > 1;
  if (hi < p.N - 1 || H > 1) q.strideX = Kg * C;
  if (lo > 0) {
    q.strideZ = Lg * C;
    q.Y = nullptr; q.strideY = 0; q.alpha = 1.0; q.beta = 0.0;
    q.zReadNext = true;
  }
  if (hi < p.N - 1) q.xJustWritten = true;
  *out = q;
  return true;
}

Plan Handle::columnsPlan(const KronProblem& p) const {
  if (p.mm != MMType::KMM || p.forward || p.opX != fastKronOp_N || p.N < 2 || p.M < 2) return Plan();
  Plan plan;
  bool grouped = false;
  for (int hi = (int)p.N - 1; hi >= 0;) {
    int lo = hi;
    const uint32_t P = p.P[hi], most = p.P[hi] == p.Q[hi] ? colsInplaceMost(P, p.dt) : 0;
    if (most) {
      int run = 1;
      while (run <= hi && p.P[hi - run] == P && p.Q[hi - run] == P) run++;
      const int groups = (run + (int)most - 1) / (int)most;
      lo = hi + 1 - (run + groups - 1) / groups;
    }
    KronProblem q;
    if (!columnsPart(p, (uint32_t)lo, (uint32_t)hi, &q)) return Plan();
    const Plan& one = select(q);
    if (one.size() != 1) return Plan();
    plan.push_back(PlanStep{(uint32_t)lo, (uint32_t)hi, one[0].kernel});
    // A last factor of its own on the plain or padded step runs on the caller's columns, an entry for every block of its rows: many
    // entries of few columns cost more than the groups behind it save (us: sgekmm 2 columns of 8x7^3x12^3 222 / 643, 6 columns of
    // 8x8x6x7x4x7x3 44 / 121, 47 columns of 6x7x7x2x3x3x7x6x2 285 / 448, dgekmm 5 columns of 8x3x7^3x6x3, 2 entries, 65 / 153; with
    // fewer entries or more columns 0.6 to 0.95 of the time).
    if (lo == hi && hi == (int)p.N - 1 && db_.kernels()[one[0].kernel].P <= 1) {
      const uint32_t wide = p.dt == DType::F32 ? 64 : 16;
      if (q.batch >= 16384 ? p.M <= wide : q.batch >= 4096 && p.M <= (p.dt == DType::F32 ? 16u : 8u)) return Plan();
    }
    if (lo < hi) grouped = true;
    hi = lo - 1;
  }
  if (!grouped) return Plan();
  // against the launches of the chain as it would run otherwise (with merged factors, one more that writes those): fewer is
  // ahead at every size measured (2 to 10 factors of 2 to 8 rows, 2 to 1024 columns, either type: 1.2 to 4.5 times but for
  // sgekmm 8^4 x 88, 14.1 / 14.0 us), as many where groups of the kernel with two LDS buffers are among them (1.4 to 2.6 times:
  // sgekmm 6^6 x 88 58.8 -> 22.2, dgekmm 5^6 x 1024 217 -> 95); as many launches of the register kernels are no slower
  // (sgekmm 8^5 x 64 19.8, 1024 columns 113)
  KronProblem q = p;
  MergeArgs unused;
  const size_t merge = mergedProblem(p, &q, &unused) ? 1 : 0;
  const Plan& other = select(q);
  bool lds = false, merged16 = merge != 0;
  for (auto& s : other) lds = lds || db_.kernels()[s.kernel].name.find("_small_fused_lds_") != std::string::npos;
  for (uint32_t i = 0; i < q.N; i++) merged16 = merged16 && q.P[i] <= 16;
  // (Small fp64 problems of 2x2 and 4x4 factors keep the plan that merges them to 16x16, which is fixed for them: dgekmm 4^6 x 64
  // 17.1 us against 9.2.)
  if (merged16 && (uint64_t)p.M * p.K() * p.batch <= (1ull << 18)) return Plan();
  return plan.size() < merge + other.size() + (lds ? 1 : 0) ? plan : Plan();
}

fastKronError Handle::runColumns(const KronProblem& p, const Plan& plan, void* temp1, void* temp2) {
  if (plan.empty() || (plan.size() > 1 && !temp1) || (plan.size() > 2 && !temp2)) return fastKronKernelNotFound;
  void* tmps[2] = {temp1, temp2};
  auto run = [&](bool dry) -> fastKronError {
    const void* x = p.X;
    for (size_t i = 0; i < plan.size(); i++) {
      const PlanStep& s = plan[i];
      KronProblem q;
      if (s.hi >= p.N || s.lo > s.hi || !columnsPart(p, s.lo, s.hi, &q)) return fastKronKernelNotFound;
      q.X = x;
      if (s.lo > 0) q.Z = tmps[i % 2];
      const Plan one(1, PlanStep{0, s.hi - s.lo, s.kernel});
      if (const fastKronError e = execute(q, one, nullptr, nullptr, dry); e != fastKronSuccess) return e;
      x = q.Z;
    }
    return fastKronSuccess;
  };
  if (run(true) != fastKronSuccess) return fastKronKernelNotFound;
  lastPlan_ = p.str();
  for (auto& s : plan) lastPlan_ += ";" + std::to_string(s.lo) + "-" + std::to_string(s.hi) + ":" + db_.kernels()[s.kernel].name;
  if (planOnly_) launchLog_.clear();
  return run(planOnly_);
}

// The online rule for the two-part plan: how many trailing factors one whole-block kernel takes.
fastKronError Handle::trySplitLeadingTrailing(const KronProblem& p, void* temp1, void* temp2) {
  if (p.mm != MMType::MKM || p.forward || p.opX != fastKronOp_N) return fastKronKernelNotFound;
  if (!temp1 || !temp2 || p.N < 3) return fastKronKernelNotFound;
  // trailing run of identical square factors that one whole-row kernel fuses:
  // fp32 8x8 (five), 16x16 (four), 32x32 (three), 64x64 (two); fp64 16x16 (three), 32x32 or 64x64 (two);
  // 9x9 ... 15x15 (three, either type); 3x3, 5x5, 6x6, 7x7 (eight, six, five, five, either type)
  const uint32_t tp = p.P[p.N - 1], tq = p.Q[p.N - 1];
  // two trailing factors of other shapes on one of the pair kernels (exact tiles for 32x64 and 64x32, padded ones up to 64), where
  // that takes fewer launches: (31x63)^3 on one row 18.3 -> 11.3 us, 10 x 50^3 31.7 -> 21.8, 80 x 63^3 176 -> 130, 10 x 6x6x50x50
  // 28.9 -> 17.2.  Not with fewer than 256 columns for the leading factors to run along (80 x 50x2x50 21.7 / 26.9), and not for
  // many blocks of 33 to 47 rows a side, which the padded step reads in whole pieces (80 x 40^3 49.2 / 52.0, 500 x 36^3 174 / 191).
  auto trailingPair = [&]() -> fastKronError {
    const uint32_t g2 = p.N - 2;
    KronProblem r1, r2;
    if (!buildSplit(p, g2, temp1, temp2, &r1, &r2)) return fastKronKernelNotFound;
    if (r2.M < 256 || (tp == tq && tp > 32 && tp < 48 && (uint64_t)r1.M * r1.batch >= 2048)) return fastKronKernelNotFound;
    const Plan& rp1 = select(r1);
    if (rp1.size() != 1 || db_.kernels()[rp1[0].kernel].fused != 2 || db_.kernels()[rp1[0].kernel].P == 0)
      return fastKronKernelNotFound;
    const Plan& rp2 = select(r2);
    const Plan& apart = select(p);
    if (1 + rp2.size() >= apart.size()) return fastKronKernelNotFound;
    // nor, from 1024 blocks on in fp64, where leading factors that make rows at least twice as long come from the padded step to the
    // plain one (dgemkm 242 x 6x50^3 70 / 86, 1071 x 7x28^3 61 / 75, 3 x 9x20^5 54 / 62; other factors 0.9 of the time; behind a
    // transposed copy the pair is what made the copy worth while)
    const uint64_t blocks = (uint64_t)r1.M * r1.batch;
    if (p.dt == DType::F64 && blocks >= 1024 && !p.xJustWritten) {
      const int plain = db_.genericKernel(p.dt);
      for (auto& s : rp2)
        if (s.kernel == plain && p.Q[s.lo] >= 2 * p.P[s.lo])
          for (auto& t : apart) if (t.lo <= s.lo && s.lo <= t.hi && t.kernel != plain) return fastKronKernelNotFound;
    }
    return runSplit(p, g2, r1, rp1, r2, rp2, temp2);
  };
  if (tq != tp || p.P[p.N - 2] != tp || p.Q[p.N - 2] != tq || (tp > 32 && tp < 64)) return trailingPair();
  uint32_t maxT = 0;
  if (tp == 32 && p.dt == DType::F32) maxT = 3;      // three 32x32 fp32 factors fused per 32768-column block
  else if (tp == 32 || tp == 64)      maxT = 2;
  else if (p.dt == DType::F32) maxT = (tp == 8) ? 5 : (tp == 16) ? 4 : 0;
  else if (tp == 16)           maxT = 3;
  else if (tp == 8)            maxT = 5;              // fp64: the whole-row kernel for five 8x8 factors
  // (few rows of 32^3, fp32: the pair kernel spreads them over more CUs than one workgroup per row does)
  if (p.dt == DType::F32 && tp == 32 && (uint64_t)p.M * (p.K() / 32768) * p.batch < 96) maxT = 2;
  // (few blocks of 16^4: the wave-per-block kernel for three factors spreads them over more CUs)
  if (p.dt == DType::F32 && tp == 16 && p.N >= 4 && (uint64_t)p.M * (p.K() / 65536) * p.batch < 96) maxT = 3;
  if (maxT == 0 && tp >= 9 && tp <= 15) maxT = 3;       // zero-padded form of the 16x16x3 wave-per-block kernel
  if (maxT == 0 && tp >= 17 && tp <= 31) maxT = 2;      // zero-padded form of the 32x32 pair kernel
  bool inplace = false;
  if (maxT == 0 && (tp == 3 || tp == 5 || tp == 6 || tp == 7)) {
    // rows longer than the in-place kernel's LDS: as many trailing factors as it holds (3^8, 5^6, 6^5, 7^5), which are blocks
    // of 6561 columns and more for the leading ones
    inplace = true;
    for (uint64_t bytes = dtypeSize(p.dt) * tp; bytes + 16 <= 160 * 1024 && maxT < kMaxFused; bytes *= tp) maxT++;
  }
  if (maxT == 0) return fastKronKernelNotFound;
  uint32_t nT = 0;
  while (nT < maxT && nT < p.N && p.P[p.N - 1 - nT] == tp && p.Q[p.N - 1 - nT] == tp) nT++;
  if (nT < 2 || nT == p.N) return fastKronKernelNotFound;         // a chain of nT factors alone is a whole-row problem
  // (sgemkm 1000 x 5^7 527 -> 342 us, 1 x 5^7 26 -> 14, 1000 x 3^9 128 -> 76, 1000 x 6^6 313 -> 177, 200 x 7^6 183 -> 120,
  // dgemkm 100 x 7^6 185 -> 126, all against groups of the kernel with two LDS buffers.  Three and more leading factors lose,
  // 50 x 3^11 87 -> 125.  fp64 blocks of 6^5 and 7^5 take a CU each (these figures in passes of one digit; 6^5 has two a pass since): 7^6 is ahead from 96
  // blocks on (14 rows 50 -> 39 us, 13 rows 37 / 37), 6^6 only where the groups' pieces no longer fit the CUs at once, from 208
  // on (16 rows 19.5 / 22.5, 33 rows 27.1 / 27.3, 38 rows 38.6 / 29.0; 32 x 2x2x6^5 25.0 / 31.1, 57 rows 40.8 / 37.0).)
  if (inplace && (nT != maxT || p.N - nT > 2)) return fastKronKernelNotFound;
  if (inplace && p.dt == DType::F64 && tp >= 6) {
    uint64_t blocks = (uint64_t)p.M * p.batch;
    for (uint32_t i = 0; i < p.N - nT; i++) blocks *= p.P[i];
    if (blocks < (tp == 6 ? 208 : 96)) return fastKronKernelNotFound;
  }
  if (p.dt == DType::F64 && tp == 8 && nT != 5) return fastKronKernelNotFound;   // (that kernel takes exactly five)
  const uint32_t g = p.N - nT;
  KronProblem q1, q2;
  if (!buildSplit(p, g, temp1, temp2, &q1, &q2)) return fastKronKernelNotFound;
  const Plan& plan1 = select(q1);
  if (plan1.size() != 1 || db_.kernels()[plan1[0].kernel].P == 0) return fastKronKernelNotFound;
  const Plan& plan2 = select(q2);
  return runSplit(p, g, q1, plan1, q2, plan2, temp2);
}

// A tuned record with explicit merge / split fields for this problem, if the file has one.
bool Handle::lookupChoice(const KronProblem& p, Choice* c) const {
  int merge = -1, transposeX = 0;
  uint32_t split = 0;
  Plan plan;
  if (!db_.lookupTuned(p.str(), &plan, &merge, &split, &transposeX) || merge < 0) return false;
  c->merge = merge == 1; c->columns = merge == 2; c->split = split; c->plan = plan; c->transposeX = transposeX != 0;
  return true;
}

// Runs a tuned choice; fastKronKernelNotFound when it does not fit this call (the caller then selects online).
fastKronError Handle::runChoice(const KronProblem& p0, const Choice& c, void* temp1, void* temp2, const CallWorkspace* ws) {
  if (c.transposeX) {
    KronProblem pn;
    void* xt = nullptr;
    if (!transposedProblem(p0, temp1, temp2, &pn, &xt)) return fastKronKernelNotFound;
    if (!temp2 && (c.split || c.plan.size() != 1)) return fastKronKernelNotFound;      // the copy sits in temp1 then
    Choice rest = c;
    rest.transposeX = false;
    if (!planOnly_ && launchTransposeX(p0, xt, pn.strideX) != hipSuccess) return fastKronInvalidArgument;
    fastKronError e = runChoice(pn, rest, temp1, temp2, ws);
    if (e == fastKronSuccess) noteTranspose(p0);
    return e;
  }
  KronProblem p = p0;
  if (c.columns) {
    if (p.mm != MMType::KMM || p.forward || p.opX != fastKronOp_N || !db_.orderedPlan(p, c.plan)) return fastKronKernelNotFound;
    for (auto& s : c.plan) {
      KronProblem q;
      if (!columnsPart(p, s.lo, s.hi, &q) || !db_.validPlan(q, Plan(1, PlanStep{0, s.hi - s.lo, s.kernel}), dev_)) return fastKronKernelNotFound;
    }
    return runColumns(p, c.plan, temp1, temp2);
  }
  if (c.merge) {
    KronProblem merged;
    if (!mergeSmallFactors(p0, &merged, ws)) return fastKronKernelNotFound;
    p = merged;
  }
  if (c.split) {
    KronProblem q1, q2;
    if (!buildSplit(p, c.split, temp1, temp2, &q1, &q2)) return fastKronKernelNotFound;
    Plan plan1, plan2;
    for (auto& s : c.plan) {
      if (s.lo >= c.split) plan1.push_back(PlanStep{s.lo - c.split, s.hi - c.split, s.kernel});
      else if (s.hi < c.split) plan2.push_back(s);
      else return fastKronKernelNotFound;
    }
    if (!db_.validPlan(q1, plan1, dev_) || !db_.validPlan(q2, plan2, dev_)) return fastKronKernelNotFound;
    return runSplit(p, c.split, q1, plan1, q2, plan2, temp2);
  }
  if (!db_.validPlan(p, c.plan, dev_)) return fastKronKernelNotFound;
  fastKronError e = execute(p, c.plan, temp1, temp2, true);
  if (e != fastKronSuccess) return e;
  lastPlan_ = p.str();
  for (auto& s : c.plan)
    lastPlan_ += ";" + std::to_string(s.lo) + "-" + std::to_string(s.hi) + ":" + db_.kernels()[s.kernel].name;
  if (planOnly_) { launchLog_.clear(); return execute(p, c.plan, temp1, temp2, true); }
  return execute(p, c.plan, temp1, temp2);
}

// Everything of a launch's arguments that follows from the problem and the factor range; the caller
// fills in the input/output buffers.
StepArgs makeStepArgs(const KronProblem& p, uint32_t lo, uint32_t hi, bool first, bool last) {
  StepArgs a{};
  a.nf = hi - lo + 1;
  a.M = p.M; a.batch = p.batch;
  a.Kin = p.colsBefore(hi);
  a.Kout = p.colsAfter(lo);
  for (uint32_t j = 0; j < a.nf && j < kMaxFused; j++) {
    const uint32_t fi = hi - j;
    a.f[j] = p.F[fi]; a.f_batch[j] = p.strideF[fi];
    a.p[j] = p.P[fi]; a.q[j] = p.Q[fi];
    // Storage of op(F): MKM factors are P x Q, KMM factors are Q x P; opF = T stores the transpose
    // (reference tests/testBase.h:264-268,295-299).
    const bool pMajor = (p.mm == MMType::MKM) == (p.opF == fastKronOp_N);
    a.f_sp[j] = pMajor ? (int64_t)p.Q[fi] : 1;
    a.f_sq[j] = pMajor ? 1 : (int64_t)p.P[fi];
  }
  const bool rowMajor = (p.mm == MMType::MKM);      // rows contiguous along the columns
  auto setLd = [&](int64_t& ldm, int64_t& ldc, uint64_t cols, bool transposed) {
    const bool rm = transposed ? !rowMajor : rowMajor;
    if (rm) { ldm = (int64_t)cols; ldc = 1; } else { ldm = 1; ldc = (int64_t)p.M; }
  };
  setLd(a.in_ldm, a.in_ldc, a.Kin, first && p.opX == fastKronOp_T);
  setLd(a.out_ldm, a.out_ldc, a.Kout, false);
  if (last) {
    a.epilogue = 1; a.alpha = p.alpha; a.beta = p.beta;
    a.y = (p.beta != 0.0) ? p.Y : nullptr;          // beta is skipped when Y is null, reference kernel.h:158-159
    a.y_batch = p.strideY;
    setLd(a.y_ldm, a.y_ldc, p.L(), false);
  }
  return a;
}

// With dryRun the launches are only validated (kernel-specific checks on the concrete buffers);
// fastKronKernelNotFound then means "this plan cannot run on these buffers".
fastKronError Handle::execute(const KronProblem& p, const Plan& plan, void* temp1, void* temp2, bool dryRun,
                              int* refused) {
  const size_t n = plan.size();
  if (n == 0) return fastKronKernelNotFound;
  const uint64_t L = p.L();

  // Ping-pong plan of reference src/kmm/kmmalgo.cpp:82-110: launch l < n-1 writes tmps[l % 2]; when
  // only one temporary is given, Z is the other one, placed so that the last intermediate is not Z.
  void* tmps[2] = {temp1, temp2};
  bool zIsTmp[2] = {false, false};
  if (!p.forward && n > 1 && temp2 == nullptr) {
    if (n % 2 == 1) { tmps[1] = temp1; tmps[0] = p.Z; zIsTmp[0] = true; }
    else            { tmps[1] = p.Z; zIsTmp[1] = true; }
    if (n == 2) { tmps[1] = nullptr; zIsTmp[1] = false; }     // a 2-launch plan never touches the second one
  }

  // capacity of a temporary by the API's contract: the widest step output of every batch entry
  uint64_t tempElems = 0;
  if (!p.forward) {
    size_t ye = 0, te = 0;
    if (sizes(p.M, p.N, p.P, p.Q, &ye, &te) == fastKronSuccess) tempElems = (uint64_t)te * p.batch;
  }
  const void* in = p.X;
  uint64_t inBatch = p.strideX;
  for (size_t l = 0; l < n; l++) {
    const PlanStep& s = plan[l];
    const KernelInfo& k = db_.kernels()[s.kernel];
    const bool first = (l == 0), last = (l + 1 == n);
    if (s.hi - s.lo + 1 > kMaxFused) return fastKronKernelNotFound;
    StepArgs a = makeStepArgs(p, s.lo, s.hi, first, last);
    a.in = in; a.in_batch = inBatch;
    if (p.inner && !k.outer) { if (refused) *refused = s.kernel; return fastKronKernelNotFound; }
    if (last) {
      a.out = p.Z; a.out_batch = p.strideZ;
    } else if (p.forward) {
      a.out = p.inter[s.lo - 1];
      a.out_batch = p.haveStrideInter ? p.strideInter[s.lo - 1] : (uint64_t)p.M * a.Kout;
    } else {
      const int t = (int)(l % 2);
      a.out = tmps[t];
      a.out_batch = (uint64_t)p.M * a.Kout;
      if (zIsTmp[t]) {
        // Z doubles as scratch: the intermediate has to fit the per-batch Z region.
        if (a.Kout > L || (p.batch > 1 && p.strideZ < (uint64_t)p.M * L)) return fastKronInvalidArgument;
        if (p.batch > 1) a.out_batch = p.strideZ;
      }
      if (a.out == nullptr) return fastKronInvalidArgument;
    }
    if (p.inner) {
      a.inner = p.inner;
      a.outer.in = first ? p.outerX : p.inner * a.in_batch;
      a.outer.out = last ? p.outerZ : p.inner * a.out_batch;
      a.outer.y = p.outerY;
    }
    {
      // Non-temporal hints (StepArgs::stream_in / stream_out).  Measured: an intermediate of 134 MB is read back
      // from the memory-side cache by the next launch (non-temporal stores cost 4 % there), one of 268 MB is not
      // (they gain 2 %); X and Z of a launch that moves 268 MB or more with nothing cached gain 2.5 to 4 %, also
      // when Z itself is small (8 x 512 x (32x16)^3: 67 MB of Z behind 537 MB of X, 126.2 -> 121.9 us).
      constexpr uint64_t kStreamFrom = 96ull << 20, kBeyondCache = 192ull << 20;
      const uint64_t es8 = dtypeSize(p.dt);
      const uint64_t inBytes = (uint64_t)p.M * a.Kin * p.batch * es8, outBytes = (uint64_t)p.M * a.Kout * p.batch * es8;
      const uint64_t moved = inBytes + outBytes + (a.y ? outBytes : 0);
      const bool inFromCaller = first && !p.xJustWritten, outToCaller = (last || p.forward) && !p.zReadNext;
      a.stream_in = inFromCaller ? (moved >= kStreamFrom && inBytes >= kStreamFrom / 2) : inBytes > kBeyondCache;
      a.stream_out = outToCaller ? moved >= kStreamFrom : outBytes > kBeyondCache;
    }
    {
      // A temporary that this launch neither reads nor writes, for kernels that keep an intermediate of their own:
      // the first launch reads X and the last writes Z, so one of the two temporaries is idle then.
      void* idle = nullptr;
      if (!p.forward && (first || last)) {
        for (void* t : {temp1, temp2})
          if (t && t != a.in && t != a.out && t != (const void*)p.Z && t != p.X && t != p.Y && !idle) idle = t;
      }
      a.scratch = idle; a.scratch_elems = idle ? tempElems : 0;
      a.sync = callWs_ ? nullptr : syncArea();
    }
    if (logLevel() >= 2)
      printf("[fastkron]   launch %zu: factors [%u,%u] Kin=%llu Kout=%llu kernel %s\n", l, s.lo, s.hi,
             (unsigned long long)a.Kin, (unsigned long long)a.Kout, k.name.c_str());
    // The batch index is a grid dimension (at most 65535): larger batches go out in chunks of that many.
    constexpr uint32_t kMaxGridBatch = 65535;
    const size_t es = dtypeSize(p.dt);
    for (uint32_t b0 = 0; b0 < a.batch; b0 += kMaxGridBatch) {
      StepArgs c = a;
      c.batch = a.batch - b0 < kMaxGridBatch ? a.batch - b0 : kMaxGridBatch;
      c.in = (const char*)a.in + (size_t)b0 * a.in_batch * es;
      c.out = (char*)a.out + (size_t)b0 * a.out_batch * es;
      if (a.y) c.y = (const char*)a.y + (size_t)b0 * a.y_batch * es;
      for (uint32_t j = 0; j < a.nf && j < kMaxFused; j++)
        c.f[j] = (const char*)a.f[j] + (size_t)b0 * a.f_batch[j] * es;
      if (dryRun) {
        StepArgs c2 = c;                                                // (alignment of both batch dimensions)
        if (c.inner) { c2.in_batch = c.outer.in; c2.out_batch = c.outer.out; c2.y_batch = c.outer.y; }
        if (k.check && (!k.check(k, c) || (c.inner && !k.check(k, c2)))) {  // every chunk: its base pointers differ
          if (refused) *refused = s.kernel;
          return fastKronKernelNotFound;
        }
        if (planOnly_) {
          char line[768];
          int n = snprintf(line, sizeof(line), "kernel=%s lo=%u hi=%u M=%u batch=%u Kin=%llu Kout=%llu in=%p out=%p y=%p "
                           "in_batch=%llu out_batch=%llu y_batch=%llu stream_in=%u stream_out=%u f_batch=", k.name.c_str(), s.lo, s.hi, c.M, c.batch,
                           (unsigned long long)c.Kin, (unsigned long long)c.Kout, c.in, c.out, c.y,
                           (unsigned long long)c.in_batch, (unsigned long long)c.out_batch, (unsigned long long)c.y_batch,
                           c.stream_in, c.stream_out);
          launchLog_.append(line, n > 0 ? (size_t)n : 0);
          for (uint32_t j = 0; j < c.nf && j < kMaxFused; j++)
            launchLog_ += (j ? "," : "") + std::to_string(c.f_batch[j]);
          if (c.inner)
            launchLog_ += " inner=" + std::to_string(c.inner) + " outer_in=" + std::to_string(c.outer.in) + " outer_out=" +
                          std::to_string(c.outer.out) + " outer_y=" + std::to_string(c.outer.y);
          launchLog_ += "\n";
        }
        continue;
      }
      if (k.usesSync) {
        // the counter area is one more piece of device state of the handle: a later call on another stream is
        // ordered behind this launch (orderWorkspaceBehind)
        if (mergeWsUsed_ && mergeWsStream_ != stream_) orderWorkspaceBehind(stream_);
        mergeWsStream_ = stream_; mergeWsUsed_ = true;
      }
      hipError_t he = k.launch(k, c, stream_);
      if (he != hipSuccess) {
        fprintf(stderr, "[fastkron] launch of %s failed: %s\n", k.name.c_str(), hipGetErrorString(he));
        return fastKronInvalidArgument;               // reference cuda_kernel_db.cu:296-301
      }
    }
    in = a.out; inBatch = a.out_batch;
  }
  return fastKronSuccess;
}

}  // namespace fk
