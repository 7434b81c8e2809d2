// Host side of libfermihip: device memory, the tensor-contraction engine, the closed-shell
// DF-CCSD residual, the DIIS-accelerated iteration and the (T) driver, plus the C ABI.
//
// The CCSD residual is a factorised form (Fov/Foo/Fvv, Loo/Lvv, Woooo, Wvoov/Wvovo
// intermediates) of the closed-shell term list of Fermi.jl's RCCSDHelper.jl:57-220; it is
// the same function of (T1, T2) and is checked against a term-by-term restatement of that
// file.  The T2 numerator is accumulated as P and symmetrised at the end,
// newT2 = P + P[j,i,b,a] (RCCSDHelper.jl:190).
#include "fh_host.h"
#include "fh_internal.h"
#include "../../include/fermihip.h"

#include <rocblas/rocblas.h>
#include <rocsolver/rocsolver.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>
#include <random>
#include <sstream>
#include <thread>
#include <type_traits>

namespace fh {

static thread_local std::string g_last_error;
void set_error(const std::string& m) { g_last_error = m; }

// ------------------------------------------------------------------ pool
Pool::~Pool() {
  int cur = 0;
  (void)hipGetDevice(&cur);
  (void)hipSetDevice(device_);
  for (auto& kv : free_) (void)hipFree(kv.second);
  for (auto& kv : live_) (void)hipFree(kv.first);
  (void)hipSetDevice(cur);
}
void* Pool::get(size_t bytes) {
  bytes = (bytes + 255) & ~size_t(255);
  auto it = free_.lower_bound(bytes);
  // reuse a free block of at most 25% more than asked
  if (it != free_.end() && it->first <= bytes + bytes / 4) {
    void* p = it->second;
    size_t sz = it->first;
    free_.erase(it);
    live_[p] = sz;
    in_use_ += sz;
    peak_ = std::max(peak_, in_use_);
    return p;
  }
  void* p = nullptr;
  hipError_t e = hipMalloc(&p, bytes);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    release_free();
    e = hipMalloc(&p, bytes);
    if (e != hipSuccess && give_back) {
      (void)hipGetLastError();
      give_back();
      e = hipMalloc(&p, bytes);
    }
    if (e != hipSuccess) {
      (void)hipGetLastError();
      throw Error{-4, "out of device memory allocating " + std::to_string(bytes) + " bytes"};
    }
  }
  live_[p] = bytes;
  in_use_ += bytes;
  peak_ = std::max(peak_, in_use_);
  return p;
}
void Pool::put(void* p) {
  auto it = live_.find(p);
  if (it == live_.end()) return;
  in_use_ -= it->second;
  free_.insert({it->second, p});
  live_.erase(it);
}
void Pool::release_free() {
  for (auto& kv : free_) (void)hipFree(kv.second);
  free_.clear();
}

// ------------------------------------------------------------------ context
struct Phase {
  double ms = 0.0;
  double flops = 0.0;
  double bytes = 0.0;  // algorithmic HBM bytes of the bandwidth-bound phases
  int calls = 0;
};

struct IterRow {
  int ite;
  double e, de, rms, ms;
  bool diis;
};

// Timed spans on the context stream, read back at the next synchronisation point by flush_timers; between
// those, timing waits only for work that many spans have been queued behind.
struct EventRt {
  using Event = hipEvent_t;
  using Stream = hipStream_t;
  static bool create(Event& e) { return hipEventCreate(&e) == hipSuccess; }
  static void destroy(Event e) { (void)hipEventDestroy(e); }
  static bool record(Event e, Stream s) { return hipEventRecord(e, s) == hipSuccess; }
  static bool wait(Event e) { return hipEventSynchronize(e) == hipSuccess; }
  static bool elapsed(float& ms, Event a, Event b) { return hipEventElapsedTime(&ms, a, b) == hipSuccess; }
};

struct BlasHandle {
  rocblas_handle h = nullptr;
  BlasHandle() = default;
  BlasHandle(const BlasHandle&) = delete;
  BlasHandle& operator=(const BlasHandle&) = delete;
  ~BlasHandle() { reset(); }
  void reset() {
    if (h) (void)rocblas_destroy_handle(h);
    h = nullptr;
  }
};

// Pinned chunks for large copies between the device and pageable host memory (copy_staged): 16 MiB, lent by the contexts
// of the process to one another.  (One in each context cost its first such copy 2 ms.)
struct HostStage {
  static constexpr int kThreads = 4;
  static constexpr size_t kChunk = (size_t)2 << 20;
  const int device;
  char* mem = nullptr;
  hipEvent_t ev[kThreads][2] = {};
  explicit HostStage(int d) : device(d) {}
  bool init() {
    void* p = nullptr;
    if (hipHostMalloc(&p, 2 * kThreads * kChunk, hipHostMallocDefault) != hipSuccess) return false;
    mem = static_cast<char*>(p);
    for (auto& t : ev)
      for (hipEvent_t& e : t)
        if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return false;
    return true;
  }
  char* buf(int t, int k) { return mem + (2 * t + k) * kChunk; }
  HostStage(const HostStage&) = delete;
  HostStage& operator=(const HostStage&) = delete;
  ~HostStage() {
    for (auto& t : ev)
      for (hipEvent_t e : t)
        if (e) (void)hipEventDestroy(e);
    if (mem) (void)hipHostFree(mem);
  }
};
static IdlePool<HostStage>& stages() {
  static auto* const p = new IdlePool<HostStage>;   // not torn down at exit, after the HIP runtime
  return *p;
}
struct StageUser {
  StageUser() { stages().enter(); }
  ~StageUser() { stages().leave(); }
  StageUser(const StageUser&) = delete;
  StageUser& operator=(const StageUser&) = delete;
};

struct Ctx {
  int device = 0;
  hipStream_t s = nullptr;
  StageUser stage_user;
  size_t unstaged = 0;   // chunks_worth_making
  BlasHandle blas;   // of the eigensolver, made on first use; given back when an allocation would fail and no solver lives
  int solvers = 0;
  // declared before every Buf member, so that it is destroyed after all of them
  std::unique_ptr<Pool> pool;
  int o = 0, v = 0, naux = 0;
  bool have_df = false, prepared = false;
  bool ov_only = false;  // fh_set_df was given Bov alone (what Fermi's DF-MP2 computes, RMP2a.jl:49-54)
  // fh_set_mo: the conventional (Chonky) MO blocks were handed over instead of B tensors
  // (RCCSDa.jl:25-35); Fia (Fock.jl:32) enters the guess and the energy when given
  bool conventional = false, have_fia = false;
  Buf Fia;
  int lowp = 0;  // residual contractions: 0 FP64 MFMA, 1 FP32 MFMA, 2 split-BF16x3 MFMA (large GEMMs)
  Buf eo, ev, Boo, Bov, Bvv;
  // 4-index blocks (Julia index order, column-major)
  Buf OOOO, OOOV, OOVV, OVOV, OVVV;
  // constants of the residual: LX[k,c,l,d] = 2 (kc|ld) - (kd|lc) and, n2 further, (kd|lc); the ladder's operand
  // Vs[cd, ab] over pairs (prepare_ladder) and Pt[c,d,a,k] = (kd|ac); FP32 copies of LX and Vs for the
  // reduced-precision residual (made on first use)
  Buf LX, Vs, Pt, LX32, Vs32;
  // Lkl[k,l,c,d] = LX[k,c,l,d] and Okl[k,l,i,c] = (ki|lc): the slices of slice_sum
  Buf Lkl, Okl;
  // what T1 multiplies: Lo1[l,c,k,i] = 2 (ki|lc) - (li|kc), L1[k,c,i,a] = 2 (kc|ia) - (ki|ac)
  Buf Lo1, L1;
  // GEMM operands made from the integral blocks above (a permuted FP64 copy, or an FP32 copy for
  // split-BF16x3): the same for every CC iteration, so made once and kept, up to opcache_cap
  // bytes; key "<block>|<index order>|<d or f>"
  std::map<std::string, Buf> opcache;
  size_t opcache_bytes = 0, opcache_cap = 0;
  // device-resident amplitudes (last guess / solve)
  Buf T1, T2;
  bool have_amp = false;
  // scratch for reductions
  Buf partials, scal;
  // learned T2 guess: network parameters (FP32), feature mean / inverse scale, occupied pair
  // distances [o,o]; attached per molecule (fh_set_df detaches it)
  Buf mlp_P, mlp_xm, mlp_xs, pair_d;
  int mlp_h = 0;
  double mlp_ys = 0.0;
  bool have_model = false;
  std::map<std::string, Phase> phases;
  Spans<EventRt> spans;
  std::vector<IterRow> iters;
  double last_energy = 0.0, last_et = 0.0;

  int64_t nov() const { return (int64_t)o * v; }
  int64_t n2() const { return (int64_t)o * o * v * v; }
};

static auto add_span(Ctx& c) {
  return [&c](const Spans<EventRt>::Span& p, float ms) {
    Phase& ph = c.phases[p.name];
    ph.ms += ms;
    ph.flops += p.flops;
    ph.bytes += p.bytes;
    ph.calls += 1;
  };
}
// RAII span timer
struct Timer {
  Ctx& c;
  Spans<EventRt>::Span p;
  hipStream_t st;
  Timer(Ctx& cc, const std::string& n, double f = 0.0, double bytes = 0.0, hipStream_t on = nullptr)
      : c(cc), st(on ? on : cc.s) {
    p.name = n;
    p.flops = f;
    p.bytes = bytes;
    if (!c.spans.begin(p, st)) throw Error{-2, std::string("HIP event: ") + hipGetErrorString(hipGetLastError())};
  }
  Timer(const Timer&) = delete;
  Timer& operator=(const Timer&) = delete;
  ~Timer() { c.spans.end(p, st, add_span(c)); }
};

// resolve recorded spans (call after the stream has been synchronised)
static void flush_timers(Ctx& c) { c.spans.flush(add_span(c)); }

static Buf dalloc(Ctx& c, int64_t n) { return Buf(c.pool.get(), (size_t)std::max<int64_t>(n, 1) * sizeof(double)); }
struct StagedCopy {
  static constexpr int kThreads = HostStage::kThreads;
  static constexpr size_t kChunk = HostStage::kChunk;
  Ctx& c;
  HostStage& st;
  char* dev;
  bool to_host;
  std::atomic<int> err{(int)hipSuccess};
  bool ok(hipError_t e) {
    if (e != hipSuccess) err = (int)e;
    return e == hipSuccess;
  }
  char* buf(int t, int k) { return st.buf(t, k); }
  bool enter() { return ok(hipSetDevice(c.device)); }
  bool start(int t, int k, size_t at, size_t n) {
    return ok(to_host ? hipMemcpyAsync(buf(t, k), dev + at, n, hipMemcpyDeviceToHost, c.s)
                      : hipMemcpyAsync(dev + at, buf(t, k), n, hipMemcpyHostToDevice, c.s));
  }
  bool mark(int t, int k) { return ok(hipEventRecord(st.ev[t][k], c.s)); }
  bool wait(int t, int k) { return ok(hipEventSynchronize(st.ev[t][k])); }
  void drain() { (void)hipStreamSynchronize(c.s); }
};
// Copy of n bytes between the device and pageable host memory in pinned chunks (copy_chunked; pages of new host memory
// are made by four threads at once instead of one).  false: not taken (chunks_pay, chunks_worth_making, memory that
// the runtime knows, which it copies directly, or no pinned memory).  Returns with the host memory free for other use.
// (mu nu|la si) of two water molecules, 42 MB into new memory: 4.7 ms with one pageable copy, 2.2 ms so, 0.6 of them
// kernels.
static bool copy_staged(Ctx& c, char* dev, char* host, size_t n, bool to_host) {
  if (!chunks_pay(n, to_host)) return false;
  hipPointerAttribute_t at{};
  if (hipPointerGetAttributes(&at, host) == hipSuccess) {
    if (at.type != hipMemoryTypeUnregistered) return false;
  } else {
    (void)hipGetLastError();
  }
  std::unique_ptr<HostStage> st = stages().take(c.device);
  if (!st) {
    if (!chunks_worth_making(c.unstaged, n, to_host)) return false;
    st = std::make_unique<HostStage>(c.device);
    if (!st->init()) {
      (void)hipGetLastError();
      return false;
    }
  }
  StagedCopy rt{c, *st, dev, to_host};
  if (!copy_chunked(rt, host, n, to_host)) FH_HIP((hipError_t)rt.err.load());
  stages().give(std::move(st));
  return true;
}
static void h2d(Ctx& c, double* d, const double* h, int64_t n) {
  if (copy_staged(c, reinterpret_cast<char*>(d), reinterpret_cast<char*>(const_cast<double*>(h)), n * sizeof(double), false)) return;
  FH_HIP(hipMemcpyAsync(d, h, n * sizeof(double), hipMemcpyHostToDevice, c.s));
}
static void d2h(Ctx& c, double* h, const double* d, int64_t n) {
  if (copy_staged(c, reinterpret_cast<char*>(const_cast<double*>(d)), reinterpret_cast<char*>(h), n * sizeof(double), true)) return;
  FH_HIP(hipMemcpyAsync(h, d, n * sizeof(double), hipMemcpyDeviceToHost, c.s));
  FH_HIP(hipStreamSynchronize(c.s));
}
static void d2d(Ctx& c, double* d, const double* s, int64_t n) {
  FH_HIP(hipMemcpyAsync(d, s, n * sizeof(double), hipMemcpyDeviceToDevice, c.s));
}
static double read_scalar(Ctx& c, const double* d) {
  double h = 0.0;
  FH_HIP(hipMemcpyAsync(&h, d, sizeof(double), hipMemcpyDeviceToHost, c.s));
  FH_HIP(hipStreamSynchronize(c.s));
  return h;
}

// ------------------------------------------------------------------ contraction engine
// C[ic] = alpha * sum A[ia] B[ib] + beta * C[ic]  (einsum-style single-letter indices,
// column-major tensors in the index order of the strings).  Evaluated as
// permute -> MFMA GEMM -> permute, skipping every permute whose operand is already in a
// GEMM-ready layout (including transposed operands).
struct Letters {
  std::string s;
  const TView* t;
  int64_t dim(char ch) const {
    auto p = s.find(ch);
    return t->dim[p];
  }
};

static int64_t prod_dims(const Letters& L, const std::string& sub) {
  int64_t n = 1;
  for (char ch : sub) n *= L.dim(ch);
  return n;
}

// input strides of `from` (column-major) listed in the order of `to`
static void strides_for(const TView& from, const std::string& fromL, const std::string& toL, int64_t* istr,
                        int64_t* odim) {
  int64_t st[6];
  int64_t acc = 1;
  for (int d = 0; d < from.nd; ++d) { st[d] = acc; acc *= from.dim[d]; }
  for (size_t d = 0; d < toL.size(); ++d) {
    auto p = fromL.find(toL[d]);
    istr[d] = st[p];
    odim[d] = from.dim[p];
  }
}

static void permute_to(Ctx& c, const TView& in, const std::string& inL, double* out, const std::string& outL,
                       double alpha, double beta) {
  int64_t istr[6], odim[6];
  strides_for(in, inL, outL, istr, odim);
  permute_f64(c.s, (int)outL.size(), odim, istr, alpha, in.p, beta, out);
}

static bool is_concat(const std::string& full, const std::string& first, const std::string& second) {
  return full == first + second;
}

// the integral blocks, whose copies contract() keeps
static const char* block_name(const Ctx& c, const TView& X) {
  return X.p == c.OVOV.d() ? "ovov" : X.p == c.OVVV.d() ? "ovvv" : X.p == c.OOOV.d() ? "ooov"
         : X.p == c.OOVV.d() ? "oovv" : X.p == c.OOOO.d() ? "oooo" : X.p == c.LX.d() ? "Lovov"
         : X.p == c.Pt.d() ? "Pt" : nullptr;
}

static void contract(Ctx& c, double alpha, const TView& A, const std::string& ia, const TView& B,
                     const std::string& ib, double beta, const TView& C, const std::string& ic) {
  FH_CHECK((int)ia.size() == A.nd && (int)ib.size() == B.nd && (int)ic.size() == C.nd, -3,
           "contract: index string rank mismatch " + ia + "," + ib + "->" + ic);
  Letters LA{ia, &A}, LB{ib, &B}, LC{ic, &C};
  std::string M, N, K;
  for (char ch : ic) {
    const bool inA = ia.find(ch) != std::string::npos, inB = ib.find(ch) != std::string::npos;
    FH_CHECK(inA != inB, -3, std::string("contract: output index in both/neither operand: ") + ch);
    if (inA) M += ch; else N += ch;
    FH_CHECK((inA ? LA.dim(ch) : LB.dim(ch)) == LC.dim(ch), -3, std::string("contract: size mismatch for ") + ch);
  }
  for (char ch : ia)
    if (ic.find(ch) == std::string::npos) {
      FH_CHECK(ib.find(ch) != std::string::npos, -3, std::string("contract: trace index unsupported: ") + ch);
      FH_CHECK(LA.dim(ch) == LB.dim(ch), -3, std::string("contract: size mismatch for ") + ch);
      K += ch;
    }
  for (char ch : ib)
    FH_CHECK(ic.find(ch) != std::string::npos || ia.find(ch) != std::string::npos, -3,
             std::string("contract: trace index unsupported: ") + ch);

  // output handling: direct (C = M++N), swapped (C = N++M) or via a temporary
  int cmode = 0;  // 0 direct, 1 swapped, 2 temp
  auto sorted = [](std::string x) { std::sort(x.begin(), x.end()); return x; };
  {
    const std::string c1 = ic.substr(0, M.size()), c2 = ic.substr(M.size());
    const std::string d1 = ic.substr(0, N.size()), d2 = ic.substr(N.size());
    if (sorted(c1) == sorted(M) && sorted(c2) == sorted(N)) { cmode = 0; M = c1; N = c2; }
    else if (sorted(d1) == sorted(N) && sorted(d2) == sorted(M)) { cmode = 1; N = d1; M = d2; }
    else {
      cmode = 2;
      // keep operand orders so that A/B may be used as stored
      std::string m2, n2;
      for (char ch : ia) if (M.find(ch) != std::string::npos) m2 += ch;
      for (char ch : ib) if (N.find(ch) != std::string::npos) n2 += ch;
      M = m2; N = n2;
    }
  }
  // choose the K order so that as many operands as possible are GEMM-ready
  std::string KA, KB;
  for (char ch : ia) if (K.find(ch) != std::string::npos) KA += ch;
  for (char ch : ib) if (K.find(ch) != std::string::npos) KB += ch;
  auto fitsA = [&](const std::string& k) { return is_concat(ia, M, k) || is_concat(ia, k, M); };
  auto fitsB = [&](const std::string& k) { return is_concat(ib, k, N) || is_concat(ib, N, k); };
  // (a copy of an integral block is cached below, one of an amplitude made each time)
  std::string Kord = KA;
  if (!(fitsA(KA) && fitsB(KA)) && fitsA(KB) && fitsB(KB)) Kord = KB;
  else if (!fitsA(KA) && fitsB(KB)) Kord = KB;
  else if (!fitsB(KA) && fitsB(KB) && block_name(c, A) && !block_name(c, B)) Kord = KB;

  int64_t Msz = 1, Nsz = 1, Ksz = 1;
  for (char ch : M) Msz *= LA.dim(ch);
  for (char ch : N) Nsz *= LB.dim(ch);
  for (char ch : Kord) Ksz *= LA.dim(ch);

  const int64_t wsz = gemm_splitk_elems(Msz, Nsz, Ksz, 1);
  Buf work;
  if (wsz) work = dalloc(c, wsz);
  // split-BF16x3 for the o^3 v^3-class GEMMs of the mixed phase, on FP32 copies of the operands
  // (half the operand traffic of FP64 loads); smaller GEMMs, the split-K shapes and those of fewer than 64 rows or
  // columns, most of a 128 x 128 tile idle, stay on FP32 MFMA (o x o v^2 x v at o = 28, v = 133: 328 us in split-BF16x3)
  const bool bf3 = c.lowp == 2 && wsz == 0 && std::min(Msz, Nsz) >= 64 && (double)Msz * (double)Nsz * (double)Ksz >= 1e9;

  // The GEMM's copy of an operand: the tensor itself when its index order is GEMM-ready and the
  // GEMM reads FP64, else a permuted and/or FP32 copy.  Copies of the integral blocks go to the
  // operand cache and serve the later calls (every CC iteration makes the same ones).
  auto operand = [&](const TView& X, const std::string& ix, bool ready, const std::string& layout, Buf& tmp,
                     Buf& tmpf) -> const void* {
    if (ready && !bf3) return X.p;
    const char* blk = block_name(c, X);
    std::string key;
    if (blk) {
      // the source index string is part of the key: two contractions that bind the letters to the
      // block's axes differently can ask for the same target layout string
      key = std::string(blk) + "|" + ix + ">" + (ready ? ix : layout) + (bf3 ? "|f" : "|d");
      auto it = c.opcache.find(key);
      if (it != c.opcache.end()) return it->second.p;
    }
    const int64_t n = X.size();
    const double* src = X.p;
    if (!ready) {
      tmp = dalloc(c, n);
      permute_to(c, X, ix, tmp.d(), layout, 1.0, 0.0);
      src = tmp.d();
    }
    Buf* made = &tmp;
    if (bf3) {
      tmpf = Buf(c.pool.get(), (size_t)n * sizeof(float));
      cast_f64_to_f32(c.s, n, src, tmpf.f());
      made = &tmpf;
    }
    const void* out = made->p;
    if (blk) {
      if (!c.opcache_cap) {
        size_t fr = 0, tot = 0;
        FH_HIP(hipMemGetInfo(&fr, &tot));
        c.opcache_cap = std::max<size_t>(1, std::min<size_t>(fr / 4, (size_t)48 << 30));
      }
      if (c.opcache_bytes + made->bytes <= c.opcache_cap) {
        c.opcache_bytes += made->bytes;
        c.opcache[key] = std::move(*made);
      }
    }
    return out;
  };
  // A as logical Msz x Ksz, B as Ksz x Nsz
  Buf tA, tB, tAf, tBf, tC;
  bool transA = false, readyA = true;
  int64_t lda;
  if (is_concat(ia, M, Kord)) { lda = std::max<int64_t>(Msz, 1); }
  else if (is_concat(ia, Kord, M)) { transA = true; lda = std::max<int64_t>(Ksz, 1); }
  else { readyA = false; lda = std::max<int64_t>(Msz, 1); }
  const void* pA = operand(A, ia, readyA, M + Kord, tA, tAf);
  bool transB = false, readyB = true;
  int64_t ldb;
  if (is_concat(ib, Kord, N)) { ldb = std::max<int64_t>(Ksz, 1); }
  else if (is_concat(ib, N, Kord)) { transB = true; ldb = std::max<int64_t>(Nsz, 1); }
  else { readyB = false; ldb = std::max<int64_t>(Ksz, 1); }
  const void* pB = operand(B, ib, readyB, Kord + N, tB, tBf);
  auto gemm = [&](bool ta, bool tb, int64_t m, int64_t n, double al, const void* a, int64_t la, const void* b,
                  int64_t lb, double be, const double* cc, double* d, int64_t ld) {
    if (bf3) {
      const int64_t w3 = gemm_bf3_splitk_elems(ta, tb, m, n, Ksz, 1, 0);
      if (w3) work = dalloc(c, w3);
      gemm_bf3(c.s, ta, tb, m, n, Ksz, al, static_cast<const float*>(a), la, 0, static_cast<const float*>(b), lb, 0, be,
               cc, ld, d, ld, 0, 1, 0, work.d(), w3);
    } else
      gemm_f64(c.s, ta, tb, m, n, Ksz, al, static_cast<const double*>(a), la, 0, static_cast<const double*>(b), lb, 0,
               be, cc, ld, 0, d, ld, 0, 1, 0, work.d(), wsz, c.lowp != 0);
  };
  if (cmode == 0) {
    gemm(transA, transB, Msz, Nsz, alpha, pA, lda, pB, ldb, beta, C.p, C.p, Msz);
  } else if (cmode == 1) {
    // C^T (Nsz x Msz) = op(B)^T op(A)^T
    gemm(!transB, !transA, Nsz, Msz, alpha, pB, ldb, pA, lda, beta, C.p, C.p, Nsz);
  } else {
    tC = dalloc(c, Msz * Nsz);
    gemm(transA, transB, Msz, Nsz, 1.0, pA, lda, pB, ldb, 0.0, nullptr, tC.d(), Msz);
    TView T;
    T.p = tC.d();
    T.nd = (int)(M.size() + N.size());
    int q = 0;
    for (char ch : M) T.dim[q++] = LA.dim(ch);
    for (char ch : N) T.dim[q++] = LB.dim(ch);
    permute_to(c, T, M + N, C.p, ic, alpha, beta);
  }
}

// out[M, N] (+)= alpha sum_z A_z^T B_z over nz slices, A_z [K, M] and B_z [K, N] with K contiguous: index orders
// [k.., m, z] of amplitudes, which one GEMM over (k.., z) would need permuted first.  One batched GEMM into slices
// and their sum.
static void slice_sum(Ctx& c, int64_t M, int64_t N, int64_t K, int64_t nz, double alpha, const double* A, const double* B,
                      double beta, double* out) {
  Buf w = dalloc(c, M * N * nz);
  gemm_f64(c.s, true, false, M, N, K, 1.0, A, K, K * M, B, K, K * N, 0.0, nullptr, 0, 0, w.d(), M, M * N, nz, 0, nullptr, 0,
           c.lowp != 0);
  splitk_reduce_f64(c.s, M, N, nz, w.d(), alpha, beta, out, M, 0, out, M, 0, 1);
}

// out[outL] = alpha * in[inL] + beta * out
static void perm(Ctx& c, const TView& in, const std::string& inL, const TView& out, const std::string& outL,
                 double alpha, double beta) {
  FH_CHECK((int)inL.size() == in.nd && (int)outL.size() == out.nd, -3, "perm: rank mismatch");
  permute_to(c, in, inL, out.p, outL, alpha, beta);
}

// ------------------------------------------------------------------ integrals
static void require_df(Ctx& c, bool full = true) {
  FH_CHECK(c.have_df, -6, "no DF tensors: call fh_set_df first");
  FH_CHECK(!full || !c.ov_only, -6, "only Bov was given to fh_set_df: this entry point needs Boo and Bvv too");
}

static void prepare(Ctx& c) {
  require_df(c);
  if (c.prepared) return;
  if (c.conventional) {  // the blocks came with fh_set_mo
    c.prepared = true;
    return;
  }
  const int keep = c.lowp;
  c.lowp = 0;  // integrals are assembled in FP64
  const int64_t o = c.o, v = c.v, Q = c.naux;
  Timer t(c, "integrals", 2.0 * Q * (double)(o * o * o * o + o * o * o * v + o * o * v * v + o * v * o * v +
                                              o * v * v * v));
  TView Boo = tv(c.Boo.d(), {Q, o, o}), Bov = tv(c.Bov.d(), {Q, o, v}), Bvv = tv(c.Bvv.d(), {Q, v, v});
  c.OOOO = dalloc(c, o * o * o * o);
  c.OOOV = dalloc(c, o * o * o * v);
  c.OOVV = dalloc(c, o * o * v * v);
  c.OVOV = dalloc(c, o * v * o * v);
  c.OVVV = dalloc(c, o * v * v * v);
  // DFERI.jl:83,109,134,151,177
  contract(c, 1.0, Boo, "Qij", Boo, "Qkl", 0.0, tv(c.OOOO.d(), {o, o, o, o}), "ijkl");
  contract(c, 1.0, Boo, "Qij", Bov, "Qka", 0.0, tv(c.OOOV.d(), {o, o, o, v}), "ijka");
  contract(c, 1.0, Boo, "Qij", Bvv, "Qab", 0.0, tv(c.OOVV.d(), {o, o, v, v}), "ijab");
  contract(c, 1.0, Bov, "Qia", Bov, "Qjb", 0.0, tv(c.OVOV.d(), {o, v, o, v}), "iajb");
  contract(c, 1.0, Bov, "Qia", Bvv, "Qbc", 0.0, tv(c.OVVV.d(), {o, v, v, v}), "iabc");
  c.L1.reset();   // the residual's constants follow on first use (prepare_rings, prepare_ladder)
  c.Vs.reset();
  c.Vs32.reset();
  c.Pt.reset();
  c.opcache.clear();  // copies of the previous blocks
  c.opcache_bytes = 0;
  c.prepared = true;
  c.lowp = keep;
}

// The residual's constants of the blocks without VVVV (built on the first residual; (T) does not need them, 4 o^2 v^2 of
// memory): L[k,c,l,d] = 2 (kc|ld) - (kd|lc) and the exchange block (kd|lc) of the ring products, and the forms below them.
static void prepare_rings(Ctx& c) {
  prepare(c);
  if (c.L1.p) return;   // the last one
  const int64_t o = c.o, v = c.v;
  c.LX = dalloc(c, 2 * c.n2());
  TView ovov = tv(c.OVOV.d(), {o, v, o, v});
  perm(c, ovov, "kdlc", tv(c.LX.d() + c.n2(), {o, v, o, v}), "kcld", 1.0, 0.0);
  d2d(c, c.LX.d(), c.LX.d() + c.n2(), c.n2());
  axpby_f64(c.s, c.n2(), 2.0, c.OVOV.d(), -1.0, c.LX.d());
  c.LX32.reset();
  c.Lkl = dalloc(c, c.n2());
  perm(c, tv(c.LX.d(), {o, v, o, v}), "kcld", tv(c.Lkl.d(), {o, o, v, v}), "klcd", 1.0, 0.0);
  c.Okl = dalloc(c, o * o * o * v);
  perm(c, tv(c.OOOV.d(), {o, o, o, v}), "kilc", tv(c.Okl.d(), {o, o, o, v}), "klic", 1.0, 0.0);
  c.Lo1 = dalloc(c, o * o * o * v);
  perm(c, tv(c.OOOV.d(), {o, o, o, v}), "kilc", tv(c.Lo1.d(), {o, v, o, o}), "lcki", 2.0, 0.0);
  perm(c, tv(c.OOOV.d(), {o, o, o, v}), "likc", tv(c.Lo1.d(), {o, v, o, o}), "lcki", -1.0, 1.0);
  c.L1 = dalloc(c, c.n2());
  d2d(c, c.L1.d(), c.OVOV.d(), c.n2());
  perm(c, tv(c.OOVV.d(), {o, o, v, v}), "kiac", tv(c.L1.d(), {o, v, o, v}), "kcia", -1.0, 2.0);
}

// The PP ladder's operands (built on the first residual; (T) does not need them): Vs[cd, ab] = (ca|db) +- (da|cb)
// over c >= d, a >= b (symmetric, then antisymmetric combinations; k_vv_pairs) and Pt[c,d,a,k] = (kd|ac).
// S = tau V needs only the symmetric and antisymmetric parts of tau in (c, d) against those of V, a quarter of
// the flops of the full v^2 x v^2 product; the T1 dressing of V is applied to the o^2 v o product with Pt instead.
static void prepare_ladder(Ctx& c) {
  prepare(c);
  if (c.Vs.p && c.Pt.p) return;
  const int keep = c.lowp;
  c.lowp = 0;
  const int64_t o = c.o, v = c.v, Q = c.naux, np = v * (v + 1) / 2, ldv = vv_pairs_ld(v);
  if (!c.Vs.p) {  // DF: from Bvv (fh_set_mo makes Vs from the conventional VVVV block)
    // (ca|db) for a block of a and every b up to its last, at most 1 GiB at a time
    const int64_t na = std::max<int64_t>(1, std::min<int64_t>(((int64_t)1 << 27) / (v * v * v), std::max<int64_t>(8, v / 8)));
    Timer t(c, "integrals_vvvv", 1.0 * Q * (double)(v * v * v * v));
    Buf Vs = dalloc(c, 2 * ldv * np), T = dalloc(c, std::min(na, v) * v * v * v);
    for (int64_t a0 = 0; a0 < v; a0 += na) {
      const int64_t m = std::min(na, v - a0);
      gemm_f64(c.s, true, false, v * m, v * (a0 + m), Q, 1.0, c.Bvv.d() + Q * v * a0, Q, 0, c.Bvv.d(), Q, 0, 0.0, nullptr, 0,
               0, T.d(), v * m, 0);
      vv_pairs(c.s, (int)v, (int)a0, (int)m, T.d(), v, v * m, v * v * m, false, Vs.d());
    }
    c.Vs = std::move(Vs);   // only whole: T may have failed to be allocated
  }
  c.Pt = dalloc(c, v * v * v * o);
  perm(c, tv(c.OVVV.d(), {o, v, v, v}), "kdac", tv(c.Pt.d(), {v, v, v, o}), "cdak", 1.0, 0.0);
  c.lowp = keep;
}

// ------------------------------------------------------------------ CCSD numerators
// R1 = numerator of the T1 update (RCCSDHelper.jl:57-85); R2 = numerator of the T2 update
// (RCCSDHelper.jl:123-220), both without the diagonal Fock term.
// t1_only: the T1 numerator alone (R2 is not touched)
static void residual(Ctx& c, const double* t1p, const double* t2p, double* R1, double* R2, bool t1_only = false) {
  prepare_rings(c);
  if (!t1_only) prepare_ladder(c);
  const int64_t o = c.o, v = c.v;
  const double o_ = (double)o, v_ = (double)v;
  Timer tm(c, "residual", 0.0);
  TView t1 = tv(const_cast<double*>(t1p), {o, v}), t2 = tv(const_cast<double*>(t2p), {o, o, v, v});
  TView ovov = tv(c.OVOV.d(), {o, v, o, v}), oooo = tv(c.OOOO.d(), {o, o, o, o}), oovv = tv(c.OOVV.d(), {o, o, v, v});
  TView ovvv = tv(c.OVVV.d(), {o, v, v, v}), ooov = tv(c.OOOV.d(), {o, o, o, v}), Lovov = tv(c.LX.d(), {o, v, o, v});
  TView r1 = tv(R1, {o, v});
  const int64_t n2 = c.n2(), ov = o * v, np = v * (v + 1) / 2, mp = o * (o + 1) / 2, ldv = vv_pairs_ld(v);

  Buf bFov = dalloc(c, o * v), bLoo = dalloc(c, o * o), bLvv = dalloc(c, v * v);
  TView Fov = tv(bFov, {o, v}), Loo = tv(bLoo, {o, o}), Lvv = tv(bLvv, {v, v});
  // forms of the amplitudes (k_amp_forms).  Split-BF16x3 takes the ring operands in FP32 where its GEMM is used
  // (the o^3 v^3 products of at least 1e9 elements, as in contract); the ladder's pairs are FP32 in both
  // reduced precisions
  const bool ring32 = c.lowp == 2 && (double)ov * (double)ov * (double)ov >= 1e9;
  Buf bu = dalloc(c, n2), btau, bring, bpair;
  if (t1_only) {
    amp_forms<double, double>(c.s, (int)o, (int)v, t1p, t2p, bu.d(), nullptr, nullptr, nullptr);
  } else {
    btau = dalloc(c, n2);
    bring = Buf(c.pool.get(), (size_t)(2 * n2) * (ring32 ? sizeof(float) : sizeof(double)));
    bpair = Buf(c.pool.get(), (size_t)(2 * mp * np) * (c.lowp ? sizeof(float) : sizeof(double)));
    if (ring32) amp_forms<float, float>(c.s, (int)o, (int)v, t1p, t2p, bu.d(), btau.d(), bring.f(), bpair.f());
    else if (c.lowp) amp_forms<double, float>(c.s, (int)o, (int)v, t1p, t2p, bu.d(), btau.d(), bring.d(), bpair.f());
    else amp_forms<double, double>(c.s, (int)o, (int)v, t1p, t2p, bu.d(), btau.d(), bring.d(), bpair.d());
  }
  TView u = tv(bu, {o, o, v, v});

  // Fov[k,c] = L[k,c,l,d] t1[l,d]
  // Loo[k,i] = L[k,c,l,d] t2[i,l,c,d] + (2 (ki|lc) - (li|kc)) t1[l,c] + Fov[k,c] t1[i,c] with L t2 = (kc|ld) u[i,l,c,d]
  // Lvv[a,c] = -L[k,c,l,d] t2[k,l,a,d] - t1[k,a] Fov[k,c] + 2 (kd|ac) t1[k,d] - (kc|ad) t1[k,d]
  contract(c, 1.0, Lovov, "kcld", t1, "ld", 0.0, Fov, "kc");
  if (!t1_only && !ring32)
    contract(c, 1.0, ovov, "kcld", tv(bring.d(), {o, v, o, v}), "icld", 0.0, Loo, "ki");
  else
    contract(c, 1.0, ovov, "kcld", u, "ilcd", 0.0, Loo, "ki");
  contract(c, 1.0, tv(c.Lo1.d(), {o, v, o, o}), "lcki", t1, "lc", 1.0, Loo, "ki");
  slice_sum(c, v, v, o * o, v, -1.0, t2p, c.Lkl.d(), 0.0, Lvv.p);
  contract(c, -1.0, t1, "ka", Fov, "kc", 1.0, Lvv, "ac");
  contract(c, 2.0, ovvv, "kdac", t1, "kd", 1.0, Lvv, "ac");
  contract(c, -1.0, ovvv, "kcad", t1, "kd", 1.0, Lvv, "ac");

  // ---- T1 numerator (Fov[k,c] t1[i,c] t1[k,a] appears with both signs: Loo takes it after its product here)
  contract(c, 1.0, Lvv, "ac", t1, "ic", 0.0, r1, "ia");
  contract(c, -1.0, Loo, "ki", t1, "ka", 1.0, r1, "ia");
  contract(c, 1.0, tv(c.L1.d(), {o, v, o, v}), "kcia", t1, "kc", 1.0, r1, "ia");
  if (!t1_only && !ring32)
    contract(c, 1.0, Fov, "kc", tv(bring.d(), {o, v, o, v}), "kcia", 1.0, r1, "ia");
  else
    contract(c, 1.0, Fov, "kc", u, "kica", 1.0, r1, "ia");
  contract(c, 1.0, ovvv, "kdac", u, "ikcd", 1.0, r1, "ia");
  slice_sum(c, o, v, o * o, v, -1.0, c.Okl.d(), u.p, 1.0, r1.p);
  if (t1_only) return;
  bu.reset();
  contract(c, 1.0, Fov, "kc", t1, "ic", 1.0, Loo, "ki");

  // ---- T2 numerator: P, the ring products and the ladder, then R2 = P + P[j,i,b,a] + ... (k_t2_numerator)
  TView tau = tv(btau, {o, o, v, v});
  Buf bP = dalloc(c, n2);
  TView P = tv(bP, {o, o, v, v});
  perm(c, ovov, "iajb", P, "ijab", 0.5, 0.0);                       // (ia|jb)  (:134)
  // (a term may enter as itself or with (i,a) and (j,b) exchanged: each in the form whose GEMM writes P in place)
  contract(c, 1.0, t1, "ic", ovvv, "jbca", 1.0, P, "ijab");          // T1 x (ia|cb)
  // Y[i,j,a,k], the part of P that T1 completes as -Y[i,j,a,k] t1[k,b]: (ka|ij) terms here, the ladder's below
  Buf bY = dalloc(c, o * o * v * o);
  TView Y = tv(bY, {o, o, v, o});
  perm(c, ooov, "jkia", Y, "ijak", 1.0, 0.0);
  contract(c, 1.0, t1, "ic", oovv, "kjac", 1.0, Y, "ijak");
  contract(c, 1.0, ovov, "kcia", t1, "jc", 1.0, Y, "ijak");
  {
    // Woooo[k,l,i,j] = (ki|lj) + (ki|lc) t1[j,c] + (lj|kc) t1[i,c] + (kc|ld) tau[i,j,c,d]
    Buf bw = dalloc(c, o * o * o * o);
    TView W = tv(bw, {o, o, o, o});
    perm(c, oooo, "kilj", W, "klij", 1.0, 0.0);
    contract(c, 1.0, ooov, "kilc", t1, "jc", 1.0, W, "klij");
    contract(c, 1.0, ooov, "ljkc", t1, "ic", 1.0, W, "klij");
    contract(c, 1.0, ovov, "kcld", tau, "ijcd", 1.0, W, "klij");
    contract(c, 0.5, W, "klij", tau, "klab", 1.0, P, "ijab");
  }
  // particle-particle ladder sum_cd tau[i,j,c,d] ((ca|db) - (kd|ac) t1[k,b] - (kc|bd) t1[k,a]): the first part over
  // packed pairs (prepare_ladder), the others as Y += tau[i,j,c,d] (kd|ac)
  Buf bS = dalloc(c, 2 * mp * np);
  {
    const double fl = 4.0 * (double)mp * (double)np * (double)np;
    if (c.lowp && !c.Vs32.p) {
      c.Vs32 = Buf(c.pool.get(), (size_t)(2 * ldv * np) * sizeof(float));
      cast_f64_to_f32(c.s, 2 * ldv * np, c.Vs.d(), c.Vs32.f());
    }
    const int64_t wl = c.lowp == 2 ? gemm_bf3_splitk_elems(false, false, mp, np, np, 2, 1) : gemm_splitk_elems(mp, np, np, 2);
    Buf work;
    if (wl) work = dalloc(c, wl);
    Timer tl(c, c.lowp == 2 ? "ladder_bf16x3" : (c.lowp ? "ladder_fp32" : "ladder"), fl);
    if (!c.lowp)
      gemm_f64(c.s, false, false, mp, np, np, 1.0, bpair.d(), mp, mp * np, c.Vs.d(), ldv, ldv * np, 0.0, nullptr, 0, 0,
               bS.d(), mp, mp * np, 2, /*tag: PP ladder*/ 1, work.d(), wl);
    else if (c.lowp == 2)
      gemm_bf3(c.s, false, false, mp, np, np, 1.0, bpair.f(), mp, mp * np, c.Vs32.f(), ldv, ldv * np, 0.0, nullptr, 0,
               bS.d(), mp, mp * np, 2, 1, work.d(), wl);
    else
      gemm_f32_fd(c.s, mp, np, np, 1.0, bpair.f(), mp, mp * np, c.Vs32.f(), ldv, ldv * np, 0.0, nullptr, 0, bS.d(), mp,
                  mp * np, 2, 1, work.d(), wl);
  }
  bpair.reset();
  {
    Timer tl(c, "ladder_t1", 2.0 * (double)n2 * (double)ov + 2.0 * (double)n2 * o_);
    contract(c, 1.0, tau, "ijcd", tv(c.Pt.d(), {v, v, v, o}), "cdak", 1.0, Y, "ijak");
    contract(c, -1.0, Y, "ijak", t1, "kb", 1.0, P, "ijab");
  }
  // Lvv[a,c] t2[i,j,c,b]: a product for each b
  {
    const int64_t wl = gemm_splitk_elems(o * o, v, v, v);
    Buf work;
    if (wl) work = dalloc(c, wl);
    gemm_f64(c.s, false, true, o * o, v, v, 1.0, t2p, o * o, o * o * v, Lvv.p, v, 0, 1.0, P.p, o * o, o * o * v, P.p, o * o,
             o * o * v, v, 0, work.d(), wl, c.lowp != 0);
  }
  contract(c, -1.0, Loo, "ki", t2, "kjab", 1.0, P, "ijab");
  // Rings.  With A = Wvoov[i,a,k,c] and B = Wvovo[i,a,k,c] (operators of the ring and crossed ring) the three
  // applications A u - B t2 - (crossed) B t2 are
  //   C u / 2 - Z / 2 - Z[ibja],  C = 2 A - B,  Z[iajb] = B[iakc] t2[kjbc],
  // and the (kc|ld) t2 parts of C and B are L u / 2 and -(kd|lc) t2[ilda] / 2: four o^3 v^3 products over (o v)
  // square matrices in [i,a,j,b] order, in two batches of two.
  Buf bD = dalloc(c, 2 * n2);
  {
    Timer tr(c, c.lowp == 2 ? "ring_bf16x3" : (c.lowp ? "ring_fp32" : "ring"), 4.0 * 2.0 * o_ * o_ * o_ * v_ * v_ * v_);
    Buf bW = dalloc(c, 2 * n2), bXX = dalloc(c, o * o * o * v);
    TView Cw = tv(bW.d(), {o, v, o, v}), Bw = tv(bW.d() + n2, {o, v, o, v});
    perm(c, oovv, "kiac", Bw, "iakc", 1.0, 0.0);
    contract(c, 1.0, t1, "id", ovvv, "kdac", 1.0, Bw, "iakc");
    TView Z = tv(bXX, {o, o, o, v});
    // Z[k,i,l,c] = (ki|lc) + (lc|kd) t1[i,d]
    perm(c, ooov, "kilc", Z, "kilc", 1.0, 0.0);
    contract(c, 1.0, ovov, "lckd", t1, "id", 1.0, Z, "kilc");
    contract(c, -1.0, Z, "kilc", t1, "la", 1.0, Bw, "iakc");
    // C = 2 A - B: 2 (ia|kc) + 2 (kc|ad) t1[i,d] - 2 ((li|kc) + (ld|kc) t1[i,d]) t1[l,a] - B
    d2d(c, Cw.p, Bw.p, n2);
    axpby_f64(c.s, n2, 2.0, c.OVOV.d(), -1.0, Cw.p);
    contract(c, 2.0, t1, "id", ovvv, "kcad", 1.0, Cw, "iakc");
    perm(c, ooov, "likc", Z, "likc", 1.0, 0.0);
    contract(c, 1.0, ovov, "ldkc", t1, "id", 1.0, Z, "likc");
    contract(c, -2.0, Z, "likc", t1, "la", 1.0, Cw, "iakc");
    // [C | B] += 1/2 [u | -t2[ilda]] [L | (lc|kd)], then [D | F] = [C | B] [u | -t2[kjbc]]
    if (ring32) {
      if (!c.LX32.p) {
        c.LX32 = Buf(c.pool.get(), (size_t)(2 * n2) * sizeof(float));
        cast_f64_to_f32(c.s, 2 * n2, c.LX.d(), c.LX32.f());
      }
      gemm_bf3(c.s, false, false, ov, ov, ov, 0.5, bring.f(), ov, n2, c.LX32.f(), ov, n2, 1.0, bW.d(), ov, bW.d(), ov, n2, 2, 0);
      Buf bW32(c.pool.get(), (size_t)(2 * n2) * sizeof(float));
      cast_f64_to_f32(c.s, 2 * n2, bW.d(), bW32.f());
      gemm_bf3(c.s, false, false, ov, ov, ov, 1.0, bW32.f(), ov, n2, bring.f(), ov, n2, 0.0, nullptr, 0, bD.d(), ov, n2, 2, 0);
    } else {
      const int64_t wl = gemm_splitk_elems(ov, ov, ov, 2);
      Buf work;
      if (wl) work = dalloc(c, wl);
      gemm_f64(c.s, false, false, ov, ov, ov, 0.5, bring.d(), ov, n2, c.LX.d(), ov, n2, 1.0, bW.d(), ov, n2, bW.d(), ov, n2,
               2, 0, work.d(), wl, c.lowp != 0);
      gemm_f64(c.s, false, false, ov, ov, ov, 1.0, bW.d(), ov, n2, bring.d(), ov, n2, 0.0, nullptr, 0, 0, bD.d(), ov, n2, 2,
               0, work.d(), wl, c.lowp != 0);
    }
  }
  t2_numerator(c.s, (int)o, (int)v, P.p, bD.d(), bD.d() + n2, bS.d(), R2);   // (:190)
}

static double energy(Ctx& c, const double* t1, const double* t2) {
  prepare(c);
  if (!c.partials.p) c.partials = dalloc(c, 4096);
  if (!c.scal.p) c.scal = dalloc(c, 64);
  {
    // reads T2 and (kc|ld) once each (T1 is o v): 16 B per o^2 v^2 element
    Timer t(c, "cc_energy", 0.0, 16.0 * (double)c.n2());
    cc_energy(c.s, c.o, c.v, t1, t2, c.OVOV.d(), c.partials.d(), c.scal.d());
  }
  if (c.have_fia) {
    // the conventional-integral variant adds 2 sum f[k,c] T1[k,c] (RCCSDHelper.jl:32-49)
    dot_f64(c.s, c.nov(), c.Fia.d(), t1, c.partials.d() + 2048, c.scal.d() + 3);
    double h[4];
    FH_HIP(hipMemcpyAsync(h, c.scal.d(), 4 * sizeof(double), hipMemcpyDeviceToHost, c.s));
    FH_HIP(hipStreamSynchronize(c.s));
    return h[0] + 2.0 * h[3];
  }
  return read_scalar(c, c.scal.d());
}

// newT = residual(T) ./ D; returns rms of (newT1 - T1), (newT2 - T2); errors optionally kept
// New amplitudes; the sums of their squared changes (T1, T2) go to c.scal[0], [1]
static void update_amp(Ctx& c, const double* t1, const double* t2, double* n1, double* n2, void* e1, void* e2, bool f32) {
  residual(c, t1, t2, n1, n2);
  if (!c.partials.p) c.partials = dalloc(c, 4096);
  if (!c.scal.p) c.scal = dalloc(c, 64);
  int64_t nb = 0;
  jacobi_update(c.s, c.o, c.v, false, c.eo.d(), c.ev.d(), n1, t1, e1, f32, c.partials.d(), &nb);
  sum_partials(c.s, nb, c.partials.d(), c.scal.d());
  {
    // T2 update: read the numerator and the old T2, write the new T2 (24 B) and the error (4 or 8 B)
    Timer t(c, "jacobi", 0.0, (24.0 + (e2 ? (f32 ? 4.0 : 8.0) : 0.0)) * (double)c.n2());
    jacobi_update(c.s, c.o, c.v, true, c.eo.d(), c.ev.d(), n2, t2, e2, f32, c.partials.d() + 2048, &nb);
    sum_partials(c.s, nb, c.partials.d() + 2048, c.scal.d() + 1);
  }
}

// DF-MP2 correlation energy RMP2_energy (RMP2a.jl:91-144) from Bov and the orbital energies alone:
// the reference's pairs i <= j, every pair and tile of (ia|jb) reduced to energy where it is made
// (fh_mp2.hip), so nothing but the partial sums is stored.
static double mp2_energy(Ctx& c) {
  require_df(c, false);
  FH_CHECK(!c.conventional, -6, "fh_mp2_energy: the DF-MP2 energy needs BOV; this context holds conventional blocks");
  const int o = c.o, v = c.v;
  Timer t(c, "df_mp2", (double)c.naux * (double)o * (o + 1.0) * (double)v * (double)v);
  const int64_t np = mp2_partials(o, v);
  Buf part = dalloc(c, np);
  mp2_pair_energy(c.s, o, v, c.naux, c.Bov.d(), c.eo.d(), c.ev.d(), part.d());
  if (!c.scal.p) c.scal = dalloc(c, 64);
  sum_partials(c.s, np, part.d(), c.scal.d() + 2);
  return read_scalar(c, c.scal.d() + 2);
}

// ------------------------------------------------------------------ allocation-free DF-MP2 energy
// fh_mp2_energy_noalloc keeps its intermediates (the partial sums) in this file-scope device array
// instead of allocating them.  Each GPU holds its
// own copy (128 MiB) from the library's load to the end of the process.  In host code `scratch` is
// only a host-side stand-in for the symbol: its device address on each device comes from
// hipGetSymbolAddress at fh_create (with that device current) and is kept in g_scratch[device].
constexpr int64_t kNoAllocDoubles = (int64_t)16 << 20;
static __device__ __align__(256) double scratch[kNoAllocDoubles];
constexpr int kNoAllocMaxDevices = 64;
static std::mutex g_scratch_mu;
static double* g_scratch[kNoAllocMaxDevices] = {};

// once per device, with that device current
static void init_noalloc_scratch(int device) {
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (device < 0 || device >= kNoAllocMaxDevices || g_scratch[device]) return;
  void* p = nullptr;
  FH_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  g_scratch[device] = static_cast<double*>(p);
}

static double* noalloc_scratch(int device) {
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  return (device >= 0 && device < kNoAllocMaxDevices) ? g_scratch[device] : nullptr;
}

// The sizes that the entry point takes: those whose [Q, b, j] copy of Bov, (ia|jb) blocks of some nj values of j and up
// to 2048 partial sums a block would fit the scratch array.  The pair kernel needs its partial sums only (at most 16384),
// but callers size their problems by this limit, and a size that was refused is refused.
static bool noalloc_mp2_fits(int64_t o, int64_t v, int64_t Q) {
  const int64_t ov = o * v;
  for (int64_t nj = std::min<int64_t>(o, std::max<int64_t>(1, (kNoAllocDoubles - Q * ov) / (ov * v))); nj >= 1; --nj)
    if (Q * ov + ov * v * nj + (o + nj - 1) / nj * std::min<int64_t>(v * nj, 2048) <= kNoAllocDoubles) return true;
  return false;
}

// The DF-MP2 energy of mp2_energy() from device-resident eps_o, eps_v, Bov into the device double
// *E, the partial sums in the scratch array.  Nothing in it has to start at zero: the pair kernel
// writes every partial sum.
static void mp2_energy_noalloc(Ctx& c, int o, int v, int naux, const double* eo, const double* ev, const double* Bov,
                               double* E) {
  double* part = noalloc_scratch(c.device);
  FH_CHECK(part != nullptr, -6, "fh_mp2_energy_noalloc: no scratch address for this device (fh_create sets it)");
  FH_CHECK(noalloc_mp2_fits(o, v, naux), -1,
           "fh_mp2_energy_noalloc: naux o v + o v^2 + partial sums exceed the 128 MiB scratch (16777216 doubles)");
  mp2_pair_energy(c.s, o, v, naux, Bov, eo, ev, part);
  sum_partials(c.s, mp2_partials(o, v), part, E);
}

static void mp2_guess(Ctx& c) {
  prepare(c);
  const int64_t o = c.o, v = c.v;
  if (!c.T1.p) c.T1 = dalloc(c, o * v);
  if (!c.T2.p) c.T2 = dalloc(c, c.n2());
  perm(c, tv(c.OVOV.d(), {o, v, o, v}), "iajb", tv(c.T2.d(), {o, o, v, v}), "ijab", 1.0, 0.0);
  if (!c.partials.p) c.partials = dalloc(c, 4096);
  int64_t nb = 0;
  Buf zero = dalloc(c, c.n2());
  fill_f64(c.s, c.n2(), 0.0, zero.d());
  jacobi_update(c.s, c.o, c.v, true, c.eo.d(), c.ev.d(), c.T2.d(), zero.d(), nullptr, false, c.partials.d(), &nb);
  // T1 = Fia ./ D1 (RCCSDa.jl:53,84): zero for canonical RHF orbitals (Fock.jl:95), the given Fia of
  // a conventional context (Fock.jl:32)
  if (c.have_fia) {
    d2d(c, c.T1.d(), c.Fia.d(), o * v);
    jacobi_update(c.s, c.o, c.v, false, c.eo.d(), c.ev.d(), c.T1.d(), zero.d(), nullptr, false, c.partials.d(), &nb);
  } else {
    fill_f64(c.s, o * v, 0.0, c.T1.d());
  }
  c.have_amp = true;
}

// learned guess: MP2 amplitudes plus the network's symmetrised correction, evaluated in chunks
// T1 = R1(T1 = 0, T2) / D1 at the guess's T2: the first-order T1 (the T1 that the first CC
// iteration from T1 = 0 would produce), so that the iterations start with both amplitude sets
// close to the solution
static void first_order_t1(Ctx& c) {
  Timer t(c, "t1_first_order", 0.0);
  const int keep = c.lowp;
  c.lowp = 0;
  Buf r1 = dalloc(c, c.nov()), zero = dalloc(c, c.nov());
  fill_f64(c.s, c.nov(), 0.0, zero.d());
  residual(c, zero.d(), c.T2.d(), r1.d(), nullptr, true);
  if (!c.partials.p) c.partials = dalloc(c, 4096);
  int64_t nb = 0;
  jacobi_update(c.s, c.o, c.v, false, c.eo.d(), c.ev.d(), r1.d(), zero.d(), nullptr, false, c.partials.d(), &nb);
  d2d(c, c.T1.d(), r1.d(), c.nov());
  c.lowp = keep;
}

static void learned_guess(Ctx& c) {
  FH_CHECK(c.have_model, -6, "no T2-guess model: call fh_set_t2_model after fh_set_df");
  mp2_guess(c);
  Timer t(c, "t2_guess_learned", 0.0);
  const int h = c.mlp_h;
  const int64_t n = c.n2();
  if (t2_mlp_fused_available(h)) {
    Buf Y(c.pool.get(), (size_t)n * sizeof(float)), ws(c.pool.get(), t2_mlp_fused_scratch_bytes());
    t2_mlp_fused(c.s, (int)c.o, (int)c.v, c.T2.d(), c.eo.d(), c.ev.d(), c.pair_d.d(), c.mlp_xm.f(), c.mlp_xs.f(),
                 c.mlp_P.f(), ws.p, Y.f());
    t2_learned_apply(c.s, (int)c.o, (int)c.v, c.mlp_ys, Y.f(), c.T2.d());
    return;
  }
  // other widths: layer by layer (FP32-MFMA GEMMs), in chunks of amplitudes
  const int64_t C = std::min<int64_t>(n, (int64_t)1 << 20);
  Buf X(c.pool.get(), (size_t)(6 * C) * sizeof(float)), A(c.pool.get(), (size_t)(3 * h * C) * sizeof(float));
  Buf Y(c.pool.get(), (size_t)n * sizeof(float));
  float* A1 = A.f();
  float* A2 = A1 + (int64_t)h * C;
  float* A3 = A2 + (int64_t)h * C;
  for (int64_t e0 = 0; e0 < n; e0 += C) {
    const int64_t m = std::min<int64_t>(C, n - e0);
    t2_features(c.s, (int)c.o, (int)c.v, e0, m, c.T2.d(), c.eo.d(), c.ev.d(), c.pair_d.d(), c.mlp_xm.f(),
                c.mlp_xs.f(), X.f());
    mlp_forward(c.s, h, c.mlp_P.f(), m, X.f(), A1, A2, A3, Y.f() + e0);
  }
  t2_learned_apply(c.s, (int)c.o, (int)c.v, c.mlp_ys, Y.f(), c.T2.d());
}

// ------------------------------------------------------------------ DIIS (DIIS.jl:21-96)
struct DIIS {
  Ctx& c;
  int64_t n;
  int maxv;
  bool f32;
  std::vector<Buf> vecs, errs;
  std::vector<std::vector<double>> B;   // B[a][b] = errs[a] . errs[b], b <= a
  Buf part;
  int slot;                             // the newest row's place in c.scal, until resolve() takes it from a host copy
  bool pending = false;
  const char* phase;  // timer name of the vector work (nullptr: untimed)
  DIIS(Ctx& cc, int64_t nn, int m, bool f, int sl, const char* ph = nullptr)
      : c(cc), n(nn), maxv(m), f32(f), slot(sl), phase(ph) {
    part = dalloc(c, 8 * reduce_blocks_needed(n));
    if (!c.scal.p) c.scal = dalloc(c, 64);
  }
  double esz() const { return f32 ? 4.0 : 8.0; }
  std::unique_ptr<Timer> timer(double bytes) {
    return std::unique_ptr<Timer>(phase ? new Timer(c, phase, 0.0, bytes) : nullptr);
  }
  // the products of the newest error vector, from a host copy of c.scal made after push()
  void resolve(const double* scal) {
    if (!pending) return;
    B.emplace_back(scal + slot, scal + slot + errs.size());
    pending = false;
  }
  // push! takes ownership of the error buffer and copies the vector
  void push(const double* vec, Buf&& err) {
    if ((int)vecs.size() + 1 > maxv) {
      int idx = 0;
      double best = -1.0;
      for (size_t q = 0; q < errs.size(); ++q) {
        const double nq = std::sqrt(B[q][q]);
        if (nq > best) { best = nq; idx = (int)q; }   // findmax: first maximum
      }
      vecs.erase(vecs.begin() + idx);
      errs.erase(errs.begin() + idx);
      B.erase(B.begin() + idx);
      for (size_t q = idx; q < B.size(); ++q) B[q].erase(B[q].begin() + idx);
    }
    Buf vb = dalloc(c, n);
    {
      auto t = timer(16.0 * (double)n);
      d2d(c, vb.d(), vec, n);
    }
    vecs.push_back(std::move(vb));
    errs.push_back(std::move(err));
    const void* xs[8];
    for (size_t q = 0; q < errs.size(); ++q) xs[q] = errs[q].p;
    auto t = timer(esz() * (double)errs.size() * (double)n);
    dots(c.s, n, (int)errs.size(), xs, errs.back().p, f32, part.d(), c.scal.d() + slot);
    pending = true;
  }
  void extrapolate(double* out, bool add_res) {
    const int m = (int)vecs.size();
    FH_CHECK(m >= 2, -3, "DIIS cannot extrapolate from one vector");
    const int N = m + 1;
    std::vector<double> A(N * N, 1.0), x(N, 0.0);
    A[(N - 1) * N + (N - 1)] = 0.0;
    for (int a = 0; a < m; ++a)
      for (int b = 0; b <= a; ++b) A[a * N + b] = A[b * N + a] = B[a][b];
    x[N - 1] = 1.0;
    // B \ rhs by LU with partial pivoting (row-major)
    for (int k = 0; k < N; ++k) {
      int p = k;
      for (int r = k + 1; r < N; ++r)
        if (std::fabs(A[r * N + k]) > std::fabs(A[p * N + k])) p = r;
      if (p != k) {
        for (int cc = 0; cc < N; ++cc) std::swap(A[k * N + cc], A[p * N + cc]);
        std::swap(x[k], x[p]);
      }
      FH_CHECK(A[k * N + k] != 0.0, -5, "DIIS: singular B matrix");
      for (int r = k + 1; r < N; ++r) {
        const double f = A[r * N + k] / A[k * N + k];
        for (int cc = k; cc < N; ++cc) A[r * N + cc] -= f * A[k * N + cc];
        x[r] -= f * x[k];
      }
    }
    for (int k = N - 1; k >= 0; --k) {
      double sacc = x[k];
      for (int cc = k + 1; cc < N; ++cc) sacc -= A[k * N + cc] * x[cc];
      x[k] = sacc / A[k * N + k];
    }
    std::vector<const double*> xs(m);
    std::vector<const void*> es(m);
    for (int q = 0; q < m; ++q) { xs[q] = vecs[q].d(); es[q] = errs[q].p; }
    auto t = timer((8.0 * m + (add_res ? esz() * m : 0.0) + 8.0) * (double)n);
    lincomb(c.s, n, m, xs.data(), x.data(), es.data(), f32, add_res, out);
  }
};

// ------------------------------------------------------------------ DF-RHF SCF (RHFa.jl:67-223)
// Symmetric eigensolver on the device (rocSOLVER syevd, the divide-and-conquer LAPACK method):
// A (n x n, column-major) is overwritten by the eigenvectors, w gets the eigenvalues ascending, as
// eigen(Symmetric(A), sortby = x -> x) orders them.
//
// Up to n = 1024 the context keeps the rocBLAS handle and with it the solver's workspace (some 170 MiB), which a
// handle of one call allocates and frees each time, until an allocation would fail (Pool::give_back); above, a handle
// lives as long as the solver.
//
// From n = 3 to 160, what a workgroup's registers hold, the matrix is made tridiagonal and the eigenvectors of T turned
// back by fh_eigen.hip, rocSOLVER does what lies between: n = 96 0.15 + 0.03 ms for the two against 0.62 + 0.2 in dsyevd,
// the whole SCF of 24, 64, 96, 128, 160 functions 7.0, 10.5, 13.6, 16.9, 21.0 ms against 10.7, 21.8, 20.5, 26.9, 36.9.
struct Eigen {
  Ctx& c;
  struct Alive {
    int& n;
    explicit Alive(int& m) : n(m) { ++n; }
    ~Alive() { --n; }
  } alive;
  BlasHandle own;
  rocblas_handle h = nullptr;
  Buf work, info, tau, Z;
  int n;
  Eigen(Ctx& cc, int nn) : c(cc), alive(cc.solvers), n(nn) {
    BlasHandle& b = n <= 1024 ? c.blas : own;
    if (!b.h) FH_CHECK(rocblas_create_handle(&b.h) == rocblas_status_success, -2, "rocblas_create_handle failed");
    h = b.h;
    FH_CHECK(rocblas_set_stream(h, c.s) == rocblas_status_success, -2, "rocblas_set_stream failed");
    work = dalloc(c, n);
    info = dalloc(c, 1);
    if (tridiag_fits(n)) {
      tau = dalloc(c, n);
      Z = dalloc(c, 2 * (int64_t)n * n);
    }
  }
  void run(double* A, double* w) {
    if (tridiag_fits(n)) {
      double* const V = Z.d() + (int64_t)n * n;
      tridiag(c.s, n, A, V, w, work.d(), tau.d());
      FH_CHECK(rocsolver_dstedc(h, rocblas_evect_tridiagonal, n, w, work.d(), Z.d(), n,
                                reinterpret_cast<rocblas_int*>(info.p)) == rocblas_status_success, -2,
               "rocsolver_dstedc failed");
      tridiag_apply(c.s, n, V, tau.d(), Z.d(), A);
    } else {
      FH_CHECK(rocsolver_dsyevd(h, rocblas_evect_original, rocblas_fill_upper, n, A, n, w, work.d(),
                                reinterpret_cast<rocblas_int*>(info.p)) == rocblas_status_success, -2,
               "rocsolver_dsyevd failed");
    }
    rocblas_int hi = 0;
    FH_HIP(hipMemcpyAsync(&hi, info.p, sizeof(hi), hipMemcpyDeviceToHost, c.s));
    FH_HIP(hipStreamSynchronize(c.s));
    FH_CHECK(hi == 0, -5, "eigensolver did not converge (info " + std::to_string(hi) + ")");
  }
};

// C = alpha op(A) op(B) + beta C for the SCF's small dense matrices (FP64 MFMA; split-K workspace
// from the pool when the shape asks for it)
static void mm(Ctx& c, bool ta, bool tb, int64_t M, int64_t N, int64_t K, double alpha, const double* A, int64_t lda,
               const double* B, int64_t ldb, double beta, double* C, int64_t ldc) {
  const int64_t wsz = gemm_splitk_elems(M, N, K, 1);
  Buf work;
  if (wsz) work = dalloc(c, wsz);
  gemm_f64(c.s, ta, tb, M, N, K, alpha, A, lda, 0, B, ldb, 0, beta, beta != 0.0 ? C : nullptr, ldc, 0, C, ldc, 0, 1,
           0, work.p ? work.d() : nullptr, wsz);
}

static double dotd(Ctx& c, int64_t n, const double* x, const double* y, int slot) {
  dot_f64(c.s, n, x, y, c.partials.d(), c.scal.d() + slot);
  return read_scalar(c, c.scal.d() + slot);
}

// out = in^T (n x n)
static void transpose_sq(Ctx& c, int64_t n, const double* in, double alpha, double beta, double* out) {
  const int64_t od[2] = {n, n}, is[2] = {n, 1};
  permute_f64(c.s, 2, od, is, alpha, in, beta, out);
}

// RHF(ints, C, Lambda, ::RHFa) with DF integrals: S, H = T + V [n,n], b[Q,mu,nu] in HBM.
// b == nullptr: conventional integrals, eri[(m,n),(r,s)] = (mn|rs) and eri_x[(m,n),(r,s)] = (mr|ns) (n^2 x n^2)
static void rhf(Ctx& c, const fh_scf_opts& op, int n, int naux, int no, double Vnuc, const double* S, const double* H,
                const double* b, double* eps_out, double* C_out, fh_scf_result& res, const double* eri = nullptr,
                const double* eri_x = nullptr) {
  const int64_t nn = (int64_t)n * n, Q = naux;
  if (!c.partials.p) c.partials = dalloc(c, 4096);
  if (!c.scal.p) c.scal = dalloc(c, 64);
  Eigen eig(c, n);
  Buf L = dalloc(c, nn), F = dalloc(c, nn), Ft = dalloc(c, nn), Cm = dalloc(c, nn), D = dalloc(c, nn),
      Dold = dalloc(c, nn), Ftil = dalloc(c, nn), Dtil = dalloc(c, nn), T1 = dalloc(c, nn), T2 = dalloc(c, nn),
      J = dalloc(c, nn), K = dalloc(c, nn), w = dalloc(c, n), X = dalloc(c, Q), Z = dalloc(c, Q * no * n);
  // Lambda = S^-1/2 = U diag(d)^-1/2 U^T (RHFHelper.jl:9,36)
  {
    Timer t(c, "scf_guess");
    d2d(c, T1.d(), S, nn);
    eig.run(T1.d(), w.d());
    double dmin = 0.0;
    FH_HIP(hipMemcpyAsync(&dmin, w.d(), sizeof(double), hipMemcpyDeviceToHost, c.s));
    FH_HIP(hipStreamSynchronize(c.s));
    FH_CHECK(dmin > 0.0, -1, "fh_rhf: overlap matrix is not positive definite");
    scale_cols_rsqrt(c.s, n, T1.d(), w.d(), T2.d());
    mm(c, false, true, n, n, n, 1.0, T2.d(), n, T1.d(), n, 0.0, L.d(), n);
    // guess Fock matrix: GWH (RHFHelper.jl:44-51) or the core Hamiltonian (RHFHelper.jl:10)
    if (op.guess == 0) gwh_fock(c.s, n, S, H, F.d());
    else d2d(c, F.d(), H, nn);
  }
  // Ft = L^T F L; eps, Ct = eigen(Ft); C = L Ct; D = Co Co^T
  auto orbitals = [&](const double* Fm) {
    Timer t(c, "scf_diag", 4.0 * (double)nn * n + 2.0 * (double)nn * no);
    mm(c, false, false, n, n, n, 1.0, Fm, n, L.d(), n, 0.0, T1.d(), n);
    mm(c, true, false, n, n, n, 1.0, L.d(), n, T1.d(), n, 0.0, Ft.d(), n);
    eig.run(Ft.d(), w.d());
    mm(c, false, false, n, n, n, 1.0, L.d(), n, Ft.d(), n, 0.0, Cm.d(), n);
    mm(c, false, true, n, n, no, 1.0, Cm.d(), n, Cm.d(), n, 0.0, D.d(), n);
  };
  // build_fock! with DF integrals (RHFHelper.jl:88-93): F = H + 2 J - K with
  // J[m,n] = b[Q,m,n] (b[Q,r,s] D[r,s]) and, since D = Co Co^T, K[m,n] = Z[Q,i,m] Z[Q,i,n] with
  // Z[Q,i,m] = b[Q,m,r] Co[r,i] (one strided-batched GEMM over m)
  auto fock = [&]() {
    if (!b) {
      // conventional build_fock! (RHFHelper.jl:68-73): J = (mn|rs) D[r,s], K = (mr|ns) D[r,s], two GEMVs
      Timer t(c, "scf_fock", 4.0 * (double)nn * nn);
      mm(c, false, false, nn, 1, nn, 1.0, eri, nn, D.d(), nn, 0.0, J.d(), nn);
      mm(c, false, false, nn, 1, nn, 1.0, eri_x, nn, D.d(), nn, 0.0, K.d(), nn);
      d2d(c, F.d(), H, nn);
      axpby_f64(c.s, nn, 2.0, J.d(), 1.0, F.d());
      axpby_f64(c.s, nn, -1.0, K.d(), 1.0, F.d());
      return;
    }
    Timer t(c, "scf_fock", 4.0 * (double)Q * nn + 2.0 * (double)Q * nn * no + 2.0 * (double)nn * Q * no);
    mm(c, false, false, Q, 1, nn, 1.0, b, Q, D.d(), nn, 0.0, X.d(), Q);
    mm(c, true, false, nn, 1, Q, 1.0, b, Q, X.d(), Q, 0.0, J.d(), nn);
    const int64_t wsz = gemm_splitk_elems(Q, no, n, n);
    Buf work;
    if (wsz) work = dalloc(c, wsz);
    gemm_f64(c.s, false, false, Q, no, n, 1.0, b, Q * (int64_t)n, Q, Cm.d(), n, 0, 0.0, nullptr, 0, 0, Z.d(), Q,
             Q * no, n, 0, work.p ? work.d() : nullptr, wsz);
    mm(c, true, false, n, n, Q * no, 1.0, Z.d(), Q * no, Z.d(), Q * no, 0.0, K.d(), n);
    d2d(c, F.d(), H, nn);
    axpby_f64(c.s, nn, 2.0, J.d(), 1.0, F.d());
    axpby_f64(c.s, nn, -1.0, K.d(), 1.0, F.d());
  };
  orbitals(F.d());
  // the loop starts from the guess orbitals' density (RHFa.jl:118-127)
  fock();
  d2d(c, Ftil.d(), F.d(), nn);
  d2d(c, Dtil.d(), D.d(), nn);
  d2d(c, Dold.d(), D.d(), nn);
  std::unique_ptr<DIIS> dm;
  if (op.diis) dm.reset(new DIIS(c, nn, op.ndiis, false, 16));
  int ite = 1;
  double E = 0.0, dE = 1.0, Drms = 1.0;
  bool converged = false;
  while (ite <= op.scf_max_iter) {
    orbitals(F.d());                                              // RHFa.jl:137-147
    fock();                                                       // :150
    dot_f64(c.s, nn, D.d(), H, c.partials.d(), c.scal.d() + 8);
    dot_f64(c.s, nn, D.d(), F.d(), c.partials.d(), c.scal.d() + 9);
    d2d(c, T1.d(), D.d(), nn);                                    // Drms (:189-190)
    axpby_f64(c.s, nn, -1.0, Dold.d(), 1.0, T1.d());
    dot_f64(c.s, nn, T1.d(), T1.d(), c.partials.d(), c.scal.d() + 10);
    if (dm) {                                                     // err = L^T (F D S - S D F) L  (:157-160)
      mm(c, false, false, n, n, n, 1.0, F.d(), n, D.d(), n, 0.0, T1.d(), n);       // F D
      mm(c, false, false, n, n, n, 1.0, T1.d(), n, S, n, 0.0, T2.d(), n);          // F D S
      mm(c, false, false, n, n, n, 1.0, S, n, D.d(), n, 0.0, J.d(), n);            // S D (J is free here)
      mm(c, false, false, n, n, n, -1.0, J.d(), n, F.d(), n, 1.0, T2.d(), n);      // - S D F
      mm(c, false, false, n, n, n, 1.0, T2.d(), n, L.d(), n, 0.0, T1.d(), n);
      Buf err = dalloc(c, nn);
      mm(c, true, false, n, n, n, 1.0, L.d(), n, T1.d(), n, 0.0, err.d(), n);
      dm->push(F.d(), std::move(err));
    }
    double h[24];                                                 // both energies, Drms and the DIIS row in one copy
    d2h(c, h, c.scal.d(), 24);
    const double Enew = h[8] + h[9] + Vnuc;                       // :151-154
    if (dm) dm->resolve(h);
    if (op.oda && Drms > op.oda_cutoff && ite < op.oda_shutoff) {   // ODA (:163-180)
      d2d(c, T1.d(), D.d(), nn);
      axpby_f64(c.s, nn, -1.0, Dtil.d(), 1.0, T1.d());            // dD = D - D~
      transpose_sq(c, n, T1.d(), 1.0, 0.0, T2.d());               // tr(A dD) = sum A .* dD^T
      const double sv = dotd(c, nn, Ftil.d(), T2.d(), 11);
      const double cv = dotd(c, nn, F.d(), T2.d(), 12) - sv;
      const double lam = (cv <= -sv / (2.0 * cv)) ? 1.0 : -sv / (2.0 * cv);
      axpby_f64(c.s, nn, lam, F.d(), 1.0 - lam, Ftil.d());
      axpby_f64(c.s, nn, lam, D.d(), 1.0 - lam, Dtil.d());
      d2d(c, F.d(), Ftil.d(), nn);
    } else if (dm && ite > op.diis_start) {                       // DIIS (:183-186)
      dm->extrapolate(F.d(), false);
    }
    Drms = std::sqrt(h[10] / (double)nn);
    dE = Enew - E;
    E = Enew;
    d2d(c, Dold.d(), D.d(), nn);
    ++ite;
    if (std::fabs(dE) < op.scf_e_conv && Drms < op.scf_max_rms && ite > 5) {   // :200-203
      converged = true;
      break;
    }
  }
  FH_CHECK(std::isfinite(E), -5, "fh_rhf: non-finite energy");
  if (eps_out) d2h(c, eps_out, w.d(), n);
  if (C_out) d2h(c, C_out, Cm.d(), nn);
  res.energy = E;
  res.e_conv = dE;
  res.d_rms = Drms;
  res.niter = ite - 1;
  res.converged = converged ? 1 : 0;
}

static void solve(Ctx& c, const fh_cc_opts& op, fh_cc_result& res) {
  prepare(c);
  FH_CHECK(c.have_amp, -6, "no starting amplitudes");
  FH_CHECK(op.cc_max_iter >= 0 && op.cc_ndiis >= 1 && op.cc_ndiis <= 8 && op.cc_diis_relax >= 1, -1,
           "invalid CC options");
  FH_CHECK(op.precision_mode >= 0 && op.precision_mode <= 2, -1,
           "precision_mode must be 0 (FP64), 1 (FP32 then FP64) or 2 (split-BF16x3 then FP64)");
  FH_CHECK(op.max_restarts >= 0 && op.fault_inject >= 0, -1, "max_restarts and fault_inject must be >= 0");
  const int64_t n1 = c.nov(), n2 = c.n2();
  const double epsT = 2.220446049250313e-16;
  double e_conv = op.cc_e_conv, max_rms = op.cc_max_rms;
  if ((e_conv < epsT || max_rms < epsT) && !op.precision_override) e_conv = max_rms = epsT;   // RCCSDa.jl:139-146
  const bool do_diis = op.cc_diis != 0;
  const bool f32 = op.diis_prec != 0;
  const double dp = op.cc_damp_ratio;
  std::unique_ptr<DIIS> dm1(new DIIS(c, n1, op.cc_ndiis, f32, 16)), dm2(new DIIS(c, n2, op.cc_ndiis, f32, 24, "diis"));
  c.iters.clear();
  // mixed precision: the residual's contractions run at `level` (2 split-BF16x3 or 1 FP32, then
  // 0 FP64).  A reduced-precision phase ends when |dE| and rms fall below its switch thresholds,
  // or when its rms has not reached a new minimum for kStall iterations (the precision's own
  // noise floor).  Each switch starts a fresh DIIS subspace: the error vectors of the lower
  // precision describe its own fixed point, which extrapolation would otherwise pull back to.
  // The FP64 phase polishes to the final criteria (or for polish_iters iterations).
  constexpr int kStall = 4;
  int level = op.precision_mode, stall = 0;
  double best_rms = 1e300;
  int polish_done = 0, niter_mixed = 0, niter_bf3 = 0, restarts = 0;
  bool injected = false;
  const double sw_e = std::max(op.mixed_e_switch, e_conv), sw_rms = std::max(op.mixed_rms_switch, max_rms);
  const double sw_e2 = std::max(op.bf3_e_switch, e_conv), sw_rms2 = std::max(op.bf3_rms_switch, max_rms);

  Buf nT1 = std::move(c.T1), nT2 = std::move(c.T2);     // newT (guess)
  // the context holds no amplitudes until the loop has ended normally: an error (non-finite
  // amplitudes, singular DIIS, out of memory) leaves have_amp false and the reduced-precision level
  // reset, so a later call that needs amplitudes fails with -6 instead of reading freed buffers
  c.have_amp = false;
  struct LevelGuard {
    Ctx& c;
    ~LevelGuard() { c.lowp = 0; }
  } level_guard{c};
  Buf oT1 = dalloc(c, n1), oT2 = dalloc(c, n2);         // T
  double Ecc = energy(c, nT1.d(), nT2.d());            // :160
  res.guess_energy = Ecc;
  double dE = 1.0, rms = 1.0;
  int ite = 1;
  if (op.verbose) std::printf("%10s    %15s    %12s    %12s    %10s    %5s\n", "Iteration", "CC Energy", "dE", "Max RMS", "time (s)", "diis");
  while (true) {
    while (level > 0 && ((std::fabs(dE) < (level == 2 ? sw_e2 : sw_e) && rms < (level == 2 ? sw_rms2 : sw_rms)) ||
                         stall >= kStall)) {
      level = 0;                                           // FP64 polish
      dm1.reset(new DIIS(c, n1, op.cc_ndiis, f32, 16));
      dm2.reset(new DIIS(c, n2, op.cc_ndiis, f32, 24, "diis"));
      dE = 1.0;
      rms = 1.0;
      stall = 0;
      best_rms = 1e300;
    }
    if (level == 0) {
      if (!(std::fabs(dE) > e_conv || rms > max_rms)) break;                                   // :178
      if (op.precision_mode > 0 && op.polish_iters >= 0 && polish_done >= op.polish_iters) break;
    }
    if (ite > op.cc_max_iter) break;
    c.lowp = level;
    auto t0 = std::chrono::steady_clock::now();
    std::swap(oT1, nT1);                                                                        // :185-186
    std::swap(oT2, nT2);
    if (!nT1.p) nT1 = dalloc(c, n1);
    if (!nT2.p) nT2 = dalloc(c, n2);
    const double oldE = Ecc;
    Buf e1, e2;
    if (do_diis) {
      e1 = Buf(c.pool.get(), (size_t)n1 * (f32 ? 4 : 8));
      e2 = Buf(c.pool.get(), (size_t)n2 * (f32 ? 4 : 8));
    }
    update_amp(c, oT1.d(), oT2.d(), nT1.d(), nT2.d(), e1.p, e2.p, f32);                         // :190-194
    c.lowp = 0;
    if (op.fault_inject > 0 && ite == op.fault_inject && !injected) {      // test hook: one NaN in the new T2
      const double nan = std::nan("");
      FH_HIP(hipMemcpyAsync(nT2.d() + n2 / 2, &nan, sizeof(double), hipMemcpyHostToDevice, c.s));
      FH_HIP(hipStreamSynchronize(c.s));
      injected = true;
    }
    bool diis = false;
    if (do_diis) {
      dm1->push(nT1.d(), std::move(e1));                                                        // :199-202
      dm2->push(nT2.d(), std::move(e2));
    }
    // the changes and both rows of products in one copy
    double h[32];
    d2h(c, h, c.scal.d(), 32);
    const double r1 = std::sqrt(h[0] / (double)n1), r2 = std::sqrt(h[1] / (double)n2);
    if (do_diis) {
      dm1->resolve(h);
      dm2->resolve(h);
      if (ite >= op.diis_start && ite % op.cc_diis_relax == 0 &&                             // :204
          (op.precision_mode == 0 || dm2->vecs.size() >= 2)) {
        dm2->extrapolate(nT2.d(), true);                                                        // :206
        dm1->extrapolate(nT1.d(), true);                                                        // :207
        diis = true;
      }
    }
    if (dp > 0) {                                                                               // :213-216
      axpby_f64(c.s, n1, dp, oT1.d(), 1.0 - dp, nT1.d());
      axpby_f64(c.s, n2, dp, oT2.d(), 1.0 - dp, nT2.d());
    }
    Ecc = energy(c, nT1.d(), nT2.d());                                                          // :218
    rms = std::max(r1, r2);
    if (!(std::isfinite(Ecc) && std::isfinite(rms)) && restarts < op.max_restarts) {
      // restart from this iteration's (finite) input amplitudes in FP64 with fresh DIIS subspaces
      ++restarts;
      if (op.verbose) std::printf("    %-5d    non-finite energy or amplitudes: restart %d from the last finite amplitudes (FP64)\n", ite, restarts);
      d2d(c, nT1.d(), oT1.d(), n1);
      d2d(c, nT2.d(), oT2.d(), n2);
      Ecc = oldE;
      level = 0;
      dm1.reset(new DIIS(c, n1, op.cc_ndiis, f32, 16));
      dm2.reset(new DIIS(c, n2, op.cc_ndiis, f32, 24, "diis"));
      dE = 1.0;
      rms = 1.0;
      stall = 0;
      best_rms = 1e300;
      ++ite;
      continue;
    }
    dE = Ecc - oldE;
    if (rms < best_rms) {
      best_rms = rms;
      stall = 0;
    } else {
      ++stall;
    }
    if (level > 0) ++niter_mixed;
    if (level == 2) ++niter_bf3;
    if (level == 0 && op.precision_mode > 0) ++polish_done;
    const double ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    c.iters.push_back({ite, Ecc, dE, rms, ms, diis});
    if (op.verbose) std::printf("    %-5d    %-15.10f    %+12.10f    %-12.10f    %-10.5f    %s%s\n", ite, Ecc, dE, rms, ms / 1e3, diis ? "true" : "false", level == 2 ? " bf16x3" : (level == 1 ? " fp32" : ""));
    FH_CHECK(std::isfinite(Ecc) && std::isfinite(rms), -5, "non-finite CC energy or amplitudes at iteration " + std::to_string(ite));
    ++ite;
  }
  c.lowp = 0;
  res.correlation = Ecc;
  res.e_conv = dE;
  res.t_conv = rms;
  res.niter = ite - 1;
  res.niter_mixed = niter_mixed;
  res.niter_bf3 = niter_bf3;
  res.restarts = restarts;
  res.converged = (level == 0 && std::fabs(dE) < e_conv && rms < max_rms) ? 1 : 0;            // :231
  c.T1 = std::move(nT1);
  c.T2 = std::move(nT2);
  c.have_amp = true;
  c.last_energy = Ecc;
}

// ------------------------------------------------------------------ (T), ijk.jl:20-150
__global__ __launch_bounds__(1024) void k_accumulate(int64_t n, const double* __restrict__ partials, double* __restrict__ acc) {
  // single block; fixed order -> deterministic
  __shared__ double red[1024];
  double t = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += 1024) t += partials[i];
  red[threadIdx.x] = t;
  __syncthreads();
  for (int st = 512; st > 0; st >>= 1) {
    if ((int)threadIdx.x < st) red[threadIdx.x] += red[threadIdx.x + st];
    __syncthreads();
  }
  if (threadIdx.x == 0) *acc += red[0];
}

// (T) with W stored as T (double: FP64 path; float: FP32 MFMA W build, or split-BF16x3 when bf3).
// Triples t0 .. t0+nt-1 of the reference's loop order (for i, for j <= i, for k <= j; ijk.jl:49,63,83),
// t(i,j,k) = i(i+1)(i+2)/6 + j(j+1)/2 + k; nt < 0: all triples.
//
// The triples go in chunks of W slots, several (i, j) pairs to a chunk; each chunk is two W-build launches
// (fh_triples.hip) and one energy launch over device tables that are made and uploaded once.
template <typename T>
static double triples_t(Ctx& c, bool bf3, int64_t t0 = 0, int64_t nt = -1) {
  prepare(c);
  FH_CHECK(c.have_amp, -6, "no amplitudes for (T)");
  const bool lowp = std::is_same<T, float>::value;
  const int fmt = bf3 ? 2 : (lowp ? 1 : 0);
  const int64_t o = c.o, v = c.v, vv = v * v, v3 = vv * v;
  const double o_ = (double)o, v_ = (double)v;
  const double ntrip_all = o_ * (o_ + 1) * (o_ + 2) / 6.0;
  const double ntrip = nt < 0 ? ntrip_all : std::max(0.0, std::min((double)nt, ntrip_all - (double)t0));
  const std::string sfx = bf3 ? "_bf16x3" : (lowp ? "_fp32" : "");
  Timer tall(c, "triples" + sfx, ntrip * 12.0 * (v_ * v_ * v_ * v_ + o_ * v_ * v_ * v_));

  // runs of consecutive k of one (i, j)
  struct Run {
    int i, j, k0, nk;
  };
  std::vector<Run> runs;
  int64_t ntot = 0;
  const int64_t tend = nt < 0 ? INT64_MAX : t0 + nt;
  for (int64_t i = 0; i < o; ++i)
    for (int64_t j = 0; j <= i; ++j) {
      const int64_t base = i * (i + 1) * (i + 2) / 6 + j * (j + 1) / 2;  // t(i, j, 0)
      const int64_t kbeg = std::max<int64_t>(0, t0 - base);
      int64_t kend = (i == j) ? j : j + 1;  // i=j=k has zero weight (ijk.jl:133)
      if (tend - base < kend) kend = std::max<int64_t>(0, tend - base);
      if (kend > kbeg) {
        runs.push_back({(int)i, (int)j, (int)kbeg, (int)(kend - kbeg)});
        ntot += kend - kbeg;
      }
    }
  if (runs.empty()) return c.last_et = 0.0;

  const TriplesTiles tt = triples_tiles(fmt, (int)o, (int)v, (double)ntot / (double)runs.size());
  const int64_t KC = triples_chunk_slots((int)v, (int)sizeof(T), tt, ntot);

  // tables of every chunk: W slots, column tiles of the first launch, energy runs
  struct Chunk {
    int64_t slots, cols, eruns;  // offsets (ints) into the table
    int nslot, ncol, nerun;
  };
  std::vector<int> tab, orb;
  std::vector<Chunk> chunks;
  triples_orbits((int)v, orb);
  const int64_t norb = (int64_t)orb.size() / 3;
  int max_erun = 0;
  for (size_t r = 0, done = 0; r < runs.size();) {
    std::vector<Run> in;
    int64_t ns = 0;
    while (r < runs.size() && ns < KC) {
      const int take = (int)std::min<int64_t>(runs[r].nk - (int64_t)done, KC - ns);
      in.push_back({runs[r].i, runs[r].j, runs[r].k0 + (int)done, take});
      ns += take;
      done += take;
      if ((int)done == runs[r].nk) { ++r; done = 0; }
    }
    Chunk ch;
    ch.nslot = (int)ns;
    ch.slots = (int64_t)tab.size();
    for (const Run& q : in)
      for (int k = q.k0; k < q.k0 + q.nk; ++k) tab.insert(tab.end(), {q.i, q.j, k, 0});
    ch.cols = (int64_t)tab.size();
    int slot = 0;
    for (const Run& q : in) {
      triples_col_tiles(tt, (int)v, q.i, q.j, q.k0, q.nk, slot, tab);
      slot += q.nk;
    }
    ch.ncol = (int)(((int64_t)tab.size() - ch.cols) / 8);
    ch.eruns = (int64_t)tab.size();
    const int kpw = triples_energy_kpw((int)norb, (int)ns);
    slot = 0;
    for (const Run& q : in) {
      const int np = (q.nk + kpw - 1) / kpw;
      for (int p = 0; p < np; ++p) {
        const int b = q.nk * p / np, e = q.nk * (p + 1) / np;
        tab.insert(tab.end(), {q.i, q.j, q.k0 + b, e - b, slot + b, 0, 0, 0});
      }
      slot += q.nk;
    }
    ch.nerun = (int)(((int64_t)tab.size() - ch.eruns) / 8);
    max_erun = std::max(max_erun, ch.nerun);
    chunks.push_back(ch);
  }
  Buf orbits(c.pool.get(), orb.size() * sizeof(int)), table(c.pool.get(), tab.size() * sizeof(int));
  FH_HIP(hipMemcpyAsync(orbits.p, orb.data(), orb.size() * sizeof(int), hipMemcpyHostToDevice, c.s));
  FH_HIP(hipMemcpyAsync(table.p, tab.data(), tab.size() * sizeof(int), hipMemcpyHostToDevice, c.s));
  FH_HIP(hipStreamSynchronize(c.s));
  const int* dtab = static_cast<const int*>(table.p);

  // operands: AV and its row-swapped copy share one allocation, BVp and BVq likewise
  const int64_t nd = triples_pitch_elems((int)o, (int)v), avsz = vv * o * nd, bvsz = nd * v * o * o;
  Buf AVall(c.pool.get(), (size_t)(2 * avsz) * sizeof(T)), BVqp(c.pool.get(), (size_t)(2 * bvsz) * sizeof(T));
  TriplesOperands op;
  op.av = AVall.p;
  op.avs = static_cast<T*>(AVall.p) + avsz;
  op.bvq = BVqp.p;
  op.bvp = static_cast<T*>(BVqp.p) + bvsz;
  triples_operands(c.s, fmt, (int)o, (int)v, c.OVVV.d(), c.T2.d(), c.OOOV.d(), op.av, op.avs, op.bvp, op.bvq);
  Buf T1p = dalloc(c, v * o), vvb = dalloc(c, triples_vv_blocked_elems((int)o, (int)v));
  {
    Buf vvoo = dalloc(c, vv * o * o);
    perm(c, tv(c.T1.d(), {o, v}), "ia", tv(T1p.d(), {v, o}), "ai", 1.0, 0.0);
    perm(c, tv(c.OVOV.d(), {o, v, o, v}), "iajb", tv(vvoo.d(), {v, v, o, o}), "abij", 1.0, 0.0);
    triples_block_vv(c.s, (int)o, (int)v, vvoo.d(), vvb.d());
  }
  Buf Wbuf(c.pool.get(), (size_t)(triples_plane((int)v) * v * std::min(KC, ntot)) * sizeof(T));
  T* W = static_cast<T*>(Wbuf.p);
  Buf part = dalloc(c, norb * max_erun + 16);
  Buf acc = dalloc(c, 1);
  fill_f64(c.s, 1, 0.0, acc.d());
  for (const Chunk& ch : chunks) {
    const double fcls = 2.0 * v_ * v_ * v_ * (v_ + o_) * (double)ch.nslot;  // one permutation class
    {
      Timer tg(c, "triples_gemm" + sfx, 6.0 * fcls);
      {
        Timer tf(c, "triples_w_first" + sfx, 2.0 * fcls);
        triples_w_first(c.s, fmt, (int)o, (int)v, tt, op, W, dtab + ch.cols, ch.ncol);
      }
      Timer tr(c, "triples_w_slices" + sfx, 4.0 * fcls);
      triples_w_slices(c.s, fmt, (int)o, (int)v, tt, op, W, dtab + ch.slots, ch.nslot);
    }
    // algorithmic bytes: the chunk's W read once
    Timer te(c, "triples_energy" + sfx, 0.0, (double)sizeof(T) * (double)v3 * (double)ch.nslot);
    triples_energy(c.s, (int)o, (int)v, ch.nerun, dtab + ch.eruns, W, (int)norb, static_cast<const int*>(orbits.p),
                   T1p.d(), vvb.d(), c.eo.d(), c.ev.d(), part.d());
    hipLaunchKernelGGL(k_accumulate, dim3(1), dim3(1024), 0, c.s, norb * ch.nerun, part.d(), acc.d());
    FH_HIP(hipGetLastError());
  }
  const double Et = read_scalar(c, acc.d());
  c.last_et = Et;
  return Et;
}

// prec_mode 0: FP64; 1: FP32 MFMA W build; 2: split-BF16x3 MFMA W build
static double triples(Ctx& c, int prec_mode, int64_t t0 = 0, int64_t nt = -1) {
  return prec_mode == 0 ? triples_t<double>(c, false, t0, nt) : triples_t<float>(c, prec_mode == 2, t0, nt);
}

}  // namespace fh

// ====================================================================== C ABI
using namespace fh;

struct fh_ctx {
  Ctx c;
};

// thrown after a call completed with a documented fallback: the call returns 1 (message in fh_last_error)
struct Fallback {};

template <typename F>
static int guarded(F&& f) {
  try {
    f();
    return 0;
  } catch (const Fallback&) {
    return 1;
  } catch (const Error& e) {
    set_error(e.msg);
    return e.code;
  } catch (const std::exception& e) {
    set_error(e.what());
    return -3;
  }
}

struct DeviceGuard {
  int prev = 0;
  explicit DeviceGuard(int d) { (void)hipGetDevice(&prev); (void)hipSetDevice(d); }
  ~DeviceGuard() { (void)hipSetDevice(prev); }
};

extern "C" {

void fh_default_opts(fh_cc_opts* p) {
  if (!p) return;
  p->cc_max_iter = 50;
  p->cc_e_conv = 1e-10;
  p->cc_max_rms = 1e-10;
  p->cc_diis = 1;
  p->cc_ndiis = 3;
  p->diis_start = 3;
  p->cc_diis_relax = 3;
  p->diis_prec = 1;
  p->cc_damp_ratio = 0.0;
  p->precision_override = 0;
  p->verbose = 0;
  p->precision_mode = 0;
  p->polish_iters = -1;
  p->mixed_e_switch = 1e-9;
  p->mixed_rms_switch = 1e-9;
  p->bf3_e_switch = 1e-7;
  p->bf3_rms_switch = 1e-8;
  p->max_restarts = 1;
  p->fault_inject = 0;
}

const char* fh_last_error(void) { return g_last_error.c_str(); }

int fh_create(fh_ctx** out, int device) {
  return guarded([&] {
    FH_CHECK(out != nullptr, -1, "fh_create: null output pointer");
    *out = nullptr;
    int n = 0;
    FH_HIP(hipGetDeviceCount(&n));
    FH_CHECK(device >= 0 && device < n, -1, "fh_create: no HIP device " + std::to_string(device));
    DeviceGuard g(device);
    auto* x = new fh_ctx();
    x->c.device = device;
    x->c.pool.reset(new Pool(device));
    x->c.pool->give_back = [c = &x->c] {
      if (c->solvers || !c->blas.h) return;
      (void)hipStreamSynchronize(c->s);
      c->blas.reset();
    };
    hipError_t e = hipStreamCreateWithFlags(&x->c.s, hipStreamNonBlocking);
    if (e != hipSuccess) { delete x; throw Error{-2, std::string("hipStreamCreate: ") + hipGetErrorString(e)}; }
    try {
      init_noalloc_scratch(device);  // the device address of this device's scratch array
    } catch (...) {
      (void)hipStreamDestroy(x->c.s);
      delete x;
      throw;
    }
    *out = x;
  });
}

void fh_destroy(fh_ctx* x) {
  if (!x) return;
  DeviceGuard g(x->c.device);
  (void)hipStreamSynchronize(x->c.s);
  flush_timers(x->c);
  hipStream_t s = x->c.s;
  delete x;  // Ctx members go in reverse declaration order: every Buf before the pool
  (void)hipStreamDestroy(s);
}

// Forget the previous molecule (integral blocks, operand copies, amplitudes, guess network) and
// take the orbital energies of the next one.
static void new_molecule(Ctx& c, int o, int v, int naux, const double* eps_o, const double* eps_v, const char* who) {
  for (int i = 0; i < o; ++i)
    for (int a = 0; a < v; ++a)
      FH_CHECK(eps_o[i] < eps_v[a], -1, std::string(who) + ": occupied orbital energy above a virtual one");
  c.have_df = false;
  c.prepared = false;
  c.have_amp = false;
  c.OOOO.reset(); c.OOOV.reset(); c.OOVV.reset(); c.OVOV.reset(); c.OVVV.reset();
  c.LX.reset(); c.LX32.reset(); c.Vs.reset(); c.Vs32.reset(); c.Pt.reset(); c.T1.reset(); c.T2.reset();
  c.Lkl.reset(); c.Okl.reset(); c.Lo1.reset(); c.L1.reset();
  c.Boo.reset(); c.Bov.reset(); c.Bvv.reset();
  c.opcache.clear(); c.opcache_bytes = 0;
  c.have_model = false; c.pair_d.reset();
  c.conventional = false; c.have_fia = false; c.Fia.reset();
  c.o = o; c.v = v; c.naux = naux;
  c.eo = dalloc(c, o); c.ev = dalloc(c, v);
  h2d(c, c.eo.d(), eps_o, o);
  h2d(c, c.ev.d(), eps_v, v);
}

int fh_set_df(fh_ctx* x, int o, int v, int naux, const double* eps_o, const double* eps_v, const double* Boo,
              const double* Bov, const double* Bvv) {
  return guarded([&] {
    FH_CHECK(x != nullptr, -1, "fh_set_df: null context");
    FH_CHECK(o >= 1 && v >= 1 && naux >= 1, -1, "fh_set_df: invalid dimensions");
    FH_CHECK(eps_o && eps_v && Bov, -1, "fh_set_df: null array");
    FH_CHECK((Boo == nullptr) == (Bvv == nullptr), -1, "fh_set_df: give both Boo and Bvv, or neither (DF-MP2 only)");
    DeviceGuard g(x->c.device);
    Ctx& c = x->c;
    new_molecule(c, o, v, naux, eps_o, eps_v, "fh_set_df");
    const int64_t Q = naux;
    c.ov_only = Boo == nullptr;
    c.Bov = dalloc(c, Q * o * v);
    h2d(c, c.Bov.d(), Bov, Q * o * v);
    if (!c.ov_only) {
      c.Boo = dalloc(c, Q * o * o); c.Bvv = dalloc(c, Q * v * v);
      h2d(c, c.Boo.d(), Boo, Q * o * o);
      h2d(c, c.Bvv.d(), Bvv, Q * v * v);
    }
    FH_HIP(hipStreamSynchronize(c.s));
    c.have_df = true;
  });
}

// The conventional (Chonky) integral path of RCCSD(moints, aoints, ::RCCSDa), RCCSDa.jl:25-35: the six
// 4-index MO blocks are handed over as computed by compute_OOOO! ... compute_VVVV! (Chonky.jl) and
// Fd / Fia of compute_F! (Fock.jl:1-36).  VVVV goes straight into the ladder's operand layout, the pairs
// Vs[cd, ab] of VVVV[c,a,d,b] (the conventional ladder tau[i,j,c,d] VVVV[c,a,d,b],
// RCCSDHelper.jl:194-202); the other blocks are kept in the reference's index order.
int fh_set_mo(fh_ctx* x, int o, int v, const double* eps_o, const double* eps_v, const double* Fia,
              const double* OOOO, const double* OOOV, const double* OOVV, const double* OVOV, const double* OVVV,
              const double* VVVV) {
  return guarded([&] {
    FH_CHECK(x != nullptr, -1, "fh_set_mo: null context");
    FH_CHECK(o >= 1 && v >= 1, -1, "fh_set_mo: invalid dimensions");
    FH_CHECK(eps_o && eps_v && OOOO && OOOV && OOVV && OVOV && OVVV && VVVV, -1, "fh_set_mo: null array");
    FH_CHECK((double)v * v * v * v < 9.0e18 / 8, -1, "fh_set_mo: VVVV too large");
    DeviceGuard g(x->c.device);
    Ctx& c = x->c;
    new_molecule(c, o, v, 0, eps_o, eps_v, "fh_set_mo");
    const int64_t O = o, V = v;
    auto up = [&](Buf& b, const double* h, int64_t n) { b = dalloc(c, n); h2d(c, b.d(), h, n); };
    up(c.OOOO, OOOO, O * O * O * O);
    up(c.OOOV, OOOV, O * O * O * V);
    up(c.OOVV, OOVV, O * O * V * V);
    up(c.OVOV, OVOV, O * V * O * V);
    up(c.OVVV, OVVV, O * V * V * V);
    {
      Buf tmp;
      up(tmp, VVVV, V * V * V * V);
      c.Vs = dalloc(c, V * (V + 1) * vv_pairs_ld(v));
      vv_pairs(c.s, v, 0, v, tmp.d(), V, V * V, V * V * V, true, c.Vs.d());
      FH_HIP(hipStreamSynchronize(c.s));
    }
    if (Fia) {
      up(c.Fia, Fia, O * V);
      c.have_fia = true;
    }
    FH_HIP(hipStreamSynchronize(c.s));
    c.conventional = true;
    c.ov_only = false;
    c.have_df = true;
  });
}

// AO -> MO DF transforms compute_BOO! / compute_BOV! / compute_BVV! (DFERI.jl:15-69) on the
// device.  One FP64 MFMA GEMM makes the half-transformed H[Q,mu,q] = sum_nu b[Q,mu,nu] C[nu,q] for
// the active MOs q (K = nbf), then three strided-batched GEMMs (one batch entry per second MO
// index, K = nbf) give B[Q,p,q] = sum_mu H[Q,mu,q] C[mu,p] for the oo, ov and vv blocks.
int fh_set_df_ao(fh_ctx* x, int nbf, int naux, int ndocc, int drop_occ, int drop_vir, const double* eps,
                 const double* C, const double* bAO) {
  return guarded([&] {
    FH_CHECK(x != nullptr, -1, "fh_set_df_ao: null context");
    FH_CHECK(eps && C && bAO, -1, "fh_set_df_ao: null array");
    FH_CHECK(nbf >= 2 && naux >= 1 && ndocc >= 1 && ndocc < nbf, -1, "fh_set_df_ao: invalid dimensions");
    // RMP2a.jl:62-68: frozen core below ndocc, inactive virtuals below nvir
    FH_CHECK(drop_occ >= 0 && drop_occ < ndocc, -1,
             "fh_set_df_ao: invalid number of frozen orbitals " + std::to_string(drop_occ) + " for " +
                 std::to_string(ndocc) + " doubly occupied orbitals");
    FH_CHECK(drop_vir >= 0 && drop_vir < nbf - ndocc, -1,
             "fh_set_df_ao: invalid number of inactive virtual orbitals " + std::to_string(drop_vir) + " for " +
                 std::to_string(nbf - ndocc) + " total virtual orbitals");
    FH_CHECK((double)naux * nbf * nbf < 9.0e18 / 8, -1, "fh_set_df_ao: AO tensor too large");
    DeviceGuard g(x->c.device);
    Ctx& c = x->c;
    const int o = ndocc - drop_occ, v = nbf - drop_vir - ndocc, nact = o + v;
    new_molecule(c, o, v, naux, eps + drop_occ, eps + ndocc, "fh_set_df_ao");  // Fock.jl:81-94
    c.ov_only = false;
    const int64_t Q = naux, n = nbf;
    Buf dC = dalloc(c, n * n);
    h2d(c, dC.d(), C, n * n);
    Buf b = dalloc(c, Q * n * n);
    h2d(c, b.d(), bAO, Q * n * n);
    c.Boo = dalloc(c, Q * o * o);
    c.Bov = dalloc(c, Q * o * v);
    c.Bvv = dalloc(c, Q * v * v);
    {
      Timer t(c, "ao_to_mo", 2.0 * (double)Q * n * n * nact + 2.0 * (double)Q * n * ((double)o * o + (double)o * v +
                                                                                        (double)v * v));
      Buf H = dalloc(c, Q * n * nact);
      {
        const int64_t wsz = gemm_splitk_elems(Q * n, nact, n, 1);
        Buf work;
        if (wsz) work = dalloc(c, wsz);
        gemm_f64(c.s, false, false, Q * n, nact, n, 1.0, b.d(), Q * n, 0, dC.d() + n * drop_occ, n, 0, 0.0, nullptr, 0,
                 0, H.d(), Q * n, 0, 1, 0, work.p ? work.d() : nullptr, wsz);
      }
      b.reset();
      const double* Co = dC.d() + n * drop_occ;
      const double* Cv = dC.d() + n * ndocc;
      auto half = [&](const double* Hq, int nq, const double* Cp, int np, double* B) {
        const int64_t wsz = gemm_splitk_elems(Q, np, n, nq);
        Buf work;
        if (wsz) work = dalloc(c, wsz);
        gemm_f64(c.s, false, false, Q, np, n, 1.0, Hq, Q, Q * n, Cp, n, 0, 0.0, nullptr, 0, 0, B, Q, Q * np, nq, 0,
                 work.p ? work.d() : nullptr, wsz);
      };
      half(H.d(), o, Co, o, c.Boo.d());                   // Bij[Q,i,j]  (DFERI.jl:25-27)
      half(H.d() + Q * n * o, v, Co, o, c.Bov.d());       // Bia[Q,i,a]  (DFERI.jl:46-48)
      half(H.d() + Q * n * o, v, Cv, v, c.Bvv.d());       // Bab[Q,a,b]  (DFERI.jl:64-66)
    }
    FH_HIP(hipStreamSynchronize(c.s));
    flush_timers(c);
    c.have_df = true;
  });
}

void fh_default_scf_opts(fh_scf_opts* p) {
  if (!p) return;
  p->scf_max_iter = 50;
  p->scf_e_conv = 1e-10;
  p->scf_max_rms = 1e-9;
  p->diis = 1;
  p->ndiis = 8;
  p->diis_start = 3;
  p->oda = 1;
  p->oda_cutoff = 1e-1;
  p->oda_shutoff = 20;
  p->guess = 0;
}

int fh_rhf(fh_ctx* x, const fh_scf_opts* opts, int nbf, int naux, int ndocc, double Vnuc, const double* S,
           const double* H, const double* bAO, double* eps, double* C, fh_scf_result* res) {
  return guarded([&] {
    FH_CHECK(x != nullptr && opts != nullptr && res != nullptr, -1, "fh_rhf: null argument");
    FH_CHECK(S && H && bAO, -1, "fh_rhf: null array");
    FH_CHECK(nbf >= 1 && naux >= 1 && ndocc >= 1 && ndocc <= nbf, -1, "fh_rhf: invalid dimensions");
    FH_CHECK((double)naux * nbf * nbf < 9.0e18 / 8, -1, "fh_rhf: AO tensor too large");
    const fh_scf_opts& op = *opts;
    FH_CHECK(op.scf_max_iter >= 0 && (!op.diis || (op.ndiis >= 2 && op.ndiis <= 8)) && (op.guess == 0 || op.guess == 1),
             -1, "fh_rhf: invalid options (ndiis 2..8, guess 0 = gwh or 1 = core)");
    DeviceGuard g(x->c.device);
    Ctx& c = x->c;
    const int64_t nn = (int64_t)nbf * nbf;
    Buf dS = dalloc(c, nn), dH = dalloc(c, nn), db = dalloc(c, (int64_t)naux * nn);
    h2d(c, dS.d(), S, nn);
    h2d(c, dH.d(), H, nn);
    h2d(c, db.d(), bAO, (int64_t)naux * nn);
    *res = fh_scf_result{};
    {
      Timer t(c, "scf");
      rhf(c, op, nbf, naux, ndocc, Vnuc, dS.d(), dH.d(), db.d(), eps, C, *res);
    }
    FH_HIP(hipStreamSynchronize(c.s));
    flush_timers(c);
  });
}

// RHF with conventional integrals (the Chonky / SparseERI path of RHFa.jl:14-223, build_fock! of
// RHFHelper.jl:68-73): eri[mu,nu,la,si] = (mu nu|la si) in HBM with a (mu la|nu si)-ordered copy for K.
int fh_rhf_conv(fh_ctx* x, const fh_scf_opts* opts, int nbf, int ndocc, double Vnuc, const double* S, const double* H,
                const double* eri, double* eps, double* C, fh_scf_result* res) {
  return guarded([&] {
    FH_CHECK(x != nullptr && opts != nullptr && res != nullptr, -1, "fh_rhf_conv: null argument");
    FH_CHECK(S && H && eri, -1, "fh_rhf_conv: null array");
    FH_CHECK(nbf >= 1 && ndocc >= 1 && ndocc <= nbf, -1, "fh_rhf_conv: invalid dimensions");
    FH_CHECK((double)nbf * nbf * nbf * nbf < 4.0e9, -1, "fh_rhf_conv: 4-index tensor too large (nbf^4 >= 4e9)");
    const fh_scf_opts& op = *opts;
    FH_CHECK(op.scf_max_iter >= 0 && (!op.diis || (op.ndiis >= 2 && op.ndiis <= 8)) && (op.guess == 0 || op.guess == 1),
             -1, "fh_rhf_conv: invalid options (ndiis 2..8, guess 0 = gwh or 1 = core)");
    DeviceGuard g(x->c.device);
    Ctx& c = x->c;
    const int64_t n = nbf, nn = n * n;
    Buf dS = dalloc(c, nn), dH = dalloc(c, nn), dE = dalloc(c, nn * nn), dX = dalloc(c, nn * nn);
    h2d(c, dS.d(), S, nn);
    h2d(c, dH.d(), H, nn);
    h2d(c, dE.d(), eri, nn * nn);
    perm(c, tv(dE.d(), {n, n, n, n}), "mrns", tv(dX.d(), {n, n, n, n}), "mnrs", 1.0, 0.0);
    *res = fh_scf_result{};
    {
      Timer t(c, "scf");
      rhf(c, op, nbf, 0, ndocc, Vnuc, dS.d(), dH.d(), nullptr, eps, C, *res, dE.d(), dX.d());
    }
    FH_HIP(hipStreamSynchronize(c.s));
    flush_timers(c);
  });
}

// The DF fit of compute_ERI! (AtomicIntegrals.jl:31-41): Jh = J^-1/2 = U diag(d)^-1/2 U^T from the
// eigenpairs of the Coulomb metric, then b[Q,(mu,nu)] = sum_P Jh[P,Q] Pqp[(mu,nu),P] as one FP64 MFMA
// GEMM (M = naux, N = nbf^2, K = naux) that writes b with Q fastest.
int fh_df_fit(fh_ctx* x, int nbf, int naux, const double* J, const double* Pqp, double* b) {
  return guarded([&] {
    FH_CHECK(x != nullptr && J && Pqp && b, -1, "fh_df_fit: null argument");
    FH_CHECK(nbf >= 1 && naux >= 1, -1, "fh_df_fit: invalid dimensions");
    FH_CHECK((double)naux * nbf * nbf < 9.0e18 / 8, -1, "fh_df_fit: AO tensor too large");
    DeviceGuard g(x->c.device);
    Ctx& c = x->c;
    const int64_t Q = naux, nn = (int64_t)nbf * nbf;
    Buf dJ = dalloc(c, Q * Q), U = dalloc(c, Q * Q), Us = dalloc(c, Q * Q), w = dalloc(c, Q), dP = dalloc(c, nn * Q),
        db = dalloc(c, nn * Q);
    h2d(c, dJ.d(), J, Q * Q);
    h2d(c, dP.d(), Pqp, nn * Q);
    {
      Timer t(c, "df_fit", 4.0 * (double)Q * Q * Q + 2.0 * (double)Q * Q * nn);
      Eigen eig(c, naux);
      d2d(c, U.d(), dJ.d(), Q * Q);
      eig.run(U.d(), w.d());
      double dmin = 0.0;
      FH_HIP(hipMemcpyAsync(&dmin, w.d(), sizeof(double), hipMemcpyDeviceToHost, c.s));
      FH_HIP(hipStreamSynchronize(c.s));
      FH_CHECK(dmin > 0.0, -1, "fh_df_fit: Coulomb metric J is not positive definite");
      scale_cols_rsqrt(c.s, naux, U.d(), w.d(), Us.d());
      mm(c, false, true, Q, Q, Q, 1.0, Us.d(), Q, U.d(), Q, 0.0, dJ.d(), Q);   // Jh (into dJ)
      mm(c, true, true, Q, nn, Q, 1.0, dJ.d(), Q, dP.d(), nn, 0.0, db.d(), Q);
    }
    d2h(c, b, db.d(), nn * Q);
    flush_timers(c);
  });
}

// Conventional 4-index AO -> MO transform (Chonky.jl:1-131): out[i,j,k,l] = eri[mu,nu,rho,sigma]
// C1[mu,i] C2[nu,j] C3[rho,k] C4[sigma,l] as four quarter transforms, each one FP64 MFMA GEMM (the
// middle two strided-batched over the indices not yet transformed).
int fh_ao2mo_4index(fh_ctx* x, int nbf, int n1, const double* C1, int n2, const double* C2, int n3, const double* C3,
                    int n4, const double* C4, const double* eri, double* out) {
  return guarded([&] {
    FH_CHECK(x != nullptr && C1 && C2 && C3 && C4 && eri && out, -1, "fh_ao2mo_4index: null argument");
    FH_CHECK(nbf >= 1 && n1 >= 1 && n2 >= 1 && n3 >= 1 && n4 >= 1 && n1 <= nbf && n2 <= nbf && n3 <= nbf && n4 <= nbf,
             -1, "fh_ao2mo_4index: invalid dimensions");
    const int64_t n = nbf, nn = n * n, n3a = nn * n, n4a = nn * nn;
    FH_CHECK((double)n4a < 9.0e18 / 8, -1, "fh_ao2mo_4index: AO tensor too large");
    DeviceGuard g(x->c.device);
    Ctx& c = x->c;
    auto up = [&](const double* h, int64_t cnt) { Buf b = dalloc(c, cnt); h2d(c, b.d(), h, cnt); return b; };
    Buf dC1 = up(C1, n * n1), dC2 = up(C2, n * n2), dC3 = up(C3, n * n3), dC4 = up(C4, n * n4), dE = up(eri, n4a);
    const int64_t m12 = (int64_t)n1 * n2, m123 = m12 * n3, nout = m123 * n4;
    Buf X1 = dalloc(c, (int64_t)n1 * n3a), X2 = dalloc(c, m12 * nn), X3 = dalloc(c, m123 * n), dO = dalloc(c, nout);
    {
      Timer t(c, "ao2mo_4index", 2.0 * ((double)n1 * n4a + (double)m12 * n3a + (double)m123 * nn + (double)nout * n));
      auto gemm = [&](bool ta, int64_t M, int64_t N, int64_t K, const double* A, int64_t lda, int64_t sA, const double* B,
                      int64_t ldb, double* D, int64_t ldd, int64_t sD, int64_t batch) {
        const int64_t wsz = gemm_splitk_elems(M, N, K, batch);
        Buf work;
        if (wsz) work = dalloc(c, wsz);
        gemm_f64(c.s, ta, false, M, N, K, 1.0, A, lda, sA, B, ldb, 0, 0.0, nullptr, 0, 0, D, ldd, sD, batch, 0,
                 work.p ? work.d() : nullptr, wsz);
      };
      // X1[i,(nu rho sigma)] = C1[mu,i] eri[mu,(nu rho sigma)]
      gemm(true, n1, n3a, n, dC1.d(), n, 0, dE.d(), n, X1.d(), n1, 0, 1);
      // X2[(i,j),(rho sigma)] = X1[i,nu,(rho sigma)] C2[nu,j], one batch entry per (rho, sigma), issued in
      // launches of at most 32768 entries (the GEMM grid's batch limit)
      for (int64_t b0 = 0; b0 < nn; b0 += 32768) {
        const int64_t nb = std::min<int64_t>(32768, nn - b0);
        gemm(false, n1, n2, n, X1.d() + b0 * n1 * n, n1, (int64_t)n1 * n, dC2.d(), n, X2.d() + b0 * m12, n1, m12, nb);
      }
      // X3[(i,j,k),sigma] = X2[(i,j),rho,sigma] C3[rho,k], one batch entry per sigma
      gemm(false, m12, n3, n, X2.d(), m12, m12 * n, dC3.d(), n, X3.d(), m12, m123, n);
      // out[(i,j,k),l] = X3[(i,j,k),sigma] C4[sigma,l]
      gemm(false, m123, n4, n, X3.d(), m123, 0, dC4.d(), n, dO.d(), m123, 0, 1);
    }
    d2h(c, out, dO.d(), nout);
    flush_timers(c);
  });
}

int fh_get_df(fh_ctx* x, double* Boo, double* Bov, double* Bvv) {
  return guarded([&] {
    FH_CHECK(x != nullptr, -1, "null context");
    DeviceGuard g(x->c.device);
    Ctx& c = x->c;
    require_df(c, false);
    FH_CHECK(!c.conventional, -6, "fh_get_df: the context holds conventional MO blocks (fh_set_mo), no DF tensors");
    const int64_t Q = c.naux, o = c.o, v = c.v;
    FH_CHECK(!(c.ov_only && (Boo || Bvv)), -6, "only Bov was given to fh_set_df");
    if (Boo) d2h(c, Boo, c.Boo.d(), Q * o * o);
    if (Bov) d2h(c, Bov, c.Bov.d(), Q * o * v);
    if (Bvv) d2h(c, Bvv, c.Bvv.d(), Q * v * v);
  });
}

int fh_mp2_energy(fh_ctx* x, double* E) {
  return guarded([&] {
    FH_CHECK(x != nullptr && E != nullptr, -1, "null argument");
    DeviceGuard g(x->c.device);
    Ctx& c = x->c;
    *E = mp2_energy(c);
    flush_timers(c);
    FH_CHECK(std::isfinite(*E), -5, "non-finite energy");
  });
}

int fh_mp2_energy_noalloc(fh_ctx* x, int o, int v, int naux, const double* eps_o, const double* eps_v,
                          const double* Bov, double* E) {
  return guarded([&] {
    FH_CHECK(x != nullptr && eps_o && eps_v && Bov && E, -1, "fh_mp2_energy_noalloc: null argument");
    FH_CHECK(o >= 1 && v >= 1 && naux >= 1, -1, "fh_mp2_energy_noalloc: invalid dimensions");
    DeviceGuard g(x->c.device);
    Ctx& c = x->c;
    mp2_energy_noalloc(c, o, v, naux, eps_o, eps_v, Bov, E);
    double h = 0.0;
    FH_HIP(hipMemcpyAsync(&h, E, sizeof(double), hipMemcpyDeviceToHost, c.s));
    FH_HIP(hipStreamSynchronize(c.s));
    FH_CHECK(std::isfinite(h), -5, "fh_mp2_energy_noalloc: non-finite energy");
  });
}

int fh_prepare(fh_ctx* x) {
  return guarded([&] {
    FH_CHECK(x != nullptr, -1, "null context");
    DeviceGuard g(x->c.device);
    prepare_rings(x->c);
    prepare_ladder(x->c);
    FH_HIP(hipStreamSynchronize(x->c.s));
    flush_timers(x->c);
  });
}

static void upload_amp(Ctx& c, const double* T1, const double* T2) {
  if (!c.T1.p) c.T1 = dalloc(c, c.nov());
  if (!c.T2.p) c.T2 = dalloc(c, c.n2());
  h2d(c, c.T1.d(), T1, c.nov());
  h2d(c, c.T2.d(), T2, c.n2());
  c.have_amp = true;
}

int fh_t2_guess(fh_ctx* x, int kind, double* T1, double* T2) {
  return guarded([&] {
    FH_CHECK(x != nullptr, -1, "null context");
    FH_CHECK(kind >= 0 && kind <= 3, -1,
             "fh_t2_guess: kind must be 0 (MP2) or 1 (learned), plus 2 for the first-order T1");
    DeviceGuard g(x->c.device);
    Ctx& c = x->c;
    require_df(c);
    bool fell_back = false;
    if (kind & 1) {
      // the MP2 guess is the fallback of the learned one: no network attached, or a guess whose
      // energy is not finite
      if (c.have_model) {
        learned_guess(c);
        if (!std::isfinite(energy(c, c.T1.d(), c.T2.d()))) { mp2_guess(c); fell_back = true; }
      } else {
        mp2_guess(c);
        fell_back = true;
      }
    } else {
      mp2_guess(c);
    }
    if (fell_back) set_error("fh_t2_guess: the learned guess was not available; the MP2 guess was used");
    if (kind & 2) first_order_t1(c);
    if (T1) d2h(c, T1, c.T1.d(), c.nov());
    if (T2) d2h(c, T2, c.T2.d(), c.n2());
    FH_HIP(hipStreamSynchronize(c.s));
    flush_timers(c);
    if (fell_back) throw Fallback{};
  });
}

int fh_ccsd_energy(fh_ctx* x, const double* T1, const double* T2, double* E) {
  return guarded([&] {
    FH_CHECK(x != nullptr && E != nullptr, -1, "null argument");
    DeviceGuard g(x->c.device);
    Ctx& c = x->c;
    require_df(c);
    FH_CHECK((T1 == nullptr) == (T2 == nullptr), -1, "T1 and T2 must both be given or both NULL");
    if (T1) {
      Buf a = dalloc(c, c.nov()), b = dalloc(c, c.n2());
      h2d(c, a.d(), T1, c.nov());
      h2d(c, b.d(), T2, c.n2());
      *E = energy(c, a.d(), b.d());
    } else {
      FH_CHECK(c.have_amp, -6, "no device-resident amplitudes");
      *E = energy(c, c.T1.d(), c.T2.d());
    }
    flush_timers(c);
    FH_CHECK(std::isfinite(*E), -5, "non-finite energy");
  });
}

int fh_ccsd_residual(fh_ctx* x, const double* T1, const double* T2, double* n1, double* n2) {
  return guarded([&] {
    FH_CHECK(x && T1 && T2 && n1 && n2, -1, "null argument");
    DeviceGuard g(x->c.device);
    Ctx& c = x->c;
    require_df(c);
    Buf a = dalloc(c, c.nov()), b = dalloc(c, c.n2()), ra = dalloc(c, c.nov()), rb = dalloc(c, c.n2());
    h2d(c, a.d(), T1, c.nov());
    h2d(c, b.d(), T2, c.n2());
    update_amp(c, a.d(), b.d(), ra.d(), rb.d(), nullptr, nullptr, false);
    d2h(c, n1, ra.d(), c.nov());
    d2h(c, n2, rb.d(), c.n2());
    flush_timers(c);
  });
}

int fh_ccsd_solve(fh_ctx* x, const fh_cc_opts* opts, double* T1, double* T2, fh_cc_result* res) {
  return guarded([&] {
    FH_CHECK(x && res, -1, "null argument");
    FH_CHECK((T1 == nullptr) == (T2 == nullptr), -1, "T1 and T2 must both be given or both NULL");
    DeviceGuard g(x->c.device);
    Ctx& c = x->c;
    require_df(c);
    fh_cc_opts op;
    fh_default_opts(&op);
    if (opts) op = *opts;
    if (T1) upload_amp(c, T1, T2);
    else if (!c.have_amp) mp2_guess(c);
    std::memset(res, 0, sizeof(*res));
    solve(c, op, *res);
    if (T1) {
      d2h(c, T1, c.T1.d(), c.nov());
      d2h(c, T2, c.T2.d(), c.n2());
    }
    FH_HIP(hipStreamSynchronize(c.s));
    flush_timers(c);
  });
}

int fh_triples(fh_ctx* x, int prec_mode, const double* T1, const double* T2, double* Et) {
  return guarded([&] {
    FH_CHECK(x && Et, -1, "null argument");
    FH_CHECK(prec_mode >= 0 && prec_mode <= 2, -1,
             "fh_triples: prec_mode must be 0 (FP64), 1 (FP32 W build) or 2 (split-BF16x3 W build)");
    FH_CHECK((T1 == nullptr) == (T2 == nullptr), -1, "T1 and T2 must both be given or both NULL");
    DeviceGuard g(x->c.device);
    Ctx& c = x->c;
    require_df(c);
    if (T1) upload_amp(c, T1, T2);
    *Et = triples(c, prec_mode);
    flush_timers(c);
    FH_CHECK(std::isfinite(*Et), -5, "non-finite (T) energy");
  });
}

int fh_triples_range(fh_ctx* x, int prec_mode, const double* T1, const double* T2, long long first, long long count,
                     double* Et) {
  return guarded([&] {
    FH_CHECK(x && Et, -1, "null argument");
    FH_CHECK(prec_mode >= 0 && prec_mode <= 2, -1,
             "fh_triples_range: prec_mode must be 0 (FP64), 1 (FP32 W build) or 2 (split-BF16x3 W build)");
    FH_CHECK((T1 == nullptr) == (T2 == nullptr), -1, "T1 and T2 must both be given or both NULL");
    DeviceGuard g(x->c.device);
    Ctx& c = x->c;
    require_df(c);
    const long long o = c.o, ntrip = o * (o + 1) * (o + 2) / 6;
    FH_CHECK(first >= 0 && count >= 0 && first <= ntrip && count <= ntrip - first, -1,
             "fh_triples_range: triples " + std::to_string(first) + " + " + std::to_string(count) + " outside 0.." +
                 std::to_string(ntrip));
    if (T1) upload_amp(c, T1, T2);
    *Et = triples(c, prec_mode, first, count);
    flush_timers(c);
    FH_CHECK(std::isfinite(*Et), -5, "non-finite (T) energy");
  });
}

int fh_stats(fh_ctx* x, char* json, size_t cap) {
  return guarded([&] {
    FH_CHECK(x && json && cap > 0, -1, "null argument");
    Ctx& c = x->c;
    DeviceGuard g(c.device);
    FH_HIP(hipStreamSynchronize(c.s));
    flush_timers(c);
    std::ostringstream s;
    s.precision(17);
    s << "{\"o\":" << c.o << ",\"v\":" << c.v << ",\"naux\":" << c.naux << ",\"pool_peak_bytes\":" << c.pool->peak()
      << ",\"phases\":{";
    bool first = true;
    for (auto& kv : c.phases) {
      if (!first) s << ",";
      first = false;
      s << "\"" << kv.first << "\":{\"ms\":" << kv.second.ms << ",\"flops\":" << kv.second.flops
        << ",\"bytes\":" << kv.second.bytes << ",\"calls\":" << kv.second.calls << "}";
    }
    s << "},\"iterations\":[";
    for (size_t q = 0; q < c.iters.size(); ++q) {
      const IterRow& r = c.iters[q];
      if (q) s << ",";
      s << "[" << r.ite << "," << r.e << "," << r.de << "," << r.rms << "," << r.ms << "," << (r.diis ? "true" : "false") << "]";
    }
    s << "]}";
    const std::string out = s.str();
    FH_CHECK(out.size() + 1 <= cap, -1, "fh_stats: buffer too small (" + std::to_string(out.size() + 1) + " bytes needed)");
    std::memcpy(json, out.c_str(), out.size() + 1);
  });
}

}  // extern "C"

// ---------------------------------------------------------------- Gaussian basis sets and integrals
// A basis set: contracted shells with their primitive coefficients normalised on the host (the
// role of GaussianBasis.jl's BasisSet for AtomicIntegrals.jl:18-45).
struct fh_basis {
  int spherical = 1, nbf = 0, maxl = 0;
  std::vector<int> l, nprim, poff, foff;
  std::vector<double> center, exps, coefs;  // coefs: of unnormalised x^l primitives (normalised contraction)
  std::vector<int> fun;                     // per function: (shell, component)
};

namespace fh {
static double dfact(int n) {
  double r = 1.0;
  for (; n > 1; n -= 2) r *= n;
  return r;
}
// Cartesian exponents, x-major (x^l, x^{l-1} y, x^{l-1} z, ...)
static std::vector<std::array<int, 3>> cart_list(int l) {
  std::vector<std::array<int, 3>> out;
  for (int lx = l; lx >= 0; --lx)
    for (int ly = l - lx; ly >= 0; --ly) out.push_back({lx, ly, l - lx - ly});
  return out;
}
// <x^a y^b z^c | x^a' y^b' z^c'> of one primitive normalised for x^l, relative to <x^l|x^l>
static double cart_ovl(const std::array<int, 3>& e1, const std::array<int, 3>& e2) {
  const int l = e1[0] + e1[1] + e1[2];
  double r = 1.0;
  for (int d = 0; d < 3; ++d) {
    if ((e1[d] + e2[d]) % 2) return 0.0;
    r *= dfact(e1[d] + e2[d] - 1);
  }
  return r / dfact(2 * l - 1);
}
// normalised real solid harmonics (m = -l .. l) over the Cartesian components, l <= 3:
// p: x, y, z; d: xy, yz, 2z^2-x^2-y^2, xz, x^2-y^2; f: 3x^2y-y^3, xyz, y(4z^2-x^2-y^2),
// z(2z^2-3x^2-3y^2), x(4z^2-x^2-y^2), z(x^2-y^2), x^3-3xy^2
static void solid_table(double* tab /*[4][7][10]*/) {
  struct Term { int m, x, y, z; double c; };
  static const std::vector<std::vector<Term>> T = {
      {{0, 0, 0, 0, 1.0}},
      {{0, 1, 0, 0, 1.0}, {1, 0, 1, 0, 1.0}, {2, 0, 0, 1, 1.0}},
      {{0, 1, 1, 0, 1.0}, {1, 0, 1, 1, 1.0}, {2, 0, 0, 2, 2.0}, {2, 2, 0, 0, -1.0}, {2, 0, 2, 0, -1.0},
       {3, 1, 0, 1, 1.0}, {4, 2, 0, 0, 1.0}, {4, 0, 2, 0, -1.0}},
      {{0, 2, 1, 0, 3.0}, {0, 0, 3, 0, -1.0}, {1, 1, 1, 1, 1.0}, {2, 0, 1, 2, 4.0}, {2, 2, 1, 0, -1.0},
       {2, 0, 3, 0, -1.0}, {3, 0, 0, 3, 2.0}, {3, 2, 0, 1, -3.0}, {3, 0, 2, 1, -3.0}, {4, 1, 0, 2, 4.0},
       {4, 3, 0, 0, -1.0}, {4, 1, 2, 0, -1.0}, {5, 2, 0, 1, 1.0}, {5, 0, 2, 1, -1.0}, {6, 3, 0, 0, 1.0},
       {6, 1, 2, 0, -3.0}}};
  std::fill(tab, tab + 4 * 7 * 10, 0.0);
  for (int l = 0; l <= 3; ++l) {
    const auto cl = cart_list(l);
    for (const Term& t : T[l]) {
      for (size_t k = 0; k < cl.size(); ++k)
        if (cl[k][0] == t.x && cl[k][1] == t.y && cl[k][2] == t.z) tab[(l * 7 + t.m) * 10 + k] = t.c;
    }
    for (int m = 0; m < 2 * l + 1; ++m) {
      double n2 = 0.0;
      for (size_t i = 0; i < cl.size(); ++i)
        for (size_t j = 0; j < cl.size(); ++j) n2 += tab[(l * 7 + m) * 10 + i] * tab[(l * 7 + m) * 10 + j] * cart_ovl(cl[i], cl[j]);
      for (size_t i = 0; i < cl.size(); ++i) tab[(l * 7 + m) * 10 + i] /= std::sqrt(n2);
    }
  }
}

// the device copy of a basis set for one call
struct DevBasis {
  Buf shells, ex, cf;
  std::vector<char> host;
};
static DevBasis upload_basis(Ctx& c, const fh_basis& b) {
  DevBasis d;
  const size_t sz = integrals_shell_bytes(), ns = b.l.size();
  d.host.resize(sz * ns);
  for (size_t i = 0; i < ns; ++i)
    integrals_pack_shell(d.host.data() + i * sz, b.l[i], b.nprim[i], b.poff[i], b.foff[i], &b.center[3 * i]);
  d.shells = Buf(c.pool.get(), std::max<size_t>(d.host.size(), 1));
  FH_HIP(hipMemcpyAsync(d.shells.p, d.host.data(), d.host.size(), hipMemcpyHostToDevice, c.s));
  d.ex = dalloc(c, (int64_t)b.exps.size());
  d.cf = dalloc(c, (int64_t)b.coefs.size());
  h2d(c, d.ex.d(), b.exps.data(), (int64_t)b.exps.size());
  h2d(c, d.cf.d(), b.coefs.data(), (int64_t)b.coefs.size());
  return d;
}
static std::vector<char> sph_tab(int spherical) {
  double t[4 * 7 * 10];
  solid_table(t);
  std::vector<char> out(integrals_table_bytes());
  integrals_pack_table(out.data(), t, spherical);
  return out;
}
static IntBasis int_basis(const fh_basis& b) {
  return {(int)b.l.size(), b.nbf, b.spherical, (int)b.exps.size(), b.l.data(), b.nprim.data(), b.poff.data(), b.foff.data(),
          b.center.data(), b.exps.data(), b.coefs.data()};
}
}  // namespace fh

extern "C" {

int fh_basis_create(fh_basis** out, int nshell, const int* l, const int* nprim, const double* center,
                    const double* exps, const double* coefs, int spherical) {
  return guarded([&] {
    FH_CHECK(out != nullptr, -1, "null argument");
    *out = nullptr;
    FH_CHECK(nshell >= 1 && l && nprim && center && exps && coefs, -1, "fh_basis_create: invalid arguments");
    std::unique_ptr<fh_basis> b(new fh_basis());
    b->spherical = spherical ? 1 : 0;
    int off = 0, f = 0;
    for (int i = 0; i < nshell; ++i) {
      FH_CHECK(l[i] >= 0 && l[i] <= integrals_max_l_aux(), -1,
               "fh_basis_create: angular momentum " + std::to_string(l[i]) + " above f");
      FH_CHECK(nprim[i] >= 1 && nprim[i] <= 64, -1, "fh_basis_create: 1..64 primitives per shell");
      const int L = l[i];
      std::vector<double> c(nprim[i]);
      for (int k = 0; k < nprim[i]; ++k) {
        const double a = exps[off + k];
        FH_CHECK(a > 0.0 && std::isfinite(a) && std::isfinite(coefs[off + k]), -1, "fh_basis_create: invalid exponent");
        c[k] = coefs[off + k] * std::pow(2.0 * a / M_PI, 0.75) * std::pow(4.0 * a, 0.5 * L) / std::sqrt(dfact(2 * L - 1));
      }
      double s = 0.0;
      for (int k = 0; k < nprim[i]; ++k)
        for (int q = 0; q < nprim[i]; ++q) {
          const double p = exps[off + k] + exps[off + q];
          s += c[k] * c[q] * std::pow(M_PI / p, 1.5) * dfact(2 * L - 1) / std::pow(2.0 * p, L);
        }
      FH_CHECK(s > 0.0, -1, "fh_basis_create: contraction of zero norm");
      for (int k = 0; k < nprim[i]; ++k) {
        b->exps.push_back(exps[off + k]);
        b->coefs.push_back(c[k] / std::sqrt(s));
      }
      b->l.push_back(L);
      b->nprim.push_back(nprim[i]);
      b->poff.push_back(off);
      b->foff.push_back(f);
      for (int d = 0; d < 3; ++d) b->center.push_back(center[3 * i + d]);
      const int nf = spherical ? 2 * L + 1 : (L + 1) * (L + 2) / 2;
      for (int m = 0; m < nf; ++m) { b->fun.push_back(i); b->fun.push_back(m); }
      f += nf;
      off += nprim[i];
      b->maxl = std::max(b->maxl, L);
    }
    b->nbf = f;
    *out = b.release();
  });
}

int fh_basis_nbf(const fh_basis* b) { return b ? b->nbf : 0; }

void fh_basis_destroy(fh_basis* b) { delete b; }

// S, T, V (overlap / kinetic / nuclear of AtomicIntegrals.jl:16-29): any output may be NULL
int fh_one_electron(fh_ctx* x, const fh_basis* b, int natom, const double* Z, const double* xyz, double* S, double* T,
                    double* V) {
  return guarded([&] {
    FH_CHECK(x && b, -1, "null argument");
    FH_CHECK(natom >= 0 && (natom == 0 || (Z && xyz)), -1, "fh_one_electron: invalid atoms");
    DeviceGuard g(x->c.device);
    Ctx& c = x->c;
    const int n = b->nbf;
    DevBasis d = upload_basis(c, *b);
    const auto tab = sph_tab(b->spherical);
    Buf dZ = dalloc(c, std::max(natom, 1)), dX = dalloc(c, 3 * std::max(natom, 1));
    if (natom) { h2d(c, dZ.d(), Z, natom); h2d(c, dX.d(), xyz, 3 * natom); }
    Buf dS = dalloc(c, (int64_t)n * n), dT = dalloc(c, (int64_t)n * n), dV = dalloc(c, (int64_t)n * n);
    {
      Timer t(c, "ao_one_electron");
      integrals_one_electron(c.s, (int)b->l.size(), d.shells.p, d.ex.d(), d.cf.d(), natom, dZ.d(), dX.d(), tab.data(),
                             n, dS.d(), dT.d(), dV.d());
    }
    if (S) d2h(c, S, dS.d(), (int64_t)n * n);
    if (T) d2h(c, T, dT.d(), (int64_t)n * n);
    if (V) d2h(c, V, dV.d(), (int64_t)n * n);
    FH_HIP(hipStreamSynchronize(c.s));
    flush_timers(c);
  });
}

// dipole integrals <mu| r - origin |nu> (GaussianBasis.dipole, as FourthMoment.jl:74 uses it)
int fh_dipole(fh_ctx* x, const fh_basis* b, const double* origin, double* Dx, double* Dy, double* Dz) {
  return guarded([&] {
    FH_CHECK(x && b && Dx && Dy && Dz, -1, "null argument");
    DeviceGuard g(x->c.device);
    Ctx& c = x->c;
    const int64_t n = b->nbf;
    const double zero[3] = {0.0, 0.0, 0.0};
    DevBasis d = upload_basis(c, *b);
    const auto tab = sph_tab(b->spherical);
    Buf o1 = dalloc(c, n * n), o2 = dalloc(c, n * n), o3 = dalloc(c, n * n);
    integrals_dipole(c.s, (int)b->l.size(), d.shells.p, d.ex.d(), d.cf.d(), origin ? origin : zero, tab.data(), (int)n,
                     o1.d(), o2.d(), o3.d());
    d2h(c, Dx, o1.d(), n * n);
    d2h(c, Dy, o2.d(), n * n);
    d2h(c, Dz, o3.d(), n * n);
  });
}

// (mu nu|la si), eri[nbf^4] column-major (ERI_2e4c, AtomicIntegrals.jl:43-46)
int fh_eri_2e4c(fh_ctx* x, const fh_basis* b, double* eri) {
  return guarded([&] {
    FH_CHECK(x && b && eri, -1, "null argument");
    FH_CHECK(b->maxl <= integrals_max_l_orbital(), -1, "fh_eri_2e4c: orbital shells up to d");
    const int64_t n = b->nbf;
    FH_CHECK((double)n * n * n * n < 4.0e9, -1, "fh_eri_2e4c: 4-index tensor too large (nbf^4 >= 4e9)");
    DeviceGuard g(x->c.device);
    Ctx& c = x->c;
    const auto tab = sph_tab(b->spherical);
    IntScratch sc;
    Buf out = dalloc(c, n * n * n * n);
    {
      Timer t(c, "ao_eri_4c");
      integrals_eri4c(c.s, c.pool.get(), sc, int_basis(*b), tab.data(), out.d());
    }
    d2h(c, eri, out.d(), n * n * n * n);
    flush_timers(c);
  });
}

// Pqp[mu, nu, P] = (mu nu|P) (ERI_2e3c(bs, auxbs), AtomicIntegrals.jl:36)
int fh_eri_2e3c(fh_ctx* x, const fh_basis* b, const fh_basis* aux, double* Pqp) {
  return guarded([&] {
    FH_CHECK(x && b && aux && Pqp, -1, "null argument");
    FH_CHECK(b->maxl <= integrals_max_l_orbital(), -1, "fh_eri_2e3c: orbital shells up to d");
    FH_CHECK(b->spherical == aux->spherical, -1, "fh_eri_2e3c: both sets spherical or both Cartesian");
    const int64_t n = b->nbf, Q = aux->nbf;
    DeviceGuard g(x->c.device);
    Ctx& c = x->c;
    const auto tab = sph_tab(b->spherical);
    IntScratch sc;
    Buf out = dalloc(c, n * n * Q);
    {
      Timer t(c, "ao_eri_3c");
      integrals_eri3c(c.s, c.pool.get(), sc, int_basis(*b), int_basis(*aux), tab.data(), out.d());
    }
    d2h(c, Pqp, out.d(), n * n * Q);
    flush_timers(c);
  });
}

// J[P, Q] = (P|Q) (ERI_2e2c(auxbs), AtomicIntegrals.jl:35)
int fh_eri_2e2c(fh_ctx* x, const fh_basis* aux, double* J) {
  return guarded([&] {
    FH_CHECK(x && aux && J, -1, "null argument");
    const int64_t Q = aux->nbf;
    DeviceGuard g(x->c.device);
    Ctx& c = x->c;
    const auto tab = sph_tab(aux->spherical);
    IntScratch sc;
    Buf out = dalloc(c, Q * Q);
    {
      Timer t(c, "ao_eri_2c");
      integrals_eri2c(c.s, c.pool.get(), sc, int_basis(*aux), tab.data(), out.d());
    }
    d2h(c, J, out.d(), Q * Q);
    flush_timers(c);
  });
}

// ---------------------------------------------------------------- learned T2 guess network
struct fh_mlp {
  int device = 0;
  hipStream_t s = nullptr;
  std::unique_ptr<Pool> pool;  // declared before the Bufs: destroyed after them
  int h = 0;
  int64_t step = 0;
  Buf P, G, m, v;
};

static void mlp_upload(fh_mlp* n, void* dst, const void* src, size_t bytes) {
  FH_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, n->s));
}

int fh_mlp_create(fh_mlp** out, int device, int hidden, unsigned long long seed) {
  return guarded([&] {
    FH_CHECK(out != nullptr, -1, "null argument");
    FH_CHECK(hidden > 0 && 256 % hidden == 0, -1, "fh_mlp_create: hidden width must divide 256");
    *out = nullptr;
    DeviceGuard g(device);
    std::unique_ptr<fh_mlp> n(new fh_mlp());
    n->device = device;
    FH_HIP(hipSetDevice(device));
    FH_HIP(hipStreamCreate(&n->s));
    n->pool.reset(new Pool(device));
    n->h = hidden;
    const size_t np = mlp_nparams(hidden);
    n->P = Buf(n->pool.get(), np * sizeof(float));
    n->G = Buf(n->pool.get(), np * sizeof(float));
    n->m = Buf(n->pool.get(), np * sizeof(float));
    n->v = Buf(n->pool.get(), np * sizeof(float));
    // Glorot-uniform weights, zero biases
    std::vector<float> p(np, 0.0f);
    std::mt19937_64 rng(seed);
    const MlpOffsets o = mlp_offsets(hidden);
    auto glorot = [&](size_t off, int fan_out, int fan_in) {
      std::uniform_real_distribution<float> u(-1.0f, 1.0f);
      const float a = std::sqrt(6.0f / (float)(fan_in + fan_out));
      for (size_t k = 0; k < (size_t)fan_out * fan_in; ++k) p[off + k] = a * u(rng);
    };
    glorot(o.W1, hidden, 6);
    glorot(o.W2, hidden, hidden);
    glorot(o.W3, hidden, hidden);
    glorot(o.w4, 1, hidden);
    mlp_upload(n.get(), n->P.p, p.data(), np * sizeof(float));
    std::vector<float> z(np, 0.0f);
    mlp_upload(n.get(), n->m.p, z.data(), np * sizeof(float));
    mlp_upload(n.get(), n->v.p, z.data(), np * sizeof(float));
    FH_HIP(hipStreamSynchronize(n->s));
    *out = n.release();
  });
}

size_t fh_mlp_num_params(const fh_mlp* n) { return n ? mlp_nparams(n->h) : 0; }

int fh_mlp_get_params(fh_mlp* n, float* params) {
  return guarded([&] {
    FH_CHECK(n != nullptr && params != nullptr, -1, "null argument");
    DeviceGuard g(n->device);
    FH_HIP(hipMemcpyAsync(params, n->P.p, mlp_nparams(n->h) * sizeof(float), hipMemcpyDeviceToHost, n->s));
    FH_HIP(hipStreamSynchronize(n->s));
  });
}

int fh_mlp_set_params(fh_mlp* n, const float* params) {
  return guarded([&] {
    FH_CHECK(n != nullptr && params != nullptr, -1, "null argument");
    DeviceGuard g(n->device);
    for (size_t k = 0; k < mlp_nparams(n->h); ++k)
      FH_CHECK(std::isfinite(params[k]), -5, "fh_mlp_set_params: non-finite parameter");
    mlp_upload(n, n->P.p, params, mlp_nparams(n->h) * sizeof(float));
    n->step = 0;
    std::vector<float> z(mlp_nparams(n->h), 0.0f);
    mlp_upload(n, n->m.p, z.data(), z.size() * sizeof(float));
    mlp_upload(n, n->v.p, z.data(), z.size() * sizeof(float));
    FH_HIP(hipStreamSynchronize(n->s));
  });
}

int fh_mlp_forward(fh_mlp* n, long long ns, const float* X, float* Y) {
  return guarded([&] {
    FH_CHECK(n != nullptr && X != nullptr && Y != nullptr && ns >= 0, -1, "invalid argument");
    DeviceGuard g(n->device);
    if (ns == 0) return;
    const int h = n->h;
    const int64_t C = std::min<int64_t>(ns, (int64_t)1 << 20);
    Buf dX(n->pool.get(), (size_t)(6 * C) * sizeof(float)), A(n->pool.get(), (size_t)(3 * h * C) * sizeof(float));
    Buf dY(n->pool.get(), (size_t)C * sizeof(float));
    for (int64_t e0 = 0; e0 < ns; e0 += C) {
      const int64_t m = std::min<int64_t>(C, ns - e0);
      mlp_upload(n, dX.p, X + 6 * e0, (size_t)(6 * m) * sizeof(float));
      mlp_forward(n->s, h, n->P.f(), m, dX.f(), A.f(), A.f() + h * C, A.f() + 2 * h * C, dY.f());
      FH_HIP(hipMemcpyAsync(Y + e0, dY.p, (size_t)m * sizeof(float), hipMemcpyDeviceToHost, n->s));
    }
    FH_HIP(hipStreamSynchronize(n->s));
  });
}

// one batch on the device: forward + backward into n->G; batch loss sum (B*L) into *lsum (device)
static void mlp_batch(fh_mlp* n, int64_t B, const float* X, const float* T, Buf& A, Buf& dy, Buf& dAZ, Buf& part,
                      Buf& lpart, double* lsum) {
  const int h = n->h;
  float* A1 = A.f();
  float* A2 = A1 + (int64_t)h * B;
  float* A3 = A2 + (int64_t)h * B;
  float* y = A3 + (int64_t)h * B;
  mlp_forward(n->s, h, n->P.f(), B, X, A1, A2, A3, y);
  int64_t nl = 0;
  mlp_backward(n->s, h, n->P.f(), B, X, T, A1, A2, A3, y, dy.f(), dAZ.f(), dAZ.f() + (int64_t)h * B, n->G.f(), part.f(),
               lpart.d(), &nl);
  sum_partials(n->s, nl, lpart.d(), lsum);
}

struct MlpWork {
  Buf A, dy, dAZ, part, lpart;
  MlpWork(fh_mlp* n, int64_t B)
      : A(n->pool.get(), (size_t)((3 * n->h + 1) * B) * sizeof(float)),
        dy(n->pool.get(), (size_t)B * sizeof(float)),
        dAZ(n->pool.get(), (size_t)(2 * n->h * B) * sizeof(float)),
        part(n->pool.get(), (size_t)mlp_partial_elems(n->h, B) * sizeof(float)),
        lpart(n->pool.get(), (size_t)kMlpLossPartials * sizeof(double)) {}
};

int fh_mlp_loss_grad(fh_mlp* n, long long ns, const float* X, const float* T, double* loss, float* grad) {
  return guarded([&] {
    FH_CHECK(n != nullptr && X != nullptr && T != nullptr && ns > 0, -1, "invalid argument");
    DeviceGuard g(n->device);
    Buf dX(n->pool.get(), (size_t)(6 * ns) * sizeof(float)), dT(n->pool.get(), (size_t)ns * sizeof(float));
    Buf ls(n->pool.get(), sizeof(double));
    mlp_upload(n, dX.p, X, (size_t)(6 * ns) * sizeof(float));
    mlp_upload(n, dT.p, T, (size_t)ns * sizeof(float));
    MlpWork w(n, ns);
    mlp_batch(n, ns, dX.f(), dT.f(), w.A, w.dy, w.dAZ, w.part, w.lpart, ls.d());
    double l = 0.0;
    FH_HIP(hipMemcpyAsync(&l, ls.p, sizeof(double), hipMemcpyDeviceToHost, n->s));
    if (grad) FH_HIP(hipMemcpyAsync(grad, n->G.p, mlp_nparams(n->h) * sizeof(float), hipMemcpyDeviceToHost, n->s));
    FH_HIP(hipStreamSynchronize(n->s));
    if (loss) *loss = l / (double)ns;
  });
}

int fh_mlp_train(fh_mlp* n, long long ns, const float* X, const float* T, int epochs, int batch, float lr,
                 unsigned long long seed, double* epoch_loss) {
  return guarded([&] {
    FH_CHECK(n != nullptr && X != nullptr && T != nullptr && ns > 0 && epochs >= 0 && batch > 0 && lr > 0.0f, -1,
             "invalid argument");
    DeviceGuard g(n->device);
    Buf dX(n->pool.get(), (size_t)(6 * ns) * sizeof(float)), dT(n->pool.get(), (size_t)ns * sizeof(float));
    mlp_upload(n, dX.p, X, (size_t)(6 * ns) * sizeof(float));
    mlp_upload(n, dT.p, T, (size_t)ns * sizeof(float));
    const int64_t B = std::min<int64_t>(batch, ns);
    const int64_t nbat = (ns + B - 1) / B;
    MlpWork w(n, B);
    Buf Xb(n->pool.get(), (size_t)(6 * B) * sizeof(float)), Tb(n->pool.get(), (size_t)B * sizeof(float));
    Buf perm(n->pool.get(), (size_t)ns * sizeof(int64_t)), ls(n->pool.get(), (size_t)nbat * sizeof(double));
    std::vector<int64_t> hp(ns);
    std::vector<double> hl(nbat);
    std::mt19937_64 rng(seed);
    const size_t np = mlp_nparams(n->h);
    for (int ep = 0; ep < epochs; ++ep) {
      for (int64_t k = 0; k < ns; ++k) hp[k] = k;
      std::shuffle(hp.begin(), hp.end(), rng);
      mlp_upload(n, perm.p, hp.data(), (size_t)ns * sizeof(int64_t));
      for (int64_t b = 0; b < nbat; ++b) {
        const int64_t off = b * B, m = std::min<int64_t>(B, ns - off);
        mlp_gather(n->s, m, off, static_cast<const int64_t*>(perm.p), dX.f(), dT.f(), Xb.f(), Tb.f());
        mlp_batch(n, m, Xb.f(), Tb.f(), w.A, w.dy, w.dAZ, w.part, w.lpart, ls.d() + b);
        mlp_adam(n->s, (int64_t)np, n->P.f(), n->G.f(), n->m.f(), n->v.f(), lr, ++n->step);
      }
      FH_HIP(hipMemcpyAsync(hl.data(), ls.p, (size_t)nbat * sizeof(double), hipMemcpyDeviceToHost, n->s));
      FH_HIP(hipStreamSynchronize(n->s));
      double tot = 0.0;
      for (double q : hl) tot += q;
      FH_CHECK(std::isfinite(tot), -5, "fh_mlp_train: non-finite loss");
      if (epoch_loss) epoch_loss[ep] = tot / (double)ns;
    }
  });
}

void fh_mlp_destroy(fh_mlp* n) {
  if (!n) return;
  DeviceGuard g(n->device);
  (void)hipStreamSynchronize(n->s);
  hipStream_t s = n->s;
  delete n;
  (void)hipStreamDestroy(s);
}

// Attach the network parameters and normalisation (host arrays) to a context: the part of
// fh_set_t2_model / fh_load_t2_model after the parameters are known.
static void attach_t2_model(Ctx& c, int h, const float* params_host, const float* params_dev, const float* x_mean,
                            const float* x_scale, double y_scale, const double* pair_dist) {
  require_df(c);
  FH_CHECK(std::isfinite(y_scale), -1, "t2 model: non-finite y_scale");
  const size_t np = mlp_nparams(h);
  c.mlp_P = Buf(c.pool.get(), np * sizeof(float));
  if (params_dev) FH_HIP(hipMemcpyAsync(c.mlp_P.p, params_dev, np * sizeof(float), hipMemcpyDeviceToDevice, c.s));
  else FH_HIP(hipMemcpyAsync(c.mlp_P.p, params_host, np * sizeof(float), hipMemcpyHostToDevice, c.s));
  c.mlp_xm = Buf(c.pool.get(), 6 * sizeof(float));
  c.mlp_xs = Buf(c.pool.get(), 6 * sizeof(float));
  FH_HIP(hipMemcpyAsync(c.mlp_xm.p, x_mean, 6 * sizeof(float), hipMemcpyHostToDevice, c.s));
  FH_HIP(hipMemcpyAsync(c.mlp_xs.p, x_scale, 6 * sizeof(float), hipMemcpyHostToDevice, c.s));
  c.pair_d = dalloc(c, c.o * c.o);
  if (pair_dist) FH_HIP(hipMemcpyAsync(c.pair_d.p, pair_dist, (size_t)(c.o * c.o) * sizeof(double), hipMemcpyHostToDevice, c.s));
  else fill_f64(c.s, c.o * c.o, 0.0, c.pair_d.d());
  FH_HIP(hipStreamSynchronize(c.s));
  c.mlp_h = h;
  c.mlp_ys = y_scale;
  c.have_model = true;
}

// Model file of the learned guess (little-endian): "FHT2MLP1", int32 hidden, int32 nparams,
// float32 x_mean[6], float32 x_scale[6], float64 y_scale, float32 params[nparams].
int fh_load_t2_model(fh_ctx* x, const char* path, const double* pair_dist) {
  return guarded([&] {
    FH_CHECK(x != nullptr && path != nullptr, -1, "null argument");
    DeviceGuard g(x->c.device);
    Ctx& c = x->c;
    std::unique_ptr<FILE, int (*)(FILE*)> f(std::fopen(path, "rb"), &std::fclose);
    FH_CHECK(f != nullptr, -1, std::string("fh_load_t2_model: cannot open ") + path);
    char magic[8];
    int32_t h = 0, np = 0;
    float xm[6], xs[6];
    double ys = 0.0;
    auto rd = [&](void* dst, size_t bytes) {
      FH_CHECK(std::fread(dst, 1, bytes, f.get()) == bytes, -1, std::string("fh_load_t2_model: truncated file ") + path);
    };
    rd(magic, 8);
    FH_CHECK(std::memcmp(magic, "FHT2MLP1", 8) == 0, -1, std::string("fh_load_t2_model: not a model file: ") + path);
    rd(&h, 4);
    rd(&np, 4);
    FH_CHECK(h > 0 && h <= 1024 && 256 % h == 0 && (size_t)np == mlp_nparams(h), -1,
             "fh_load_t2_model: inconsistent width / parameter count");
    rd(xm, sizeof(xm));
    rd(xs, sizeof(xs));
    rd(&ys, sizeof(ys));
    std::vector<float> params((size_t)np);
    rd(params.data(), params.size() * sizeof(float));
    for (float q : params) FH_CHECK(std::isfinite(q), -5, "fh_load_t2_model: non-finite parameter");
    attach_t2_model(c, h, params.data(), nullptr, xm, xs, ys, pair_dist);
  });
}

int fh_set_t2_model(fh_ctx* x, const fh_mlp* net, const float* x_mean, const float* x_scale, double y_scale,
                    const double* pair_dist) {
  return guarded([&] {
    FH_CHECK(x != nullptr && net != nullptr && x_mean != nullptr && x_scale != nullptr, -1, "null argument");
    DeviceGuard g(x->c.device);
    FH_HIP(hipStreamSynchronize(net->s));
    attach_t2_model(x->c, net->h, nullptr, net->P.f(), x_mean, x_scale, y_scale, pair_dist);
  });
}

}  // extern "C"
