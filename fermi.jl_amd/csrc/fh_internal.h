// Internal declarations shared by the libfermihip translation units.
// All tensors are column-major (first index fastest), like the Julia arrays that
// cross the C-ABI.  Everything here runs on one HIP stream owned by the context.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstddef>
#include <functional>
#include <string>
#include <vector>
#include <map>

namespace fh {

// ---------------------------------------------------------------- errors
struct Error {
  int code;
  std::string msg;
};
void set_error(const std::string& m);
#define FH_HIP(x)                                                                    \
  do {                                                                               \
    hipError_t e_ = (x);                                                             \
    if (e_ != hipSuccess)                                                            \
      throw ::fh::Error{-2, std::string("HIP error ") + hipGetErrorString(e_) + " at " + __FILE__ + ":" + std::to_string(__LINE__)}; \
  } while (0)
#define FH_CHECK(cond, code, msg)                  \
  do {                                             \
    if (!(cond)) throw ::fh::Error{(code), (msg)}; \
  } while (0)

// ---------------------------------------------------------------- device memory pool
// Size-bucketed caching allocator: buffers are returned to a free list and reused;
// nothing is released to HIP until the pool is destroyed or an allocation would fail.
class Pool {
 public:
  explicit Pool(int device) : device_(device) {}
  ~Pool();
  void* get(size_t bytes);
  void put(void* p);
  size_t in_use() const { return in_use_; }
  size_t peak() const { return peak_; }
  void release_free();
  // what else can be freed when an allocation still fails without the free list
  std::function<void()> give_back;
 private:
  int device_;
  std::multimap<size_t, void*> free_;
  std::map<void*, size_t> live_;
  size_t in_use_ = 0, peak_ = 0;
};

// Owning device buffer handed out by the pool.
struct Buf {
  Pool* pool = nullptr;
  void* p = nullptr;
  size_t bytes = 0;
  Buf() = default;
  Buf(Pool* pl, size_t b) : pool(pl), p(b ? pl->get(b) : nullptr), bytes(b) {}
  Buf(const Buf&) = delete;
  Buf& operator=(const Buf&) = delete;
  Buf(Buf&& o) noexcept { *this = std::move(o); }
  Buf& operator=(Buf&& o) noexcept {
    if (this != &o) { reset(); pool = o.pool; p = o.p; bytes = o.bytes; o.p = nullptr; o.bytes = 0; }
    return *this;
  }
  ~Buf() { reset(); }
  void reset() { if (p && pool) pool->put(p); p = nullptr; bytes = 0; }
  double* d() const { return static_cast<double*>(p); }
  float* f() const { return static_cast<float*>(p); }
};

// A column-major FP64 tensor view (up to 6 modes).
struct TView {
  double* p = nullptr;
  int nd = 0;
  int64_t dim[6] = {1, 1, 1, 1, 1, 1};
  int64_t size() const { int64_t s = 1; for (int i = 0; i < nd; ++i) s *= dim[i]; return s; }
};
inline TView tv(double* p, std::initializer_list<int64_t> dims) {
  TView t; t.p = p; t.nd = 0;
  for (int64_t d : dims) t.dim[t.nd++] = d;
  return t;
}
// a view of a scratch buffer: refused when the tensor does not fit the buffer
inline TView tv(const Buf& b, std::initializer_list<int64_t> dims) {
  TView t = tv(b.d(), dims);
  FH_CHECK((size_t)t.size() * sizeof(double) <= b.bytes, -3, "tensor view larger than its scratch buffer");
  return t;
}

// ---------------------------------------------------------------- kernel launchers
// D = alpha * op(A) * op(B) + beta * C  (column-major, FP64 MFMA); C may alias D.
// Strided batches: A_i = A + i*sA etc.
void gemm_f64(hipStream_t s, bool ta, bool tb, int64_t M, int64_t N, int64_t K, double alpha,
              const double* A, int64_t lda, int64_t sA, const double* B, int64_t ldb, int64_t sB,
              double beta, const double* C, int64_t ldc, int64_t sC, double* D, int64_t ldd, int64_t sD,
              int64_t batch = 1, int tag = 0, double* work = nullptr, int64_t work_elems = 0,
              bool f32 = false);
// f32 = true: operands rounded to FP32 in LDS, FP32 MFMA with FP32 accumulation (mixed precision)

// FP32-MFMA GEMM (NN) with FP32 operands in HBM and FP64 output
void gemm_f32_fd(hipStream_t s, int64_t M, int64_t N, int64_t K, double alpha, const float* A, int64_t lda, int64_t sA,
                 const float* B, int64_t ldb, int64_t sB, double beta, const double* C, int64_t ldc, double* D, int64_t ldd,
                 int64_t sD, int64_t batch, int tag, double* work = nullptr, int64_t work_elems = 0);
// FP32 operands and output, any transposition, C = alpha op(A) op(B) + beta C (tag 3)
void gemm_f32(hipStream_t s, bool ta, bool tb, int64_t M, int64_t N, int64_t K, double alpha, const float* A,
              int64_t lda, const float* B, int64_t ldb, double beta, float* C, int64_t ldc, float* work = nullptr,
              int64_t work_elems = 0);
// FP32 network layer: D = tanh(A B + bias[row]) (tag 4)
void gemm_f32_tanh(hipStream_t s, int64_t M, int64_t N, int64_t K, const float* A, int64_t lda, const float* B, int64_t ldb,
                   const float* bias, float* D, int64_t ldd);
// split-BF16x3 MFMA GEMM (three bf16 products per FP32 product, FP32 accumulation) on FP32 operands with FP64
// output: tag 0 any transposition, tag 1 (the PP ladder) untransposed; the tags give distinct kernel symbols
void gemm_bf3(hipStream_t s, bool ta, bool tb, int64_t M, int64_t N, int64_t K, double alpha, const float* A,
              int64_t lda, int64_t sA, const float* B, int64_t ldb, int64_t sB, double beta, const double* C, int64_t ldc,
              double* D, int64_t ldd, int64_t sD, int64_t batch, int tag, double* work = nullptr,
              int64_t work_elems = 0);
// its workspace (doubles) to split K for this shape (0: no split)
int64_t gemm_bf3_splitk_elems(bool ta, bool tb, int64_t M, int64_t N, int64_t K, int64_t batch, int tag);
// D = alpha sum_s W_s + beta C over the S slices W [M N][batch][S] of a product cut along K
void splitk_reduce_f64(hipStream_t s, int64_t M, int64_t N, int64_t S, const double* W, double alpha, double beta,
                       const double* C, int64_t ldc, int64_t sC, double* D, int64_t ldd, int64_t sD, int64_t batch);

// ---------------------------------------------------------------- (T) W build (fh_triples.hip)
// elements of an (a, b) plane of W, in panels of 8 a: [a / 8][b][a % 8]
__host__ __device__ inline int64_t triples_plane(int v) { return (int64_t)8 * ((v + 7) / 8) * v; }
// fmt: 0 FP64, 1 FP32, 2 split-BF16x3 (W in FP32).  Operands hold triples_pitch_elems(o, v) values of k per
// row (8 bytes each for fmt 0, else 4): av, avs v^2 o rows each, bvp, bvq v o^2 rows each.
struct TriplesOperands {
  void *av, *avs, *bvp, *bvq;
};
struct TriplesTiles {
  int grain, nb, per, nt;            // slices: blocks of `grain`, at most `per` of them per tile, nt tiles along v
  int nb_first, per_first, nt_first; // first launch: the same, nt_first tiles along v^2
};
int64_t triples_pitch_elems(int o, int v);
void triples_operands(hipStream_t s, int fmt, int o, int v, const double* ovvv, const double* t2, const double* ooov,
                      void* av, void* avs, void* bvp, void* bvq);
TriplesTiles triples_tiles(int fmt, int o, int v, double nk);  // nk: mean k per run
// W slots (triples) of a chunk, out of ntot
int64_t triples_chunk_slots(int v, int elem, const TriplesTiles& tt, int64_t ntot);
// appends the column tiles of the run k0 .. k0 + nk - 1 of (i, j), its W slots from `slot`: 8 ints each
void triples_col_tiles(const TriplesTiles& t, int v, int i, int j, int k0, int nk, int slot, std::vector<int>& out);
// W[plane(a, b) of c of a slot, v planes a slot] = classes abc + bac; then += the other four (slots: 4 ints (i, j, k, 0) each)
void triples_w_first(hipStream_t s, int fmt, int o, int v, const TriplesTiles& tt, const TriplesOperands& op, void* W,
                     const int* cols, int ncol);
void triples_w_slices(hipStream_t s, int fmt, int o, int v, const TriplesTiles& tt, const TriplesOperands& op, void* W,
                      const int* slots, int nslot);
// ---------------------------------------------------------------- T2-guess network (fh_mlp.hip)
struct MlpOffsets {
  size_t W1, b1, W2, b2, W3, b3, w4, b4;
};
size_t mlp_nparams(int h);
MlpOffsets mlp_offsets(int h);
int64_t mlp_partial_elems(int h, int64_t B);  // floats of the bias-gradient scratch for batch B
// forward of a batch X[6,B] -> activations A1..A3 [h,B] and outputs y[B]
void mlp_forward(hipStream_t s, int h, const float* P, int64_t B, const float* X, float* A1, float* A2, float* A3,
                 float* y);
// gradient G of L = 1/(2B) sum (y - T)^2 after mlp_forward; dy[B], dA/dZ [h,B] scratch; lpart gets
// *nlpart partial sums of B*L (at most kMlpLossPartials doubles, one a workgroup of the output layer's pass)
constexpr int kMlpLossPartials = 1024;
void mlp_backward(hipStream_t s, int h, const float* P, int64_t B, const float* X, const float* T, const float* A1,
                  const float* A2, const float* A3, const float* y, float* dy, float* dA, float* dZ, float* G,
                  float* part, double* lpart, int64_t* nlpart);
void mlp_adam(hipStream_t s, int64_t n, float* P, const float* G, float* m, float* v, float lr, int64_t t);
void mlp_gather(hipStream_t s, int64_t B, int64_t off, const int64_t* perm, const float* X, const float* T, float* Xb,
                float* Tb);
void t2_features(hipStream_t s, int o, int v, int64_t e0, int64_t n, const double* t2, const double* eo,
                 const double* ev, const double* dij, const float* xm, const float* xs, float* X);
void t2_learned_apply(hipStream_t s, int o, int v, double ys, const float* Y, double* t2);
// network output Y[o,o,v,v] for all amplitudes in one fused kernel (hidden width 128 only; wsplit:
// t2_mlp_fused_scratch_bytes() of device memory for the bf16 weight planes)
bool t2_mlp_fused_available(int h);
size_t t2_mlp_fused_scratch_bytes();
void t2_mlp_fused(hipStream_t s, int o, int v, const double* t2, const double* eo, const double* ev, const double* dij,
                  const float* xm, const float* xs, const float* P, void* wsplit, float* Y);

// workspace (elements of the partial sums' type) that the GEMMs would use to split K for this shape (0: no split)
int64_t gemm_splitk_elems(int64_t M, int64_t N, int64_t K, int64_t batch);
// tag selects a distinct kernel symbol for profiling: 0 generic, 1 PP ladder

// out[perm] = alpha * in + beta * out: out dim d has size odim[d] and reads input with stride istr[d].
void permute_f64(hipStream_t s, int nd, const int64_t* odim, const int64_t* istr, double alpha,
                 const double* in, double beta, double* out);

void axpby_f64(hipStream_t s, int64_t n, double a, const double* x, double b, double* y);  // y = a x + b y
void fill_f64(hipStream_t s, int64_t n, double v, double* y);
// amplitude forms of the CCSD residual's GEMMs, any output null: u, tau [ijab]; ring [iajb] x 2 (u, -t2[ijba]);
// pair [ij, ab] over i >= j, a >= b, x 2 (symmetric, antisymmetric)
template <typename TR, typename TP>
void amp_forms(hipStream_t s, int o, int v, const double* t1, const double* t2, double* u, double* tau, TR* ring, TP* pair);
// the PP ladder's operand V[cd,ab] +- V[dc,ab] over c >= d, a >= b for a0 <= a < a0 + na (see k_vv_pairs), columns
// vv_pairs_ld(v) apart
int64_t vv_pairs_ld(int64_t v);
void vv_pairs(hipStream_t s, int v, int a0, int na, const double* T, int64_t sa, int64_t sd, int64_t sb, bool sym, double* out);
// T2 numerator from P[ijab], the ring products D, F [iajb] and the packed ladder Sp [ij, ab] x 2
void t2_numerator(hipStream_t s, int o, int v, const double* P, const double* D, const double* F, const double* Sp, double* R2);
// T1/T2 Jacobi update: new = R / D (D from eps on the fly); writes new into R, err = new - old
// (as FP64 or FP32) and per-block partial sums of err^2.
void jacobi_update(hipStream_t s, int o, int v, bool is_t2, const double* eo, const double* ev, double* R,
                   const double* old, void* err, bool err_f32, double* partials, int64_t* nblocks);
int64_t reduce_blocks_needed(int64_t n);
// deterministic FP64 dot products: partial sums per block, then one final block.
void dot_f64(hipStream_t s, int64_t n, const double* x, const double* y, double* partials, double* result);
// result[q] = x_q . y (FP64 sums) for up to 8 FP64 or FP32 vectors; partials: nv reduce_blocks_needed(n)
void dots(hipStream_t s, int64_t n, int nv, const void* const* xs, const void* y, bool f32, double* partials,
          double* result);
void sum_partials(hipStream_t s, int64_t n, const double* partials, double* result);
// y = sum_i c_i x_i (+ sum_i c_i e_i) for up to 8 FP64 vectors and 8 FP64/FP32 error vectors
void lincomb(hipStream_t s, int64_t n, int nv, const double* const* xs, const double* cs,
             const void* const* es, bool err_f32, bool add_err, double* y);
void cast_f64_to_f32(hipStream_t s, int64_t n, const double* x, float* y);
// closed-shell CC energy (RCCSDHelper.jl:8-23) -> partials + final sum into result
void cc_energy(hipStream_t s, int o, int v, const double* t1, const double* t2, const double* ovov,
               double* partials, double* result);

// DF-MP2 energy (RMP2a.jl:91-144, fh_mp2.hip) from Bov[Q, i, a] -> mp2_partials(o, v) FP64 partial sums
int64_t mp2_partials(int o, int v);
void mp2_pair_energy(hipStream_t s, int o, int v, int Q, const double* Bov, const double* eo, const double* ev,
                     double* partials);

// Symmetric A (n x n, its upper triangle) -> T (d, e) = Q^T A Q, the reflectors of Q in the columns of V [n, n] and
// tau (fh_eigen.hip); out = Q Z
inline bool tridiag_fits(int n) { return n >= 3 && n <= 160; }
void tridiag(hipStream_t s, int n, const double* A, double* V, double* d, double* e, double* tau);
void tridiag_apply(hipStream_t s, int n, const double* V, const double* tau, const double* Z, double* out);
// SCF: out = U diag(w)^-1/2 (n x n, column-major); GWH guess Fock matrix (RHFHelper.jl:44-51)
void scale_cols_rsqrt(hipStream_t s, int n, const double* U, const double* w, double* out);
void gwh_fock(hipStream_t s, int n, const double* S, const double* H, double* F);

// (T) energy of nrun runs of k (8 ints each: i, j, k0, nk, W slot of k0): W
// holds the W intermediate of ijk.jl:108-115; one FP64 partial per orbit and run.
// orbits: device list of cube-block triples (A>=B>=C), 3 ints each (triples_orbits)
int triples_orbit_count(int v);
void triples_orbits(int v, std::vector<int>& out);
// vvb: the (ia|jb) blocks in 8x8 tiles, made by triples_block_vv from vvoo[a,b,i,j]
// (triples_vv_blocked_elems doubles)
int64_t triples_vv_blocked_elems(int o, int v);
void triples_block_vv(hipStream_t s, int o, int v, const double* vvoo, double* vvb);
// k values per run: long enough to amortise the k-independent staging, short enough to fill the chip
int triples_energy_kpw(int norb, int nslot);
template <typename TW>  // W stored as double (FP64 path) or float (FP32 W build)
void triples_energy(hipStream_t s, int o, int v, int nrun, const int* runs, const TW* W, int norb, const int* orbits,
                    const double* t1p, const double* vvb, const double* eo, const double* ev, double* partials);

// ---------------------------------------------------------------- Gaussian integrals (fh_integrals.hip)
// shells: packed records (integrals_pack_shell, integrals_shell_bytes each); tab: packed spherical
// table (integrals_pack_table)
size_t integrals_shell_bytes();
size_t integrals_table_bytes();
int integrals_max_l_orbital();
int integrals_max_l_aux();
void integrals_pack_shell(void* dst, int l, int nprim, int poff, int foff, const double* center);
void integrals_pack_table(void* dst, const double* c, int spherical);
void integrals_one_electron(hipStream_t s, int nshell, const void* shells, const double* ex, const double* cf,
                            int natom, const double* Z, const double* xyz, const void* tab, int nbf, double* S,
                            double* T, double* V);
void integrals_dipole(hipStream_t s, int nshell, const void* shells, const double* ex, const double* cf,
                      const double* origin, const void* tab, int nbf, double* Dx, double* Dy, double* Dz);
// a basis set as the host holds it: nexp primitives, shell i's from poff[i] on, its functions from foff[i] on
struct IntBasis {
  int nshell, nbf, spherical, nexp;
  const int *l, *nprim, *poff, *foff;
  const double *center, *exps, *coefs;
};
// lists and tables of a Coulomb integral call: kept until the stream has been synchronised
struct IntScratch {
  std::vector<char> host;
  Buf lists, tables;
};
// (mu nu|P), (P|Q) and (mu nu|la si) into out (orbital shells up to d, fitting shells up to f)
void integrals_eri3c(hipStream_t s, Pool* pool, IntScratch& sc, const IntBasis& b, const IntBasis& aux, const void* tab,
                     double* out);
void integrals_eri2c(hipStream_t s, Pool* pool, IntScratch& sc, const IntBasis& aux, const void* tab, double* out);
void integrals_eri4c(hipStream_t s, Pool* pool, IntScratch& sc, const IntBasis& b, const void* tab, double* out);

}  // namespace fh
