// Dense GEMM on CDNA4 matrix cores: D = alpha * op(A) * op(B) + beta * C, column-major.
//
// Workgroup: 256 threads = 4 wavefronts in a 2x2 arrangement; each wavefront owns a
// (BM/2)x(BN/2) block of the output as 16x16 MFMA accumulators.  Operand tiles are staged
// through LDS with double buffering (global loads for stage s+1 are in flight while stage s
// is multiplied).  Both tiles lie k-contiguous in LDS, whatever the source's order: a lane's
// fragments are 16-byte reads of two (FP64) or four (FP32) of k, and the padded rows put 16 of
// them on distinct banks, as they do the stores.  A full step has no bounds check.  (An m-major
// tile of A with 8-byte reads, checked loads and scattered stores for a k-contiguous source left
// the matrix pipes busy 52 % of the time, bank conflicts as many cycles as the MFMAs: TN
// 7600 x 7600 x 840 in FP64 2.74 ms (35 TFLOP/s), so 2.03 ms (48 TFLOP/s, pipes busy 80 %).)
//
// Precision variants (template F32 and the global element types TI / TO):
//   F32 = false: FP64 operands, v_mfma_f64_16x16x4f64, FP64 accumulation (TI = TO = double);
//   F32 = true : operands rounded to FP32 when staged into LDS (TI may be double or float),
//                v_mfma_f32_16x16x4f32 with FP32 accumulation, alpha/beta epilogue in FP64,
//                output stored as TO (double or float).
//
// Tile -> workgroup mapping: consecutive workgroup ids land on different XCDs (round robin
// over 8), so the linear id is first remapped such that each XCD receives a contiguous range
// of tiles.  Within that order tiles are rastered M-fastest (tiles sharing a column block of
// B are neighbours), or -- when A is the larger operand -- in groups of gn N-tiles whose B
// blocks fit in L2: each group sweeps all M-tiles, so B stays in L2 and A is streamed once
// per group instead of once per N-tile.
#include "fh_host.h"
#include "fh_internal.h"

#include <algorithm>
#include <type_traits>

namespace fh {

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <int BM, int BN, int BK, bool TA, bool TB, int OCC, int TAG, bool F32, typename TI, typename TO>
__global__ __launch_bounds__(256, OCC) void k_gemm(
    int64_t M, int64_t N, int64_t K, double alpha, const TI* __restrict__ A, int64_t lda, int64_t sA,
    const TI* __restrict__ B, int64_t ldb, int64_t sB, double beta, const TO* C, int64_t ldc, int64_t sC, TO* D,
    int64_t ldd, int64_t sD, int tilesM, int tilesN, int64_t kchunk, int gn) {
  static_assert(F32 || std::is_same<TI, double>::value, "FP64 MFMA needs FP64 operands");
  using T = typename std::conditional<F32, float, double>::type;
  using Acc = typename std::conditional<F32, f32x4, f64x4>::type;
  constexpr int WM = BM / 2, WN = BN / 2, MB = WM / 16, NB = WN / 16;
  // an LDS read holds KV of k of a row, k group g = lane / 16 of a wavefront KV g .. KV g + KV - 1 of 4 KV (the order
  // of k is the same for both operands, so any will do); KS is the row stride that spreads 16 rows over all banks
  constexpr int KV = F32 && BK > 8 ? 4 : 2, KS = BK + (F32 ? 4 : 2);
  constexpr int LA = BM * BK / 512, LB = BN * BK / 512;   // pairs of k that a thread copies
  typedef T TV __attribute__((ext_vector_type(KV)));
  typedef T T2 __attribute__((ext_vector_type(2)));
  typedef TI TI2 __attribute__((ext_vector_type(2), aligned(sizeof(TI))));
  __shared__ __attribute__((aligned(16))) T As[2][BM][KS];
  __shared__ __attribute__((aligned(16))) T Bs[2][BN][KS];

  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int wm = wid & 1, wn = wid >> 1;

  // XCD-aware remap of the linear tile id, then the raster
  const int64_t nwg = (int64_t)tilesM * tilesN;
  const int64_t w = blockIdx.x;
  const int64_t q = nwg >> 3, r = nwg & 7, x = w & 7;
  const int64_t L = x * q + (x < r ? x : r) + (w >> 3);
  int64_t mt, nt;
  if (gn <= 0) {
    mt = L % tilesM;
    nt = L / tilesM;
  } else {
    const int64_t g = L / ((int64_t)tilesM * gn);
    const int64_t rem = L - g * (int64_t)tilesM * gn;
    const int64_t wdt = (tilesN - g * gn < gn) ? tilesN - g * gn : gn;
    mt = rem / wdt;
    nt = g * gn + rem % wdt;
  }
  const int64_t m0 = mt * BM, n0 = nt * BN;

  const int64_t bz = blockIdx.y, kz = blockIdx.z;
  A += bz * sA;
  B += bz * sB;
  if (kchunk > 0) {
    // split-K: slice kz covers k in [kz*kchunk, min(K, (kz+1)*kchunk)) and writes its own D slice
    const int64_t kb = kz * kchunk;
    K = (K - kb < kchunk) ? K - kb : kchunk;
    A += TA ? kb : lda * kb;
    B += TB ? ldb * kb : kb;
  }
  if (C) C += bz * sC;
  D += (kz * gridDim.y + bz) * sD;
  // The thread's pairs of consecutive k: row (or column) index r and pair index kp; lanes run along the contiguous
  // axis of the source.  Source pointers advance by BK of k a step.  Rows and columns outside the output read its
  // last ones (their products go to elements that are not stored), so a full step has no bounds check.
  auto rowA = [&](int t) { const int e = tid + 256 * t; return TA ? e / (BK / 2) : e % BM; };
  auto kpA = [&](int t) { const int e = tid + 256 * t; return TA ? e % (BK / 2) : e / BM; };
  auto rowB = [&](int t) { const int e = tid + 256 * t; return TB ? e % BN : e / (BK / 2); };
  auto kpB = [&](int t) { const int e = tid + 256 * t; return TB ? e / BN : e % (BK / 2); };
  TI2 ra[LA], rb[LB];
  const TI *pa[LA], *pb[LB];
  const int64_t skA = TA ? 1 : lda, skB = TB ? ldb : 1;   // stride of k
#pragma unroll
  for (int t = 0; t < LA; ++t) {
    const int64_t gm = m0 + rowA(t) < M ? m0 + rowA(t) : M - 1;
    pa[t] = A + gm * (TA ? lda : 1) + 2 * kpA(t) * skA;
  }
#pragma unroll
  for (int t = 0; t < LB; ++t) {
    const int64_t gc = n0 + rowB(t) < N ? n0 + rowB(t) : N - 1;
    pb[t] = B + gc * (TB ? 1 : ldb) + 2 * kpB(t) * skB;
  }
  auto gload = [&]() {
#pragma unroll
    for (int t = 0; t < LA; ++t) {
      if constexpr (TA) ra[t] = *reinterpret_cast<const TI2*>(pa[t]);
      else ra[t] = TI2{pa[t][0], pa[t][lda]};
      pa[t] += BK * skA;
    }
#pragma unroll
    for (int t = 0; t < LB; ++t) {
      if constexpr (!TB) rb[t] = *reinterpret_cast<const TI2*>(pb[t]);
      else rb[t] = TI2{pb[t][0], pb[t][ldb]};
      pb[t] += BK * skB;
    }
  };
  // the last step when BK does not divide K: kr (1 .. BK - 1) of k are left; the others read the first and count
  // as zero
  auto gload_tail = [&](int kr) {
    auto get = [&](const TI* p, int64_t sk, int k) {
      const TI v = p[k < kr ? 0 : -(int64_t)k * sk];
      return k < kr ? v : TI(0);
    };
#pragma unroll
    for (int t = 0; t < LA; ++t) ra[t] = TI2{get(pa[t], skA, 2 * kpA(t)), get(pa[t] + skA, skA, 2 * kpA(t) + 1)};
#pragma unroll
    for (int t = 0; t < LB; ++t) rb[t] = TI2{get(pb[t], skB, 2 * kpB(t)), get(pb[t] + skB, skB, 2 * kpB(t) + 1)};
  };
  auto sstore = [&](int buf) {
#pragma unroll
    for (int t = 0; t < LA; ++t)
      *reinterpret_cast<T2*>(&As[buf][rowA(t)][2 * kpA(t)]) = T2{(T)ra[t][0], (T)ra[t][1]};
#pragma unroll
    for (int t = 0; t < LB; ++t)
      *reinterpret_cast<T2*>(&Bs[buf][rowB(t)][2 * kpB(t)]) = T2{(T)rb[t][0], (T)rb[t][1]};
  };

  Acc acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = Acc{0, 0, 0, 0};

  const int64_t nst = (K + BK - 1) / BK;
  const int kr = (int)(K % BK);
  auto fetch = [&](int64_t st) {
    if (st + 1 == nst && kr) gload_tail(kr); else gload();
  };
  if (nst) {
    fetch(0);
    sstore(0);
  }
  __syncthreads();
  for (int64_t s = 0; s < nst; ++s) {
    const int buf = s & 1;
    if (s + 1 < nst) fetch(s + 1);
#pragma unroll
    for (int ks = 0; ks < BK; ks += 4 * KV) {
      TV af[MB], bf[NB];
#pragma unroll
      for (int i = 0; i < MB; ++i)
        af[i] = *reinterpret_cast<const TV*>(&As[buf][wm * WM + i * 16 + (lane & 15)][ks + KV * (lane >> 4)]);
#pragma unroll
      for (int j = 0; j < NB; ++j)
        bf[j] = *reinterpret_cast<const TV*>(&Bs[buf][wn * WN + j * 16 + (lane & 15)][ks + KV * (lane >> 4)]);
#pragma unroll
      for (int q = 0; q < KV; ++q)
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
          for (int j = 0; j < NB; ++j) {
            // B fragment as the first MFMA operand, so the accumulator lanes run along M
            if constexpr (F32) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(bf[j][q], af[i][q], acc[i][j], 0, 0, 0);
            else acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bf[j][q], af[i][q], acc[i][j], 0, 0, 0);
          }
    }
    if (s + 1 < nst) sstore(buf ^ 1);
    __syncthreads();
  }

  // epilogue: the accumulator of block (i, j) holds, in lane l and register r, the element at row l & 15 and
  // column (l >> 4) + 4 r (FP64 MFMA) or 4 (l >> 4) + r (FP32 MFMA) of the 16x16 block.  With beta != 0 every C
  // value of the thread is loaded (unconditionally, an element outside D reading C[0]) before the first
  // store.
  auto at = [&](int i, int j, int rr, int64_t& row, int64_t& col) {
    row = m0 + wm * WM + i * 16 + (lane & 15);
    col = n0 + wn * WN + j * 16 + (F32 ? 4 * (lane >> 4) + rr : (lane >> 4) + 4 * rr);
    return row < M && col < N;
  };
  if constexpr (TAG == 4) {
    // a network layer: D = tanh(A B + bias), the bias of a row in C
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
          int64_t row, col;
          if (at(i, j, rr, row, col)) D[row + ldd * col] = tanhf((float)acc[i][j][rr] + C[row]);
        }
  } else if (beta != 0.0) {
    TO cv[MB][NB][4];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
          int64_t row, col;
          const bool in = at(i, j, rr, row, col);
          cv[i][j][rr] = C[in ? row + ldc * col : 0];
        }
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
          int64_t row, col;
          if (at(i, j, rr, row, col))
            D[row + ldd * col] = (TO)(alpha * (double)acc[i][j][rr] + beta * (double)cv[i][j][rr]);
        }
  } else {
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
          int64_t row, col;
          if (at(i, j, rr, row, col)) D[row + ldd * col] = (TO)(alpha * (double)acc[i][j][rr]);
        }
  }
}

// L2 budget of the B blocks of one raster group (bytes)
static constexpr int64_t kGroupBytes = 1 << 20;

template <int BM, int BN, int BK, bool TA, bool TB, int TAG, bool F32, typename TI, typename TO>
static void launch(hipStream_t s, int64_t M, int64_t N, int64_t K, double alpha, const TI* A, int64_t lda, int64_t sA,
                   const TI* B, int64_t ldb, int64_t sB, double beta, const TO* C, int64_t ldc, int64_t sC, TO* D,
                   int64_t ldd, int64_t sD, int64_t batch, int64_t kchunk) {
  const int64_t tm = (M + BM - 1) / BM, tn = (N + BN - 1) / BN;
  FH_CHECK(tm * tn <= max_workgroups(256) && batch < 65536, -3, "gemm grid too large");
  dim3 grid((unsigned)(tm * tn), (unsigned)batch, (unsigned)(kchunk > 0 ? (K + kchunk - 1) / kchunk : 1));
  // A larger than B: group N-tiles so that a group's B blocks stay in L2
  int gn = 0;
  if (M > N) {
    const int64_t kl = kchunk > 0 ? kchunk : K;
    const int64_t per = std::max<int64_t>(1, kl * BN * (int64_t)sizeof(TI));
    gn = (int)std::max<int64_t>(1, std::min<int64_t>(tn, kGroupBytes / per));
  }
  constexpr int OCC = BM == 32 && !F32 ? 3 : 4;   // workgroups per CU that the LDS holds
  hipLaunchKernelGGL((k_gemm<BM, BN, BK, TA, TB, OCC, TAG, F32, TI, TO>), grid, dim3(256), 0, s, M, N, K, alpha, A, lda,
                     sA, B, ldb, sB, beta, C, ldc, sC, D, ldd, sD, (int)tm, (int)tn, kchunk, gn);
  FH_HIP(hipGetLastError());
}

// How a shape is cut.  64x64 tiles at up to four workgroups per CU measured fastest wherever there are enough of
// them (the latency of the next operand tile is hidden by the other workgroups); BK = 8 when the per-tile K loop
// is short.  Below 1.5 tiles per CU the K loop of a tile is exposed, so K is cut into slices of at least 128
// towards four workgroups per CU; a K under 384 is not, as the reduction (about 4 us) costs what it saves.
// Measured in FP64: (136, 2926, 2926) in a batch of two, 276 tiles, 286 us uncut, 160 us in three slices and 9 us to
// add them; one tile with K = 1805 110 us uncut, 6 + 4 us cut.
// A shape that leaves the chip under 256 workgroups even so is bound by the latency of a K step, about 1 us
// whatever its depth: 32x32 tiles in K steps of 32 spread it over more CUs in a quarter of the steps (the products
// of the residual at o = 5, v = 19: 10 us each with 64x64 tiles in steps of 8, 5 us so).  So does every shape under
// 1.5 tiles a CU with 32 < K <= 256, which has no K to cut and few steps to hide the latency of the first ones in: eight
// CC iterations at o = 16, v = 76 11.2 ms against 11.5 with 64x64 tiles, the network's gradient of 8192 samples (layers
// of K = 128) 219 us against 243; o = 5, v = 19, o = 10, v = 40 and o = 28, v = 133 the same either way.
struct GemmPlan {
  bool small;
  int64_t slices;
};
static GemmPlan gemm_plan(int64_t M, int64_t N, int64_t K, int64_t batch) {
  const int64_t tiles = ((M + 63) / 64) * ((N + 63) / 64) * batch;
  if (tiles >= 384) return {false, 1};
  if (K > 32 && K <= 256) return {true, 1};
  const int64_t most = K < 384 ? 1 : K / 128;
  if (tiles * most >= 256) return {false, std::min<int64_t>(std::max<int64_t>(1, 1024 / tiles), most)};
  const int64_t tiles32 = ((M + 31) / 32) * ((N + 31) / 32) * batch;
  return {true, std::min<int64_t>(std::max<int64_t>(1, 512 / tiles32), most)};
}

template <bool TA, bool TB, int TAG, bool F32, typename TI, typename TO>
static void pick(hipStream_t s, bool small, int64_t M, int64_t N, int64_t K, double alpha, const TI* A, int64_t lda,
                 int64_t sA, const TI* B, int64_t ldb, int64_t sB, double beta, const TO* C, int64_t ldc, int64_t sC,
                 TO* D, int64_t ldd, int64_t sD, int64_t batch, int64_t kchunk) {
  const int64_t kl = kchunk > 0 ? kchunk : K;
  if (small)
    launch<32, 32, 32, TA, TB, TAG, F32, TI, TO>(s, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, D, ldd,
                                                 sD, batch, kchunk);
  else if (kl <= 512)
    launch<64, 64, 8, TA, TB, TAG, F32, TI, TO>(s, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, D, ldd, sD,
                                                batch, kchunk);
  else
    launch<64, 64, 16, TA, TB, TAG, F32, TI, TO>(s, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, D, ldd,
                                                 sD, batch, kchunk);
}

int64_t gemm_splitk_elems(int64_t M, int64_t N, int64_t K, int64_t batch) {
  if (M <= 0 || N <= 0 || batch <= 0) return 0;
  const int64_t sl = gemm_plan(M, N, K, batch).slices;
  return sl > 1 ? sl * M * N * batch : 0;
}

// D = alpha sum over the S slices of W [M N][batch][S] + beta C, summed in FP64
template <typename T>
__global__ __launch_bounds__(256) void k_splitk_reduce(int64_t M, int64_t N, int64_t S, const T* __restrict__ W,
                                                       double alpha, double beta, const T* C, int64_t ldc, int64_t sC,
                                                       T* D, int64_t ldd, int64_t sD) {
  const int64_t n = M * N, st = n * gridDim.y;
  W += n * blockIdx.y;
  C += sC * blockIdx.y;
  D += sD * blockIdx.y;
  for (int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x; idx < n; idx += (int64_t)gridDim.x * 256) {
    const int64_t m = idx % M, c = idx / M;
    double acc = 0.0;
#pragma unroll 8
    for (int64_t q = 0; q < S; ++q) acc += (double)W[idx + q * st];
    double val = alpha * acc;
    if (beta != 0.0) val += beta * (double)C[m + ldc * c];
    D[m + ldd * c] = (T)val;
  }
}

template <typename T>
static void splitk_reduce(hipStream_t s, int64_t M, int64_t N, int64_t S, const T* W, double alpha, double beta,
                          const T* C, int64_t ldc, int64_t sC, T* D, int64_t ldd, int64_t sD, int64_t batch) {
  const int64_t g = std::min<int64_t>((M * N + 255) / 256, 65536);
  hipLaunchKernelGGL((k_splitk_reduce<T>), dim3((unsigned)g, (unsigned)batch), dim3(256), 0, s, M, N, S, W, alpha,
                     beta, C, ldc, sC, D, ldd, sD);
  FH_HIP(hipGetLastError());
}

void splitk_reduce_f64(hipStream_t s, int64_t M, int64_t N, int64_t S, const double* W, double alpha, double beta,
                       const double* C, int64_t ldc, int64_t sC, double* D, int64_t ldd, int64_t sD, int64_t batch) {
  splitk_reduce<double>(s, M, N, S, W, alpha, beta, C, ldc, sC, D, ldd, sD, batch);
}

static void check_args(int64_t M, int64_t K, int64_t N, bool ta, bool tb, int64_t lda, int64_t ldb, int64_t ldd,
                       double beta, const void* C, int64_t ldc) {
  FH_CHECK(K >= 0, -3, "gemm: negative K");
  FH_CHECK(lda >= (ta ? (K > 0 ? K : 1) : M) && ldb >= (tb ? N : (K > 0 ? K : 1)) && ldd >= M, -3,
           "gemm: leading dimension too small");
  FH_CHECK(beta == 0.0 || (C != nullptr && ldc >= M), -3, "gemm: C missing");
}

void gemm_f64(hipStream_t s, bool ta, bool tb, int64_t M, int64_t N, int64_t K, double alpha, const double* A,
              int64_t lda, int64_t sA, const double* B, int64_t ldb, int64_t sB, double beta, const double* C,
              int64_t ldc, int64_t sC, double* D, int64_t ldd, int64_t sD, int64_t batch, int tag, double* work,
              int64_t work_elems, bool f32) {
  if (M <= 0 || N <= 0 || batch <= 0) return;
  check_args(M, K, N, ta, tb, lda, ldb, ldd, beta, C, ldc);
  const GemmPlan plan = gemm_plan(M, N, K, batch);
  const bool split = plan.slices > 1 && work != nullptr && work_elems >= plan.slices * M * N * batch;
  const int64_t kchunk = split ? (K + plan.slices - 1) / plan.slices : 0;
  const double al = split ? 1.0 : alpha, be = split ? 0.0 : beta;
  const double* Cc = split ? nullptr : C;
  double* Dd = split ? work : D;
  const int64_t lddd = split ? M : ldd, sDD = split ? M * N : sD;
#define FH_PICK2(TA_, TB_, F_)                                                                                      \
  do {                                                                                                              \
    if (tag == 1)                                                                                                   \
      pick<TA_, TB_, 1, F_, double, double>(s, plan.small, M, N, K, al, A, lda, sA, B, ldb, sB, be, Cc, ldc, sC, Dd,  \
                                            lddd, sDD, batch, kchunk);                                              \
    else                                                                                                            \
      pick<TA_, TB_, 0, F_, double, double>(s, plan.small, M, N, K, al, A, lda, sA, B, ldb, sB, be, Cc, ldc, sC, Dd,  \
                                            lddd, sDD, batch, kchunk);                                              \
  } while (0)
#define FH_PICK(TA_, TB_)              \
  do {                                 \
    if (f32) FH_PICK2(TA_, TB_, true); \
    else FH_PICK2(TA_, TB_, false);    \
  } while (0)
  if (ta) {
    if (tb) FH_PICK(true, true); else FH_PICK(true, false);
  } else {
    if (tb) FH_PICK(false, true); else FH_PICK(false, false);
  }
#undef FH_PICK
#undef FH_PICK2
  if (split)
    splitk_reduce<double>(s, M, N, (K + kchunk - 1) / kchunk, work, alpha, beta, C, ldc, sC, D, ldd, sD, batch);
}

// FP32-MFMA GEMM with FP32 operands in HBM and FP64 output (NN)
void gemm_f32_fd(hipStream_t s, int64_t M, int64_t N, int64_t K, double alpha, const float* A, int64_t lda, int64_t sA,
                 const float* B, int64_t ldb, int64_t sB, double beta, const double* C, int64_t ldc, double* D, int64_t ldd,
                 int64_t sD, int64_t batch, int tag, double* work, int64_t work_elems) {
  if (M <= 0 || N <= 0 || batch <= 0) return;
  check_args(M, K, N, false, false, lda, ldb, ldd, beta, C, ldc);
  const GemmPlan plan = gemm_plan(M, N, K, batch);
  const bool split = plan.slices > 1 && work != nullptr && work_elems >= plan.slices * M * N * batch;
  const int64_t kchunk = split ? (K + plan.slices - 1) / plan.slices : 0;
  auto run = [&](auto tagc) {
    if (split)
      pick<false, false, decltype(tagc)::value, true, float, double>(s, plan.small, M, N, K, 1.0, A, lda, sA, B, ldb, sB,
                                                                     0.0, nullptr, 0, 0, work, M, M * N, batch, kchunk);
    else
      pick<false, false, decltype(tagc)::value, true, float, double>(s, plan.small, M, N, K, alpha, A, lda, sA, B, ldb,
                                                                     sB, beta, C, ldc, sD, D, ldd, sD, batch, 0);
  };
  if (tag == 1) run(std::integral_constant<int, 1>()); else run(std::integral_constant<int, 0>());
  if (split)
    splitk_reduce<double>(s, M, N, (K + kchunk - 1) / kchunk, work, alpha, beta, C, ldc, sD, D, ldd, sD, batch);
}

// FP32 operands and output, any transposition (the T2-guess network's layers; tag 3)
void gemm_f32(hipStream_t s, bool ta, bool tb, int64_t M, int64_t N, int64_t K, double alpha, const float* A,
              int64_t lda, const float* B, int64_t ldb, double beta, float* C, int64_t ldc, float* work,
              int64_t work_elems) {
  if (M <= 0 || N <= 0) return;
  check_args(M, K, N, ta, tb, lda, ldb, ldc, beta, C, ldc);
  const GemmPlan plan = gemm_plan(M, N, K, 1);
  const bool split = plan.slices > 1 && work != nullptr && work_elems >= plan.slices * M * N;
  const int64_t kchunk = split ? (K + plan.slices - 1) / plan.slices : 0;
#define FH_F32(TA_, TB_)                                                                                             \
  pick<TA_, TB_, 3, true, float, float>(s, plan.small, M, N, K, split ? 1.0 : alpha, A, lda, 0, B, ldb, 0,           \
                                        split ? 0.0 : beta, split ? nullptr : C, ldc, 0, split ? work : C,           \
                                        split ? M : ldc, split ? M * N : 0, 1, kchunk)
  if (ta) {
    if (tb) FH_F32(true, true); else FH_F32(true, false);
  } else {
    if (tb) FH_F32(false, true); else FH_F32(false, false);
  }
#undef FH_F32
  if (split) splitk_reduce<float>(s, M, N, (K + kchunk - 1) / kchunk, work, alpha, beta, C, ldc, 0, C, ldc, 0, 1);
}

void gemm_f32_tanh(hipStream_t s, int64_t M, int64_t N, int64_t K, const float* A, int64_t lda, const float* B, int64_t ldb,
                   const float* bias, float* D, int64_t ldd) {
  if (M <= 0 || N <= 0) return;
  check_args(M, K, N, false, false, lda, ldb, ldd, 0.0, nullptr, 0);
  pick<false, false, 4, true, float, float>(s, gemm_plan(M, N, K, 1).small, M, N, K, 1.0, A, lda, 0, B, ldb, 0, 0.0, bias,
                                            0, 0, D, ldd, 0, 1, 0);
}

}  // namespace fh
