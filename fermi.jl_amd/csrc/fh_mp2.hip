// DF-MP2 correlation energy (RMP2a.jl:91-144) in one kernel from Bov[Q, i, a]:
//   E = sum_{i <= j} w_ij sum_ab X[a,b] (2 X[a,b] - X[b,a]) / (e_i + e_j - e_a - e_b),  X[a,b] = (ia|jb) = B_i^T B_j,
// w = 1 for i = j, else 2.  A workgroup takes an orbital pair and a tile of X with its transposed partner, both as
// FP64 MFMA products, and reduces them to energy in registers: no (ia|jb) in memory, and half the products of the
// whole o v x o v matrix.  The partner of an off-diagonal tile is computed transposed (B_j rows a, B_i rows b), so that
// X[a,b] and X[b,a] meet in the same register of the same lane; a diagonal tile is its own partner, through LDS.
//
// Bound by the FP64 matrix pipes: o = 40, v = 190, Q = 840 (50 GFLOP) 1.04 ms, 48 TFLOP/s, against 2.7 ms for the GEMM of
// the whole matrix, its (ia|jb) of 462 MB and a pass that reduced them (2.0 ms with the GEMM's present kernel);
// o = 5, v = 19 38 us against 50.
#include "fh_internal.h"

#include <algorithm>

namespace fh {
namespace {
typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));
typedef double f64x2u __attribute__((ext_vector_type(2), aligned(8)));

constexpr int64_t kMaxBlocks = 16384;

// index of the triangle x <= y, y (y + 1) / 2 + x, and back
__host__ __device__ inline int64_t tri(int64_t n) { return n * (n + 1) / 2; }
__device__ inline void untri(int64_t q, int64_t& x, int64_t& y) {
  y = (int64_t)((sqrt(8.0 * (double)q + 1.0) - 1.0) * 0.5);
  while (tri(y) > q) --y;
  while (tri(y + 1) <= q) ++y;
  x = q - tri(y);
}
}  // namespace

template <int BT, int BK>
__global__ __launch_bounds__(256, BT == 64 ? 3 : 4) void k_mp2(int o, int v, int Q, const double* __restrict__ B,
                                                const double* __restrict__ eo, const double* __restrict__ ev,
                                                int64_t nitem, double* __restrict__ partials) {
  constexpr int WB = BT / 32, KS = BK + 2, LD = BT * BK / 512;
  static_assert(4 * BT * KS >= BT * (BT + 1), "the diagonal tile fits the operand buffers");
  __shared__ __attribute__((aligned(16))) double lds[4 * BT * KS];
  __shared__ double red[4];
  double(*As)[BT][KS] = reinterpret_cast<double(*)[BT][KS]>(lds);
  double(*Bs)[BT][KS] = reinterpret_cast<double(*)[BT][KS]>(lds + 2 * BT * KS);
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wid & 1, wn = wid >> 1;
  const int64_t nt = (v + BT - 1) / BT, noff = tri(nt - 1), ld = (int64_t)Q * o;
  const int nst = (Q + BK - 1) / BK, kr = Q % BK;

  // acc += (rows of Ap) (rows of Bp)^T; wavefront (wm, wn) owns the 16-blocks of parity wm, wn, and skips those outside
  // the tile's ma x mb valid rows and columns
  auto product = [&](const double* Ap, int ma, const double* Bp, int mb, f64x4 (&acc)[WB][WB]) {
    const double *pa[LD], *pb[LD];
    f64x2 ra[LD], rb[LD];
#pragma unroll
    for (int t = 0; t < LD; ++t) {
      const int e = tid + 256 * t, row = e / (BK / 2), kp = e % (BK / 2);
      pa[t] = Ap + ld * min(row, ma - 1) + 2 * kp;
      pb[t] = Bp + ld * min(row, mb - 1) + 2 * kp;
    }
    auto fetch = [&](int st) {
      if (st + 1 == nst && kr) {
        // kr of k are left: the others read the first and count as zero
#pragma unroll
        for (int t = 0; t < LD; ++t) {
          const int k = 2 * ((tid + 256 * t) % (BK / 2));
          auto get = [&](const double* p, int kk) { return kk < kr ? p[kk - k] : 0.0; };
          ra[t] = f64x2{get(pa[t], k), get(pa[t], k + 1)};
          rb[t] = f64x2{get(pb[t], k), get(pb[t], k + 1)};
        }
      } else {
#pragma unroll
        for (int t = 0; t < LD; ++t) {
          ra[t] = *reinterpret_cast<const f64x2u*>(pa[t]);
          rb[t] = *reinterpret_cast<const f64x2u*>(pb[t]);
          pa[t] += BK;
          pb[t] += BK;
        }
      }
    };
    auto store = [&](int buf) {
#pragma unroll
      for (int t = 0; t < LD; ++t) {
        const int e = tid + 256 * t, row = e / (BK / 2), kp = e % (BK / 2);
        *reinterpret_cast<f64x2*>(&As[buf][row][2 * kp]) = ra[t];
        *reinterpret_cast<f64x2*>(&Bs[buf][row][2 * kp]) = rb[t];
      }
    };
    const int ni = (ma - 16 * wm + 31) / 32, nj = (mb - 16 * wn + 31) / 32;   // valid blocks of the wavefront
    fetch(0);
    __syncthreads();   // the buffers' last readers
    store(0);
    __syncthreads();
    for (int st = 0; st < nst; ++st) {
      const int buf = st & 1;
      if (st + 1 < nst) fetch(st + 1);
      auto step = [&](auto full) {
#pragma unroll
        for (int ks = 0; ks < BK; ks += 8) {
          f64x2 af[WB], bf[WB];
#pragma unroll
          for (int i = 0; i < WB; ++i) {
            af[i] = *reinterpret_cast<const f64x2*>(&As[buf][(2 * i + wm) * 16 + (lane & 15)][ks + 2 * (lane >> 4)]);
            bf[i] = *reinterpret_cast<const f64x2*>(&Bs[buf][(2 * i + wn) * 16 + (lane & 15)][ks + 2 * (lane >> 4)]);
          }
#pragma unroll
          for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int i = 0; i < WB; ++i)
#pragma unroll
              for (int j = 0; j < WB; ++j)
                if (decltype(full)::value || (i < ni && j < nj))
                  acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bf[j][q], af[i][q], acc[i][j], 0, 0, 0);
        }
      };
      if (ni >= WB && nj >= WB) step(std::true_type());
      else if (ni > 0 && nj > 0) step(std::false_type());
      if (st + 1 < nst) store(buf ^ 1);
      __syncthreads();
    }
  };

  double e = 0.0;
  for (int64_t it = blockIdx.x; it < nitem; it += gridDim.x) {
    const int64_t tp = it / tri(o);
    int64_t i, j, ta, tb;
    untri(it % tri(o), i, j);
    // off-diagonal tiles (two products) first
    if (tp < noff) {
      untri(tp, ta, tb);
      ++tb;
    } else {
      ta = tb = tp - noff;
    }
    const int a0 = (int)ta * BT, b0 = (int)tb * BT, ma = min(BT, v - a0), mb = min(BT, v - b0);
    const double *Bi = B + (int64_t)Q * i, *Bj = B + (int64_t)Q * j;
    f64x4 X[WB][WB], Y[WB][WB];
#pragma unroll
    for (int p = 0; p < WB; ++p)
#pragma unroll
      for (int q = 0; q < WB; ++q) X[p][q] = Y[p][q] = f64x4{0, 0, 0, 0};
    product(Bi + ld * a0, ma, Bj + ld * b0, mb, X);
    const bool diag = ta == tb;
    if (!diag) {
      product(Bj + ld * a0, ma, Bi + ld * b0, mb, Y);
    } else {
      __syncthreads();
#pragma unroll
      for (int p = 0; p < WB; ++p)
#pragma unroll
        for (int q = 0; q < WB; ++q)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            lds[((2 * p + wm) * 16 + (lane & 15)) + (BT + 1) * ((2 * q + wn) * 16 + (lane >> 4) + 4 * r)] = X[p][q][r];
      __syncthreads();
#pragma unroll
      for (int p = 0; p < WB; ++p)
#pragma unroll
        for (int q = 0; q < WB; ++q)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            Y[p][q][r] = lds[(BT + 1) * ((2 * p + wm) * 16 + (lane & 15)) + ((2 * q + wn) * 16 + (lane >> 4) + 4 * r)];
    }
    const double eij = eo[i] + eo[j], wt = i == j ? 1.0 : 2.0;
    double s = 0.0;
#pragma unroll
    for (int p = 0; p < WB; ++p)
#pragma unroll
      for (int q = 0; q < WB; ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int a = (2 * p + wm) * 16 + (lane & 15), b = (2 * q + wn) * 16 + (lane >> 4) + 4 * r;
          if (a < ma && b < mb) {
            const double x = X[p][q][r], y = Y[p][q][r], d = eij - ev[a0 + a] - ev[b0 + b];
            s += (diag ? x * (2.0 * x - y) : 2.0 * (x * x + y * y - x * y)) / d;
          }
        }
    e += wt * s;
  }
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) e += __shfl_xor(e, m, 64);
  if (lane == 0) red[wid] = e;
  __syncthreads();
  if (tid == 0) partials[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// 64 x 64 tiles, or 32 x 32 with K steps of 32 where those would be too few to hide their latency, under some six a CU
// (naux = 4.2 (o + v): o = 12, v = 70 52 us against 71, o = 20, v = 150 205 against 232, o = 40, v = 100 336 against 327).
// The items go tile by tile over the pairs: in 8 x 8 blocks of pairs an XCD (its L2 to share their rows) o = 40,
// v = 190 took 1.32 ms, 1.18 so, and few blocks left XCDs idle (o = 20, v = 100: 167 us, 114 so).
struct Mp2Plan {
  int tile;
  int64_t items;
};
static Mp2Plan mp2_plan(int o, int v) {
  const int64_t n64 = tri((v + 63) / 64) * tri(o);
  if (v <= 32 || n64 < 1400) return {32, tri((v + 31) / 32) * tri(o)};
  return {64, n64};
}
int64_t mp2_partials(int o, int v) { return std::min(mp2_plan(o, v).items, kMaxBlocks); }

void mp2_pair_energy(hipStream_t s, int o, int v, int Q, const double* Bov, const double* eo, const double* ev,
                     double* partials) {
  const Mp2Plan p = mp2_plan(o, v);
  const dim3 grid((unsigned)std::min(p.items, kMaxBlocks)), block(256);
  if (p.tile == 32)
    hipLaunchKernelGGL((k_mp2<32, 32>), grid, block, 0, s, o, v, Q, Bov, eo, ev, p.items, partials);
  else
    hipLaunchKernelGGL((k_mp2<64, 16>), grid, block, 0, s, o, v, Q, Bov, eo, ev, p.items, partials);
  FH_HIP(hipGetLastError());
}

}  // namespace fh
