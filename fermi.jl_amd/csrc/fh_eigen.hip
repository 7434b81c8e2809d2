// Householder tridiagonalisation of a small symmetric matrix and its back transformation: the two O(n^3) ends of the
// SCF's eigensolver (the tridiagonal problem between them is rocSOLVER's stedc).
//
// Q^T A Q = T with Q = H(n-1) ... H(1), H(k) = 1 - tau v v^T, v zero from row k on and v[k-1] = 1, from the last column
// up, beta = -sign(alpha) |x| (LAPACK's dsytd2 for an upper triangle: the same T and Q up to rounding, so the
// eigenvectors keep their signs).
#include "fh_internal.h"

namespace fh {

namespace {

// sum over the 16 lanes of a DPP row, the same in each of them
template <int CTRL>
__device__ __forceinline__ double dpp_add(double x) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xf, 0xf, false);
  return x + __hiloint2double(hi, lo);
}
__device__ __forceinline__ double sum16(double x) {
  x = dpp_add<0xB1>(x);    // quad_perm [1, 0, 3, 2]
  x = dpp_add<0x4E>(x);    // quad_perm [2, 3, 0, 1]
  x = dpp_add<0x141>(x);   // row_half_mirror
  return dpp_add<0x140>(x);  // row_mirror
}

}  // namespace

// One workgroup, the whole (symmetric, both triangles) matrix in its registers: lane l of wave w holds rows l % 16 + 16 s
// of columns 4 w + l / 16 + 32 j, so a product A v is a sum over 16 lanes and the rank-2 update needs no exchange.  Per
// column the owner's copy in LDS, the reflector in every wave (no wave waits for another's square root and divisions),
// the product into LDS, the update: two barriers.  Bound by those serial steps: n columns, one after the other, 1.6 us each;
// n = 96: 150 us against 620 of rocSOLVER's sytd2, which goes through memory.
template <int NC>
__global__ __launch_bounds__(512) void k_tridiag(int n, const double* __restrict__ A, double* __restrict__ V,
                                                 double* __restrict__ d, double* __restrict__ e,
                                                 double* __restrict__ tau) {
  constexpr int NS = 2 * NC;
  __shared__ double xb[2][32 * NC], pb[32 * NC];
  const int tid = threadIdx.x, l = tid & 63, w = tid >> 6, rl = l & 15, cl = 4 * w + (l >> 4);
  double a[NC][NS];
#pragma unroll
  for (int j = 0; j < NC; ++j)
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int r = rl + 16 * s, c = cl + 32 * j;
      a[j][s] = r < n && c < n ? A[r <= c ? r + (int64_t)n * c : c + (int64_t)n * r] : 0.0;
    }
  // rows 0 .. c of column c
  auto put = [&](int c) {
#pragma unroll
    for (int j = 0; j < NC; ++j)
      if (c == cl + 32 * j) {
#pragma unroll
        for (int s = 0; s < NS; ++s)
          if (rl + 16 * s <= c) xb[c & 1][rl + 16 * s] = a[j][s];
      }
  };
  put(n - 1);
  for (int k = n - 1; k >= 1; --k) {
    __syncthreads();
    const double* x = xb[k & 1];
    double alpha = x[k - 1], v[NS], vc[NC], ss, up = 1.0;
    auto squares = [&] {
      ss = 0.0;
#pragma unroll
      for (int s = 0; s < NS; ++s) ss = fma(v[s], v[s], ss);
      ss = sum16(ss);
    };
#pragma unroll
    for (int s = 0; s < NS; ++s) v[s] = rl + 16 * s < k - 1 ? x[rl + 16 * s] : 0.0;
    squares();
    // A column whose squares come near the ends of the exponent's range is taken times a power of two: the coupling of
    // two molecules far apart, 1e-160 of the rest, has squares of a few bits, with which H is not orthogonal.
    const double norm2 = fma(alpha, alpha, ss);
    if (norm2 < 0x1p-900 || norm2 > 0x1p900) {
      up = norm2 < 1.0 ? 0x1p600 : 0x1p-600;
      alpha *= up;
#pragma unroll
      for (int s = 0; s < NS; ++s) v[s] *= up;
      squares();
    }
    double beta = alpha, t = 0.0, sc = 0.0;  // x = 0: H = 1
    if (ss != 0.0) {
      beta = -copysign(sqrt(fma(alpha, alpha, ss)), alpha);
      t = (beta - alpha) / beta;
      sc = 1.0 / (alpha - beta);
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) v[s] = rl + 16 * s == k - 1 ? 1.0 : v[s] * sc;
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const int c = cl + 32 * j;
      vc[j] = 0.0;
      if (32 * j >= k) continue;
      vc[j] = c < k - 1 ? x[c] * up * sc : c == k - 1 ? 1.0 : 0.0;
      double q0 = 0.0, q1 = 0.0;
#pragma unroll
      for (int s = 0; s < NS; s += 2) {
        q0 = fma(a[j][s], v[s], q0);
        q1 = fma(a[j][s + 1], v[s + 1], q1);
      }
      q0 = sum16(q0 + q1) * t;
      if (rl == 0 && c < k) pb[c] = q0;
    }
    if (tid < 16) {
#pragma unroll
      for (int s = 0; s < NS; ++s)
        if (rl + 16 * s < k) V[rl + 16 * s + (int64_t)n * k] = v[s];
    }
    if (tid == 0) {
      d[k] = x[k];
      e[k - 1] = beta / up;
      tau[k - 1] = t;
    }
    __syncthreads();
    double p[NS], dt = 0.0;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      p[s] = rl + 16 * s < k ? pb[rl + 16 * s] : 0.0;
      dt = fma(p[s], v[s], dt);
    }
    const double al = -0.5 * t * sum16(dt);
#pragma unroll
    for (int s = 0; s < NS; ++s) p[s] = fma(al, v[s], p[s]);
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const int c = cl + 32 * j;
      if (32 * j >= k) continue;
      const double pc = c < k ? fma(al, vc[j], pb[c]) : 0.0;
#pragma unroll
      for (int s = 0; s < NS; ++s) a[j][s] = fma(-v[s], pc, fma(-p[s], vc[j], a[j][s]));
    }
    put(k - 1);
  }
  __syncthreads();
  if (tid == 0) d[0] = xb[0][0];
}

// out = Q Z: 16 lanes a column of Z, four columns a workgroup, the reflectors in turn from L2, four ahead.  Serial in the
// reflectors as well: n = 96 33 us, where ormtr's dozen launches take 200.
template <int NC>
__global__ __launch_bounds__(64) void k_tridiag_apply(int n, const double* __restrict__ V, const double* __restrict__ tau,
                                                      const double* __restrict__ Z, double* __restrict__ out) {
  constexpr int NS = 2 * NC, AHEAD = 4;
  const int rl = threadIdx.x & 15, c = 4 * blockIdx.x + (threadIdx.x >> 4);
  double z[NS], v[AHEAD][NS], t[AHEAD];
#pragma unroll
  for (int s = 0; s < NS; ++s) z[s] = rl + 16 * s < n && c < n ? Z[rl + 16 * s + (int64_t)n * c] : 0.0;
  auto load = [&](int u, int k) {
    t[u] = k < n ? tau[k - 1] : 0.0;
#pragma unroll
    for (int s = 0; s < NS; ++s) v[u][s] = k < n && rl + 16 * s < k ? V[rl + 16 * s + (int64_t)n * k] : 0.0;
  };
#pragma unroll
  for (int u = 0; u < AHEAD; ++u) load(u, 1 + u);
  for (int k = 1; k < n; k += AHEAD) {
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      double q0 = 0.0, q1 = 0.0;
#pragma unroll
      for (int s = 0; s < NS; s += 2) {
        q0 = fma(v[u][s], z[s], q0);
        q1 = fma(v[u][s + 1], z[s + 1], q1);
      }
      const double f = -t[u] * sum16(q0 + q1);
#pragma unroll
      for (int s = 0; s < NS; ++s) z[s] = fma(f, v[u][s], z[s]);
      load(u, k + u + AHEAD);
    }
  }
#pragma unroll
  for (int s = 0; s < NS; ++s)
    if (rl + 16 * s < n && c < n) out[rl + 16 * s + (int64_t)n * c] = z[s];
}

#define FH_BY_SIZE(K, ...)                                            \
  do {                                                                \
    if (n <= 32) hipLaunchKernelGGL((K<1>), __VA_ARGS__);             \
    else if (n <= 64) hipLaunchKernelGGL((K<2>), __VA_ARGS__);        \
    else if (n <= 96) hipLaunchKernelGGL((K<3>), __VA_ARGS__);        \
    else if (n <= 128) hipLaunchKernelGGL((K<4>), __VA_ARGS__);       \
    else hipLaunchKernelGGL((K<5>), __VA_ARGS__);                     \
    FH_HIP(hipGetLastError());                                        \
  } while (0)
void tridiag(hipStream_t s, int n, const double* A, double* V, double* d, double* e, double* tau) {
  FH_CHECK(tridiag_fits(n), -3, "tridiag: size");
  FH_BY_SIZE(k_tridiag, dim3(1), dim3(512), 0, s, n, A, V, d, e, tau);
}
void tridiag_apply(hipStream_t s, int n, const double* V, const double* tau, const double* Z, double* out) {
  FH_CHECK(tridiag_fits(n), -3, "tridiag: size");
  FH_BY_SIZE(k_tridiag_apply, dim3((n + 3) / 4), dim3(64), 0, s, n, V, tau, Z, out);
}
#undef FH_BY_SIZE

}  // namespace fh
