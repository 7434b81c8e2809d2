// Bandwidth-bound kernels of the DF-RCCSD(T) engine: tensor permutes, amplitude
// updates with on-the-fly denominators, deterministic FP64 reductions, DIIS linear
// combinations and the CC energy.
//
// Reductions are deterministic: every kernel writes one FP64 partial per workgroup
// (fixed grid for a given length) and a single workgroup adds the partials in a fixed
// order, so repeated runs give bitwise-identical results.
#include "fh_internal.h"

namespace fh {

static constexpr int RB = 256;        // threads per reduction block
static constexpr int64_t RMAX = 2048; // max partials per reduction

int64_t reduce_blocks_needed(int64_t n) {
  int64_t b = (n + RB * 4 - 1) / (RB * 4);
  if (b < 1) b = 1;
  if (b > RMAX) b = RMAX;
  return b;
}

static __device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// block-wide sum, result valid in thread 0
static __device__ __forceinline__ double block_sum(double v) {
  __shared__ double red[RB / 64];
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) red[w] = v;
  __syncthreads();
  double t = 0.0;
  if (threadIdx.x == 0) {
#pragma unroll
    for (int i = 0; i < RB / 64; ++i) t += red[i];
  }
  return t;
}

// ------------------------------------------------------------------ permute
struct PermArgs {
  int nd;
  int64_t odim[6], istr[6], ostr[6];
};

// out element per thread; used when output dim 0 reads the input with unit stride
__global__ __launch_bounds__(256) void k_permute_simple(PermArgs a, int64_t n, double alpha, const double* __restrict__ in,
                                                        double beta, double* __restrict__ out) {
  for (int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x; idx < n; idx += (int64_t)gridDim.x * 256) {
    int64_t rem = idx, off = 0;
#pragma unroll
    for (int d = 0; d < 6; ++d) {
      if (d < a.nd) {
        const int64_t c = rem % a.odim[d];
        rem /= a.odim[d];
        off += c * a.istr[d];
      }
    }
    double v = alpha * in[off];
    if (beta != 0.0) v += beta * out[idx];
    out[idx] = v;
  }
}

// The same with 32-bit index arithmetic (tensors of fewer than 2^31 elements, input offsets below
// 2^31): each coordinate comes from a division by an invariant integer done as a multiply-high and a
// shift (Granlund & Montgomery, PLDI 1994: q = (umulhi(n, m) + n) >> s with s = ceil(log2 d) and
// m = floor(2^32 (2^s - d) / d) + 1, exact for n < 2^31), instead of six 64-bit divisions per element.
struct PermArgs32 {
  int nd;
  uint32_t odim[6], istr[6], m[6], sh[6];
};
__global__ __launch_bounds__(256) void k_permute_simple32(PermArgs32 a, uint32_t n, double alpha,
                                                          const double* __restrict__ in, double beta,
                                                          double* __restrict__ out) {
  for (uint32_t idx = blockIdx.x * 256u + threadIdx.x; idx < n; idx += gridDim.x * 256u) {
    uint32_t rem = idx, off = 0;
#pragma unroll
    for (int d = 0; d < 6; ++d) {
      if (d < a.nd) {
        const uint32_t q = (__umulhi(rem, a.m[d]) + rem) >> a.sh[d];
        off += (rem - q * a.odim[d]) * a.istr[d];
        rem = q;
      }
    }
    double v = alpha * in[off];
    if (beta != 0.0) v += beta * out[idx];
    out[idx] = v;
  }
}

// 32x32 tiles over (output dim 0, output dim p) where dim p is the input's unit-stride dim:
// reads are coalesced along p, writes along output dim 0.  Each workgroup iteration moves two tiles
// (eight loads per thread in flight before the barrier).
__global__ __launch_bounds__(256) void k_permute_tiled(PermArgs a, int p, int64_t nrest, int64_t t0, int64_t tp,
                                                       double alpha, const double* __restrict__ in, double beta,
                                                       double* __restrict__ out) {
  __shared__ double tile[2][32][33];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int64_t ntiles = nrest * t0 * tp;
  for (int64_t base = 2 * (int64_t)blockIdx.x; base < ntiles; base += 2 * (int64_t)gridDim.x) {
    int64_t b0[2], bp[2], ioff[2], ooff[2];
    bool live[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      live[u] = base + u < ntiles;
      const int64_t blk = live[u] ? base + u : base;
      b0[u] = blk % t0;
      bp[u] = (blk / t0) % tp;
      // decompose the remaining dims
      int64_t rem = blk / (t0 * tp), io = 0, oo = 0;
      for (int d = 1; d < a.nd; ++d) {
        if (d == p) continue;
        const int64_t c = rem % a.odim[d];
        rem /= a.odim[d];
        io += c * a.istr[d];
        oo += c * a.ostr[d];
      }
      ioff[u] = io;
      ooff[u] = oo;
    }
    // load: threads consecutive along p
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t i0 = b0[u] * 32 + ty + 8 * r, ip = bp[u] * 32 + tx;
        if (live[u] && i0 < a.odim[0] && ip < a.odim[p]) tile[u][ty + 8 * r][tx] = in[ioff[u] + i0 * a.istr[0] + ip];
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t i0 = b0[u] * 32 + tx, ip = bp[u] * 32 + ty + 8 * r;
        if (live[u] && i0 < a.odim[0] && ip < a.odim[p]) {
          const int64_t o = ooff[u] + i0 + ip * a.ostr[p];
          double v = alpha * tile[u][tx][ty + 8 * r];
          if (beta != 0.0) v += beta * out[o];
          out[o] = v;
        }
      }
    }
    __syncthreads();
  }
}

void permute_f64(hipStream_t s, int nd, const int64_t* odim, const int64_t* istr, double alpha, const double* in,
                 double beta, double* out) {
  FH_CHECK(nd >= 1 && nd <= 6, -3, "permute: rank out of range");
  PermArgs a;
  a.nd = nd;
  int64_t n = 1;
  for (int d = 0; d < 6; ++d) { a.odim[d] = 1; a.istr[d] = 0; a.ostr[d] = 0; }
  for (int d = 0; d < nd; ++d) {
    a.odim[d] = odim[d];
    a.istr[d] = istr[d];
    a.ostr[d] = n;
    n *= odim[d];
  }
  if (n == 0) return;
  int p = -1;
  if (a.istr[0] != 1 || a.odim[0] == 1) {
    for (int d = 1; d < nd; ++d)
      if (a.istr[d] == 1 && a.odim[d] > 1) p = d;
  }
  if (p < 0 || a.odim[0] < 8) {
    int64_t g = (n + 255) / 256;
    if (g > 65536 * 4) g = 65536 * 4;
    int64_t maxoff = 0;
    for (int d = 0; d < nd; ++d) maxoff += (a.odim[d] - 1) * a.istr[d];
    bool small = n < (int64_t(1) << 31) && maxoff < (int64_t(1) << 31);
    for (int d = 0; d < nd; ++d) small = small && a.istr[d] >= 0;
    if (small) {
      PermArgs32 b;
      b.nd = nd;
      for (int d = 0; d < 6; ++d) {
        const uint32_t dv = d < nd ? (uint32_t)a.odim[d] : 1u;
        uint32_t sh = 0;
        while ((uint64_t(1) << sh) < dv) ++sh;
        b.odim[d] = dv;
        b.istr[d] = d < nd ? (uint32_t)a.istr[d] : 0u;
        b.sh[d] = sh;
        b.m[d] = (uint32_t)(((uint64_t(1) << 32) * ((uint64_t(1) << sh) - dv)) / dv + 1);
      }
      hipLaunchKernelGGL(k_permute_simple32, dim3((unsigned)g), dim3(256), 0, s, b, (uint32_t)n, alpha, in, beta, out);
    } else {
      hipLaunchKernelGGL(k_permute_simple, dim3((unsigned)g), dim3(256), 0, s, a, n, alpha, in, beta, out);
    }
  } else {
    const int64_t t0 = (a.odim[0] + 31) / 32, tp = (a.odim[p] + 31) / 32;
    const int64_t nrest = n / (a.odim[0] * a.odim[p]);
    int64_t g = (nrest * t0 * tp + 1) / 2;
    if (g > 65536 * 4) g = 65536 * 4;
    hipLaunchKernelGGL(k_permute_tiled, dim3((unsigned)g), dim3(256), 0, s, a, p, nrest, t0, tp, alpha, in, beta, out);
  }
  FH_HIP(hipGetLastError());
}

// ------------------------------------------------------------------ elementwise
__global__ void k_axpby(int64_t n, double a, const double* __restrict__ x, double b, double* __restrict__ y) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
    y[i] = (b == 0.0) ? a * x[i] : a * x[i] + b * y[i];
}
__global__ void k_fill(int64_t n, double v, double* __restrict__ y) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) y[i] = v;
}
static unsigned grid_for(int64_t n) {
  int64_t g = (n + 255) / 256;
  if (g > 65536) g = 65536;
  if (g < 1) g = 1;
  return (unsigned)g;
}
void axpby_f64(hipStream_t s, int64_t n, double a, const double* x, double b, double* y) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_axpby, dim3(grid_for(n)), dim3(256), 0, s, n, a, x, b, y);
  FH_HIP(hipGetLastError());
}
void fill_f64(hipStream_t s, int64_t n, double v, double* y) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_fill, dim3(grid_for(n)), dim3(256), 0, s, n, v, y);
  FH_HIP(hipGetLastError());
}

// ------------------------------------------------------------------ CCSD residual: operand forms and assembly
// Every form of the amplitudes that the residual's GEMMs read, from one read of T2 (each T2[:,:,a,b] tile with its
// partner [:,:,b,a]; any output may be null):
//   u[i,j,a,b] = 2 t2[ijab] - t2[ijba],  tau[i,j,a,b] = t2 + t1[ia] t1[jb],
//   ring[i,a,j,b] = u[ijab] and, n2 further, -t2[ijba],
//   pair[ij, ab] (i >= j, a >= b) = ts[ijab] + ts[ijba] (a > b; ts[ijaa] for a = b) and, Mp Kp further,
//   ts[ijab] - ts[ijba], with ts = (tau[ijab] + tau[jiba]) / 2.
template <typename TR, typename TP>
__global__ __launch_bounds__(256) void k_amp_forms(int o, int v, const double* __restrict__ t1, const double* __restrict__ t2,
                                                   double* __restrict__ u, double* __restrict__ tau, TR* __restrict__ ring,
                                                   TP* __restrict__ pair) {
  const int64_t oo = (int64_t)o * o, n2 = oo * v * v, ov = (int64_t)o * v;
  const int64_t np = (int64_t)v * (v + 1) / 2, mp = oo / 2 + (o + 1) / 2;
  const int64_t nblk = (oo + 255) / 256;
  for (int64_t w = blockIdx.x; w < np * nblk; w += gridDim.x) {
    const int64_t p = w / nblk;
    const int e = (int)(w - p * nblk) * 256 + threadIdx.x;
    int a = (int)((sqrt(8.0 * (double)p + 1.0) - 1.0) * 0.5);
    while ((int64_t)a * (a + 1) / 2 > p) --a;
    while ((int64_t)(a + 1) * (a + 2) / 2 <= p) ++a;
    const int b = (int)(p - (int64_t)a * (a + 1) / 2);
    if (e >= oo) continue;
    const int i = e % o, j = e / o, et = j + o * i;
    const int64_t ab = oo * (a + (int64_t)v * b), ba = oo * (b + (int64_t)v * a);
    const double x = t2[ab + e], y = t2[ba + e];
    const double xt = pair ? t2[ba + et] : 0.0, yt = pair ? t2[ab + et] : 0.0;
    const double s = t1[i + (int64_t)o * a] * t1[j + (int64_t)o * b], r = t1[i + (int64_t)o * b] * t1[j + (int64_t)o * a];
    if (u) {
      u[ab + e] = 2.0 * x - y;
      u[ba + e] = 2.0 * y - x;
    }
    if (tau) {
      tau[ab + e] = x + s;
      tau[ba + e] = y + r;
    }
    if (ring) {
      const int64_t f = i + (int64_t)o * a + ov * j + ov * o * b, g = i + (int64_t)o * b + ov * j + ov * o * a;
      ring[f] = (TR)(2.0 * x - y);
      ring[g] = (TR)(2.0 * y - x);
      ring[n2 + f] = (TR)(-y);
      ring[n2 + g] = (TR)(-x);
    }
    if (pair && i >= j) {
      const double ta = 0.5 * (x + xt) + s, tb = 0.5 * (y + yt) + r;
      const int64_t m = (int64_t)i * (i + 1) / 2 + j + mp * p;
      pair[m] = (TP)(a == b ? ta : ta + tb);
      pair[m + mp * np] = (TP)(a == b ? 0.0 : ta - tb);
    }
  }
}
template <typename TR, typename TP>
void amp_forms(hipStream_t s, int o, int v, const double* t1, const double* t2, double* u, double* tau, TR* ring, TP* pair) {
  const int64_t w = (int64_t)v * (v + 1) / 2 * (((int64_t)o * o + 255) / 256);
  hipLaunchKernelGGL((k_amp_forms<TR, TP>), dim3((unsigned)std::min<int64_t>(w, 65536)), dim3(256), 0, s, o, v, t1, t2, u,
                     tau, ring, pair);
  FH_HIP(hipGetLastError());
}
template void amp_forms<double, double>(hipStream_t, int, int, const double*, const double*, double*, double*, double*, double*);
template void amp_forms<double, float>(hipStream_t, int, int, const double*, const double*, double*, double*, double*, float*);
template void amp_forms<float, float>(hipStream_t, int, int, const double*, const double*, double*, double*, float*, float*);

// The PP ladder's operand over pairs c >= d, a >= b: with V[cd,ab] = (ca|db) = T(c, a, d, b) (element c + v-strides,
// T at sa a + sd d + sb b from its first a),
//   out[cd, ab] = V[cd,ab] + V[dc,ab]  and, behind all of them,  V[cd,ab] - V[dc,ab];
// sym: V is replaced by (V[cd,ab] + V[dc,ba]) / 2, its part that reaches the symmetrised residual (T must then
// hold every a and b).  32 x 32 tiles over (c, d): both reads run along the first index, the writes along d.
__global__ __launch_bounds__(256) void k_vv_pairs(int v, int a0, int na, const double* __restrict__ T, int64_t sa, int64_t sd,
                                                  int64_t sb, bool sym, int64_t ldv, double* __restrict__ out) {
  __shared__ double x[32][33], y[32][33];  // V[cd,ab] as [d][c], V[dc,ab] as [c][d]
  int ct = 0, q = blockIdx.x;
  while (q > ct) { q -= ct + 1; ++ct; }
  const int c0 = 32 * ct, d0 = 32 * q, tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int a = a0 + blockIdx.y, b = blockIdx.z;
  if (b > a || a >= a0 + na) return;
  const double* t = T + sa * (a - a0) + sb * b;
  const double* r = T + sa * b + sb * a;  // sym only
  for (int k = ty; k < 32; k += 8) {
    double p = 0.0, m = 0.0;
    if (c0 + tx < v && d0 + k < v) p = sym ? 0.5 * t[c0 + tx + sd * (d0 + k)] : t[c0 + tx + sd * (d0 + k)];
    if (d0 + tx < v && c0 + k < v) m = sym ? 0.5 * t[d0 + tx + sd * (c0 + k)] : t[d0 + tx + sd * (c0 + k)];
    x[k][tx] = p;
    y[k][tx] = m;
  }
  if (sym) {
    __syncthreads();
    for (int k = ty; k < 32; k += 8) {
      // + V[dc,ba] = T(d, b, c, a) to V[cd,ab], + V[cd,ba] = T(c, b, d, a) to V[dc,ab]
      if (d0 + tx < v && c0 + k < v) x[tx][k] += 0.5 * r[d0 + tx + sd * (c0 + k)];
      if (c0 + tx < v && d0 + k < v) y[tx][k] += 0.5 * r[c0 + tx + sd * (d0 + k)];
    }
  }
  __syncthreads();
  const int64_t col = ldv * ((int64_t)a * (a + 1) / 2 + b), anti = ldv * ((int64_t)v * (v + 1) / 2);
  for (int k = ty; k < 32; k += 8) {
    const int c = c0 + k, d = d0 + tx;
    if (c >= v || d > c) continue;
    const int64_t at = col + (int64_t)c * (c + 1) / 2 + d;
    out[at] = x[tx][k] + y[k][tx];
    out[at + anti] = x[tx][k] - y[k][tx];
  }
  if (c0 + 32 >= v && d0 == 0 && threadIdx.x < 4) {  // the padding of the column
    const int64_t np = (int64_t)v * (v + 1) / 2 + threadIdx.x;
    if (np < ldv) out[col + np] = out[col + anti + np] = 0.0;
  }
}
// whole 16-byte loads of FP32 columns
int64_t vv_pairs_ld(int64_t v) { return (v * (v + 1) / 2 + 3) / 4 * 4; }
void vv_pairs(hipStream_t s, int v, int a0, int na, const double* T, int64_t sa, int64_t sd, int64_t sb, bool sym, double* out) {
  const int nt = (v + 31) / 32;
  FH_CHECK(v < 65536, -3, "vv_pairs: grid too large");
  hipLaunchKernelGGL(k_vv_pairs, dim3((unsigned)(nt * (nt + 1) / 2), (unsigned)na, (unsigned)(a0 + na)), dim3(256), 0, s, v, a0,
                     na, T, sa, sd, sb, sym, vv_pairs_ld(v), out);
  FH_HIP(hipGetLastError());
}

// T2 numerator from its parts:
//   R2[ijab] = G[ijab] + G[jiba] + S[ijab],  G[ijab] = P[ijab] + (D[iajb] + F[iajb]) / 2 + F[ibja],
// D, F the two ring products in [i,a,j,b] order and S the ladder, S[ijab] = (Sp +- Sm)[ij, ab] / 2 over the packed
// pairs (+ where i >= j and a >= b agree).  One 32 x 32 (i, j) tile of an (a >= b) pair per workgroup step gives
// R2[ijab] and its mirror R2[jiba].
__global__ __launch_bounds__(256) void k_t2_numerator(int o, int v, const double* __restrict__ P, const double* __restrict__ D,
                                                      const double* __restrict__ F, const double* __restrict__ Sp,
                                                      double* __restrict__ R2) {
  __shared__ double gt[32][33];  // G[jiba] as [i][j]
  const int64_t oo = (int64_t)o * o, ov = (int64_t)o * v, np = (int64_t)v * (v + 1) / 2, mp = oo / 2 + (o + 1) / 2;
  const int nt = (o + 31) / 32, tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int64_t w = blockIdx.x; w < np * nt * nt; w += gridDim.x) {
    const int64_t p = w / (nt * nt);
    const int tl = (int)(w - p * nt * nt), i0 = 32 * (tl % nt), j0 = 32 * (tl / nt);
    int a = (int)((sqrt(8.0 * (double)p + 1.0) - 1.0) * 0.5);
    while ((int64_t)a * (a + 1) / 2 > p) --a;
    while ((int64_t)(a + 1) * (a + 2) / 2 <= p) ++a;
    const int b = (int)(p - (int64_t)a * (a + 1) / 2);
    const int64_t ab = oo * (a + (int64_t)v * b), ba = oo * (b + (int64_t)v * a);
    const int64_t rab = (int64_t)o * a + ov * o * b, rba = (int64_t)o * b + ov * o * a;  // ring offsets of (a, b), (b, a)
    __syncthreads();
    for (int k = ty; k < 32; k += 8) {
      const int j = j0 + tx, i = i0 + k;  // G[j,i,b,a]: j the unit-stride index
      if (j < o && i < o) {
        const int64_t q = j + ov * i;
        gt[k][tx] = P[ba + j + (int64_t)o * i] + 0.5 * (D[rba + q] + F[rba + q]) + F[rab + q];
      }
    }
    __syncthreads();
    for (int k = ty; k < 32; k += 8) {
      const int i = i0 + tx, j = j0 + k;
      if (i < o && j < o) {
        const int64_t q = i + ov * j;
        const int64_t m = (i >= j ? (int64_t)i * (i + 1) / 2 + j : (int64_t)j * (j + 1) / 2 + i) + mp * p;
        const double sp = Sp[m], sm = Sp[m + mp * np];
        const double r = P[ab + i + (int64_t)o * j] + 0.5 * (D[rab + q] + F[rab + q]) + F[rba + q] + gt[tx][k] +
                         0.5 * (i >= j ? sp + sm : sp - sm);
        R2[ab + i + (int64_t)o * j] = r;
        gt[tx][k] = r;
      }
    }
    if (a != b) {
      __syncthreads();
      for (int k = ty; k < 32; k += 8) {
        const int j = j0 + tx, i = i0 + k;
        if (j < o && i < o) R2[ba + j + (int64_t)o * i] = gt[k][tx];
      }
    }
  }
}
void t2_numerator(hipStream_t s, int o, int v, const double* P, const double* D, const double* F, const double* Sp, double* R2) {
  const int64_t nt = (o + 31) / 32, w = (int64_t)v * (v + 1) / 2 * nt * nt;
  hipLaunchKernelGGL(k_t2_numerator, dim3((unsigned)std::min<int64_t>(w, 65536)), dim3(256), 0, s, o, v, P, D, F, Sp, R2);
  FH_HIP(hipGetLastError());
}

// ------------------------------------------------------------------ Jacobi update (RCCSDHelper.jl:347-348)
template <bool T2, bool F32>
__global__ __launch_bounds__(RB) void k_jacobi(int o, int v, const double* __restrict__ eo, const double* __restrict__ ev,
                                               double* __restrict__ R, const double* __restrict__ old, void* err,
                                               double* __restrict__ partials) {
  const int64_t n = T2 ? (int64_t)o * o * v * v : (int64_t)o * v;
  double acc = 0.0;
  for (int64_t idx = (int64_t)blockIdx.x * RB + threadIdx.x; idx < n; idx += (int64_t)gridDim.x * RB) {
    double d;
    if (T2) {
      const int64_t i = idx % o, j = (idx / o) % o, a = (idx / ((int64_t)o * o)) % v, b = idx / ((int64_t)o * o * v);
      d = eo[i] + eo[j] - ev[a] - ev[b];
    } else {
      const int64_t i = idx % o, a = idx / o;
      d = eo[i] - ev[a];
    }
    const double nv = R[idx] / d;
    R[idx] = nv;
    const double e = nv - old[idx];
    if (err) {
      if (F32) static_cast<float*>(err)[idx] = (float)e;
      else static_cast<double*>(err)[idx] = e;
    }
    acc += e * e;
  }
  const double t = block_sum(acc);
  if (threadIdx.x == 0) partials[blockIdx.x] = t;
}
void jacobi_update(hipStream_t s, int o, int v, bool is_t2, const double* eo, const double* ev, double* R,
                   const double* old, void* err, bool err_f32, double* partials, int64_t* nblocks) {
  const int64_t n = is_t2 ? (int64_t)o * o * v * v : (int64_t)o * v;
  const int64_t g = reduce_blocks_needed(n);
  *nblocks = g;
  if (is_t2) {
    if (err_f32) hipLaunchKernelGGL((k_jacobi<true, true>), dim3(g), dim3(RB), 0, s, o, v, eo, ev, R, old, err, partials);
    else hipLaunchKernelGGL((k_jacobi<true, false>), dim3(g), dim3(RB), 0, s, o, v, eo, ev, R, old, err, partials);
  } else {
    if (err_f32) hipLaunchKernelGGL((k_jacobi<false, true>), dim3(g), dim3(RB), 0, s, o, v, eo, ev, R, old, err, partials);
    else hipLaunchKernelGGL((k_jacobi<false, false>), dim3(g), dim3(RB), 0, s, o, v, eo, ev, R, old, err, partials);
  }
  FH_HIP(hipGetLastError());
}

// ------------------------------------------------------------------ reductions
__global__ __launch_bounds__(RB) void k_dot(int64_t n, const double* __restrict__ x, const double* __restrict__ y,
                                            double* __restrict__ partials) {
  double acc = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * RB + threadIdx.x; i < n; i += (int64_t)gridDim.x * RB) acc += x[i] * y[i];
  const double t = block_sum(acc);
  if (threadIdx.x == 0) partials[blockIdx.x] = t;
}
__global__ __launch_bounds__(RB) void k_sum(int64_t n, const double* __restrict__ partials, double* __restrict__ result) {
  double acc = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += RB) acc += partials[i];
  const double t = block_sum(acc);
  if (threadIdx.x == 0) *result = t;
}
void sum_partials(hipStream_t s, int64_t n, const double* partials, double* result) {
  hipLaunchKernelGGL(k_sum, dim3(1), dim3(RB), 0, s, n, partials, result);
  FH_HIP(hipGetLastError());
}
void dot_f64(hipStream_t s, int64_t n, const double* x, const double* y, double* partials, double* result) {
  const int64_t g = reduce_blocks_needed(n);
  hipLaunchKernelGGL(k_dot, dim3(g), dim3(RB), 0, s, n, x, y, partials);
  FH_HIP(hipGetLastError());
  sum_partials(s, g, partials, result);
}
// result[q] = x_q . y for up to 8 vectors, each element of y read once: a row of the DIIS matrix in two launches and one
// read of the subspace (bound by HBM for large amplitudes, by launches for small ones: a dot and its sum per element of
// the matrix, each with a copy back, were 132 of them a solve at o = 16, v = 76, 20 us each).
struct DotsArgs {
  int nv;
  const void* x[8];
};
template <typename T>
__global__ __launch_bounds__(RB) void k_dots(int64_t n, DotsArgs a, const T* __restrict__ y, double* __restrict__ partials) {
  double acc[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  for (int64_t i = (int64_t)blockIdx.x * RB + threadIdx.x; i < n; i += (int64_t)gridDim.x * RB) {
    const double v = (double)y[i];
#pragma unroll
    for (int q = 0; q < 8; ++q)
      if (q < a.nv) acc[q] += (double)static_cast<const T*>(a.x[q])[i] * v;
  }
#pragma unroll
  for (int q = 0; q < 8; ++q)
    if (q < a.nv) {
      const double t = block_sum(acc[q]);
      if (threadIdx.x == 0) partials[(int64_t)q * gridDim.x + blockIdx.x] = t;
      __syncthreads();
    }
}
__global__ __launch_bounds__(RB) void k_sums(int64_t n, const double* __restrict__ partials, double* __restrict__ result) {
  double acc = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += RB) acc += partials[n * blockIdx.x + i];
  const double t = block_sum(acc);
  if (threadIdx.x == 0) result[blockIdx.x] = t;
}
void dots(hipStream_t s, int64_t n, int nv, const void* const* xs, const void* y, bool f32, double* partials,
          double* result) {
  FH_CHECK(nv >= 1 && nv <= 8, -3, "dots: 1..8 vectors");
  DotsArgs a;
  a.nv = nv;
  for (int q = 0; q < 8; ++q) a.x[q] = q < nv ? xs[q] : nullptr;
  const int64_t g = reduce_blocks_needed(n);
  if (f32) hipLaunchKernelGGL((k_dots<float>), dim3(g), dim3(RB), 0, s, n, a, static_cast<const float*>(y), partials);
  else hipLaunchKernelGGL((k_dots<double>), dim3(g), dim3(RB), 0, s, n, a, static_cast<const double*>(y), partials);
  FH_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_sums, dim3(nv), dim3(RB), 0, s, g, partials, result);
  FH_HIP(hipGetLastError());
}

// ------------------------------------------------------------------ DIIS extrapolation (DIIS.jl:86-93)
struct LinArgs {
  int nv;
  const double* x[8];
  const void* e[8];
  double c[8];
};
template <bool F32>
__global__ void k_lincomb(int64_t n, LinArgs a, bool add_err, double* __restrict__ y) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    double acc = 0.0;
    for (int q = 0; q < a.nv; ++q) acc += a.c[q] * a.x[q][i];
    if (add_err) {
      double ae = 0.0;
      for (int q = 0; q < a.nv; ++q)
        ae += a.c[q] * (F32 ? (double)static_cast<const float*>(a.e[q])[i] : static_cast<const double*>(a.e[q])[i]);
      acc += ae;
    }
    y[i] = acc;
  }
}
void lincomb(hipStream_t s, int64_t n, int nv, const double* const* xs, const double* cs, const void* const* es,
             bool err_f32, bool add_err, double* y) {
  FH_CHECK(nv >= 1 && nv <= 8, -3, "lincomb: 1..8 vectors");
  LinArgs a;
  a.nv = nv;
  for (int q = 0; q < 8; ++q) { a.x[q] = q < nv ? xs[q] : nullptr; a.e[q] = q < nv ? es[q] : nullptr; a.c[q] = q < nv ? cs[q] : 0.0; }
  if (err_f32) hipLaunchKernelGGL((k_lincomb<true>), dim3(grid_for(n)), dim3(256), 0, s, n, a, add_err, y);
  else hipLaunchKernelGGL((k_lincomb<false>), dim3(grid_for(n)), dim3(256), 0, s, n, a, add_err, y);
  FH_HIP(hipGetLastError());
}

__global__ void k_cast(int64_t n, const double* __restrict__ x, float* __restrict__ y) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) y[i] = (float)x[i];
}
void cast_f64_to_f32(hipStream_t s, int64_t n, const double* x, float* y) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_cast, dim3(grid_for(n)), dim3(256), 0, s, n, x, y);
  FH_HIP(hipGetLastError());
}

// ------------------------------------------------------------------ CC energy (RCCSDHelper.jl:8-23)
// E = sum_{k,c,l,d} (kc|ld) * (2 T2[k,l,c,d] - T2[l,k,c,d] - T1[l,c] T1[k,d] + 2 T1[k,c] T1[l,d]),
// iterated in the memory order of OVOV[k,c,l,d] so that the integral stream is coalesced.
__global__ __launch_bounds__(RB) void k_cc_energy(int o, int v, const double* __restrict__ t1, const double* __restrict__ t2,
                                                  const double* __restrict__ ovov, double* __restrict__ partials) {
  const int64_t n = (int64_t)o * v * o * v;
  const int64_t oo = (int64_t)o * o;
  double acc = 0.0;
  for (int64_t idx = (int64_t)blockIdx.x * RB + threadIdx.x; idx < n; idx += (int64_t)gridDim.x * RB) {
    const int64_t k = idx % o, c = (idx / o) % v, l = (idx / ((int64_t)o * v)) % o, d = idx / ((int64_t)o * v * o);
    const double t2klcd = t2[k + o * l + oo * c + oo * v * d];
    const double t2lkcd = t2[l + o * k + oo * c + oo * v * d];
    const double b = 2.0 * t2klcd - t2lkcd - t1[l + o * c] * t1[k + o * d] + 2.0 * t1[k + o * c] * t1[l + o * d];
    acc += b * ovov[idx];
  }
  const double t = block_sum(acc);
  if (threadIdx.x == 0) partials[blockIdx.x] = t;
}
// The same sum for o <= 64, one (c,d) pair at a time: the o x o tile T2[:,:,c,d] is read once,
// contiguously, into LDS (rows padded to o+1), where both T2[k,l,c,d] and T2[l,k,c,d] are read;
// OVOV[k,c,l,d] is read in runs of o along k.  A fixed grid strides over the pairs.
static constexpr int kCcTileO = 64;
__global__ __launch_bounds__(RB) void k_cc_energy_tiles(int o, int v, const double* __restrict__ t1,
                                                        const double* __restrict__ t2,
                                                        const double* __restrict__ ovov,
                                                        double* __restrict__ partials) {
  __shared__ double tile[kCcTileO * (kCcTileO + 1)];
  __shared__ double tc[kCcTileO], td[kCcTileO];
  const int oo = o * o, op = o + 1;
  const int64_t ov = (int64_t)o * v;
  double acc = 0.0;
  for (int cd = blockIdx.x; cd < v * v; cd += gridDim.x) {
    const int c = cd % v, d = cd / v;
    const double* __restrict__ t2cd = t2 + (int64_t)oo * cd;            // T2[:, :, c, d]
    __syncthreads();                                                     // previous pair's reads done
    for (int e = threadIdx.x; e < oo; e += RB) tile[(e % o) + op * (e / o)] = t2cd[e];
    if ((int)threadIdx.x < o) {
      tc[threadIdx.x] = t1[threadIdx.x + o * c];
      td[threadIdx.x] = t1[threadIdx.x + o * d];
    }
    __syncthreads();
    const double* __restrict__ vcd = ovov + (int64_t)o * c + ov * o * d;  // + k + o v l
    for (int e = threadIdx.x; e < oo; e += RB) {
      const int k = e % o, l = e / o;
      const double b = 2.0 * tile[k + op * l] - tile[l + op * k] - tc[l] * td[k] + 2.0 * tc[k] * td[l];
      acc += b * vcd[k + ov * l];
    }
  }
  const double t = block_sum(acc);
  if (threadIdx.x == 0) partials[blockIdx.x] = t;
}

void cc_energy(hipStream_t s, int o, int v, const double* t1, const double* t2, const double* ovov, double* partials,
               double* result) {
  if (o <= kCcTileO) {
    const int64_t g = std::min<int64_t>((int64_t)v * v, RMAX);
    hipLaunchKernelGGL(k_cc_energy_tiles, dim3(g), dim3(RB), 0, s, o, v, t1, t2, ovov, partials);
    FH_HIP(hipGetLastError());
    sum_partials(s, g, partials, result);
    return;
  }
  const int64_t n = (int64_t)o * v * o * v;
  const int64_t g = reduce_blocks_needed(n);
  hipLaunchKernelGGL(k_cc_energy, dim3(g), dim3(RB), 0, s, o, v, t1, t2, ovov, partials);
  FH_HIP(hipGetLastError());
  sum_partials(s, g, partials, result);
}

// ------------------------------------------------------------------ SCF helpers (RHFHelper.jl:7-59)
// out[i + n k] = U[i + n k] / sqrt(w[k])  (U diag(w)^-1/2, for S^-1/2 = U diag(w)^-1/2 U^T)
__global__ void k_scale_cols_rsqrt(int n, const double* __restrict__ U, const double* __restrict__ w,
                                   double* __restrict__ out) {
  const int64_t nn = (int64_t)n * n;
  for (int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x; idx < nn; idx += (int64_t)gridDim.x * 256)
    out[idx] = U[idx] / sqrt(w[idx / n]);
}
void scale_cols_rsqrt(hipStream_t s, int n, const double* U, const double* w, double* out) {
  hipLaunchKernelGGL(k_scale_cols_rsqrt, dim3(grid_for((int64_t)n * n)), dim3(256), 0, s, n, U, w, out);
  FH_HIP(hipGetLastError());
}
// generalised Wolfsberg-Helmholz Fock guess: F_ii = H_ii, F_ij = 0.875 S_ij (H_ii + H_jj)
__global__ void k_gwh_fock(int n, const double* __restrict__ S, const double* __restrict__ H, double* __restrict__ F) {
  const int64_t nn = (int64_t)n * n;
  for (int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x; idx < nn; idx += (int64_t)gridDim.x * 256) {
    const int i = (int)(idx % n), j = (int)(idx / n);
    F[idx] = i == j ? H[idx] : 0.875 * S[idx] * (H[(int64_t)i * (n + 1)] + H[(int64_t)j * (n + 1)]);
  }
}
void gwh_fock(hipStream_t s, int n, const double* S, const double* H, double* F) {
  hipLaunchKernelGGL(k_gwh_fock, dim3(grid_for((int64_t)n * n)), dim3(256), 0, s, n, S, H, F);
  FH_HIP(hipGetLastError());
}

}  // namespace fh
