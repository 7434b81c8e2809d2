// Integrals over contracted Gaussian shells on the device: overlap, kinetic, nuclear attraction, the
// 4-centre Coulomb integrals (mu nu|la si), and the density-fitting 3-centre (mu nu|P) and 2-centre
// (P|Q) integrals -- overlap / kinetic / nuclear / ERI_2e4c / ERI_2e3c / ERI_2e2c of GaussianBasis.jl,
// called by AtomicIntegrals.jl:18-45.
//
// McMurchie-Davidson scheme (J. Comput. Phys. 26, 218 (1978); Helgaker, Jorgensen, Olsen, Molecular
// Electronic-Structure Theory, sections 9.5-9.9): per primitive pair the Hermite expansion coefficients
// E^{ij}_t of each Cartesian factor, per primitive pair of pairs the Hermite Coulomb integrals
// R_{tuv} (t+u+v <= L) from the Boys function, then
//   (ab|cd) = 2 pi^{5/2} / (p q sqrt(p+q)) sum_{tuv} E^{ab}_{tuv} sum_{xyz} (-1)^{x+y+z} E^{cd}_{xyz} R_{t+x,u+y,v+z}
// and the one-electron forms.  A 3-centre (2-centre) integral takes the unit function as the
// missing partner; spherical components are the normalised real solid harmonics (m = -l .. l) of the
// table the host passes (fh_integrals_tables).  The Coulomb integrals run in two steps (k_pair_e,
// k_eri): the E^{ab} of every pair of shells once, then a kernel for each pair of Hermite orders.
#include "fh_host.h"
#include "fh_internal.h"

#include <algorithm>
#include <cmath>
#include <cstring>

namespace fh {

namespace {

constexpr int kMaxLOrb = 2;               // orbital shells: s, p, d
constexpr int kMaxLAux = 3;               // fitting shells: s, p, d, f
constexpr int kMaxCart = 10;              // Cartesian components of an f shell
constexpr int kMaxCartO = 6;              // ... of a d shell
constexpr int kMaxLR = 4 * kMaxLOrb;      // Hermite order of (dd|dd)
constexpr int kRSize = (kMaxLR + 1) * (kMaxLR + 2) * (kMaxLR + 3) / 6;   // 165

__device__ inline int tet(int t, int u, int v) {
  const int s = t + u + v, j = u + v;
  return s * (s + 1) * (s + 2) / 6 + j * (j + 1) / 2 + v;
}

// F_0 .. F_nmax of T: series + downward recursion below T = 30, asymptotic F_0 + upward recursion above
__device__ void boys(int nmax, double T, double* F) {
  if (T < 30.0) {
    double term = 1.0 / (2 * nmax + 1), s = term;
    for (int k = 1; k < 400; ++k) {
      term *= 2.0 * T / (2 * nmax + 2 * k + 1);
      s += term;
      if (term < 1e-17 * s) break;
    }
    const double eT = exp(-T);
    F[nmax] = eT * s;
    for (int m = nmax; m > 0; --m) F[m - 1] = (2.0 * T * F[m] + eT) / (2 * m - 1);
  } else {
    const double eT = exp(-T);
    F[0] = 0.5 * sqrt(M_PI / T) * erf(sqrt(T));
    for (int m = 0; m < nmax; ++m) F[m + 1] = ((2 * m + 1) * F[m] - eT) / (2.0 * T);
  }
}

// E[((i (lb+1) + j) (la+lb+1) + t) ST] for i <= la, j <= lb (one Cartesian axis)
template <int ST = 1>
__device__ void hermite_E(int la, int lb, double a, double b, double A, double B, double* E) {
  const double p = a + b, X = A - B, XPA = -b / p * X, XPB = a / p * X, h = 0.5 / p;
  const int nt = la + lb + 1;
  auto at = [&](int i, int j, int t) -> double& { return E[((i * (lb + 1) + j) * nt + t) * ST]; };
  for (int i = 0; i <= la; ++i)
    for (int j = 0; j <= lb; ++j)
      for (int t = 0; t < nt; ++t) at(i, j, t) = 0.0;
  at(0, 0, 0) = exp(-a * b / p * X * X);
  for (int i = 0; i <= la; ++i)
    for (int j = 0; j <= lb; ++j) {
      if (i == 0 && j == 0) continue;
      for (int t = 0; t <= i + j; ++t) {
        double v;
        if (i > 0) {
          v = XPA * at(i - 1, j, t) + (t + 1 <= i - 1 + j ? (t + 1) * at(i - 1, j, t + 1) : 0.0);
          if (t > 0) v += h * at(i - 1, j, t - 1);
        } else {
          v = XPB * at(i, j - 1, t) + (t + 1 <= i + j - 1 ? (t + 1) * at(i, j - 1, t + 1) : 0.0);
          if (t > 0) v += h * at(i, j - 1, t - 1);
        }
        at(i, j, t) = v;
      }
    }
}

// R[tet(t,u,v)] for t+u+v <= L at exponent al and distance (X,Y,Z): levels n = L .. 0 of
// R^n_{t+1,u,v} = t R^{n+1}_{t-1,u,v} + X R^{n+1}_{t,u,v} in two buffers
__device__ void hermite_R(int L, double al, double X, double Y, double Z, double* R, double* W) {
  double F[kMaxLR + 1];
  boys(L, al * (X * X + Y * Y + Z * Z), F);
  double* cur = W;   // level n + 1
  double* nxt = R;   // level n
  // level L: only R_000
  double m2a = 1.0;
  for (int n = 0; n < L; ++n) m2a *= -2.0 * al;
  cur[0] = m2a * F[L];
  for (int n = L - 1; n >= 0; --n) {
    m2a /= -2.0 * al;
    nxt[0] = m2a * F[n];
    for (int s = 1; s <= L - n; ++s)
      for (int t = s; t >= 0; --t)
        for (int u = s - t; u >= 0; --u) {
          const int v = s - t - u;
          double val;
          if (t > 0) val = X * cur[tet(t - 1, u, v)] + (t > 1 ? (t - 1) * cur[tet(t - 2, u, v)] : 0.0);
          else if (u > 0) val = Y * cur[tet(t, u - 1, v)] + (u > 1 ? (u - 1) * cur[tet(t, u - 2, v)] : 0.0);
          else val = Z * cur[tet(t, u, v - 1)] + (v > 1 ? (v - 1) * cur[tet(t, u, v - 2)] : 0.0);
          nxt[tet(t, u, v)] = val;
        }
    double* tmp = cur;
    cur = nxt;
    nxt = tmp;
  }
  if (cur != R)
    for (int q = 0; q < (L + 1) * (L + 2) * (L + 3) / 6; ++q) R[q] = cur[q];
}

__device__ inline int ncart(int l) { return (l + 1) * (l + 2) / 2; }
// Cartesian exponents of component c of shell l (x-major order, as the host table)
__device__ inline void cart_exps(int l, int c, int& x, int& y, int& z) {
  int k = 0;
  for (int lx = l; lx >= 0; --lx)
    for (int ly = l - lx; ly >= 0; --ly) {
      if (k == c) { x = lx; y = ly; z = l - lx - ly; return; }
      ++k;
    }
  x = y = z = 0;
}

}  // namespace

// ------------------------------------------------------------------ kernels
// Shells: l, nprim, prim offset, function offset, Cartesian center.  Primitive coefficients are those of
// unnormalised x^l exp(-a r^2) primitives that give a contracted function normalised for x^l.
// sph[l][m][c]: spherical transform of shell type l (Cartesian when spherical == 0: identity).
struct IntShell {
  int l, nprim, poff, foff;
  double x, y, z;
};
struct SphTab {
  double c[kMaxLAux + 1][2 * kMaxLAux + 1][kMaxCart];
  int spherical;
};

__device__ inline int nfun(const SphTab& T, int l) { return T.spherical ? 2 * l + 1 : ncart(l); }
__device__ inline double tcoef(const SphTab& T, int l, int m, int c) {
  return T.spherical ? T.c[l][m][c] : (m == c ? 1.0 : 0.0);
}

// ------------------------------------------------------------------ Coulomb integrals
namespace {
constexpr int nherm(int l) { return (l + 1) * (l + 2) * (l + 3) / 6; }   // Hermite functions of order <= l
constexpr int kNH = 2 * kMaxLOrb;                                       // Hermite order of a shell pair

// Hermite index <-> (t, u, v), as tet(), and the index of a sum of two
struct HermTab {
  int t[nherm(kMaxLR)], u[nherm(kMaxLR)], v[nherm(kMaxLR)];
  int sum[nherm(kNH)][nherm(kNH)];
};
constexpr HermTab herm_tab() {
  HermTab h{};
  int q = 0;
  for (int s = 0; s <= kMaxLR; ++s)
    for (int j = 0; j <= s; ++j)
      for (int v = 0; v <= j; ++v) {
        h.t[q] = s - j;
        h.u[q] = j - v;
        h.v[q] = v;
        ++q;
      }
  for (int a = 0; a < nherm(kNH); ++a)
    for (int b = 0; b < nherm(kNH); ++b) {
      const int t = h.t[a] + h.t[b], u = h.u[a] + h.u[b], v = h.v[a] + h.v[b], s = t + u + v, j = u + v;
      h.sum[a][b] = s * (s + 1) * (s + 2) / 6 + j * (j + 1) / 2 + v;
    }
  return h;
}
__device__ constexpr HermTab kHT = herm_tab();

// Boys functions F_0 .. F_{kMaxLR + kBoysTerms} at T = 0, 1/8 .. 32: F_n(T0 - d) = sum_k F_{n+k}(T0) d^k / k!, and
// with |d| <= 1/16 eight terms after the first leave (1/16)^9 / 9! = 4e-17 of F_{n+9}
constexpr int kBoysTerms = 8, kBoysRow = kMaxLR + kBoysTerms + 1, kBoysRows = 32 * 8 + 1;

// F_0 .. F_L of T
template <int L>
__device__ inline void boys_tab(const double* __restrict__ tab, double T, double* F) {
  if (T < 32.0) {
    const int k = (int)(8.0 * T + 0.5);
    const double d = 0.125 * k - T;
    const double* row = tab + k * kBoysRow + L;
    double f = row[kBoysTerms];
#pragma unroll
    for (int j = kBoysTerms; j > 0; --j) f = fma(d * (1.0 / j), f, row[j - 1]);
    F[L] = f;
    if constexpr (L > 0) {
      const double eT = exp(-T);
#pragma unroll
      for (int m = L; m > 0; --m) F[m - 1] = fma(2.0 * T, F[m], eT) * (1.0 / (2 * m - 1));
    }
  } else {
    // 1 - erf(sqrt T) = e^-T / sqrt(pi T) (1 - 1 / (2 T) + ..), under 2e-15 here
    const double eT = exp(-T), h = 0.5 / T;
    F[0] = 0.5 * sqrt(M_PI / T) - eT * h * (1.0 - h);
#pragma unroll
    for (int m = 0; m < L; ++m) F[m + 1] = fma(2 * m + 1, F[m], -eT) * h;
  }
}

// R of level m from R of level m + 1 in place, m = M .. 0; F holds the scaled F_m = R^m_000.  From the highest order
// down: an element of order S needs orders S - 1 and S - 2 of the level before (tet(): one less of t is order S - 1 at
// the same u + v and v).  One order a template level: a whole level of (dd|dd) is beyond the unroll limit and would
// put R into scratch memory.
template <int S>
__device__ inline void herm_orders(double X, double Y, double Z, double* R) {
  constexpr int b0 = nherm(S - 1), b1 = nherm(S - 2), b2 = nherm(S - 3);
#pragma unroll
  for (int x = 0; x < (S + 1) * (S + 2) / 2; ++x) {
    const int t = kHT.t[b0 + x], u = kHT.u[b0 + x], v = kHT.v[b0 + x], j = u + v;
    const int k1 = (j - 1) * j / 2 + v, k2 = (j - 2) * (j - 1) / 2 + v;
    if (t > 0) R[b0 + x] = t > 1 ? fma(X, R[b1 + x], (t - 1) * R[b2 + x]) : X * R[b1 + x];
    else if (u > 0) R[b0 + x] = u > 1 ? fma(Y, R[b1 + k1], (u - 1) * R[b2 + k2]) : Y * R[b1 + k1];
    else R[b0 + x] = v > 1 ? fma(Z, R[b1 + k1 - 1], (v - 1) * R[b2 + k2 - 2]) : Z * R[b1 + k1 - 1];
  }
  if constexpr (S > 1) herm_orders<S - 1>(X, Y, Z, R);
}
template <int L, int M>
__device__ inline void herm_levels(double X, double Y, double Z, const double* F, double* R) {
  herm_orders<L - M>(X, Y, Z, R);
  R[0] = F[M];
  if constexpr (M > 0) herm_levels<L, M - 1>(X, Y, Z, F, R);
}

// G[h] += (-1)^k ke[k] R[h + k] for the NK Hermite functions k of the ket (one column a template level: a nest of 35 x 35
// is beyond the unroll limit and would put R into scratch memory)
template <int NA, int NK, int K = 0>
__device__ inline void herm_sum(const double* __restrict__ ke, const double* R, double* G) {
  const double e = (kHT.t[K] + kHT.u[K] + kHT.v[K]) & 1 ? -ke[K] : ke[K];
#pragma unroll
  for (int h = 0; h < NA; ++h) G[h] = fma(e, R[kHT.sum[h][K]], G[h]);
  if constexpr (K + 1 < NK) herm_sum<NA, NK, K + 1>(ke, R, G);
}

// A pair of shells a, b (b < 0: the unit function).  Its tables E[prim][function][Hermite] start at eoff, its np
// primitive pairs' (p, P) at 4 poff; function f = i mb + j stands for the functions fa + i and fb + j.
struct PairHead {
  int64_t eoff;
  int poff, np, a, b, fa, fb, mb, nf, l, pad;
};
// One function of a ket pair: its table at eoff, est further for the next primitive pair; r and s as fa + i, fb + j.
struct Ket {
  int64_t eoff;
  int est, np, poff, r, s, pad;
};
constexpr int kPairPrims = 16;   // primitive pairs that a k_pair_e workgroup holds at a time
constexpr int kPairE = (kMaxLOrb + 1) * (kMaxLOrb + 1) * (2 * kMaxLOrb + 1);
static_assert((kMaxLAux + 1) * (kMaxLAux + 1) <= kPairE, "a single f shell fits too");

__device__ inline double3 center_of(const IntShell& s) { return double3{s.x, s.y, s.z}; }
}  // namespace

// Tables of a shell pair, one workgroup each: the Hermite coefficients of 16 primitive pairs' axes in LDS (a thread
// per axis and primitive pair), then a thread per (primitive pair, function, Hermite index) sums the Cartesian
// components with the spherical coefficients.  cf_a cf_b sqrt(2 pi^{5/2}) / p is taken in, so that a product of two
// tables needs only 1 / sqrt(p + q).
__global__ __launch_bounds__(256) void k_pair_e(const PairHead* __restrict__ heads, const IntShell* __restrict__ sh,
                                               const double* __restrict__ ex, const double* __restrict__ cf, SphTab T,
                                               double* __restrict__ E, double* __restrict__ prim) {
  __shared__ double Es[3][kPairE * kPairPrims];
  __shared__ double fac[kPairPrims];
  const PairHead hd = heads[blockIdx.x];
  const IntShell sa = sh[hd.a], sb = sh[hd.b < 0 ? hd.a : hd.b];
  const bool null = hd.b < 0;
  const int la = sa.l, lb = null ? 0 : sb.l, nt = la + lb + 1, nh = nherm(la + lb), npb = null ? 1 : sb.nprim;
  const int na = ncart(la), nb = ncart(lb), tid = threadIdx.x;
  const double3 A = center_of(sa), B = center_of(sb);
  for (int p0 = 0; p0 < hd.np; p0 += kPairPrims) {
    const int m = min(kPairPrims, hd.np - p0), q = tid % kPairPrims, axis = tid / kPairPrims;
    __syncthreads();
    if (q < m && axis < 4) {
      const int pa = (p0 + q) / npb, pb = (p0 + q) % npb;
      const double a = ex[sa.poff + pa], b = null ? 0.0 : ex[sb.poff + pb], p = a + b;
      if (axis < 3) {
        const double Ax = axis == 0 ? A.x : axis == 1 ? A.y : A.z, Bx = axis == 0 ? B.x : axis == 1 ? B.y : B.z;
        hermite_E<kPairPrims>(la, lb, a, b, Ax, Bx, &Es[axis][q]);
        prim[4 * (int64_t)(hd.poff + p0 + q) + 1 + axis] = (a * Ax + b * Bx) / p;
      } else {
        prim[4 * (int64_t)(hd.poff + p0 + q)] = p;
        fac[q] = cf[sa.poff + pa] * (null ? 1.0 : cf[sb.poff + pb]) * sqrt(2.0 * M_PI * M_PI * sqrt(M_PI)) / p;
      }
    }
    __syncthreads();
    for (int64_t e = tid; e < (int64_t)m * hd.nf * nh; e += 256) {
      const int h = (int)(e % nh), f = (int)(e / nh % hd.nf), k = (int)(e / nh / hd.nf);
      const int i = f / hd.mb, j = f % hd.mb, t = kHT.t[h], u = kHT.u[h], v = kHT.v[h];
      double sum = 0.0;
      for (int ia = 0; ia < na; ++ia) {
        const double ca = tcoef(T, la, i, ia);
        if (ca == 0.0) continue;
        int ax, ay, az;
        cart_exps(la, ia, ax, ay, az);
        for (int ib = 0; ib < nb; ++ib) {
          const double cb = null ? 1.0 : tcoef(T, lb, j, ib);
          if (cb == 0.0) continue;
          int bx, by, bz;
          cart_exps(lb, ib, bx, by, bz);
          if (t > ax + bx || u > ay + by || v > az + bz) continue;
          sum += ca * cb * Es[0][((ax * (lb + 1) + bx) * nt + t) * kPairPrims + k] *
                 Es[1][((ay * (lb + 1) + by) * nt + u) * kPairPrims + k] *
                 Es[2][((az * (lb + 1) + bz) * nt + v) * kPairPrims + k];
        }
      }
      E[hd.eoff + ((int64_t)(p0 + k) * hd.nf + f) * nh + h] = sum * fac[k];
    }
  }
}

// (ab|cd) for every function of the bra pairs `order` (Hermite order LAB) and every ket function (order LK): a lane
// is a ket function, a workgroup a bra pair and 64 kets, its NW wavefronts share the bra's primitive pairs.  A
// primitive quartet costs a lane the Boys table, R_{tuv} in registers (in place, orders descending: an element of
// level n needs only lower orders of level n + 1) and the ket sum over its Hermite functions; the bra sum follows
// once a bra primitive.  All loops over Hermite indices are unrolled, so R and G stay in registers.
// mode 2: J[mu, r]; 3: (mu nu|r) and (nu mu|r); 4: (mu nu|r s) and its images (also with bra and ket exchanged when
// swap: kets of lower order than the bra are computed once).
// Bound by the latency of the primitive loop where contractions are long, by FP64 arithmetic otherwise.  All launches
// of a call, against one thread per function of the ket with every table in scratch memory: (mu nu|la si) of two water
// molecules in cc-pVDZ (48 functions) 106 -> 0.6 ms, (mu nu|P) of four (96 x 96 x 336) 8.2 -> 0.4 ms.
template <int LAB>
constexpr int eri_waves() { return LAB == 0 ? 16 : LAB == 1 ? 8 : LAB == 2 ? 4 : 2; }
template <int LAB>
constexpr int eri_funcs() { return LAB == 0 ? 1 : LAB == 1 ? 3 : LAB == 2 ? 9 : LAB == 3 ? 18 : 36; }

template <int LAB, int LK>
__global__ __launch_bounds__(64 * eri_waves<LAB>()) void k_eri(
    const int* __restrict__ order, const PairHead* __restrict__ heads, const Ket* __restrict__ kets, int nket,
    int nchunk, int lsub, const double* __restrict__ E, const double* __restrict__ prim, const double* __restrict__ boys, int mode,
    int swap, int64_t n, double* __restrict__ out) {
  constexpr int NW = eri_waves<LAB>(), NF = eri_funcs<LAB>(), NA = nherm(LAB), NK = nherm(LK), L = LAB + LK, NR = nherm(L);
  __shared__ double acc[NW][NF][64];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int bi = blockIdx.x / nchunk, ch = blockIdx.x % nchunk;
  const PairHead hd = heads[order[bi]];
  // 64 >> lsub kets a workgroup; 1 << lsub lanes share a ket's primitive pairs
  const int nk64 = 64 >> lsub, sub = lane >> (6 - lsub);
  const int ki = ch * nk64 + (lane & (nk64 - 1));
  const Ket kt = kets[ki < nket ? ki : nket - 1];
  const int nw = hd.np < NW ? hd.np : NW;
  if (w < nw) {
    for (int f = 0; f < hd.nf; ++f) acc[w][f][lane] = 0.0;
    for (int pp = w; pp < hd.np; pp += NW) {
      const double* pr = prim + 4 * (int64_t)(hd.poff + pp);
      const double p = pr[0], Px = pr[1], Py = pr[2], Pz = pr[3];
      double G[NA];
#pragma unroll
      for (int h = 0; h < NA; ++h) G[h] = 0.0;
      for (int kp = sub; kp < kt.np; kp += 1 << lsub) {
        const double* qr = prim + 4 * (int64_t)(kt.poff + kp);
        const double q = qr[0], X = Px - qr[1], Y = Py - qr[2], Z = Pz - qr[3];
        const double ip = 1.0 / (p + q), al = p * q * ip;
        double F[L + 1], R[NR];
        boys_tab<L>(boys, al * (X * X + Y * Y + Z * Z), F);
        double sc = sqrt(ip);
#pragma unroll
        for (int m = 0; m <= L; ++m) {
          F[m] *= sc;
          sc *= -2.0 * al;
        }
        R[0] = F[L];
        if constexpr (L > 0) herm_levels<L, L - 1>(X, Y, Z, F, R);
        const double* ke = E + kt.eoff + (int64_t)kp * kt.est;
        herm_sum<NA, NK>(ke, R, G);
      }
      for (int x = nk64; x < 64; x *= 2)
#pragma unroll
        for (int h = 0; h < NA; ++h) G[h] += __shfl_xor(G[h], x, 64);
      const double* be = E + hd.eoff + (int64_t)pp * hd.nf * NA;
      for (int f = 0; f < hd.nf; ++f) {
        double s = 0.0;
#pragma unroll
        for (int h = 0; h < NA; ++h) s = fma(be[f * NA + h], G[h], s);
        acc[w][f][lane] += s;
      }
    }
  }
  __syncthreads();
  if (ki >= nket || sub) return;
  const int64_t n2 = n * n, n3 = n2 * n, r = kt.r, s = kt.s;
  for (int f = w; f < hd.nf; f += NW) {
    const int i = f / hd.mb, j = f % hd.mb;
    if (hd.a == hd.b && j > i) continue;   // the image of (j, i)
    double v = 0.0;
    for (int x = 0; x < nw; ++x) v += acc[x][f][lane];
    const int64_t mu = hd.fa + i, nu = hd.fb + j;
    if (mode == 2) {
      out[mu + n * r] = v;
    } else if (mode == 3) {
      out[mu + n * nu + n2 * r] = v;
      out[nu + n * mu + n2 * r] = v;
    } else {
      out[mu + n * nu + n2 * r + n3 * s] = v;
      out[nu + n * mu + n2 * r + n3 * s] = v;
      out[mu + n * nu + n2 * s + n3 * r] = v;
      out[nu + n * mu + n2 * s + n3 * r] = v;
      if (swap) {
        out[r + n * s + n2 * mu + n3 * nu] = v;
        out[s + n * r + n2 * mu + n3 * nu] = v;
        out[r + n * s + n2 * nu + n3 * mu] = v;
        out[s + n * r + n2 * nu + n3 * mu] = v;
      }
    }
  }
}

// transform a Cartesian block acc[ia * nb + ib] of shells (la, lb) and write out[(fa + ma) + sa_ld ...]
// through the callback
template <typename Write>
__device__ void write_block(const SphTab& T, int la, int lb, const double* acc, Write&& wr) {
  const int na = ncart(la), nb = ncart(lb), ma = nfun(T, la), mb = nfun(T, lb);
  for (int i = 0; i < ma; ++i)
    for (int j = 0; j < mb; ++j) {
      double s = 0.0;
      for (int x = 0; x < na; ++x) {
        const double cx = tcoef(T, la, i, x);
        if (cx == 0.0) continue;
        for (int y = 0; y < nb; ++y) s += cx * tcoef(T, lb, j, y) * acc[x * nb + y];
      }
      wr(i, j, s);
    }
}

// one thread per shell pair (i, j): the S, T and V blocks (V over the point charges)
__global__ void k_one_electron(int nshell, const IntShell* __restrict__ sh, const double* __restrict__ ex,
                               const double* __restrict__ cf, int natom, const double* __restrict__ Zc,
                               const double* __restrict__ xyz, SphTab T, int nbf, double* __restrict__ S,
                               double* __restrict__ Tk, double* __restrict__ V) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= nshell * nshell) return;
  const IntShell sa = sh[idx % nshell], sb = sh[idx / nshell];
  const int la = sa.l, lb = sb.l, na = ncart(la), nb = ncart(lb);
  double accS[kMaxCart * kMaxCart], accT[kMaxCart * kMaxCart], accV[kMaxCart * kMaxCart];
  for (int q = 0; q < na * nb; ++q) accS[q] = accT[q] = accV[q] = 0.0;
  double E[3][(kMaxLAux + 1) * (kMaxLAux + 3) * (2 * kMaxLAux + 3)];
  double R[kRSize], Wk[kRSize];
  const int lb2 = lb + 2, nt2 = la + lb2 + 1, L = la + lb;
  for (int pa = 0; pa < sa.nprim; ++pa)
    for (int pb = 0; pb < sb.nprim; ++pb) {
      const double a = ex[sa.poff + pa], b = ex[sb.poff + pb], k = cf[sa.poff + pa] * cf[sb.poff + pb];
      const double p = a + b;
      // E tables up to lb + 2 (the kinetic operator raises the right-hand power by two)
      hermite_E(la, lb2, a, b, sa.x, sb.x, E[0]);
      hermite_E(la, lb2, a, b, sa.y, sb.y, E[1]);
      hermite_E(la, lb2, a, b, sa.z, sb.z, E[2]);
      const double Px = (a * sa.x + b * sb.x) / p, Py = (a * sa.y + b * sb.y) / p, Pz = (a * sa.z + b * sb.z) / p;
      const double sp = sqrt(M_PI / p);
      for (int ia = 0; ia < na; ++ia) {
        int e1[3];
        cart_exps(la, ia, e1[0], e1[1], e1[2]);
        for (int ib = 0; ib < nb; ++ib) {
          int e2[3];
          cart_exps(lb, ib, e2[0], e2[1], e2[2]);
          double s1[3], t1[3];
          for (int d = 0; d < 3; ++d) {
            const int i = e1[d], j = e2[d];
            auto E0 = [&](int jj) { return E[d][(i * (lb2 + 1) + jj) * nt2 + 0] * sp; };
            s1[d] = E0(j);
            const double sm = j >= 2 ? E0(j - 2) : 0.0;
            t1[d] = -0.5 * (j * (j - 1) * sm - 2.0 * b * (2 * j + 1) * s1[d] + 4.0 * b * b * E0(j + 2));
          }
          accS[ia * nb + ib] += k * s1[0] * s1[1] * s1[2];
          accT[ia * nb + ib] += k * (t1[0] * s1[1] * s1[2] + s1[0] * t1[1] * s1[2] + s1[0] * s1[1] * t1[2]);
        }
      }
      for (int at = 0; at < natom; ++at) {
        hermite_R(L, p, Px - xyz[3 * at], Py - xyz[3 * at + 1], Pz - xyz[3 * at + 2], R, Wk);
        const double pre = -Zc[at] * 2.0 * M_PI / p * k;
        for (int ia = 0; ia < na; ++ia) {
          int e1[3];
          cart_exps(la, ia, e1[0], e1[1], e1[2]);
          for (int ib = 0; ib < nb; ++ib) {
            int e2[3];
            cart_exps(lb, ib, e2[0], e2[1], e2[2]);
            const double* ex_ = E[0] + (e1[0] * (lb2 + 1) + e2[0]) * nt2;
            const double* ey_ = E[1] + (e1[1] * (lb2 + 1) + e2[1]) * nt2;
            const double* ez_ = E[2] + (e1[2] * (lb2 + 1) + e2[2]) * nt2;
            double s = 0.0;
            for (int t = 0; t <= e1[0] + e2[0]; ++t)
              for (int u = 0; u <= e1[1] + e2[1]; ++u)
                for (int v = 0; v <= e1[2] + e2[2]; ++v) s += ex_[t] * ey_[u] * ez_[v] * R[tet(t, u, v)];
            accV[ia * nb + ib] += pre * s;
          }
        }
      }
    }
  const int64_t n = nbf;
  write_block(T, la, lb, accS, [&](int i, int j, double v) { S[(sa.foff + i) + n * (sb.foff + j)] = v; });
  write_block(T, la, lb, accT, [&](int i, int j, double v) { Tk[(sa.foff + i) + n * (sb.foff + j)] = v; });
  write_block(T, la, lb, accV, [&](int i, int j, double v) { V[(sa.foff + i) + n * (sb.foff + j)] = v; });
}

// one thread per shell pair (i, j): the dipole integrals <a| r - O |b> (x, y, z) about the origin O,
// <G_i|x - O_x|G_j> = (E^{ij}_1 + (P_x - O_x) E^{ij}_0) sqrt(pi/p) along x times the overlaps along y, z
__global__ void k_dipole(int nshell, const IntShell* __restrict__ sh, const double* __restrict__ ex,
                         const double* __restrict__ cf, double ox, double oy, double oz, SphTab T, int nbf,
                         double* __restrict__ Dx, double* __restrict__ Dy, double* __restrict__ Dz) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= nshell * nshell) return;
  const IntShell sa = sh[idx % nshell], sb = sh[idx / nshell];
  const int la = sa.l, lb = sb.l, na = ncart(la), nb = ncart(lb), nt = la + lb + 1;
  double acc[3][kMaxCart * kMaxCart];
  for (int d = 0; d < 3; ++d)
    for (int q = 0; q < na * nb; ++q) acc[d][q] = 0.0;
  double E[3][(kMaxLAux + 1) * (kMaxLAux + 1) * (2 * kMaxLAux + 1)];
  const double O[3] = {ox, oy, oz}, Ac[3] = {sa.x, sa.y, sa.z}, Bc[3] = {sb.x, sb.y, sb.z};
  for (int pa = 0; pa < sa.nprim; ++pa)
    for (int pb = 0; pb < sb.nprim; ++pb) {
      const double a = ex[sa.poff + pa], b = ex[sb.poff + pb], k = cf[sa.poff + pa] * cf[sb.poff + pb];
      const double p = a + b, sp = sqrt(M_PI / p);
      double P[3];
      for (int d = 0; d < 3; ++d) {
        hermite_E(la, lb, a, b, Ac[d], Bc[d], E[d]);
        P[d] = (a * Ac[d] + b * Bc[d]) / p;
      }
      for (int ia = 0; ia < na; ++ia) {
        int e1[3];
        cart_exps(la, ia, e1[0], e1[1], e1[2]);
        for (int ib = 0; ib < nb; ++ib) {
          int e2[3];
          cart_exps(lb, ib, e2[0], e2[1], e2[2]);
          double s1[3], m1[3];
          for (int d = 0; d < 3; ++d) {
            const double* e = E[d] + (e1[d] * (lb + 1) + e2[d]) * nt;
            s1[d] = e[0] * sp;
            m1[d] = ((e1[d] + e2[d] >= 1 ? e[1] : 0.0) + (P[d] - O[d]) * e[0]) * sp;
          }
          acc[0][ia * nb + ib] += k * m1[0] * s1[1] * s1[2];
          acc[1][ia * nb + ib] += k * s1[0] * m1[1] * s1[2];
          acc[2][ia * nb + ib] += k * s1[0] * s1[1] * m1[2];
        }
      }
    }
  const int64_t n = nbf;
  double* outs[3] = {Dx, Dy, Dz};
  for (int d = 0; d < 3; ++d)
    write_block(T, la, lb, acc[d], [&](int i, int j, double v) { outs[d][(sa.foff + i) + n * (sb.foff + j)] = v; });
}

// ------------------------------------------------------------------ host side
static unsigned blocks_for(int64_t n) { return (unsigned)((n + 127) / 128); }

void integrals_one_electron(hipStream_t s, int nshell, const void* shells, const double* ex, const double* cf,
                            int natom, const double* Z, const double* xyz, const void* tab, int nbf, double* S,
                            double* T, double* V) {
  hipLaunchKernelGGL(k_one_electron, dim3(blocks_for((int64_t)nshell * nshell)), dim3(128), 0, s, nshell,
                     static_cast<const IntShell*>(shells), ex, cf, natom, Z, xyz, *static_cast<const SphTab*>(tab), nbf,
                     S, T, V);
  FH_HIP(hipGetLastError());
}

// ------------------------------------------------------------------ Coulomb integrals: host side
namespace {
// the Boys table: F at the highest order from the series, the others downward
std::vector<double> boys_table() {
  std::vector<double> t((size_t)kBoysRows * kBoysRow);
  for (int k = 0; k < kBoysRows; ++k) {
    const double T = 0.125 * k, eT = std::exp(-T);
    const int N = kBoysRow - 1;
    double term = 1.0 / (2 * N + 1), sum = term;
    for (int m = 1; m < 400 && term > 1e-18 * sum; ++m) {
      term *= 2.0 * T / (2 * N + 2 * m + 1);
      sum += term;
    }
    double* F = t.data() + (size_t)k * kBoysRow;
    F[N] = eT * sum;
    for (int m = N; m > 0; --m) F[m - 1] = (2.0 * T * F[m] + eT) / (2 * m - 1);
  }
  return t;
}

int nfun_host(int l, int spherical) { return spherical ? 2 * l + 1 : (l + 1) * (l + 2) / 2; }

struct EriBuild {
  std::vector<IntShell> sh;
  std::vector<double> ex, cf;
  std::vector<PairHead> heads;
  std::vector<int> order[2 * kMaxLOrb + 1];   // bra pairs of each Hermite order
  std::vector<Ket> kets[2 * kMaxLOrb + 1];
  int64_t ne = 0;
  int nprim = 0;

  int add_basis(const IntBasis& b) {
    const int s0 = (int)sh.size(), p0 = (int)ex.size();
    for (int i = 0; i < b.nshell; ++i)
      sh.push_back({b.l[i], b.nprim[i], p0 + b.poff[i], b.foff[i], b.center[3 * i], b.center[3 * i + 1], b.center[3 * i + 2]});
    ex.insert(ex.end(), b.exps, b.exps + b.nexp);
    cf.insert(cf.end(), b.coefs, b.coefs + b.nexp);
    return s0;
  }
  int add_pair(int a, int b, int spherical) {
    PairHead h{};
    h.l = sh[a].l + (b < 0 ? 0 : sh[b].l);
    h.np = sh[a].nprim * (b < 0 ? 1 : sh[b].nprim);
    h.a = a;
    h.b = b;
    h.fa = sh[a].foff;
    h.fb = b < 0 ? 0 : sh[b].foff;
    h.mb = b < 0 ? 1 : nfun_host(sh[b].l, spherical);
    h.nf = nfun_host(sh[a].l, spherical) * h.mb;
    h.eoff = ne;
    h.poff = nprim;
    ne += (int64_t)h.np * h.nf * nherm(h.l);
    FH_CHECK((int64_t)nprim + h.np < ((int64_t)1 << 31), -3, "integrals: too many primitive pairs");
    nprim += h.np;
    heads.push_back(h);
    return (int)heads.size() - 1;
  }
  void add_kets(int pair) {
    const PairHead& h = heads[pair];
    const int nh = nherm(h.l);
    for (int f = 0; f < h.nf; ++f) {
      const int i = f / h.mb, j = f % h.mb;
      if (h.a == h.b && j > i) continue;
      kets[h.l].push_back({h.eoff + (int64_t)f * nh, h.nf * nh, h.np, h.poff, h.fa + i, h.fb + j, 0});
    }
  }

  // long contractions first: a launch ends with its shortest workgroups, and the lanes of a wavefront have kets of
  // like length
  void sort() {
    for (auto& o : order)
      std::stable_sort(o.begin(), o.end(), [&](int x, int y) { return heads[x].np > heads[y].np; });
    for (auto& k : kets) std::stable_sort(k.begin(), k.end(), [](const Ket& x, const Ket& y) { return x.np > y.np; });
  }
};

template <int LAB, int LK>
void eri_launch(hipStream_t s, const EriBuild& b, const int* order, const PairHead* heads, const Ket* kets,
                const double* E, const double* prim, const double* boys, int mode, int64_t n, double* out) {
  const int64_t nb = (int64_t)b.order[LAB].size(), nk = (int64_t)b.kets[LK].size();
  if (nb == 0 || nk == 0 || (mode == 4 && LAB < LK)) return;
  // lanes that share a ket: with few workgroups the longest contraction sets the time (the (ss|ss) of two water
  // molecules, up to 64 x 64 primitive pairs in 210 workgroups: 559 us with a lane a
  // ket, 85 us so)
  int lsub = 0;
  while (lsub < 5 && (nb * nk << lsub) < 64 * 1024 && (2 << lsub) <= b.kets[LK][0].np) ++lsub;
  const int64_t nch = (nk + (64 >> lsub) - 1) / (64 >> lsub);
  constexpr int NT = 64 * eri_waves<LAB>();
  FH_CHECK(nk < ((int64_t)1 << 31) && nch <= max_workgroups(NT), -3, "integrals: grid too large");
  for_launches(nb, nch, NT, [&](int64_t b0, int64_t m) {
    hipLaunchKernelGGL((k_eri<LAB, LK>), dim3((unsigned)(m * nch)), dim3(NT), 0, s, order + b0, heads, kets, (int)nk, (int)nch,
                       lsub, E, prim, boys, mode, LAB > LK ? 1 : 0, n, out);
    FH_HIP(hipGetLastError());
  });
}

void eri_run(hipStream_t s, Pool* pool, IntScratch& sc, EriBuild& b, const SphTab& tab, int mode, int64_t n, double* out) {
  b.sort();
  static const std::vector<double> boys = boys_table();
  // one upload of all lists
  auto put = [&](const void* p, size_t bytes) {
    const size_t at = (sc.host.size() + 15) / 16 * 16;
    sc.host.resize(at + bytes);
    if (bytes) std::memcpy(sc.host.data() + at, p, bytes);
    return at;
  };
  auto putv = [&](const auto& v) { return put(v.data(), v.size() * sizeof(v[0])); };
  constexpr int NL = 2 * kMaxLOrb + 1;
  const size_t oS = putv(b.sh), oX = putv(b.ex), oC = putv(b.cf), oB = putv(boys), oH = putv(b.heads);
  size_t oO[NL], oK[NL];
  for (int l = 0; l < NL; ++l) {
    oO[l] = putv(b.order[l]);
    oK[l] = putv(b.kets[l]);
  }
  sc.lists = Buf(pool, std::max<size_t>(sc.host.size(), 16));
  FH_HIP(hipMemcpyAsync(sc.lists.p, sc.host.data(), sc.host.size(), hipMemcpyHostToDevice, s));
  sc.tables = Buf(pool, (size_t)(b.ne + 4 * (int64_t)b.nprim) * sizeof(double));
  const char* d = static_cast<const char*>(sc.lists.p);
  const PairHead* heads = reinterpret_cast<const PairHead*>(d + oH);
  double *E = sc.tables.d(), *prim = E + b.ne;
  for_launches((int64_t)b.heads.size(), 1, 256, [&](int64_t h0, int64_t m) {
    hipLaunchKernelGGL(k_pair_e, dim3((unsigned)m), dim3(256), 0, s, heads + h0, reinterpret_cast<const IntShell*>(d + oS),
                       reinterpret_cast<const double*>(d + oX), reinterpret_cast<const double*>(d + oC), tab, E, prim);
    FH_HIP(hipGetLastError());
  });
  const double* bt = reinterpret_cast<const double*>(d + oB);
#define FH_ERI(A_, K_)                                                                                              \
  eri_launch<A_, K_>(s, b, reinterpret_cast<const int*>(d + oO[A_]), heads, reinterpret_cast<const Ket*>(d + oK[K_]), \
                     E, prim, bt, mode, n, out)
#define FH_ERI_BRA(A_) FH_ERI(A_, 0); FH_ERI(A_, 1); FH_ERI(A_, 2); FH_ERI(A_, 3); FH_ERI(A_, 4)
  FH_ERI_BRA(0);
  FH_ERI_BRA(1);
  FH_ERI_BRA(2);
  FH_ERI_BRA(3);
  FH_ERI_BRA(4);
#undef FH_ERI_BRA
#undef FH_ERI
}
}  // namespace

void integrals_eri3c(hipStream_t s, Pool* pool, IntScratch& sc, const IntBasis& b, const IntBasis& aux, const void* tab,
                     double* out) {
  EriBuild e;
  e.add_basis(b);
  const int a0 = e.add_basis(aux);
  for (int i = 0; i < b.nshell; ++i)
    for (int j = 0; j <= i; ++j) {
      const int p = e.add_pair(i, j, b.spherical);
      e.order[e.heads[p].l].push_back(p);
    }
  for (int k = 0; k < aux.nshell; ++k) e.add_kets(e.add_pair(a0 + k, -1, aux.spherical));
  eri_run(s, pool, sc, e, *static_cast<const SphTab*>(tab), 3, b.nbf, out);
}

void integrals_eri2c(hipStream_t s, Pool* pool, IntScratch& sc, const IntBasis& aux, const void* tab, double* out) {
  EriBuild e;
  e.add_basis(aux);
  for (int k = 0; k < aux.nshell; ++k) {
    const int p = e.add_pair(k, -1, aux.spherical);
    e.order[e.heads[p].l].push_back(p);
    e.add_kets(p);
  }
  eri_run(s, pool, sc, e, *static_cast<const SphTab*>(tab), 2, aux.nbf, out);
}

void integrals_eri4c(hipStream_t s, Pool* pool, IntScratch& sc, const IntBasis& b, const void* tab, double* out) {
  EriBuild e;
  e.add_basis(b);
  for (int i = 0; i < b.nshell; ++i)
    for (int j = 0; j <= i; ++j) {
      const int p = e.add_pair(i, j, b.spherical);
      e.order[e.heads[p].l].push_back(p);
      e.add_kets(p);
    }
  eri_run(s, pool, sc, e, *static_cast<const SphTab*>(tab), 4, b.nbf, out);
}

void integrals_dipole(hipStream_t s, int nshell, const void* shells, const double* ex, const double* cf,
                      const double* origin, const void* tab, int nbf, double* Dx, double* Dy, double* Dz) {
  hipLaunchKernelGGL(k_dipole, dim3(blocks_for((int64_t)nshell * nshell)), dim3(128), 0, s, nshell,
                     static_cast<const IntShell*>(shells), ex, cf, origin[0], origin[1], origin[2],
                     *static_cast<const SphTab*>(tab), nbf, Dx, Dy, Dz);
  FH_HIP(hipGetLastError());
}

size_t integrals_shell_bytes() { return sizeof(IntShell); }
size_t integrals_table_bytes() { return sizeof(SphTab); }
int integrals_max_l_orbital() { return kMaxLOrb; }
int integrals_max_l_aux() { return kMaxLAux; }

// host-side packing of one shell / the spherical table (the layouts above)
void integrals_pack_shell(void* dst, int l, int nprim, int poff, int foff, const double* center) {
  IntShell s;
  s.l = l;
  s.nprim = nprim;
  s.poff = poff;
  s.foff = foff;
  s.x = center[0];
  s.y = center[1];
  s.z = center[2];
  std::memcpy(dst, &s, sizeof(s));
}
void integrals_pack_table(void* dst, const double* c /*[4][7][10]*/, int spherical) {
  SphTab t;
  std::memcpy(t.c, c, sizeof(t.c));
  t.spherical = spherical;
  std::memcpy(dst, &t, sizeof(t));
}

}  // namespace fh
