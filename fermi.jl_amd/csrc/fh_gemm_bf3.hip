// Split-BF16x3 GEMM on CDNA4 matrix cores: D = alpha * op(A) * op(B) + beta * C, column-major.
//
// Every FP32 (or FP64) operand x is split when it is staged into LDS into two bfloat16 parts,
// hi = bf16(x) and lo = bf16(x - hi) (both round-to-nearest-even; x - hi is exact in FP32), and
// the product is formed from three bf16 MFMA products with FP32 accumulation:
//     A*B ~= Ahi*Bhi + Ahi*Blo + Alo*Bhi
// (the dropped Alo*Blo term and the rounding of lo leave a relative error of about 2^-16 per
// product; Henry, Tang and Heinecke, "Leveraging the bfloat16 artificial intelligence datatype
// for higher-precision computations", ARITH 2019).  Three v_mfma_f32_32x32x16_bf16 issue in the
// time of 3/16 of the FP32 MFMA work of the same tile.
//
// Workgroup: 256 threads = 4 wavefronts (2x2), BM x 128 output tile (BM = 128, three workgroups per
// CU, or 256 for large untransposed GEMMs, two), K staged BK = 16 at a time through double-buffered
// LDS (hi and lo planes of both operands).
// Each wavefront owns BM/2 x 64 as 32x32 accumulator blocks.  The MFMA is issued with the B tile
// as its first operand, so the accumulator's lane index runs along the rows of D (the output's
// unit-stride axis).  The (T) W build has kernels of its own (fh_triples.hip).
//
// Global loads: k-contiguous operands load four consecutive k per thread (one dwordx4, which needs
// the alignment of an element only); row-contiguous operands load one element per (row, k), coalesced
// across lanes.  The
// loads are branch-free (clamped rows, masks applied at the LDS store).  Tile order: the
// XCD-aware remap and the L2-grouped raster of the FP64/FP32 kernel.
#include "fh_host.h"
#include "fh_internal.h"

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <type_traits>

namespace fh {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

namespace {


// 4 values of an operand, as FP32
struct V4 {
  float x[4];
};

// two FP32 values -> packed (hi, lo) bf16 pairs
__device__ inline void split2(float a, float b, uint32_t& hi, uint32_t& lo) {
  const f32x2 v = {a, b};
  const bf16x2 h = __builtin_convertvector(v, bf16x2);
  uint32_t hb;
  __builtin_memcpy(&hb, &h, 4);
  const float ha = __uint_as_float(hb << 16), hbf = __uint_as_float(hb & 0xffff0000u);
  const f32x2 r = {a - ha, b - hbf};
  const bf16x2 l = __builtin_convertvector(r, bf16x2);
  uint32_t lb;
  __builtin_memcpy(&lb, &l, 4);
  hi = hb;
  lo = lb;
}

// split 2 values and write them to LDS rows (4 bytes per plane)
__device__ inline void put2(uint16_t* hi_plane, uint16_t* lo_plane, int off, float a, float b) {
  uint32_t h, l;
  split2(a, b, h, l);
  *reinterpret_cast<uint32_t*>(hi_plane + off) = h;
  *reinterpret_cast<uint32_t*>(lo_plane + off) = l;
}

// split 4 values and write them to LDS rows (8 bytes per plane)
__device__ inline void put4(uint16_t* hi_plane, uint16_t* lo_plane, int off, const V4& v) {
  uint32_t h0, l0, h1, l1;
  split2(v.x[0], v.x[1], h0, l0);
  split2(v.x[2], v.x[3], h1, l1);
  *reinterpret_cast<uint2*>(hi_plane + off) = make_uint2(h0, h1);
  *reinterpret_cast<uint2*>(lo_plane + off) = make_uint2(l0, l1);
}

// split 8 values (k-consecutive) and write them to LDS rows (16 bytes per plane)
__device__ inline void put8(uint16_t* hi_plane, uint16_t* lo_plane, int off, const V4& a, const V4& b) {
  uint32_t h0, l0, h1, l1, h2, l2, h3, l3;
  split2(a.x[0], a.x[1], h0, l0);
  split2(a.x[2], a.x[3], h1, l1);
  split2(b.x[0], b.x[1], h2, l2);
  split2(b.x[2], b.x[3], h3, l3);
  *reinterpret_cast<uint4*>(hi_plane + off) = make_uint4(h0, h1, h2, h3);
  *reinterpret_cast<uint4*>(lo_plane + off) = make_uint4(l0, l1, l2, l3);
}

// f(integral_constant I, integral_constant J) for I < MI, J < NJ (row-major), every index a constant
template <int I, int J, int MI, int NJ, typename F>
__device__ __forceinline__ void for_blocks(F&& f) {
  f(std::integral_constant<int, I>{}, std::integral_constant<int, J>{});
  if constexpr (J + 1 < NJ) for_blocks<I, J + 1, MI, NJ>(f);
  else if constexpr (I + 1 < MI) for_blocks<I + 1, 0, MI, NJ>(f);
}

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
__device__ inline V4 load4(const float* p) {
  const f32x4u q = *reinterpret_cast<const f32x4u*>(p);
  return V4{{q[0], q[1], q[2], q[3]}};
}

}  // namespace

// Operand tile layout in LDS: plane[row][k] (k fastest, BK + 8 bf16 per row: 16 bytes of padding),
// row = m for A, n for B.  "row-contiguous" operands (A with TA = false, B with TB = true) are
// read 4 rows x BK/8 k per thread and transposed in registers; "k-contiguous" operands are read
// 4 k of one row per load.
template <int BK, bool TA, bool TB, int TAG, typename TI, typename TO, int BM>
__global__ __launch_bounds__(256, BM == 128 ? 3 : 2) void k_gemm_bf3(int64_t M, int64_t N, int64_t K, double alpha,
                                                     const TI* __restrict__ A, int64_t lda, int64_t sA,
                                                     const TI* __restrict__ B, int64_t ldb, int64_t sB, double beta,
                                                     const TO* C, int64_t ldc, int64_t sC, TO* D, int64_t ldd,
                                                     int64_t sD, int tilesM, int tilesN, int64_t kchunk, int gn) {
  constexpr int BN = 128;        // tile width
  constexpr int kRow = BK + 8;   // LDS row (bf16)
  constexpr int KG = BK / 8;      // k per thread (row-contiguous) = loads per thread (both patterns)
  constexpr int KQ = BK / 4;      // 4-wide k groups (k-contiguous)
  constexpr int RS = 256 / KQ;    // row step (k-contiguous)
  constexpr int NJ = BN / 64;     // 32-wide accumulator blocks per wavefront along N
  constexpr int LB = BN * BK / 1024;  // B loads per thread (k-contiguous)
  constexpr int KL = KG > LB ? KG : LB;
  // BM = 256: each wavefront owns 128 rows (four 32-row blocks); row-contiguous A only
  static_assert(BM == 128 || (BM == 256 && !TA), "256-row tiles take a row-contiguous A");
  constexpr int MI = BM / 64;            // 32-row accumulator blocks per wavefront
  constexpr int RPT = 256 / BM;          // threads per A row (row-contiguous A)
  constexpr int NCH = BK / 8 / RPT;      // 8-wide k chunks per thread (row-contiguous A)
  constexpr int KGA = TA ? KG : 2 * NCH; // 4-value groups of A per thread
  __shared__ __attribute__((aligned(16))) uint16_t As[2][2][BM * kRow];  // [buf][hi/lo]
  __shared__ __attribute__((aligned(16))) uint16_t Bs[2][2][BN * kRow];

  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int wm = wid & 1, wn = wid >> 1;

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
  auto aptr = [&](int64_t gm, int64_t gk) { return TA ? A + gk + lda * gm : A + gm + lda * gk; };
  auto bptr = [&](int64_t gn_, int64_t gk) { return TB ? B + gn_ + ldb * gk : B + gk + ldb * gn_; };

  // per-thread load coordinates
  // row-contiguous pattern: rows (tid&31) + 32 i (i < 4), k KG*(tid>>5)..+KG-1; one scalar load
  //   per (row, k), coalesced across the lanes, and the LDS stores of consecutive lanes land on
  //   consecutive rows (a row stride of 4 rows would put every lane on the same few banks)
  // k-contiguous pattern:  k 4*(tid%KQ)..+3, rows tid/KQ + RS j, j < LB
  // The loads are branch-free: an element outside the operand is read at a clamped, valid
  // address and replaced by zero, so that the loads of a
  // tile issue back to back.  A k tile entirely inside K (all but the last) skips the k tests.
  // operand values of the next k tile, loaded while the current one is multiplied
  V4 ra_s[KGA], rb_s[KL];
  // zero x unless in (a mask, not a select: the compiler keeps the load unconditional)
  auto keep = [](float x, bool in) { return __uint_as_float(__float_as_uint(x) & (in ? 0xffffffffu : 0u)); };
  auto ld1 = [&](const TI* p, bool in) { return keep((float)*p, in); };
  // 4 consecutive k of row/column r of an operand, k-contiguous (p at k gk; rin: row inside)
  auto ld4 = [&](auto ptr, int64_t r, bool rin, int64_t gk) {
    V4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool in = rin && gk + e < K;
      v.x[e] = ld1(ptr(in ? r : 0, in ? gk + e : 0), in);
    }
    return v;
  };
  // Addressing hoisted out of the k loop: the thread's rows, clamped into the operand (an
  // outside row reads a valid element and is zeroed), as offsets from the tile's first row
  // (row-contiguous) or as column offsets (k-contiguous).  A full k tile then costs one pointer
  // per k column (row-contiguous) or per row (k-contiguous) and an add per element.
  constexpr int NA = TA ? KG : 1, NB = TB ? 1 : LB;
  // row-contiguous: the thread's row (M, N < 2^31, checked at launch); k-contiguous: ld * row
  int arow = 0, brow = 0;
  int64_t aoff[TA ? KG : 1], boff[TB ? 1 : LB];
  bool ain[NA], bin[NB];
  if (!TA) {
    const int64_t r = m0 + (tid % BM);
    ain[0] = r < M;
    arow = (int)(ain[0] ? r : M - 1);
  } else {
#pragma unroll
    for (int j = 0; j < KG; ++j) {
      const int64_t r = m0 + tid / KQ + RS * j;
      ain[j] = r < M;
      aoff[j] = lda * (ain[j] ? r : M - 1);
    }
  }
  if (TB) {
    const int64_t r = n0 + (tid & 127);
    bin[0] = r < N;
    brow = (int)(bin[0] ? r : N - 1);
  } else {
#pragma unroll
    for (int j = 0; j < LB; ++j) {
      const int64_t r = n0 + tid / KQ + RS * j;
      bin[j] = r < N;
      boff[j] = ldb * (bin[j] ? r : N - 1);
    }
  }
  // row-contiguous pattern: row tid & 127 of the tile, 8-wide k chunks kc0 + 2 q (q < BK / 16):
  // kc0 = tid >> 7 is the same for a whole wavefront, so a chunk's column pointer and
  // stride are uniform, the loads of one k are coalesced across the lanes' consecutive rows, and
  // each lane stores 16 contiguous bytes per plane to LDS
  const int kc0 = tid >> 7;
  // row-contiguous A: row tid % BM, 8-wide k chunks kca + RPT q (q < NCH)
  const int kca = tid / BM;
  // a k tile inside K; the values of
  // outside rows are zeroed when the tile is stored to LDS (sstore), after the MFMAs of the
  // current tile, so that the loads stay in flight meanwhile
  auto gload_full = [&](int64_t k0, V4* ra, V4* rb) {
    if (!TA) {
#pragma unroll
      for (int q = 0; q < NCH; ++q) {
        const int64_t gk = k0 + 8 * (kca + RPT * q);
        const TI* cp = A + lda * gk + arow;
#pragma unroll
        for (int e = 0; e < 8; ++e) ra[2 * q + (e >> 2)].x[e & 3] = (float)cp[lda * e];
      }
    } else {
      const int64_t gk = k0 + 4 * (tid % KQ);
#pragma unroll
      for (int j = 0; j < KG; ++j) ra[j] = load4(A + aoff[j] + gk);
    }
    if (TB) {
#pragma unroll
      for (int q = 0; q < BK / 16; ++q) {
        const int64_t gk = k0 + 8 * (kc0 + 2 * q);
        const TI* rp = B + ldb * gk + brow;
#pragma unroll
        for (int e = 0; e < 8; ++e) rb[2 * q + (e >> 2)].x[e & 3] = (float)rp[ldb * e];
      }
    } else {
      const int64_t gk = k0 + 4 * (tid % KQ);
#pragma unroll
      for (int j = 0; j < LB; ++j) rb[j] = load4(B + boff[j] + gk);
    }
  };
  // the last, partial k tile: every element checked
  auto gload_part = [&](int64_t k0, V4* ra, V4* rb) {
    if (!TA) {
#pragma unroll
      for (int q = 0; q < NCH; ++q)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int64_t gk = k0 + 8 * (kca + RPT * q) + e;
          const bool kin = gk < K;
          ra[2 * q + (e >> 2)].x[e & 3] = ld1(aptr(0, kin ? gk : 0) + arow, kin);
        }
    } else {
      const int64_t gk = k0 + 4 * (tid % KQ);
#pragma unroll
      for (int j = 0; j < KG; ++j) {
        const int64_t gm = m0 + tid / KQ + RS * j;
        ra[j] = ld4(aptr, gm, gm < M, gk);
      }
    }
    if (TB) {
#pragma unroll
      for (int q = 0; q < BK / 16; ++q)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int64_t gk = k0 + 8 * (kc0 + 2 * q) + e;
          const bool kin = gk < K;
          rb[2 * q + (e >> 2)].x[e & 3] = ld1(bptr(0, kin ? gk : 0) + brow, kin);
        }
    } else {
      const int64_t gk = k0 + 4 * (tid % KQ);
#pragma unroll
      for (int j = 0; j < LB; ++j) {
        const int64_t gcol = n0 + tid / KQ + RS * j;
        rb[j] = ld4(bptr, gcol, gcol < N, gk);
      }
    }
  };
  auto gload = [&](int64_t k0, V4* ra, V4* rb) {
    if (k0 + BK <= K) gload_full(k0, ra, rb);
    else gload_part(k0, ra, rb);
  };
  // r[2q], r[2q+1] = X[row tid & 127][k 8 (kc0 + 2q) .. +7]
  auto put_rows = [&](uint16_t* hi, uint16_t* lo, const V4* r) {
#pragma unroll
    for (int q = 0; q < BK / 16; ++q) put8(hi, lo, (tid & 127) * kRow + 8 * (kc0 + 2 * q), r[2 * q], r[2 * q + 1]);
  };
  auto put_rows_a = [&](uint16_t* hi, uint16_t* lo, const V4* r) {
#pragma unroll
    for (int q = 0; q < NCH; ++q)
      put8(hi, lo, (tid % BM) * kRow + 8 * (kca + RPT * q), r[2 * q], r[2 * q + 1]);
  };
  auto put_k = [&](uint16_t* hi, uint16_t* lo, const V4* r, int nl) {
#pragma unroll
    for (int j = 0; j < KL; ++j)
      if (j < nl) put4(hi, lo, (tid / KQ + RS * j) * kRow + 4 * (tid % KQ), r[j]);
  };
  auto sstore = [&](int buf, V4* ra, V4* rb) {
    // zero the values of rows outside the operand (loaded from a clamped address)
    if (!TA) {
#pragma unroll
      for (int j = 0; j < KGA; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) ra[j].x[i] = keep(ra[j].x[i], ain[0]);
    } else {
#pragma unroll
      for (int j = 0; j < KG; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) ra[j].x[e] = keep(ra[j].x[e], ain[j]);
    }
    if (TB) {
#pragma unroll
      for (int j = 0; j < KG; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) rb[j].x[i] = keep(rb[j].x[i], bin[0]);
    } else {
#pragma unroll
      for (int j = 0; j < LB; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) rb[j].x[e] = keep(rb[j].x[e], bin[j]);
    }
    if (!TA) put_rows_a(As[buf][0], As[buf][1], ra);
    else put_k(As[buf][0], As[buf][1], ra, KG);
    if constexpr (TB) put_rows(Bs[buf][0], Bs[buf][1], rb);
    else put_k(Bs[buf][0], Bs[buf][1], rb, LB);
  };

  // element e of the lane in block (i, j): row (l & 31), column 8 (e >> 2) + 4 (l >> 5) + (e & 3) of the block
  auto elem = [&](int i, int j, int e, int64_t& row, int64_t& col) {
    row = m0 + wm * (BM / 2) + i * 32 + (lane & 31);
    col = n0 + wn * (BN / 2) + j * 32 + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
    return row < M && col < N;
  };
  f32x16 acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  const int64_t nst = (K + BK - 1) / BK;
  const int frow = lane & 31, fk = 8 * (lane >> 5);
  // the MFMAs of the k tile in LDS buffer buf
  auto compute = [&](int buf) {
#pragma unroll
    for (int kk = 0; kk < BK / 16; ++kk) {
      bf16x8 ah[MI], al[MI], bh[NJ], bl[NJ];
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const int off = (wm * (BM / 2) + i * 32 + frow) * kRow + kk * 16 + fk;
        ah[i] = *reinterpret_cast<const bf16x8*>(&As[buf][0][off]);
        al[i] = *reinterpret_cast<const bf16x8*>(&As[buf][1][off]);
      }
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const int off = (wn * (BN / 2) + j * 32 + frow) * kRow + kk * 16 + fk;
        bh[j] = *reinterpret_cast<const bf16x8*>(&Bs[buf][0][off]);
        bl[j] = *reinterpret_cast<const bf16x8*>(&Bs[buf][1][off]);
      }
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          // B fragment as the first MFMA operand, so the accumulator lanes run along M
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bl[j], ah[i], acc[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bh[j], al[i], acc[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bh[j], ah[i], acc[i][j], 0, 0, 0);
        }
    }
  };
  gload(0, ra_s, rb_s);
  sstore(0, ra_s, rb_s);
  __syncthreads();
  for (int64_t s = 0; s < nst; ++s) {
    const int buf = s & 1;
    if (s + 1 < nst) gload((s + 1) * BK, ra_s, rb_s);
    compute(buf);
    if (s + 1 < nst) sstore(buf ^ 1, ra_s, rb_s);
    __syncthreads();
  }

  // epilogue (FP64 output).  With beta != 0 (C may alias D: in-place accumulation), per half block the
  // thread's 8 values of C are loaded (unconditionally, an element outside D reading C[0]) before the 8
  // stores, so the loads overlap instead of each waiting behind the previous store.
  for_blocks<0, 0, MI, NJ>([&](auto ii, auto jj) {
    constexpr int i = decltype(ii)::value, j = decltype(jj)::value;
    if (beta != 0.0) {
#pragma unroll
      for (int h = 0; h < 16; h += 8) {
        int64_t row[8], col[8];
        bool in[8];
        TO cv[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) in[e] = elem(i, j, h + e, row[e], col[e]);
#pragma unroll
        for (int e = 0; e < 8; ++e) cv[e] = C[in[e] ? row[e] + ldc * col[e] : 0];
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (in[e]) D[row[e] + ldd * col[e]] = (TO)(alpha * (double)acc[i][j][h + e] + beta * (double)cv[e]);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        int64_t row, col;
        if (elem(i, j, e, row, col)) D[row + ldd * col] = (TO)(alpha * (double)acc[i][j][e]);
      }
    }
  });
}

// L2 budget of the B blocks of one raster group (bytes; 1, 4 and 16 MB measured alike)
static constexpr int64_t kGroupBytesBf3 = 1 << 20;

// Tile height: 256 (each wavefront 128 rows: fewer LDS fragment reads and operand bytes per MFMA) for the PP ladder
// (272 vs 241 TFLOP/s at o = 40, v = 190) and for other NN GEMMs with M >= 1024 (the o^3 v^3 ring contractions of the
// residual, K = o v: 188 against 174 TFLOP/s at o = 40, v = 190), where two workgroups a CU are there to run; 128
// otherwise (the ladder at o = 28, v = 133, 140 tiles of 256 726 us, 560 of 128 704).  FERMIHIP_BF3_LBM / _CBM = 128 or 256 fix it for
// tags 1 / 0 (tuning).  Under 384 tiles of 128, K is cut into slices of at least 512 towards three workgroups a CU
// ((784, 3724, 17689), 210 tiles: 1.04 ms uncut, 0.49 ms in three slices).
struct Bf3Plan {
  int bm;
  int64_t slices;
};
static Bf3Plan bf3_plan(bool ta, bool tb, int tag, int64_t M, int64_t N, int64_t K, int64_t batch) {
  const bool can = !ta && !tb && (tag == 1 || M >= 1024);
  const int64_t tn = (N + 127) / 128;
  int bm = can && (M + 255) / 256 * tn * batch >= 512 ? 256 : 128;
  if (const char* env = std::getenv(tag == 1 ? "FERMIHIP_BF3_LBM" : "FERMIHIP_BF3_CBM"))
    bm = std::atoi(env) == 256 && can ? 256 : 128;
  const int64_t tiles = (M + bm - 1) / bm * tn * batch;
  const int64_t sl = bm == 256 || tiles >= 384 ? 1 : std::min<int64_t>(768 / tiles, K / 512);
  return {bm, std::max<int64_t>(1, sl)};
}
int64_t gemm_bf3_splitk_elems(bool ta, bool tb, int64_t M, int64_t N, int64_t K, int64_t batch, int tag) {
  if (M <= 0 || N <= 0 || batch <= 0) return 0;
  const int64_t sl = bf3_plan(ta, tb, tag, M, N, K, batch).slices;
  return sl > 1 ? sl * M * N * batch : 0;
}

template <bool TA, bool TB, int TAG, typename TI, typename TO>
static void launch_bf3(hipStream_t s, int bm, int64_t M, int64_t N, int64_t K, double alpha, const TI* A, int64_t lda,
                       int64_t sA, const TI* B, int64_t ldb, int64_t sB, double beta, const TO* C, int64_t ldc,
                       int64_t sC, TO* D, int64_t ldd, int64_t sD, int64_t batch, int64_t kchunk) {
  const int64_t tm = (M + bm - 1) / bm, tn = (N + 127) / 128;
  FH_CHECK(tm * tn <= max_workgroups(256) && batch < 65536, -3, "gemm grid too large");
  FH_CHECK(M < ((int64_t)1 << 31) && N < ((int64_t)1 << 31), -3, "gemm: M and N must be below 2^31");
  dim3 grid((unsigned)(tm * tn), (unsigned)batch, (unsigned)(kchunk > 0 ? (K + kchunk - 1) / kchunk : 1));
  int gn = 0;
  if (M > N) {
    const int64_t per = std::max<int64_t>(1, (kchunk > 0 ? kchunk : K) * 128 * (int64_t)sizeof(TI));
    gn = (int)std::max<int64_t>(1, std::min<int64_t>(tn, kGroupBytesBf3 / per));
  }
#define FH_BF3_GO(BM_)                                                                                              \
  hipLaunchKernelGGL((k_gemm_bf3<16, TA, TB, TAG, TI, TO, BM_>), grid, dim3(256), 0, s, M, N, K, alpha, A, lda, sA, B, \
                     ldb, sB, beta, C, ldc, sC, D, ldd, sD, (int)tm, (int)tn, kchunk, gn)
  if constexpr (!TA && !TB) {
    if (bm == 256) FH_BF3_GO(256); else FH_BF3_GO(128);
  } else {
    FH_BF3_GO(128);
  }
#undef FH_BF3_GO
  FH_HIP(hipGetLastError());
}

void gemm_bf3(hipStream_t s, bool ta, bool tb, int64_t M, int64_t N, int64_t K, double alpha, const float* A,
              int64_t lda, int64_t sA, const float* B, int64_t ldb, int64_t sB, double beta, const double* C, int64_t ldc,
              double* D, int64_t ldd, int64_t sD, int64_t batch, int tag, double* work, int64_t work_elems) {
  if (M <= 0 || N <= 0 || batch <= 0) return;
  FH_CHECK(K >= 0, -3, "gemm: negative K");
  FH_CHECK(lda >= (ta ? (K > 0 ? K : 1) : M) && ldb >= (tb ? N : (K > 0 ? K : 1)) && ldd >= M, -3,
           "gemm: leading dimension too small");
  FH_CHECK(beta == 0.0 || (C != nullptr && ldc >= M), -3, "gemm: C missing");
  FH_CHECK(tag != 1 || (!ta && !tb), -3, "gemm_bf3: the PP ladder (tag 1) takes untransposed operands");
  const Bf3Plan plan = bf3_plan(ta, tb, tag, M, N, K, batch);
  const bool split = plan.slices > 1 && work != nullptr && work_elems >= plan.slices * M * N * batch;
  const int64_t kchunk = split ? (K + plan.slices - 1) / plan.slices : 0;
#define FH_BF3(TA_, TB_, TAG_)                                                                                       \
  launch_bf3<TA_, TB_, TAG_, float, double>(s, plan.bm, M, N, K, split ? 1.0 : alpha, A, lda, sA, B, ldb, sB,        \
                                            split ? 0.0 : beta, split ? nullptr : C, ldc, sD, split ? work : D,      \
                                            split ? M : ldd, split ? M * N : sD, batch, kchunk)
  if (tag == 1) {
    FH_BF3(false, false, 1);
  } else if (ta) {
    if (tb) FH_BF3(true, true, 0); else FH_BF3(true, false, 0);
  } else {
    if (tb) FH_BF3(false, true, 0); else FH_BF3(false, false, 0);
  }
#undef FH_BF3
  if (split)
    splitk_reduce_f64(s, M, N, (K + kchunk - 1) / kchunk, work, alpha, beta, C, ldc, sD, D, ldd, sD, batch);
}

}  // namespace fh
