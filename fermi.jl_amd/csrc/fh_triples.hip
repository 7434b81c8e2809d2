// The (T) W build (ijk.jl:108-115 / ijk2.jl:109-153) on CDNA4 matrix cores.
//
// For an occupied triple (i, j, k) the six permutation classes are products of AV_n, rows (x, y), with
// Bcat_{p,q}, columns z, over k = d' (v virtuals, then o occupieds, padded with zeros to nd, a multiple of
// 8), all accumulating into one W[a, b, c]:
//   first launch   abc: AV_j[(a,b)] Bcat_{i,k}[c]  + bac: AVs_i[(a,b)] Bcat_{j,k}[c]
//                  one GEMM per run of k with M = v^2 rows (a, b) and N = v nk columns (c, k);
//   slice launch   with c fixed the other four are GEMMs with rows a and columns b (K = 4 nd):
//                  cab: AVs_i[(a,c)] Bcat_{k,j}[b] + cba: Bcat_{k,i}[a] AVs_j[(b,c)]
//                  acb: AV_k[(a,c)] Bcat_{i,j}[b]  + bca: Bcat_{j,i}[a] AV_k[(b,c)].
// So W is written once and read and written once more per chunk of triples.  An (a, b) plane of W lies in panels of 8
// a, [a / 8][b][a % 8] with a up to a multiple of 8 (triples_plane elements, the rows beyond v unused).  The rows
// (x, y) of AV and AVs lie likewise, their last panel v % 8 wide, so that the first launch's rows are the plane's
// elements in order and v^2 in number (rows up to the multiple of 8 cost v = 76 in FP64 1.2 % of the (T)).  The energy
// kernel
// then copies the 8 x 8 elements of a cube's plane as one run of whole cache lines (rows of 8 a, a quarter of a line
// each, with a fastest over all of v), and the slice launch adds to 4 a of a column at a time.  Bcat is kept as BVp (blocks
// (p, q) with p fastest) and BVq (q fastest), AV as rows (x, y) and AVs as rows (y, x).
//
// Operand layout: the k of a row are cut into groups of 8 (32 bytes, 64 for FP64), stored group-major, [group]
// [row]: a k step of 64 bytes of 16 rows is one or two contiguous runs, whole cache lines.  Row-major
// operands (64 bytes of a 128-byte line per step) had the L1 wait for lines still in flight in 68% of its
// cycles (TCP_PENDING_STALL_CYCLES) and moved every line twice.
//
// A chunk holds many (i, j) pairs: the W slots of its triples, the column tiles of its runs of k and the
// energy kernel's runs come from device tables, so one launch carries the whole chunk.  A launch per pair
// leaves a partial last round of workgroups on every pair (630 tiles on 512 places at o = 27, v = 131).
//
// Operand tiles are copied straight into a ring of LDS slots (buffer_load ... lds, 16 bytes per lane, lane l
// writing 16 l bytes past the wave-uniform LDS address), which costs no registers; a copy instruction carries
// a piece of 16 rows x 64 bytes.  The ring keeps two k steps in flight behind an explicit vector-memory wait
// and one barrier per step.
#include "fh_host.h"
#include "fh_internal.h"

#include <algorithm>
#include <cstdlib>
#include <type_traits>

namespace fh {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lds_vptr;

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 16, "vmcnt immediate");
  __builtin_amdgcn_s_waitcnt(N | (0x7 << 4) | (0xF << 8));
}
__device__ __forceinline__ void wait_vmcnt_n(int n) {  // n uniform, 0 .. 6
  if (n == 6) {  // whole 192 x 192 tiles
    wait_vmcnt<6>();
    return;
  }
  switch (n) {
    case 0: wait_vmcnt<0>(); break;
    case 1: wait_vmcnt<1>(); break;
    case 2: wait_vmcnt<2>(); break;
    case 3: wait_vmcnt<3>(); break;
    case 4: wait_vmcnt<4>(); break;
    case 5: wait_vmcnt<5>(); break;
    default: wait_vmcnt<6>(); break;
  }
}

// workgroup barrier after this wave's LDS accesses have completed (gfx950 barriers do not wait for
// them, and the compiler adds no wait before a bare s_barrier); the operand copies keep flying
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_s_waitcnt(0xF | (0x7 << 4) | (0x0 << 8) | (0x3 << 14));
  __builtin_amdgcn_s_barrier();
}

__device__ __forceinline__ unsigned lds_addr(const void* p) { return (unsigned)(uintptr_t)(lds_vptr)(p); }

// a buffer resource over a uniform base (taken from the first lane, so that it stays in scalar registers)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t uniform_rsrc(const char* p, int bytes = 0x7fffffff) {
  const uint64_t u = reinterpret_cast<uint64_t>(p);
  const uint64_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)u);
  const uint64_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(u >> 32));
  return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(lo | (hi << 32)), (short)0, bytes, 0x00020000);
}

// Fragment reads of a k step: MI + NJ blocks of 32 rows (2048 bytes apart), two 16-byte reads each: hi at pa / pb,
// lo at qa = pa ^ 16 / qb = pb ^ 16.  The compiler counts the operand copies as vector-memory operations and, unable to tell the ring
// slots apart, would wait for every copy in flight before an ordinary LDS read; these reads carry their own
// LDS wait, and their outputs are early-clobber so that no destination shares an address register while a
// read is in flight.
#define FH_RD(n, base, off) "ds_read_b128 %[" #n "], %[" #base "] offset:" #off "\n\t"
#define FH_A1 FH_RD(a0, pa, 0) FH_RD(a1, qa, 0)
#define FH_A2 FH_A1 FH_RD(a2, pa, 2048) FH_RD(a3, qa, 2048)
#define FH_A3 FH_A2 FH_RD(a4, pa, 4096) FH_RD(a5, qa, 4096)
#define FH_B1 FH_RD(b0, pb, 0) FH_RD(b1, qb, 0)
#define FH_B2 FH_B1 FH_RD(b2, pb, 2048) FH_RD(b3, qb, 2048)
#define FH_B3 FH_B2 FH_RD(b4, pb, 4096) FH_RD(b5, qb, 4096)
#define FH_OA1 [a0] "=&v"(fa[0][0]), [a1] "=&v"(fa[0][1])
#define FH_OA2 FH_OA1, [a2] "=&v"(fa[1][0]), [a3] "=&v"(fa[1][1])
#define FH_OA3 FH_OA2, [a4] "=&v"(fa[2][0]), [a5] "=&v"(fa[2][1])
#define FH_OB1 [b0] "=&v"(fb[0][0]), [b1] "=&v"(fb[0][1])
#define FH_OB2 FH_OB1, [b2] "=&v"(fb[1][0]), [b3] "=&v"(fb[1][1])
#define FH_OB3 FH_OB2, [b4] "=&v"(fb[2][0]), [b5] "=&v"(fb[2][1])
#define FH_READ(mi, nj)                                                                                        \
  if constexpr (MI == mi && NJ == nj)                                                                          \
    asm volatile(FH_A##mi FH_B##nj "s_waitcnt lgkmcnt(0)" : FH_OA##mi, FH_OB##nj : [pa] "v"(a), [qa] "v"(a ^ 16u), [pb] "v"(b), [qb] "v"(b ^ 16u) : "memory")
template <int MI, int NJ>
__device__ __forceinline__ void read_frags(unsigned a, unsigned b, f32x4 (&fa)[MI][2], f32x4 (&fb)[NJ][2]) {
  FH_READ(1, 1); FH_READ(1, 2); FH_READ(1, 3);
  FH_READ(2, 1); FH_READ(2, 2); FH_READ(2, 3);
  FH_READ(3, 1); FH_READ(3, 2); FH_READ(3, 3);
}
#undef FH_READ

// one 16-byte read of the wave's A block and one per B block, block stride 1024
#define FH_Q(j, off) FH_RD(b##j, pb, off)
#define FH_QO(j) [b##j] "=&v"(fb[j])
template <int NB>
__device__ __forceinline__ void read_rows(unsigned a, unsigned b, f32x4& fa, f32x4 (&fb)[NB]) {
  if constexpr (NB == 2)
    asm volatile(FH_RD(a0, pa, 0) FH_Q(0, 0) FH_Q(1, 1024) "s_waitcnt lgkmcnt(0)"
                 : [a0] "=&v"(fa), FH_QO(0), FH_QO(1) : [pa] "v"(a), [pb] "v"(b) : "memory");
  if constexpr (NB == 3)
    asm volatile(FH_RD(a0, pa, 0) FH_Q(0, 0) FH_Q(1, 1024) FH_Q(2, 2048) "s_waitcnt lgkmcnt(0)"
                 : [a0] "=&v"(fa), FH_QO(0), FH_QO(1), FH_QO(2) : [pa] "v"(a), [pb] "v"(b) : "memory");
  if constexpr (NB == 4)
    asm volatile(FH_RD(a0, pa, 0) FH_Q(0, 0) FH_Q(1, 1024) FH_Q(2, 2048) FH_Q(3, 3072) "s_waitcnt lgkmcnt(0)"
                 : [a0] "=&v"(fa), FH_QO(0), FH_QO(1), FH_QO(2), FH_QO(3) : [pa] "v"(a), [pb] "v"(b) : "memory");
  if constexpr (NB == 5)
    asm volatile(FH_RD(a0, pa, 0) FH_Q(0, 0) FH_Q(1, 1024) FH_Q(2, 2048) FH_Q(3, 3072) FH_Q(4, 4096)
                 "s_waitcnt lgkmcnt(0)"
                 : [a0] "=&v"(fa), FH_QO(0), FH_QO(1), FH_QO(2), FH_QO(3), FH_QO(4) : [pa] "v"(a), [pb] "v"(b) : "memory");
  if constexpr (NB == 6)
    asm volatile(FH_RD(a0, pa, 0) FH_Q(0, 0) FH_Q(1, 1024) FH_Q(2, 2048) FH_Q(3, 3072) FH_Q(4, 4096) FH_Q(5, 5120)
                 "s_waitcnt lgkmcnt(0)"
                 : [a0] "=&v"(fa), FH_QO(0), FH_QO(1), FH_QO(2), FH_QO(3), FH_QO(4), FH_QO(5)
                 : [pa] "v"(a), [pb] "v"(b) : "memory");
}

// the same for NB = 5 and 6 with the wave's extra blocks: one more A block at a2, and one (three) B blocks at b2
template <int NB>
__device__ __forceinline__ void read_rows_extra(unsigned a, unsigned b, unsigned a2, unsigned b2, f32x4& fa, f32x4 (&fb)[NB],
                                                f32x4& fx, f32x4 (&fy)[NB == 6 ? 3 : 1]) {
#define FH_X FH_RD(x, px, 0) FH_RD(y0, py, 0)
#define FH_XO [x] "=&v"(fx), [y0] "=&v"(fy[0])
#define FH_I [pa] "v"(a), [pb] "v"(b), [px] "v"(a2), [py] "v"(b2)
  if constexpr (NB == 5)
    asm volatile(FH_RD(a0, pa, 0) FH_Q(0, 0) FH_Q(1, 1024) FH_Q(2, 2048) FH_Q(3, 3072) FH_Q(4, 4096) FH_X
                 "s_waitcnt lgkmcnt(0)"
                 : [a0] "=&v"(fa), FH_QO(0), FH_QO(1), FH_QO(2), FH_QO(3), FH_QO(4), FH_XO : FH_I : "memory");
  if constexpr (NB == 6)
    asm volatile(FH_RD(a0, pa, 0) FH_Q(0, 0) FH_Q(1, 1024) FH_Q(2, 2048) FH_Q(3, 3072) FH_Q(4, 4096) FH_Q(5, 5120)
                 FH_X FH_RD(y1, py, 1024) FH_RD(y2, py, 2048) "s_waitcnt lgkmcnt(0)"
                 : [a0] "=&v"(fa), FH_QO(0), FH_QO(1), FH_QO(2), FH_QO(3), FH_QO(4), FH_QO(5), FH_XO,
                   [y1] "=&v"(fy[NB == 6 ? 1 : 0]), [y2] "=&v"(fy[NB == 6 ? 2 : 0]) : FH_I : "memory");
#undef FH_X
#undef FH_XO
#undef FH_I
}

// two FP32 values -> packed (hi, lo) bf16 pairs, hi = bf16(x), lo = bf16(x - hi)
__device__ inline void split2(float a, float b, uint32_t& hi, uint32_t& lo) {
  const f32x2 v = {a, b};
  const bf16x2 h = __builtin_convertvector(v, bf16x2);
  __builtin_memcpy(&hi, &h, 4);
  const f32x2 r = {a - __uint_as_float(hi << 16), b - __uint_as_float(hi & 0xffff0000u)};
  const bf16x2 l = __builtin_convertvector(r, bf16x2);
  __builtin_memcpy(&lo, &l, 4);
}

// Pieces of 16 rows x 64 bytes in LDS, and what lane l copies of one (its destination is 16 l bytes on).
// GB = 32: two k groups, [group][row][2 units of 16 bytes], the units of rows 8 .. 15 swapped; GB = 64: one group,
// [row][4 units], unit u of row r at u ^ (r / 4).  Either way the lanes of a copy read contiguous memory and a
// fragment read (one unit of 16 rows) falls on distinct banks.
template <int GB>
__device__ __forceinline__ int copy_row(int lane) { return GB == 32 ? (lane & 31) >> 1 : lane >> 2; }
template <int GB>
__device__ __forceinline__ int copy_group(int lane) { return GB == 32 ? lane >> 5 : 0; }
template <int GB>
__device__ __forceinline__ int copy_unit(int lane) {
  return GB == 32 ? (lane & 1) ^ ((lane >> 4) & 1) : (lane & 3) ^ ((lane >> 4) & 3);
}
// unit u of k group g of row r
template <int GB>
__device__ __forceinline__ unsigned unit_at(int r, int g, int u) {
  return GB == 32 ? (unsigned)((r >> 4) * 1024 + g * 512 + (r & 15) * 32 + (u ^ ((r >> 3) & 1)) * 16)
                  : (unsigned)((r >> 4) * 1024 + (r & 15) * 64 + (u ^ ((r >> 2) & 3)) * 16);
}

// row (x, y) of AV, and the element of a plane of W that row r is
__device__ __forceinline__ int64_t av_row(int v, int x, int y) {
  return (int64_t)8 * v * (x >> 3) + min(8, v - (x & ~7)) * y + (x & 7);
}
__device__ __forceinline__ int plane_at(int v, int r) {
  const int last = (v & ~7) * v;  // rows of the whole panels
  if (r < last) return r;
  const int w = v & 7, y = (r - last) / w;
  return last + 8 * y + (r - last - w * y);
}

// n elements in blocks of g, dealt to nt tiles of nearly equal block counts: first element of tile t
__host__ __device__ inline int tile_begin(int n, int g, int nt, int t) {
  const int nb = (n + g - 1) / g;
  return (int)((int64_t)nb * t / nt) * g;
}

}  // namespace

// ------------------------------------------------------------------ operands
// One k group of a row from 8 values at s, s + pitch, ...  FMT: 0 double, 1 float, 2 split-BF16x3 (8 bf16 hi,
// then 8 bf16 lo).
template <int FMT>
__device__ inline void put_k8(char* d, const double* s, int pitch) {
  if constexpr (FMT == 0) {
#pragma unroll
    for (int q = 0; q < 4; ++q) reinterpret_cast<double2*>(d)[q] = make_double2(s[2 * q * pitch], s[(2 * q + 1) * pitch]);
  } else if constexpr (FMT == 1) {
#pragma unroll
    for (int q = 0; q < 2; ++q)
      reinterpret_cast<float4*>(d)[q] = make_float4((float)s[4 * q * pitch], (float)s[(4 * q + 1) * pitch],
                                                    (float)s[(4 * q + 2) * pitch], (float)s[(4 * q + 3) * pitch]);
  } else {
    uint32_t h[4], l[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) split2((float)s[2 * q * pitch], (float)s[(2 * q + 1) * pitch], h[q], l[q]);
    reinterpret_cast<uint4*>(d)[0] = make_uint4(h[0], h[1], h[2], h[3]);
    reinterpret_cast<uint4*>(d)[1] = make_uint4(l[0], l[1], l[2], l[3]);
  }
}
// AV[d', (x,y), n] and AVs[d', (y,x), n]: d' < v -> (n y|x d') = OVVV[n, y, x, d']; v <= d' < v + o ->
// -T2[n, l, y, x], l = d' - v; zero up to nd.  One workgroup per 4 x 4 block of (x, y) and k group: n is the
// sources' unit-stride index and (d', row) the result's, so 32 n at a time turn in LDS, and both copies are
// written from one read in runs of 4 rows (a cache line).
template <int FMT>
__global__ __launch_bounds__(256) void k_triples_av(int o, int v, int nd, const double* __restrict__ ovvv,
                                                    const double* __restrict__ t2, char* __restrict__ av,
                                                    char* __restrict__ avs) {
  constexpr int GB = FMT == 0 ? 64 : 32;
  __shared__ double tile[8][16][33];  // [d'][x + 4 y][n]
  const int y0 = 4 * blockIdx.x, x0 = 4 * blockIdx.y, g = blockIdx.z;
  const int64_t vv = (int64_t)v * v, an = vv * (nd / 8) * GB;
  for (int n0 = 0; n0 < o; n0 += 32) {
    __syncthreads();
    for (int e = threadIdx.x; e < 8 * 16 * 32; e += 256) {
      const int n = n0 + (e & 31), y = y0 + (e >> 5 & 3), x = x0 + (e >> 7 & 3), d = 8 * g + (e >> 9);
      double val = 0.0;
      if (n < o && x < v && y < v) {
        if (d < v) val = ovvv[n + (int64_t)o * (y + (int64_t)v * (x + (int64_t)v * d))];
        else if (d < v + o) val = -t2[n + (int64_t)o * (d - v + (int64_t)o * (y + (int64_t)v * x))];
      }
      tile[e >> 9][(e >> 7 & 3) + 4 * (e >> 5 & 3)][e & 31] = val;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < 16 * 32; e += 256) {
      const int lo = e & 3, hi = e >> 2 & 3, n = e >> 4;
      if (n0 + n >= o) continue;
      if (x0 + lo < v && y0 + hi < v)
        put_k8<FMT>(av + (n0 + n) * an + (vv * g + av_row(v, x0 + lo, y0 + hi)) * GB, &tile[0][lo + 4 * hi][n], 16 * 33);
      if (y0 + lo < v && x0 + hi < v)
        put_k8<FMT>(avs + (n0 + n) * an + (vv * g + av_row(v, y0 + lo, x0 + hi)) * GB, &tile[0][hi + 4 * lo][n], 16 * 33);
    }
  }
}
// Bcat_{p,q}[d', z]: d' < v -> T2[q, p, z, d']; v <= d' < v + o -> OOOV[l, p, q, z]; zero up to nd; stored as
// BVp (block p + o q) and BVq (block q + o p).  One workgroup per 4 z, k group and 32 pairs q + o p, the
// unit-stride index of T2.
template <int FMT>
__global__ __launch_bounds__(256) void k_triples_bv(int o, int v, int nd, const double* __restrict__ t2,
                                                    const double* __restrict__ ooov, char* __restrict__ bvp,
                                                    char* __restrict__ bvq) {
  constexpr int GB = FMT == 0 ? 64 : 32;
  __shared__ double tile[8][4][33];  // [d'][z][pair]
  const int64_t bs = (int64_t)v * (nd / 8) * GB;
  const int oo = o * o, z0 = 4 * blockIdx.x, g = blockIdx.y, s0 = 32 * blockIdx.z;
  for (int e = threadIdx.x; e < 8 * 4 * 32; e += 256) {
    const int s = s0 + (e & 31), z = z0 + (e >> 5 & 3), d = 8 * g + (e >> 7);
    double val = 0.0;
    if (s < oo && z < v) {
      if (d < v) val = t2[s + (int64_t)oo * (z + (int64_t)v * d)];
      else if (d < v + o) val = ooov[d - v + (int64_t)o * (s / o + (int64_t)o * (s % o + (int64_t)o * z))];
    }
    tile[e >> 7][e >> 5 & 3][e & 31] = val;
  }
  __syncthreads();
  const int z = threadIdx.x & 3, s = threadIdx.x >> 2 & 31, q = (s0 + s) % o, p = (s0 + s) / o;
  if (s0 + s < oo && z0 + z < v) {
    char* d = threadIdx.x < 128 ? bvq + (s0 + s) * bs : bvp + (p + (int64_t)o * q) * bs;
    put_k8<FMT>(d + ((int64_t)v * g + z0 + z) * GB, &tile[0][z][s], 4 * 33);
  }
}

// ------------------------------------------------------------------ W build
// slices: W slots that share a c before the next c (1, 4, 8 and 16: 441, 436, 434 and 437 ms of slice launches at
// o = 40, v = 190)
constexpr int kSlotGroup = 8;

// What both W kernels share: the tile of a workgroup, its operands (bases at the tile's first row, per K
// segment) and its output.
struct TripW {
  const char *av, *avs, *bvp, *bvq;
  void* w;
  const int4* slots;  // (i, j, k, 0) of each W slot of the chunk
  const int4* cols;   // first launch: two int4 per column tile: (i, j, k0, slot of k0), (n0, columns, 0, 0)
  int o, v, nd;
  int nt;     // tiles along the rows (first launch: of v^2; slices: of v, the same along the columns)
  int ncol;   // first launch: column tiles; slices: W slots
  int group;  // slices: W slots of a raster group
};
template <int NSEG, int GB>
struct TripTile {
  const char *A[NSEG], *B[NSEG];  // per K segment: the operands' first group at the tile's first row / column
  int rows, cols;
  // first launch: leading dimension of the output tile; slices: of its panels.  Offset of its first element in W, and
  // elements from there to the end of its last column (first launch) or of its plane
  int64_t ldw, woff, wleft;
  int bcol, v;        // first launch: the tile's first column within its k
  int m0;             // first row
  // slices: offset of column c in a whole and in the last panel of AV, and that of the last panel's first row in Bcat
  int c8, cw, thra, thrb;
  int64_t bs;

  // whether segment s takes its A operand from AV / AVs (group stride v^2 rows) and B from Bcat (v rows), or
  // the other way round
  static __device__ __forceinline__ constexpr bool a_is_av(int s) { return NSEG == 2 || (s & 1) == 0; }

  __device__ __forceinline__ TripTile(const TripW& t, int grain) {
    // workgroup w runs on XCD w % 8: each XCD takes a contiguous range of the raster, so that
    // neighbouring tiles share their operand blocks in its L2
    const int64_t nwg = gridDim.x, w = blockIdx.x;
    const int64_t q8 = nwg >> 3, r8 = nwg & 7, x8 = w & 7;
    const int64_t L = x8 * q8 + (x8 < r8 ? x8 : r8) + (w >> 3);
    v = t.v;
    const int o = t.o;
    const int64_t pl = triples_plane(v), vv = (int64_t)v * v, an = vv * (t.nd / 8) * GB;
    bs = (int64_t)v * (t.nd / 8) * GB;
    bcol = 0;
    if constexpr (NSEG == 2) {
      const int ct = (int)(L % t.ncol), mt = (int)(L / t.ncol);
      const int4 p = t.cols[2 * ct], q = t.cols[2 * ct + 1];
      m0 = tile_begin((int)vv, grain, t.nt, mt);
      rows = min(tile_begin((int)vv, grain, t.nt, mt + 1), (int)vv) - m0;
      cols = q.y;
      const int kk = q.x / v;
      bcol = q.x - kk * v;
      A[0] = t.av + an * p.y + (int64_t)GB * m0;
      A[1] = t.avs + an * p.x + (int64_t)GB * m0;
      B[0] = t.bvq + bs * (p.z + kk + (int64_t)o * p.x);
      B[1] = t.bvq + bs * (p.z + kk + (int64_t)o * p.y);
      ldw = pl;
      woff = pl * v * p.w + pl * q.x;
      wleft = ldw * cols;
      c8 = cw = thra = thrb = 0;
    } else {
      // groups of kSlotGroup slots, then c, then the slots of the group, then the tiles of a slice: the 64
      // workgroups of an XCD in flight share AV_i, AV_j (same c) and the Bcat blocks (same slots)
      const int tt = t.nt * t.nt;
      const int64_t per = (int64_t)v * t.group * tt;
      const int gr = (int)(L / per), s0 = gr * t.group, ns = min(t.group, t.ncol - s0);
      const int rem = (int)(L - gr * per), c = rem / (ns * tt), r2 = rem - c * ns * tt, s = s0 + r2 / tt, tl = r2 % tt;
      const int4 p = t.slots[s];
      const int n0 = tile_begin(v, grain, t.nt, tl / t.nt);
      m0 = tile_begin(v, grain, t.nt, tl % t.nt);
      rows = min(tile_begin(v, grain, t.nt, tl % t.nt + 1), v) - m0;
      cols = min(tile_begin(v, grain, t.nt, tl / t.nt + 1), v) - n0;
      // the panels of rows m0 .. and n0 .. (multiples of 8) of AV, in which column c starts at c8, cw in the last, and
      // rows m0 .. and n0 .. of Bcat
      c8 = GB * 8 * c;
      cw = GB * (v & 7) * c;
      thra = GB * ((v & ~7) - m0);
      thrb = GB * ((v & ~7) - n0);
      const int64_t ca = (int64_t)GB * v * m0, cb = (int64_t)GB * v * n0;
      const int64_t ao = (int64_t)GB * m0, bo = (int64_t)GB * n0;
      A[0] = t.avs + an * p.x + ca;                            // cab: AV_i[(c,a)]
      B[0] = t.bvp + bs * (p.z + (int64_t)o * p.y) + bo;       //      Bcat_{k,j}[., b]
      A[1] = t.bvp + bs * (p.z + (int64_t)o * p.x) + ao;       // cba: Bcat_{k,i}[., a]
      B[1] = t.avs + an * p.y + cb;                            //      AV_j[(c,b)]
      A[2] = t.av + an * p.z + ca;                             // acb: AV_k[(a,c)]
      B[2] = t.bvp + bs * (p.x + (int64_t)o * p.y) + bo;       //      Bcat_{i,j}[., b]
      A[3] = t.bvp + bs * (p.y + (int64_t)o * p.x) + ao;       // bca: Bcat_{j,i}[., a]
      B[3] = t.av + an * p.z + cb;                             //      AV_k[(b,c)], in L2 from the previous segment
      ldw = 8 * v;
      woff = pl * v * s + pl * c + (int64_t)v * m0 + 8 * n0;
      wleft = pl - (int64_t)v * m0 - 8 * n0;
    }
  }
  // byte offset of column n of the tile within a k group of B
  __device__ __forceinline__ int col_off(int n) const {
    if constexpr (NSEG == 2) {
      const int q = bcol + n, kk = q / v;
      return (int)(bs * kk) + GB * (q - kk * v);
    } else {
      return GB * n;
    }
  }
};

// The k steps of a tile in order: step() calls copy(A, B, dga, dgb, odd) with resources at the step's first group,
// the lane's byte offset from there to its own group and whether the segment is an odd one (row_at).  With 32-byte
// groups a step is two groups, which may lie in two segments (an odd number of groups per segment): the lanes of the second group then copy in a
// second, masked pass, which only makes the waits that count copies stricter.  The passes end in different
// (empty) asm markers: merged into one copy with a choice of resource, they would run as a loop over the
// wave's distinct resources.
template <int NSEG, int GB>
struct Feed {
  using Tile = TripTile<NSEG, GB>;
  const char *A[NSEG - 1], *B[NSEG - 1];  // of the segments to come
  const char *pa, *pb;
  int64_t sav, sbv;  // group strides of AV and Bcat
  int ng, seg, g, second;
  int panel, c8, cw, thra, thrb;
  // Offset of a row of A (or B) in AV from that in Bcat (16 times the unit + GB times the row): a panel of 8 rows is
  // 8 v rows after the panel before it
  template <bool OF_A>
  __device__ __forceinline__ unsigned av_at(int lof) const {
    if constexpr (NSEG == 2) return (unsigned)lof;
    else return (unsigned)lof + __umul24((unsigned)lof >> (GB == 32 ? 8 : 9), (unsigned)panel) +
                (unsigned)(lof >= (OF_A ? thra : thrb) ? cw : c8);
  }
  // the same in the operand that the segment has there: A is AV in the even segments, B in the odd ones
  template <bool OF_A>
  __device__ __forceinline__ unsigned row_at(int lof, bool odd) const {
    if constexpr (NSEG == 2) {
      return (unsigned)lof;
    } else {
      const bool is_av = odd != OF_A;
      const int col = lof >= (OF_A ? thra : thrb) ? (is_av ? cw : 0) : (is_av ? c8 : 0);
      return (unsigned)lof + __umul24((unsigned)lof >> (GB == 32 ? 8 : 9), (unsigned)(is_av ? panel : 0)) + (unsigned)col;
    }
  }
  __device__ __forceinline__ Feed(const TripW& t, const Tile& tl, int lane) {
#pragma unroll
    for (int s = 0; s + 1 < NSEG; ++s) {
      A[s] = tl.A[s + 1];
      B[s] = tl.B[s + 1];
    }
    sbv = (int64_t)GB * t.v;
    sav = sbv * t.v;
    panel = GB * 8 * (t.v - 1);
    c8 = tl.c8;
    cw = tl.cw;
    thra = tl.thra;
    thrb = tl.thrb;
    ng = t.nd / 8;
    seg = g = 0;
    pa = tl.A[0];
    pb = tl.B[0];
    second = copy_group<GB>(lane);
  }
  __device__ __forceinline__ int64_t sa() const { return NSEG == 2 || (seg & 1) == 0 ? sav : sbv; }
  __device__ __forceinline__ int64_t sb() const { return NSEG == 2 || (seg & 1) == 0 ? sbv : sav; }
  __device__ __forceinline__ void next_segment() {
    ++seg;
    pa = A[0];
    pb = B[0];
#pragma unroll
    for (int s = 0; s + 2 < NSEG; ++s) {
      A[s] = A[s + 1];
      B[s] = B[s + 1];
    }
  }
  template <typename Copy>
  __device__ __forceinline__ void step(Copy&& copy) {
    constexpr int G = 64 / GB;
    if (G == 1 || g + 1 < ng) {
      copy(uniform_rsrc(pa), uniform_rsrc(pb), second ? (int)sa() : 0, second ? (int)sb() : 0, seg & 1);
      asm volatile("; step");
      g += G;
      pa += G * sa();
      pb += G * sb();
    } else {
      if (!second) {
        copy(uniform_rsrc(pa), uniform_rsrc(pb), 0, 0, seg & 1);
        asm volatile("; step, last group of a segment");
      }
      next_segment();
      if (second) {
        copy(uniform_rsrc(pa), uniform_rsrc(pb), 0, 0, seg & 1);
        asm volatile("; step, first group of a segment");
      }
      g = 1;
      pa += sa();
      pb += sb();
    }
    if (g == ng && seg + 1 < NSEG) {
      next_segment();
      g = 0;
    }
  }
};

// First launch: a wave's MI x NJ blocks at (r0, c0) of its tile, element e of lane l of block (i, j) at row l % 32 and
// column 8 (e / 4) + 4 (l / 32) + e % 4 of the block.  W goes through a buffer resource that ends with the tile's last
// column, at one running lane offset: an element outside the tile (a row beyond it starts out of range) is not
// written, with no masks and no 48 addresses.
template <int MI, int NJ>
__device__ __forceinline__ void store_blocks(const f32x16 (&acc)[MI][NJ], __amdgpu_buffer_rsrc_t rw, int r0, int c0,
                                             int rows, int ldw4, int m0, int v) {
  const int lane = threadIdx.x & 63, cl = c0 + 4 * (lane >> 5);
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int row = r0 + i * 32 + (lane & 31);
    unsigned o = row < rows ? (unsigned)(4 * plane_at(v, m0 + row) + ldw4 * cl) : 0x80000000u;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[i][j][e]), rw, o, 0, 0);
        o += (e & 3) == 3 ? 5 * ldw4 : ldw4;
        asm volatile("" : "+v"(o));  // a running sum: not folded into 48 live offsets
      }
    }
  }
}
// Slices: adds a wave's blocks to a plane of W, element e of lane l of block (i, j) at row 8 (e / 4) + 4 (l / 32) + e % 4
// and column l % 32: four consecutive elements of a panel a time, 64 lanes a run of 1 KB.  The resource ends with the
// plane, a panel beyond v starts behind it and a column beyond the tile out of range.  Per 32-row block row of the wave
// the values of W are loaded before any is stored, and the sums replace them before the first store: a store's
// data register is then not reused, which would make the next instruction wait for that store to complete.
template <int MI, int NJ>
__device__ __forceinline__ void store_slice(const f32x16 (&acc)[MI][NJ], __amdgpu_buffer_rsrc_t rw, int r0, int c0,
                                            int cols, int panel4) {
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  const int lane = threadIdx.x & 63;
  unsigned vo[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int col = c0 + 32 * j + (lane & 31);
    vo[j] = col < cols ? (unsigned)(32 * col + 16 * (lane >> 5)) : 0x80000000u;
  }
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const unsigned po = (unsigned)(panel4 * ((r0 >> 3) + 4 * i));
    f32x4 dv[NJ][4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        dv[j][q] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, vo[j] + (po + panel4 * q), 0, 0));
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) dv[j][q][e] += acc[i][j][4 * q + e];
      asm volatile("" : "+v"(dv[j][0]), "+v"(dv[j][1]), "+v"(dv[j][2]), "+v"(dv[j][3]));
    }
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, dv[j][q]), rw, vo[j] + (po + panel4 * q), 0, 0);
  }
}

// Split-BF16x3: A B ~ Ahi Bhi + Ahi Blo + Alo Bhi with FP32 accumulation (Henry, Tang and Heinecke,
// ARITH 2019), operands split once when AV and Bcat are built (32 bytes per 8 k: hi, then lo), so that a
// fragment (8 consecutive k of a row, hi and lo) is two 16-byte LDS reads and no arithmetic.  Tiles of up to
// 64 MB x 64 MB (MB = 3: two workgroups per CU; MB = 2 for v <= 128: three), 2 x 2 wavefronts of up to
// MB x MB 32 x 32 blocks.  An axis is cut into tiles of nearly equal numbers of 32-blocks and a tile's
// blocks are dealt to the two wave rows, so v = 131 costs 5 x 5 blocks, not 6 x 6; blocks, copies and
// fragment reads beyond the edge are not issued.
// Bound by the matrix cores at the rate the card sustains (a plain bf16 product of 8192^3 reaches 1122 TFLOP/s,
// 374 for three products): o = 40, v = 190: first launch 344 to 359 TFLOP/s on several cards (on one 363 so and 345 with a
// fastest over all of v in W, whose stores then begin inside a cache line; per-pair launches with row-major operands split
// in the kernel: 224), slices 335 to 352 (on one 359 so and 336 with one W element a load and store; 224);
// o = 27, v = 131: slices 202 (two batched launches of 128 x 192 tiles: 98).
template <int NSEG, int MB>
struct Bf3Tile {
  static constexpr int NS = 3, ABYTES = 64 * MB * 64, SLOT = 2 * ABYTES;
  __amdgpu_buffer_rsrc_t rw;
  char* ring;
  int lane, wid, rows, cols, nst, npa, npb, cps, ldw4, m0, v;
  int rb0, mi, cb0, nj;  // the wave's first row / column block of the tile and its block counts
  int lofa[MB], lofb[MB];

  __device__ __forceinline__ Bf3Tile(const TripW& t, const TripTile<NSEG, 32>& tl, char* lds) : ring(lds) {
    lane = threadIdx.x & 63;
    wid = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    rows = __builtin_amdgcn_readfirstlane(tl.rows);
    cols = __builtin_amdgcn_readfirstlane(tl.cols);
    // the two workgroups of a CU start half a grid of CUs apart: swapping the wave roles of every other 256
    // workgroups puts the larger and the smaller share of an odd block count on different SIMDs
    const int flip = (blockIdx.x >> 8) & 1;
    const int wm = (wid & 1) ^ flip, wn = (wid >> 1) ^ flip;
    const int nrb = (rows + 31) / 32, ncb = (cols + 31) / 32;
    rb0 = wm ? (nrb + 1) / 2 : 0;
    mi = wm ? nrb - rb0 : (nrb + 1) / 2;
    cb0 = wn ? (ncb + 1) / 2 : 0;
    nj = wn ? ncb - cb0 : (ncb + 1) / 2;
    ldw4 = 4 * (int)tl.ldw;
    m0 = __builtin_amdgcn_readfirstlane(tl.m0);
    v = t.v;
    rw = uniform_rsrc(reinterpret_cast<const char*>(static_cast<float*>(t.w) + tl.woff), 4 * (int)tl.wleft);
    nst = NSEG * t.nd / 16;
    npa = (rows + 15) / 16;
    npb = (cols + 15) / 16;
    cps = 0;
#pragma unroll
    for (int q = 0; q < MB; ++q) {
      const int r = 16 * (wid + 4 * q) + copy_row<32>(lane);
      lofa[q] = 16 * copy_unit<32>(lane) + 32 * min(r, rows - 1);
      lofb[q] = 16 * copy_unit<32>(lane) + tl.col_off(min(r, cols - 1));
      cps += (wid + 4 * q < npa) + (wid + 4 * q < npb);
    }
  }
  __device__ __forceinline__ void dma(Feed<NSEG, 32>& feed, int slot) const {
    feed.step([&](__amdgpu_buffer_rsrc_t rsa, __amdgpu_buffer_rsrc_t rsb, int dga, int dgb, bool odd) {
#pragma unroll
      for (int q = 0; q < MB; ++q)
        if (wid + 4 * q < npa)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rsa, (lds_vptr)(ring + slot * SLOT + (wid + 4 * q) * 1024), 16,
                                                   feed.template row_at<true>(lofa[q], odd) + dga, 0, 0, 0);
#pragma unroll
      for (int q = 0; q < MB; ++q)
        if (wid + 4 * q < npb)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rsb, (lds_vptr)(ring + slot * SLOT + ABYTES + (wid + 4 * q) * 1024), 16,
                                                   feed.template row_at<false>(lofb[q], odd) + dgb, 0, 0, 0);
    });
  }
  // MI x NJ blocks of this wave (0 x 0: a wave without a block, which still copies and meets the barriers).
  // Steps 0 .. NS - 2 start in flight; at step s the copies issued after step s are those of one step (none
  // at the end), and step s + 2 goes into the slot that step s - 1 left.
  template <int MI, int NJ>
  __device__ __forceinline__ void run(Feed<NSEG, 32> feed) const {
    // row l % 32 of a block, k group l / 32: units 0 (hi) and 1 (lo)
    const unsigned frag = lds_addr(ring) + unit_at<32>(lane & 31, lane >> 5, 0);
    const unsigned a_off = frag + rb0 * 2048, b_off = frag + ABYTES + cb0 * 2048;
    f32x16 acc[MI > 0 ? MI : 1][NJ > 0 ? NJ : 1];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
    dma(feed, 0);
    if (nst > 1) dma(feed, 1);
    int cur = 0, nxt = 2;
    for (int s = 0; s < nst; ++s) {
      wait_vmcnt_n(s + 1 < nst ? cps : 0);
      lds_barrier();  // step s landed for every wave; the slot of step s - 1 read by all
      if (s + 2 < nst) dma(feed, nxt);
      if constexpr (MI > 0 && NJ > 0) {
        f32x4 fa[MI][2], fb[NJ][2];
        read_frags<MI, NJ>(a_off + cur * SLOT, b_off + cur * SLOT, fa, fb);
        // the MFMA burst at raised wave priority: the other wave of the SIMD issues its LDS reads and
        // copies under it
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          const bf16x8 bh = __builtin_bit_cast(bf16x8, fb[j][0]), bl = __builtin_bit_cast(bf16x8, fb[j][1]);
          // first launch: B as the first operand, so that the accumulator's lanes run along the rows of W; slices: A, so
          // that they run along its columns and four registers are four rows (store_slice)
          auto mul = [&](int i, const bf16x8& a, const bf16x8& b) {
            if constexpr (NSEG == 2) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b, a, acc[i][j], 0, 0, 0);
            else acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[i][j], 0, 0, 0);
          };
#pragma unroll
          for (int i = 0; i < MI; ++i) mul(i, __builtin_bit_cast(bf16x8, fa[i][0]), bl);
#pragma unroll
          for (int i = 0; i < MI; ++i) mul(i, __builtin_bit_cast(bf16x8, fa[i][1]), bh);
#pragma unroll
          for (int i = 0; i < MI; ++i) mul(i, __builtin_bit_cast(bf16x8, fa[i][0]), bh);
        }
        __builtin_amdgcn_s_setprio(0);
      }
      cur = cur == NS - 1 ? 0 : cur + 1;
      nxt = nxt == NS - 1 ? 0 : nxt + 1;
    }
    if constexpr (MI > 0 && NJ > 0) {
      if constexpr (NSEG == 2) store_blocks<MI, NJ>(acc, rw, rb0 * 32, cb0 * 32, rows, ldw4, m0, v);
      else store_slice<MI, NJ>(acc, rw, rb0 * 32, cb0 * 32, cols, ldw4);
    }
  }
  template <int MI>
  __device__ __forceinline__ void run_n(const Feed<NSEG, 32>& feed) const {
    if constexpr (MB == 3) {
      if (nj == 3) {
        run<MI, 3>(feed);
        return;
      }
    }
    if (nj == 2) run<MI, 2>(feed);
    else run<MI, 1>(feed);
  }
};
template <int NSEG, int MB>
__global__ __launch_bounds__(256, MB == 3 ? 2 : 3) void k_triples_w_bf3(TripW t) {
  __shared__ __attribute__((aligned(16))) char ring[Bf3Tile<NSEG, MB>::NS * Bf3Tile<NSEG, MB>::SLOT];
  const TripTile<NSEG, 32> tl(t, 32);
  const Feed<NSEG, 32> feed(t, tl, threadIdx.x & 63);
  const Bf3Tile<NSEG, MB> tile(t, tl, ring);
  if (tile.mi == 0 || tile.nj == 0) {
    tile.template run<0, 0>(feed);
    return;
  }
  if constexpr (MB == 3) {
    if (tile.mi == 3) {
      tile.template run_n<3>(feed);
      return;
    }
  }
  if (tile.mi == 2) tile.template run_n<2>(feed);
  else tile.template run_n<1>(feed);
}

// adds N blocks of a wave of the FP32 slices to W (the tile's first element; panels of ldw elements): row block rb, column
// blocks cb, cb + 1, ...; element e of lane l at row 4 (l / 16) + e, column l % 16: a panel holds all four rows
template <int N>
__device__ __forceinline__ void add_rows4(float* W, const f32x4* blk, int rb, int cb, int rows, int cols, int ldw) {
  const int lane = threadIdx.x & 63, row = 16 * rb + 4 * (lane >> 4), col = 16 * cb + (lane & 15);
  float* const Wr = W + ldw * (row >> 3) + (row & 7) + 8 * col;
  f32x4 dv[N];
#pragma unroll
  for (int j = 0; j < N; ++j)
    dv[j] = *reinterpret_cast<const f32x4*>(row < rows && col + 16 * j < cols ? Wr + 128 * j : W);
#pragma unroll
  for (int j = 0; j < N; ++j) dv[j] += blk[j];
#pragma unroll
  for (int j = 0; j < N; ++j)
    if (row < rows && col + 16 * j < cols) *reinterpret_cast<f32x4*>(Wr + 128 * j) = dv[j];
}
// FP64 and FP32: tiles of 16 NB x 16 NB, a wavefront per 16-row block (NB column blocks), and at NB = 5 and 6 four
// wavefronts that share the last rows' blocks: the SIMDs of a CU are dealt a workgroup's wavefronts in order, so a fifth
// would always land with the first (matrix pipes busy 53 % of the time at NB = 5 with five, 63 % at NB = 6 with six;
// slices and first launch of o = 16, v = 76 in FP64 7.7 and 3.3 ms so, 5.7 and 2.7 ms with four).  An MFMA takes 64
// (FP64) or 32 (FP32) cycles, so the fragment reads (one per block and k step: a lane's 16 bytes are 2 (4) k, fed to
// 2 (4) MFMAs in turn -- the k order inside a step is free as long as A and B agree) hide behind them with four
// wavefronts per SIMD, and small tiles cost little: the tile follows v in steps of 16 instead of padding N = v = 76
// to 128.
constexpr int triples_w_waves(int nb) { return nb < 4 ? nb : 4; }
template <typename T, int NSEG, int NB>
__global__ __launch_bounds__(64 * triples_w_waves(NB), NB == 6 ? 3 : NB > 3 ? 4 : 1) void k_triples_w(TripW t) {
  constexpr bool F32 = std::is_same<T, float>::value;
  constexpr int NS = 3, ABYTES = NB * 1024, SLOT = 2 * ABYTES, KL = F32 ? 4 : 2;
  constexpr int NW = triples_w_waves(NB), NX = NB == 5 ? 2 : NB == 6 ? 3 : 0;
  using Acc = typename std::conditional<F32, f32x4, f64x4>::type;
  __shared__ __attribute__((aligned(16))) char ring[NS * SLOT];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  constexpr int GB = F32 ? 32 : 64;
  const TripTile<NSEG, GB> tl(t, 16);
  const int rows = tl.rows, cols = tl.cols;
  Feed<NSEG, GB> feed(t, tl, lane);
  const int nst = NSEG * (t.nd / 8) * GB / 64;
  // pieces of 16 rows: wid and, of NB = 5 and 6, wid + 4
  const bool second = NB > 4 && wid + 4 < NB;
  int lofa[2], lofb[2], ava[2], avb[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int r = 16 * (wid + 4 * h) + copy_row<GB>(lane);
    lofa[h] = 16 * copy_unit<GB>(lane) + GB * min(r, rows - 1);
    lofb[h] = 16 * copy_unit<GB>(lane) + tl.col_off(min(r, cols - 1));
    ava[h] = (int)feed.template av_at<true>(lofa[h]);
    avb[h] = (int)feed.template av_at<false>(lofb[h]);
  }
  auto dma = [&](int slot) {
    feed.step([&](__amdgpu_buffer_rsrc_t rsa, __amdgpu_buffer_rsrc_t rsb, int dga, int dgb, bool odd) {
      char* d = ring + slot * SLOT + wid * 1024;
#pragma unroll
      for (int h = 0; h < (NB > 4 ? 2 : 1); ++h) {
        if (h == 1 && !second) break;
        const unsigned oa = (unsigned)((NSEG == 4 && !odd ? ava[h] : lofa[h]) + dga);
        const unsigned ob = (unsigned)((NSEG == 4 && odd ? avb[h] : lofb[h]) + dgb);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsa, (lds_vptr)(d + 4096 * h), 16, oa, 0, 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsb, (lds_vptr)(d + 4096 * h + ABYTES), 16, ob, 0, 0, 0);
      }
    });
  };
  // the extra blocks: NB = 5: (4, wid) and, for one wavefront, in turn over the workgroups, (4, 4); NB = 6: three
  // of row block 4 or 5
  const bool last = NB == 5 && wid == ((int)(blockIdx.x >> 8) & 3);
  const int xr = NB == 6 ? 4 + (wid >> 1) : 4, xc = NB == 6 ? 3 * (wid & 1) : wid;
  // unit l / 16 of the step of row l % 16 (FP32: units of two groups)
  const int fu = lane >> 4;
  const unsigned frag = lds_addr(ring) + unit_at<GB>(lane & 15, F32 ? fu >> 1 : 0, F32 ? fu & 1 : fu);
  const unsigned a_off = frag + wid * 1024, b_off = frag + ABYTES;
  Acc acc[NB], accx[NX > 0 ? NX : 1];
#pragma unroll
  for (int j = 0; j < NB; ++j) acc[j] = Acc{0, 0, 0, 0};
#pragma unroll
  for (int j = 0; j < NX; ++j) accx[j] = Acc{0, 0, 0, 0};
  dma(0);
  if (nst > 1) dma(1);
  int cur = 0, nxt = 2;
  for (int s = 0; s < nst; ++s) {
    if (s + 1 >= nst) wait_vmcnt<0>();
    else if (second) wait_vmcnt<4>();
    else wait_vmcnt<2>();
    lds_barrier();
    if (s + 2 < nst) dma(nxt);
    f32x4 fa, fb[NB], fx, fy[NB == 6 ? 3 : 1];
    if constexpr (NX > 0)
      read_rows_extra<NB>(a_off + cur * SLOT, b_off + cur * SLOT, frag + xr * 1024 + cur * SLOT,
                          b_off + xc * 1024 + cur * SLOT, fa, fb, fx, fy);
    else
      read_rows<NB>(a_off + cur * SLOT, b_off + cur * SLOT, fa, fb);
    auto mul = [&](const f32x4& ua, const f32x4& ub, Acc& c, int q) {
      T ta[KL], tb[KL];
      __builtin_memcpy(ta, &ua, 16);
      __builtin_memcpy(tb, &ub, 16);
      // B as the first operand, so that the accumulator's lanes run along the rows of W; the FP32 slices A, so that
      // they run along its columns and a lane's four registers are four rows of a panel
      if constexpr (F32 && NSEG == 4) c = __builtin_amdgcn_mfma_f32_16x16x4f32(ta[q], tb[q], c, 0, 0, 0);
      else if constexpr (F32) c = __builtin_amdgcn_mfma_f32_16x16x4f32(tb[q], ta[q], c, 0, 0, 0);
      else c = __builtin_amdgcn_mfma_f64_16x16x4f64(tb[q], ta[q], c, 0, 0, 0);
    };
#pragma unroll
    for (int q = 0; q < KL; ++q) {
#pragma unroll
      for (int j = 0; j < NB; ++j) mul(fa, fb[j], acc[j], q);
      if constexpr (NB == 6) {
#pragma unroll
        for (int j = 0; j < 3; ++j) mul(fx, fy[j], accx[j], q);
      }
      if constexpr (NB == 5) mul(fx, fy[0], accx[0], q);
    }
    if constexpr (NB == 5) {
      if (last) {
#pragma unroll
        for (int q = 0; q < KL; ++q) mul(fx, fb[4], accx[1], q);
      }
    }
    cur = cur == NS - 1 ? 0 : cur + 1;
    nxt = nxt == NS - 1 ? 0 : nxt + 1;
  }
  // register e of lane l of a block: row l % 16, column (l / 16) + 4 e (FP64) or 4 (l / 16) + e (FP32); FP32 slices:
  // row 4 (l / 16) + e, column l % 16
  T* const W = static_cast<T*>(t.w) + tl.woff;
  const int ldw = (int)tl.ldw;
  auto put = [&](auto& blk, auto n, int rb, auto cb) {
    constexpr int N = decltype(n)::value;
    const int row = 16 * rb + (lane & 15);
    auto col = [&](int j, int e) { return 16 * cb(j) + (F32 ? 4 * (lane >> 4) + e : (lane >> 4) + 4 * e); };
    const int r0 = NSEG == 4 ? ldw * (row >> 3) + (row & 7) : row < rows ? plane_at(tl.v, tl.m0 + row) : 0;
    auto at = [&](int j, int e) { return r0 + (NSEG == 4 ? 8 : ldw) * col(j, e); };
    if constexpr (NSEG == 4) {
      T dv[N][4];
#pragma unroll
      for (int j = 0; j < N; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) dv[j][e] = W[row < rows && col(j, e) < cols ? at(j, e) : 0];
#pragma unroll
      for (int j = 0; j < N; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) blk[j][e] += dv[j][e];
    }
#pragma unroll
    for (int j = 0; j < N; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (row < rows && col(j, e) < cols) W[at(j, e)] = blk[j][e];
  };
  if constexpr (F32 && NSEG == 4) {
    add_rows4<NB>(W, acc, wid, 0, rows, cols, ldw);
    if constexpr (NB == 6) add_rows4<3>(W, accx, xr, xc, rows, cols, ldw);
    if constexpr (NB == 5) {
      add_rows4<1>(W, accx, 4, wid, rows, cols, ldw);
      if (last) add_rows4<1>(W, accx + 1, 4, 4, rows, cols, ldw);
    }
  } else {
    put(acc, std::integral_constant<int, NB>(), wid, [](int j) { return j; });
    if constexpr (NB == 6) put(accx, std::integral_constant<int, 3>(), xr, [&](int j) { return xc + j; });
    if constexpr (NB == 5) {
      if (last) put(accx, std::integral_constant<int, 2>(), 4, [&](int j) { return j ? 4 : wid; });
      else put(accx, std::integral_constant<int, 1>(), 4, [&](int) { return wid; });
    }
  }
}

// ------------------------------------------------------------------ (T) energy epilogue (ijk.jl:116-136)
// For one occupied triple the reference's restricted sum over a>=b>=c with weights 1/(1+d_ab+d_bc) is, with
// V = W + T1p[a,i] (jb|kc) + (ia|kc) T1p[b,j] + (ia|jb) T1p[c,k] (ijk.jl:116) and the sums S+ of V and W+ of W
// over the even orderings (abc, bca, cab) and S-, W- over the odd ones (acb, bac, cba),
//     Ef = 3 sum_p W_p V_p + W+ (S+ - 2 S-) + W- (S- - 2 S+)                    (ijk.jl:129-132)
// over D_abc, times (2 - d_ij - d_jk); a=b=c terms vanish.  W slots are v planes (a, b), c
// slowest, each in panels of 8 a.  The virtual space is cut into 8x8x8 cubes; one workgroup takes an orbit
// {A,B,C} (A>=B>=C) of cube blocks for a run of consecutive k: the six permuted cubes and the (jb|kc) and (ia|kc)
// blocks are copied straight into LDS, and a thread owns two elements (a,b,c) with all six orderings, so the
// denominator, its reciprocal and the sums are formed once per six elements of W and V never leaves the
// registers.  What does not depend on k ((ia|jb) and T1 of i and j) stays in registers.  A turn is two k (FP64 W: one): a
// thread reads all it needs of a k from LDS, and the copies of the next turn run while it computes the last k (an LDS
// read behind a copy in flight would be made to wait for it).
// o = 40, v = 190, FP32 W: 95 ms per (T), 3.3 TB/s of W (103 on a slower card; 114 with a k a turn and copies of a dword
// per lane, 162 with a fastest over all of v in W, rows of 8 a being a quarter of a cache line, and all nine (ia|jb) blocks
// of a pair copied, 260 with one ordering per thread, V cubes in LDS and a reciprocal per element); o = 27, v = 131 10.7
// (13.1, 17.7, 27.8);
// FP64 o = 16, v = 76 0.72 (0.83, 0.96, 1.5).  Bound by the copies' latency: three workgroups per CU (144 registers; at
// 128, for four, the compiler's schedule takes 160 ms); the vector units are busy for a third of the time, LDS for half.
static constexpr int CT = 8, CT3 = CT * CT * CT;

// LDS position of element (x, y, z) of a W cube, in units of 16 bytes (4 or 2 elements along x, a lane's share of a
// copy): planes of z, in which the rows turn with z and the units of a row with y.  The reads of a plane with z or y
// fixed are free of bank conflicts, those with x fixed take four passes for FP32 (a unit's four elements fall on
// different banks) and none more for FP64.
template <typename TW>
__device__ __forceinline__ int cube_off(int x, int y, int z) {
  constexpr int EU = 16 / (int)sizeof(TW), HN = 8 / EU;
  return 64 * z + 8 * ((y + z) & 7) + EU * ((x / EU) ^ (y & (HN - 1))) + x % EU;
}

// 1/d by the hardware reciprocal and two Newton steps (relative error ~1 ulp; d is a negative
// orbital-energy denominator, never zero, denormal or infinite)
__device__ __forceinline__ double rcp_nr(double d) {
  double r = __builtin_amdgcn_rcp(d);
  double e = fma(-d, r, 1.0);
  r = fma(r, e, r);
  e = fma(-d, r, 1.0);
  return fma(r, e, r);
}

template <typename TW>
__global__ __launch_bounds__(256, 3) void k_triples_energy(int o, int v, const int4* __restrict__ runs,
                                                           const TW* __restrict__ Wc, const int* __restrict__ orbits,
                                                           const double* __restrict__ t1p, const double* __restrict__ vvb,
                                                           const double* __restrict__ eo, const double* __restrict__ ev,
                                                           double* __restrict__ partials) {
  // units of 16 bytes: elements, units of a row, planes of a copy instruction, instructions of a cube
  constexpr int EU = 16 / (int)sizeof(TW), HN = 8 / EU, PZ = 8 / HN, NI = 8 / PZ;
  // values of k a turn: FP32 W has room for two in LDS with three workgroups per CU
  constexpr int KD = sizeof(TW) == 4 ? 2 : 1;
  __shared__ __attribute__((aligned(16))) TW Wl[KD][6 * CT3];
  __shared__ __attribute__((aligned(16))) double s_t1[KD][32];  // T1 of k: 8 a, b, c (and 8 unused)
  __shared__ __attribute__((aligned(16))) double s_vv[KD][2][6][CT * CT];  // [(jk) (ik)][ab ba ac ca bc cb][x + 8 y]
  __shared__ double red[4];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  // consecutive workgroups go to different XCDs: give each XCD a contiguous range of orbits, so that concurrently
  // resident orbits share their (ia|jb) blocks in its L2
  const int nwg = gridDim.x, w = blockIdx.x;
  const int ob = (w & 7) * (nwg >> 3) + min(w & 7, nwg & 7) + (w >> 3);
  const int4 run = runs[2 * blockIdx.y];
  const int i = run.x, j = run.y, k0 = run.z, nk = run.w;
  const int64_t pl = triples_plane(v);
  const TW* W = Wc + pl * v * runs[2 * blockIdx.y + 1].x;
  const int blk[3] = {orbits[3 * ob], orbits[3 * ob + 1], orbits[3 * ob + 2]};
  auto blk_of = [&](unsigned q) { return q == 0 ? blk[0] : q == 1 ? blk[1] : blk[2]; };
  // the six orderings of the orbit's blocks, (abc) (acb) (bac) (bca) (cab) (cba): 2 bits an index, 6 an ordering
  constexpr uint64_t pb = 0x192261624ull;
  // (ia|jb) of occupied pair (p, q) in 8x8 blocks: vvb + PS (p + o q) + 64 (A + nb B) + x + 8 y
  const int nb = (v + CT - 1) / CT;
  const int64_t PS = (int64_t)nb * nb * CT * CT;
  const double* vv_jk = vvb + PS * (j + (int64_t)o * k0);   // (jk) block of k0; + PS*o per k
  const double* vv_ik = vvb + PS * (i + (int64_t)o * k0);
  const double* vv_ij = vvb + PS * (i + (int64_t)o * j);

  // Copies of a k.  W: PZ planes of a cube per instruction, lane -> LDS position -> (y, z) and unit of the row; planes
  // beyond v lie behind the slot's end, where the resource ends, rows and columns beyond v are copied as they lie: the
  // elements that would use them are dropped.  vv: two 512-byte blocks per instruction.
  int clo;
  {
    const int z = PZ * (wid % NI) + lane / (8 * HN), t = lane % (8 * HN), y = (t / HN - z) & 7, h = (t % HN) ^ (y & (HN - 1));
    clo = (int)((pl * z + 8 * y + EU * h) * (int64_t)sizeof(TW));
  }
  int vlo[2];
#pragma unroll
  for (int l = 0; l < 2; ++l) {
    constexpr unsigned vx = 0x212010u, vy = 0x120201u;  // blocks of ab, ba, ac, ca, bc, cb, 4 bits each
    const int e = 4 * (2 * ((wid + 4 * l) % 3) + (lane >> 5));
    vlo[l] = (blk_of((vx >> e) & 3) + nb * blk_of((vy >> e) & 3)) * 512 + (lane & 31) * 16;
  }
  const int tlo = min(lane, 47), t1lo = (int)(blk_of(tlo >> 4) * 8 + ((tlo >> 1) & 7)) * 8 + 4 * (tlo & 1);
  auto copy = [&](int kk, int u) {
    const TW* Wk = W + pl * v * kk;
#pragma unroll
    for (int m = 0; m < 6 * NI / 4; ++m) {
      const int p = wid / NI + 4 / NI * m;
      const int64_t at = (int64_t)8 * v * blk_of(pb >> (6 * p) & 3) + 64 * blk_of(pb >> (6 * p + 2) & 3) +
                         pl * CT * blk_of(pb >> (6 * p + 4) & 3);
      const int64_t left = (pl * v - at) * (int64_t)sizeof(TW);
      const __amdgpu_buffer_rsrc_t r = uniform_rsrc(reinterpret_cast<const char*>(Wk + at), (int)min(left, (int64_t)0x7fffffff));
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          r, (lds_vptr)(reinterpret_cast<char*>(Wl[u]) + (p * NI + wid % NI) * 1024), 16, (unsigned)clo, 0, 0, 0);
    }
    const __amdgpu_buffer_rsrc_t rj = uniform_rsrc(reinterpret_cast<const char*>(vv_jk + PS * o * kk));
    const __amdgpu_buffer_rsrc_t ri = uniform_rsrc(reinterpret_cast<const char*>(vv_ik + PS * o * kk));
#pragma unroll
    for (int l = 0; l < 2; ++l) {
      const int q = wid + 4 * l;
      if (q < 3) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rj, (lds_vptr)(&s_vv[u][0][2 * q][0]), 16, (unsigned)vlo[l], 0, 0, 0);
        asm volatile("; (jk)");
      } else if (q < 6) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(ri, (lds_vptr)(&s_vv[u][1][2 * (q - 3)][0]), 16, (unsigned)vlo[l], 0, 0, 0);
        asm volatile("; (ik)");
      }
    }
    if (wid == 3) {
      // T1 of k, up to the end of T1
      const int k = k0 + kk;
      const __amdgpu_buffer_rsrc_t rt = uniform_rsrc(reinterpret_cast<const char*>(t1p + (int64_t)v * k), 8 * v * (o - k));
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rt, (lds_vptr)(&s_t1[u][0]), 4, (unsigned)t1lo, 0, 0, 0);
    }
  };
  // the thread's two elements: a and b from the lane, c from the wave and h
  const int x = lane & 7, y = lane >> 3;
  const int a = blk[0] * CT + x, b = blk[1] * CT + y;
#pragma unroll
  for (int u = 0; u < KD; ++u)
    if (u < nk) copy(u, u);
  auto t1 = [&](int e, int q) { return e < v ? t1p[e + (int64_t)v * q] : 0.0; };
  auto ij = [&](int P, int Q, int r, int q) { return vv_ij[((int64_t)(blk[P] + nb * blk[Q]) << 6) + r + 8 * q]; };
  const double ia = t1(a, i), ib = t1(b, i), ja = t1(a, j), jb = t1(b, j);
  const double ij_ab = ij(0, 1, x, y), ij_ba = ij(1, 0, y, x);
  double ic[2], jc[2], ij_ac[2], ij_ca[2], ij_bc[2], ij_cb[2], es[2];
  float wt[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int z = wid + 4 * h, c = blk[2] * CT + z;
    ic[h] = t1(c, i);
    jc[h] = t1(c, j);
    ij_ac[h] = ij(0, 2, x, z);
    ij_ca[h] = ij(2, 0, z, x);
    ij_bc[h] = ij(1, 2, y, z);
    ij_cb[h] = ij(2, 1, z, y);
    const bool in = a < v && b < v && c < v && a >= b && b >= c && a > c;
    wt[h] = in ? (a == b || b == c ? 0.5f : 1.0f) : 0.0f;
    es[h] = in ? ev[a] + ev[b] + ev[c] : 0.0;
  }
  double acc = 0.0;
  const double eij = eo[i] + eo[j];
  auto one = [&](int kk, int u) {
    const int k = k0 + kk;
    const TW* Wu = Wl[u];
    const double ka = s_t1[u][x], kb = s_t1[u][8 + y], kc[2] = {s_t1[u][16 + wid], s_t1[u][20 + wid]};
    TW wv[2][6];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int z = wid + 4 * h;
      wv[h][0] = Wu[0 * CT3 + cube_off<TW>(x, y, z)];
      wv[h][1] = Wu[1 * CT3 + cube_off<TW>(x, z, y)];
      wv[h][2] = Wu[2 * CT3 + cube_off<TW>(y, x, z)];
      wv[h][3] = Wu[3 * CT3 + cube_off<TW>(y, z, x)];
      wv[h][4] = Wu[4 * CT3 + cube_off<TW>(z, x, y)];
      wv[h][5] = Wu[5 * CT3 + cube_off<TW>(z, y, x)];
    }
    // V - W of the six orderings
    const double jk_ab = s_vv[u][0][0][x + 8 * y], jk_ba = s_vv[u][0][1][y + 8 * x];
    const double ik_ab = s_vv[u][1][0][x + 8 * y], ik_ba = s_vv[u][1][1][y + 8 * x];
    double uv[2][6];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int z = wid + 4 * h;
      const double jk_ac = s_vv[u][0][2][x + 8 * z], jk_ca = s_vv[u][0][3][z + 8 * x];
      const double jk_bc = s_vv[u][0][4][y + 8 * z], jk_cb = s_vv[u][0][5][z + 8 * y];
      const double ik_ac = s_vv[u][1][2][x + 8 * z], ik_ca = s_vv[u][1][3][z + 8 * x];
      const double ik_bc = s_vv[u][1][4][y + 8 * z], ik_cb = s_vv[u][1][5][z + 8 * y];
      uv[h][0] = fma(ia, jk_bc, fma(ik_ac, jb, ij_ab * kc[h]));
      uv[h][1] = fma(ia, jk_cb, fma(ik_ab, jc[h], ij_ac[h] * kb));
      uv[h][2] = fma(ib, jk_ac, fma(ik_bc, ja, ij_ba * kc[h]));
      uv[h][3] = fma(ib, jk_ca, fma(ik_ba, jc[h], ij_bc[h] * ka));
      uv[h][4] = fma(ic[h], jk_ab, fma(ik_cb, ja, ij_ca[h] * kb));
      uv[h][5] = fma(ic[h], jk_ba, fma(ik_ca, jb, ij_cb[h] * ka));
    }
    if (u == KD - 1) {
      lds_barrier();  // every wave has read these k
#pragma unroll
      for (int q = 0; q < KD; ++q)
        if (kk + 1 + q < nk) copy(kk + 1 + q, q);
    }
    const double D0 = eij + eo[k];
    double ak = 0.0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const double w0 = (double)wv[h][0], w1 = (double)wv[h][1], w2 = (double)wv[h][2], w3 = (double)wv[h][3],
                   w4 = (double)wv[h][4], w5 = (double)wv[h][5];
      const double v0 = w0 + uv[h][0], v1 = w1 + uv[h][1], v2 = w2 + uv[h][2], v3 = w3 + uv[h][3], v4 = w4 + uv[h][4],
                   v5 = w5 + uv[h][5];
      const double sp = v0 + v3 + v4, sm = v1 + v2 + v5, wp = w0 + w3 + w4, wm = w1 + w2 + w5;
      const double xx = fma(w0, v0, fma(w1, v1, fma(w2, v2, fma(w3, v3, fma(w4, v4, w5 * v5)))));
      const double ef = fma(3.0, xx, fma(wp, fma(-2.0, sm, sp), wm * fma(-2.0, sp, sm)));
      ak += wt[h] != 0.0f ? (double)wt[h] * ef * rcp_nr(D0 - es[h]) : 0.0;
    }
    acc += (2.0 - (i == j ? 1.0 : 0.0) - (j == k ? 1.0 : 0.0)) * ak;
  };
  for (int kk = 0; kk < nk; kk += KD) {
    wait_vmcnt<0>();
    __syncthreads();
#pragma unroll
    for (int u = 0; u < KD; ++u)
      if (kk + u < nk) one(kk + u, u);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
  if (lane == 0) red[wid] = acc;
  __syncthreads();
  if (tid == 0) partials[blockIdx.x + (int64_t)gridDim.x * blockIdx.y] = red[0] + red[1] + red[2] + red[3];
}

int triples_orbit_count(int v) {
  const int nb = (v + CT - 1) / CT;
  return nb * (nb + 1) * (nb + 2) / 6;
}

// The orbits a >= b >= c of 8-wide cubes, in blocks of 4 x 4 x 4 cube indices: the orbits of a block share their
// (jb|kc) and (ia|kc) blocks, 96 of them for up to 64 orbits of 12 each; with the orbits of a block consecutive, and
// consecutive orbits on one XCD (k_triples_energy), those reads meet in its L2.
void triples_orbits(int v, std::vector<int>& out) {
  const int nb = (v + CT - 1) / CT;
  const int ng = (nb + 3) / 4;
  out.clear();
  for (int ga = 0; ga < ng; ++ga)
    for (int gb = 0; gb <= ga; ++gb)
      for (int gc = 0; gc <= gb; ++gc)
        for (int a = 4 * ga; a < std::min(nb, 4 * ga + 4); ++a)
          for (int b = 4 * gb; b < std::min(a + 1, 4 * gb + 4); ++b)
            for (int c = 4 * gc; c < std::min(b + 1, 4 * gc + 4); ++c) {
              out.push_back(a);
              out.push_back(b);
              out.push_back(c);
            }
}

// (ia|jb) = vvoo[a + v b + v^2 (i + o j)] -> vvb in 8x8 blocks (zero-padded), so that a staged
// block is one contiguous 512-byte run
__global__ void k_block_vv(int o, int v, int nb, const double* __restrict__ vvoo, double* __restrict__ vvb) {
  const int64_t PS = (int64_t)nb * nb * CT * CT, n = PS * o * o;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) {
    const int64_t pq = e / PS;
    const int64_t r = e - pq * PS;
    const int xy = (int)(r & 63);
    const int64_t blkid = r >> 6;
    const int A = (int)(blkid % nb), B = (int)(blkid / nb);
    const int a = A * CT + (xy & 7), b = B * CT + (xy >> 3);
    vvb[e] = (a < v && b < v) ? vvoo[a + (int64_t)v * b + (int64_t)v * v * pq] : 0.0;
  }
}

int64_t triples_vv_blocked_elems(int o, int v) {
  const int64_t nb = (v + CT - 1) / CT;
  return nb * nb * CT * CT * o * o;
}

void triples_block_vv(hipStream_t s, int o, int v, const double* vvoo, double* vvb) {
  const int nb = (v + CT - 1) / CT;
  const int64_t n = triples_vv_blocked_elems(o, v);
  const int64_t g = std::min<int64_t>((n + 255) / 256, 65536 * 4);
  hipLaunchKernelGGL(k_block_vv, dim3((unsigned)g), dim3(256), 0, s, o, v, nb, vvoo, vvb);
  FH_HIP(hipGetLastError());
}

// k values per workgroup: enough workgroups to fill the chip several times over, and a run of k long enough
// to amortise the k-independent loads (runs of 8, 16, 24, 32 at o = 40, v = 190: 102, 97, 95, 95 ms;
// FERMIHIP_TRIPLES_KPW = n fixes it, for tuning and for the tests that compare runs of k)
int triples_energy_kpw(int norb, int nslot) {
  int kpw = 1;
  while (kpw < 32 && (int64_t)norb * ((nslot + 2 * kpw - 1) / (2 * kpw)) >= 4096) kpw *= 2;
  if (const char* env = std::getenv("FERMIHIP_TRIPLES_KPW")) kpw = std::max(1, std::min(64, std::atoi(env)));
  return kpw;
}

template <typename TW>
void triples_energy(hipStream_t s, int o, int v, int nrun, const int* runs, const TW* W, int norb, const int* orbits,
                    const double* t1p, const double* vvb, const double* eo, const double* ev, double* partials) {
  FH_CHECK(nrun > 0 && nrun < 65536 && norb <= max_workgroups(256), -3, "(T) energy: too many runs in a launch");
  hipLaunchKernelGGL(k_triples_energy<TW>, dim3((unsigned)norb, (unsigned)nrun), dim3(256), 0, s, o, v,
                     reinterpret_cast<const int4*>(runs), W, orbits, t1p, vvb, eo, ev, partials);
  FH_HIP(hipGetLastError());
}
template void triples_energy<double>(hipStream_t, int, int, int, const int*, const double*, int, const int*,
                                     const double*, const double*, const double*, const double*, double*);
template void triples_energy<float>(hipStream_t, int, int, int, const int*, const float*, int, const int*, const double*,
                                    const double*, const double*, const double*, double*);

// ------------------------------------------------------------------ host side of the W build
// k values per row, zero-padded to whole groups of 8, so that two segments are whole 64-byte steps
int64_t triples_pitch_elems(int o, int v) { return ((int64_t)(v + o) + 7) / 8 * 8; }

void triples_operands(hipStream_t s, int fmt, int o, int v, const double* ovvv, const double* t2, const double* ooov,
                      void* av, void* avs, void* bvp, void* bvq) {
  const int nd = (int)triples_pitch_elems(o, v);
  // along three axes: as one, v = 1300 has 17 million workgroups, more than an axis takes (max_workgroups)
  const int64_t n4 = (v + 3) / 4, ng = nd / 8, np = ((int64_t)o * o + 31) / 32;
  FH_CHECK(n4 < 65536 && ng < 65536 && np < 65536, -3, "(T) operand grid too large");
  const dim3 ga((unsigned)n4, (unsigned)n4, (unsigned)ng), gb((unsigned)n4, (unsigned)ng, (unsigned)np);
#define FH_OPS(F)                                                                                                     \
  do {                                                                                                                \
    hipLaunchKernelGGL(k_triples_av<F>, ga, dim3(256), 0, s, o, v, nd, ovvv, t2, (char*)av, (char*)avs);              \
    hipLaunchKernelGGL(k_triples_bv<F>, gb, dim3(256), 0, s, o, v, nd, t2, ooov, (char*)bvp, (char*)bvq);             \
  } while (0)
  if (fmt == 0) FH_OPS(0);
  else if (fmt == 1) FH_OPS(1);
  else FH_OPS(2);
#undef FH_OPS
  FH_HIP(hipGetLastError());
}

// Tile of an axis of n elements: fmt 2: blocks of 32, at most 2 MB of them; else blocks of 16, at most NB
TriplesTiles triples_tiles(int fmt, int o, int v, double nk) {
  TriplesTiles t;
  const int64_t vv = (int64_t)v * v;
  FH_CHECK(vv < ((int64_t)1 << 31), -3, "(T): v^2 exceeds 32 bits");
  auto tiles = [](int64_t n, int g, int per) { return (int)(((n + g - 1) / g + per - 1) / per); };
  if (fmt == 2) {
    // Tiles of up to 6 x 6 blocks of 32, and the 128 x 128 kernel (three workgroups per CU instead of two) where the
    // slices' tiles come to 4 x 4 at most: slices at o = 14, v = 60, 97, 120, 200 0.61, 2.35, 3.84, 32.3 ms, with the
    // 192 x 192 kernel 0.84, 2.95, 4.63, 41.6.  (A 160 x 160 kernel with a fourth ring slot for five blocks was 1 %
    // slower at o = 27, v = 131.)  The first launch has v^2 rows, and tiles of 4 blocks only where v fits one.
    const int nblk = (v + 31) / 32, nt = tiles(v, 32, 6);
    t.grain = 32;
    t.per = 6;
    t.nb = nblk <= 4 * nt ? 2 : 3;
    t.nb_first = v <= 128 ? 2 : 3;
  } else {
    // slices: the block count with the least padded area, wider tiles preferred (operand reuse: a tile reads 2 / NB of a
    // block per block product, at 0.3 of a product's cost).  Of NB = 2 .. 6 at v = 19, 40, 62, 76, 100, 131 and 190
    // it takes the fastest, FP64 and FP32, but for v = 131 in FP64 (3: 15.9 ms, 5: 14.2); others cost up to 2.3 times
    // as much (v = 76 in FP64 5.5 ms with 5, 13.0 with 4)
    auto best = [&](int64_t m, int64_t n) {
      int nb = 2;
      double c0 = 1e300;
      for (int b = 2; b <= 6; ++b) {
        const double pm = 16.0 * b * tiles(m, 16, b), pn = 16.0 * b * tiles(n, 16, b);
        const double cost = pm * pn * (1.0 + 0.6 / b);
        if (cost < c0) { c0 = cost; nb = b; }
      }
      return nb;
    };
    t.nb = best(v, v);
    t.nb_first = best(vv, std::max<int64_t>(1, (int64_t)(v * nk)));
    t.grain = 16;
    t.per = t.nb;
  }
  t.per_first = fmt == 2 ? 2 * t.nb_first : t.nb_first;
  // the columns of a first-launch tile are planes apart and have to fit a buffer resource: tiles of fewer blocks from
  // v = 1673 on
  while (fmt == 2 && t.per_first > 1 && triples_plane(v) * t.grain * t.per_first * 4 >= ((int64_t)1 << 31)) --t.per_first;
  t.nt = tiles(v, t.grain, t.per);
  t.nt_first = tiles(vv, t.grain, t.per_first);
  (void)o;
  return t;
}
void triples_col_tiles(const TriplesTiles& t, int v, int i, int j, int k0, int nk, int slot, std::vector<int>& out) {
  const int n = v * nk, nt = ((n + t.grain - 1) / t.grain + t.per_first - 1) / t.per_first;
  for (int q = 0; q < nt; ++q) {
    const int n0 = tile_begin(n, t.grain, nt, q), n1 = std::min(tile_begin(n, t.grain, nt, q + 1), n);
    out.insert(out.end(), {i, j, k0, slot, n0, n1 - n0, 0, 0});
  }
}

// 1 GiB of W a chunk (and 2048 slice tiles, four rounds of 512): the (T) of o = 40, v = 190 takes 960, 830,
// 782, 763 and 757 ms at 128, 256, 512, 1024 and 4096 MiB (fewer partial rounds), o = 27, v = 131 100,
// 92.0, 86.4, 84.3 and 84.5 ms.  FERMIHIP_TRIPLES_CHUNK_MB fixes it, for tests.
int64_t triples_chunk_slots(int v, int elem, const TriplesTiles& tt, int64_t ntot) {
  const int64_t slot = triples_plane(v) * v * elem, tiles = (int64_t)tt.nt * tt.nt * v;
  int64_t n = std::max(((int64_t)1 << 30) / slot, (2048 + tiles - 1) / tiles);
  if (const char* env = std::getenv("FERMIHIP_TRIPLES_CHUNK_MB")) n = (std::max<int64_t>(1, std::atoll(env)) << 20) / slot;
  n = std::min(n, std::min<int64_t>((int64_t)8e9 / slot, 60000));  // 60000: the energy launch's grid
  return std::max<int64_t>(1, std::min(n, ntot));
}

template <int NSEG>
static void launch_w(hipStream_t s, int fmt, int nb, int64_t g, const TripW& t) {
  FH_CHECK(g > 0 && g <= max_workgroups(fmt == 2 ? 256 : 64 * triples_w_waves(nb)), -3, "(T) W build: grid too large");
  const unsigned grid = (unsigned)g;
#define FH_W(T, NB) hipLaunchKernelGGL((k_triples_w<T, NSEG, NB>), dim3(grid), dim3(64 * triples_w_waves(NB)), 0, s, t)
#define FH_WT(T)               \
  switch (nb) {                \
    case 2: FH_W(T, 2); break; \
    case 3: FH_W(T, 3); break; \
    case 4: FH_W(T, 4); break; \
    case 5: FH_W(T, 5); break; \
    default: FH_W(T, 6); break; \
  }
  if (fmt == 2) {
    if (nb == 2) hipLaunchKernelGGL((k_triples_w_bf3<NSEG, 2>), dim3(grid), dim3(256), 0, s, t);
    else hipLaunchKernelGGL((k_triples_w_bf3<NSEG, 3>), dim3(grid), dim3(256), 0, s, t);
  } else if (fmt == 1) {
    FH_WT(float)
  } else {
    FH_WT(double)
  }
#undef FH_WT
#undef FH_W
  FH_HIP(hipGetLastError());
}

static TripW trip_args(int fmt, int o, int v, const TriplesTiles& tt, const TriplesOperands& op, void* W, const int* slots,
                       const int* cols) {
  TripW t;
  t.av = static_cast<const char*>(op.av);
  t.avs = static_cast<const char*>(op.avs);
  t.bvp = static_cast<const char*>(op.bvp);
  t.bvq = static_cast<const char*>(op.bvq);
  t.w = W;
  t.slots = reinterpret_cast<const int4*>(slots);
  t.cols = reinterpret_cast<const int4*>(cols);
  t.o = o;
  t.v = v;
  t.nd = (int)triples_pitch_elems(o, v);
  // offsets inside a k step of an operand tile and inside an output tile are 32-bit byte offsets
  FH_CHECK(triples_plane(v) * tt.grain * tt.per_first * (fmt == 2 ? 4 : 1) < ((int64_t)1 << 31) &&
               (192 + 2 * (int64_t)v) * t.nd * 8 < ((int64_t)1 << 31),
           -3, "(T) W build: a tile exceeds 32-bit offsets");
  return t;
}
void triples_w_first(hipStream_t s, int fmt, int o, int v, const TriplesTiles& tt, const TriplesOperands& op, void* W,
                     const int* cols, int ncol) {
  TripW t = trip_args(fmt, o, v, tt, op, W, nullptr, cols);
  t.nt = tt.nt_first;
  t.ncol = ncol;
  t.group = 1;
  const int64_t g = (int64_t)tt.nt_first * ncol;
  launch_w<2>(s, fmt, tt.nb_first, g, t);
}
void triples_w_slices(hipStream_t s, int fmt, int o, int v, const TriplesTiles& tt, const TriplesOperands& op, void* W,
                      const int* slots, int nslot) {
  TripW t = trip_args(fmt, o, v, tt, op, W, slots, nullptr);
  t.nt = tt.nt;
  t.ncol = nslot;
  t.group = kSlotGroup;
  const int64_t g = (int64_t)tt.nt * tt.nt * v * nslot;
  launch_w<4>(s, fmt, tt.nb, g, t);
}

}  // namespace fh
