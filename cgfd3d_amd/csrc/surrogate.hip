// Surrogate network kernels: BF16 MFMA GEMMs with FP32 accumulation and the
// small elementwise/reduction kernels that training needs (loss gradient,
// column sums, Adam).  Every layer of the network (the MLP and the 1-D
// transposed convolutions with kernel = stride, whose channels-last layout
// makes them plain GEMMs) runs through cgfds_gemm_bf16.
//
// Storage: bf16 values are raw 16-bit words (upper half of an IEEE binary32,
// round-to-nearest-even on conversion); matrices are row-major with explicit
// leading dimensions in elements.
#include <algorithm>
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <type_traits>

#include "cgfdh.h"
#include "cgfds.h"

int cgfdh_internal_fail(int code, const char* msg);

namespace cgfds {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

static int sfail(int code, const char* what)
{
  return cgfdh_internal_fail(code, what);
}

__device__ __forceinline__ uint16_t f2bf(float f)
{
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0;   // NaN stays NaN
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// bf16 value > 0 (the ReLU mask of a stored activation)
__device__ __forceinline__ bool bf_pos(uint16_t h) { return h != 0 && !(h & 0x8000u); }

struct GemmArgs {
  int M, N, K;
  const uint16_t* A;
  long lda;
  const uint16_t* B;
  long ldb;
  const float* bias;
  int epi;                // EPI_* below
  const uint16_t* mask;   // EPI_MASK: bf16 [M][ldm]
  long ldm;
  float* C32;
  long ldc32;
  uint16_t* C16;
  long ldc16;
  int kchunk;             // K range per blockIdx.z, multiple of 32
  float* work;            // split-K partials [gridDim.z][M][N] (then no epilogue)
  int vec16;              // mask and C16 rows allow 16-byte accesses
  int order, mt, nt, S;   // block order (below), row and column tiles, K splits
  // column sums of B (opA transposed, B not: the bias gradient beside the
  // weight gradient): [N], or with work its partials behind the products'
  float* csum;
  // moment-tensor contraction of the rows (N <= BN): y[r][t][c] = sum over k of
  // mten[r / rps][k] * C[r][t][k][c], k below nk, c below nc
  const float* mten;
  float* y;
  int nk, nc, rps;
};

// The order of the blocks.  Blocks go to the 8 XCDs in turn, each with its own
// L2, and those that read the same rows belong on one of them, close together:
// ORD_ROWS the column tiles of a row tile, ORD_SPLIT all tiles of one range of
// the contraction.  us in plain order and so: 262144 x 512 x 256 232, 216;
// 1048576 x 512 x 128 722, 671; 256 x 512 x 32768 in 16 splits 41, 38; too few
// row tiles or splits would leave XCDs idle and stay in plain order.
enum { ORD_PLAIN = 0, ORD_ROWS = 1, ORD_SPLIT = 2 };

// a launch holds below 2^32 threads in x: more blocks than these go on in y
constexpr unsigned GRID_X = 1u << 20;

static dim3 gemm_grid(long blocks)
{
  return dim3((unsigned)std::min(blocks, (long)GRID_X), (unsigned)((blocks + GRID_X - 1) / GRID_X));
}

__device__ __forceinline__ bool gemm_tile(const GemmArgs& g, int& x, int& y, int& z)
{
  const unsigned f = blockIdx.y * GRID_X + blockIdx.x, q = f / 8, xcd = f % 8;
  if (g.order == ORD_ROWS) {
    x = q / g.nt * 8 + xcd;
    y = q % g.nt;
    z = 0;
    return x < g.mt;
  }
  const unsigned tiles = (unsigned)g.mt * g.nt;
  const unsigned t = g.order == ORD_SPLIT ? q % tiles : f % tiles;
  z = g.order == ORD_SPLIT ? q / tiles * 8 + xcd : f / tiles;
  x = t % g.mt;
  y = t / g.mt;
  return z < g.S;
}

constexpr int MT_MAX = 8;   // basis terms of a moment-tensor output

enum { EPI_NONE = 0, EPI_RELU = 1, EPI_MASK = 2 };

// ---------------------------------------------------------------------------
// GEMM
// ---------------------------------------------------------------------------

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));

constexpr unsigned OUT = ~15u;   // an offset past every operand: loads zeros

__device__ const uint16_t zero16[8] __attribute__((aligned(16))) = {};

// One operand's tile, loaded straight to LDS 16 bytes a lane.  KC: the
// contraction index is the contiguous one, R rows of BK; otherwise BK rows of R.
// Inside a row the 16-byte chunks are exchanged by an exclusive or with bits of
// the row, so that the 16 rows (KC) or the 4 x 2 rows (not KC) a fragment reads
// at one chunk lie in different banks.  WIDE: leading dimensions beyond the
// 32-bit offsets, by 64-bit addresses.
template <bool KC, int R, int BK, int NT, bool WIDE> struct Operand {
  static constexpr int ROWS = KC ? R : BK, COLS = KC ? BK : R;
  static constexpr int CH = COLS / 8;             // chunks of a row
  static constexpr int N = ROWS * CH / NT;        // loads of a thread
  static_assert(ROWS * CH % NT == 0 && (CH & (CH - 1)) == 0, "");

  // whether the rows of a wave's load are too far apart for a lane's 32-bit
  // byte offset: 64 / CH rows, 16 of a tile of 32 columns, so from leading
  // dimensions of 143 million on there and 307 or 716 million elsewhere
  static bool too_wide(long ld) { return ld > (long)(OUT / 2 - 8 * CH) / (64 / CH - 1); }

  static __device__ __forceinline__ int swz(int r)
  {
    if (KC) return r & (CH < 8 ? CH - 1 : 7);
    return ((r & 3) << 1 & (CH - 1)) ^ (CH >= 16 ? (r >> 3 & 1) << 3 : 0);
  }

  // the tile at contraction index k of the operand whose first row (KC) or
  // column is r0 of nr
  static __device__ __forceinline__ void load(const uint16_t* base, long ld, int r0, int nr, int k,
                                              int ke, uint16_t* lds)
  {
    const uint16_t* p = base + (KC ? (long)r0 * ld + k : (long)k * ld + r0);
    const int t = threadIdx.x, w = __builtin_amdgcn_readfirstlane(t >> 6);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      // the wave's first row by scalar arithmetic, the lanes' distance to it (at
      // most 16 rows) in the 32-bit offset
      const int rw = (i * NT + w * 64) / CH;
      const int id = i * NT + t, r = id / CH, c = (id % CH) ^ swz(r);
      const bool ok = KC ? (r0 + r < nr && k + 8 * c < ke) : (k + r < ke && r0 + 8 * c < nr);
      if (WIDE) {
        const uint16_t* q = ok ? p + (r * ld + 8 * c) : zero16;
        __builtin_amdgcn_global_load_lds(
            (const __attribute__((address_space(1))) void*)q,
            (__attribute__((address_space(3))) void*)(lds + (long)(i * NT + w * 64) * 8), 16, 0, 0);
        continue;
      }
      const __amdgpu_buffer_rsrc_t q = __builtin_amdgcn_make_buffer_rsrc(
          (void*)(p + rw * ld), 0, (int)0xfffffff0, 0x00020000);
      const unsigned off = ok ? (unsigned)((r - rw) * (unsigned)ld + 8 * c) * 2u : OUT;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          q, (__attribute__((address_space(3))) void*)(lds + (long)(i * NT + w * 64) * 8), 16,
          (int)off, 0, 0, 0);
    }
  }

  // the MFMA fragment of rows r .. r+15 at contraction indices kk .. kk+31:
  // lane l holds row l%16, k = 8*(l/16) .. +7
  static __device__ __forceinline__ bf16x8 frag(const uint16_t* lds, int r, int kk)
  {
    const int l = threadIdx.x & 63, l16 = l & 15, g = l >> 4;
    if (KC) {
      const int row = r + l16;
      return *(const bf16x8*)(lds + (row * CH + (((kk >> 3) + g) ^ swz(row))) * 8);
    }
    // the transposing read gives each lane of 16 one column of the 4 rows of
    // 16 that they address together
    const int k = kk + 8 * g + (l16 >> 2), col = r + 4 * (l16 & 3);
    const uint16_t* a = lds + (k * CH + ((col >> 3) ^ swz(k))) * 8 + (col & 7);
    union {
      s16x4 h[2];
      bf16x8 v;
    } u;
    typedef __attribute__((address_space(3))) s16x4* lp;
    u.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp)a);
    u.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp)(a + 4 * CH * 8));
    return u.v;
  }
};

// C[M][N] = sum_k opA[m][k] * opB[k][n].  opA = A ([M][K]) or, TA, A^T with A
// stored [K][M]; opB = B ([K][N]) or, TB, B^T with B stored [N][K].
// WM x WN waves over a BM x BN tile, each BM/WM x BN/WN in MFMA 16x16x32 tiles;
// NS stages of BK in a ring, NS - 1 of them in flight.  The products are formed
// as (B^T A^T): a lane then holds 4 neighbouring columns of one row of C, which
// leave in one 16- or 8-byte store.
template <int TA, int TB, int BM, int BN, int BK, int NS, int WM, int WN, bool WIDE = false>
__global__ __launch_bounds__(64 * WM * WN) void gemm_bf16_kernel(GemmArgs g)
{
  constexpr int NT = 64 * WM * WN;
  using OA = Operand<!TA, BM, BK, NT, WIDE>;
  using OB = Operand<TB, BN, BK, NT, WIDE>;
  constexpr int FM = BM / WM / 16, FN = BN / WN / 16;
  // the ring; behind the products the waves' output rows
  constexpr int RING = NS * (BM + BN) * BK, ROWS = BM * BN + 8 * BM * WN;
  __shared__ __attribute__((aligned(16))) uint16_t sm[RING > ROWS ? RING : ROWS];
  uint16_t *const As = sm, *const Bs = sm + NS * BM * BK;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int tx, ty, tz;
  if (!gemm_tile(g, tx, ty, tz)) return;
  const int m0 = tx * BM, n0 = ty * BN;
  const int kb = tz * g.kchunk;
  const int ke = min(g.K, kb + g.kchunk);
  const int wm = w / WN * (BM / WM), wn = w % WN * (BN / WN);
  // columns of 16 this wave has to form
  const int nj = min(FN, (g.N - n0 - wn + 15) / 16);
  // the waves of the first row tile that form the column sums of B
  const bool cs = TA && !TB && g.csum && m0 == 0 && wm == 0;
  f32x4 sums[FN];
  const bf16x8 ones = {(__bf16)1.f, (__bf16)1.f, (__bf16)1.f, (__bf16)1.f,
                       (__bf16)1.f, (__bf16)1.f, (__bf16)1.f, (__bf16)1.f};
#pragma unroll
  for (int j = 0; j < FN; ++j) sums[j] = (f32x4){0.f, 0.f, 0.f, 0.f};

  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

  const int nk = (ke - kb + BK - 1) / BK;
  auto load = [&](int s) {
    OA::load(g.A, g.lda, m0, g.M, kb + s * BK, ke, As + s % NS * (BM * BK));
    OB::load(g.B, g.ldb, n0, g.N, kb + s * BK, ke, Bs + s % NS * (BN * BK));
  };
  // what the epilogue adds is requested before the products: asked for behind
  // them it is a chain of latencies, longer than a short contraction itself
  f32x4 bias[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int c = n0 + wn + 16 * j + 4 * (lane >> 4);
    bias[j] = g.bias && c < g.N ? *(const f32x4u*)(g.bias + c) : (f32x4){0.f, 0.f, 0.f, 0.f};
  }
  constexpr int MTS = BN == 128 ? BM * MT_MAX : 1;
  __shared__ float ms[MTS];                    // moment tensors of the tile's samples
  const int smp0 = g.y ? m0 / g.rps : 0;
  if (BN == 128 && g.y) {
    const int n = ((min(m0 + BM, g.M) - 1) / g.rps - smp0 + 1) * g.nk;
    for (int q = threadIdx.x; q < n; q += NT) ms[q] = g.mten[(long)smp0 * g.nk + q];
  }
#pragma unroll
  for (int s = 0; s < NS - 1; ++s)
    if (s < nk) load(s);
  for (int s = 0; s < nk; ++s) {
    if (s + NS - 1 < nk) {
      load(s + NS - 1);
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NS - 1) * (OA::N + OB::N)) : "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    }
    const uint16_t *pa = As + s % NS * (BM * BK), *pb = Bs + s % NS * (BN * BK);
#pragma unroll
    for (int kk = 0; kk < BK; kk += 32) {
      bf16x8 a[FM], b[FN];
#pragma unroll
      for (int i = 0; i < FM; ++i) a[i] = OA::frag(pa, wm + 16 * i, kk);
#pragma unroll
      for (int j = 0; j < FN; ++j)
        if (j < nj) b[j] = OB::frag(pb, wn + 16 * j, kk);
#pragma unroll
      for (int j = 0; j < FN; ++j)
        if (j < nj) {
#pragma unroll
          for (int i = 0; i < FM; ++i)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], a[i], acc[i][j], 0, 0, 0);
        }
      if (TA && !TB && cs) {
#pragma unroll
        for (int j = 0; j < FN; ++j)
          if (j < nj) sums[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], ones, sums[j], 0, 0, 0);
      }
    }
    // the stage is read before it is loaded again
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  }

  // (every load has landed and been read: the stages' LDS is free)
  // D layout of a 16x16 MFMA tile: lane l holds rows (here columns of C)
  // 4*(l/16)+e, column (row of C) l%16
  if (TA && !TB && cs && (lane & 15) == 0) {
    float* o = g.work ? g.work + (long)g.S * g.M * g.N + (long)tz * g.N : g.csum;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int c = n0 + wn + 16 * j + 4 * (lane >> 4);
      if (c < g.N) *(f32x4u*)(o + c) = sums[j];
    }
  }
  // bf16 rows leave through the wave's own LDS, so that a store writes whole
  // 128-byte lines and not 32 bytes of each of 16 rows
  constexpr int WR = BM / WM, WC = BN / WN, WS = WC + 8;
  static_assert(WM * WN * WR * WS == ROWS, "");
  uint16_t* const st = sm + w * WR * WS;
  constexpr int CH = WC / 8, NQ = WR * CH / 64;  // 16-byte pieces of a row, of a lane
  static_assert(WR * CH % 64 == 0, "");
  u16x8 keep[NQ];
  float* const ct = (float*)sm;                // the block's rows for the contraction
  const bool staged = g.C16 && g.vec16 && !g.work;
  const bool masked = staged && g.epi == EPI_MASK;
  if (masked) {
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int q = i * 64 + lane, r = min(m0 + wm + q / CH, g.M - 1);
      const int c = min(n0 + wn + q % CH * 8, g.N - 8);
      keep[i] = *(const u16x8*)(g.mask + (long)r * g.ldm + c);
    }
  }
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int cw = 16 * j + 4 * (lane >> 4), c = n0 + wn + cw;
    if (c >= g.N) continue;          // N is a multiple of 8: all four or none
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int rw = 16 * i + (lane & 15), r = m0 + wm + rw;
      if (r >= g.M) continue;
      f32x4 v = acc[i][j];
      if (g.work) {
        *(f32x4u*)(g.work + ((long)tz * g.M + r) * g.N + c) = v;
        continue;
      }
      if (g.bias) v = v + bias[j];
      if (BN == 128 && g.y) {
        *(f32x4*)(ct + (wm + rw) * g.N + c) = v;
        continue;
      }
      if (g.epi == EPI_RELU) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = v[e] > 0.f ? v[e] : 0.f;
      }
      if (g.epi == EPI_MASK && (!staged || g.C32)) {
        const uint16_t* q = g.mask + (long)r * g.ldm + c;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = bf_pos(q[e]) ? v[e] : 0.f;
      }
      if (g.C32) *(f32x4u*)(g.C32 + (long)r * g.ldc32 + c) = v;
      if (g.C16) {
        u16x4 h;
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = f2bf(v[e]);
        if (staged) {
          *(u16x4*)(st + rw * WS + cw) = h;
        } else {
          uint16_t* q = g.C16 + (long)r * g.ldc16 + c;
          for (int e = 0; e < 4; ++e) q[e] = h[e];
        }
      }
    }
  }
  if (staged) {
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int q = i * 64 + lane, rw = q / CH, r = m0 + wm + rw, c = n0 + wn + q % CH * 8;
      u16x8 h = *(const u16x8*)(st + rw * WS + q % CH * 8);
      if (masked) {
#pragma unroll
        for (int e = 0; e < 8; ++e) h[e] = bf_pos(keep[i][e]) ? h[e] : (uint16_t)0;
      }
      if (r < g.M && c < g.N) *(u16x8*)(g.C16 + (long)r * g.ldc16 + c) = h;
    }
  }
  if (BN == 128 && g.y) {
    __syncthreads();
    const int rows = min(BM, g.M - m0), n4 = g.N / 4, no = g.N / g.nk;
    for (int q = threadIdx.x; q < rows * n4; q += NT) {
      const int r = q / n4, c = (q - r * n4) * 4;
      *(f32x4u*)(g.C32 + (long)(m0 + r) * g.ldc32 + c) = *(const f32x4*)(ct + r * g.N + c);
    }
    for (int q = threadIdx.x; q < rows * no; q += NT) {
      const int r = q / no, o = q - r * no, t = o / g.nc, c = o - t * g.nc;
      const float* m = ms + ((m0 + r) / g.rps - smp0) * g.nk;
      const float* a = ct + r * g.N + t * g.nk * g.nc + c;
      float v = m[0] * a[0];
      for (int k = 1; k < g.nk; ++k) v = v + m[k] * a[k * g.nc];
      g.y[(long)(m0 + r) * no + o] = v;
    }
  }
}

// out[r][c] = sum over s of work[s][r][c], and csum[c] the same of the partials
// [S][N] behind them.  G threads share an output's partials, every G-th each,
// and a tree over them closes it: the order is fixed (deterministic), and a sum
// of 128 or 256 partials is no serial chain of loads.  A thread holds E
// neighbouring outputs, E a divisor of N.  128 partials of 128 x 72 values took
// 31 us and 256 of 512 values 60 us with one thread an output, 5 us now.
template <int E>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(int S, int M, int N, int G,
                                                           const float* work, float* out,
                                                           long ldo, float* csum)
{
  typedef float vec __attribute__((ext_vector_type(E)));
  typedef float vecu __attribute__((ext_vector_type(E), aligned(4)));
  __shared__ vec part[256];
  const int L = 256 / G, l = threadIdx.x % L, zg = threadIdx.x / L;
  const long n = (long)M * N, i = ((long)blockIdx.x * L + l) * E;
  const long end = n + (csum ? N : 0);
  vec s = (vec)(0.f);
  if (i < end) {
    const float* p = i < n ? work + i : work + S * n + (i - n);
    const long step = i < n ? n : N;
#pragma unroll 4
    for (int z = zg; z < S; z += G) s = s + *(const vecu*)(p + z * step);
  }
  part[threadIdx.x] = s;
  __syncthreads();
  for (int h = G / 2; h > 0; h >>= 1) {
    if (zg < h) part[threadIdx.x] = part[threadIdx.x] + part[threadIdx.x + h * L];
    __syncthreads();
  }
  if (zg || i >= end) return;
  float* o = i < n ? out + i / N * ldo + i % N : csum + (i - n);
  *(vecu*)o = part[l];
}

static void launch_reduce(hipStream_t st, int S, int M, int N, const float* work, float* out,
                          long ldo, float* csum)
{
  const long n = (long)M * N + (csum ? N : 0), outs = N % 4 == 0 ? n / 4 : n;
  int G = 1;
  while (G < 32 && G * 4 <= S && outs * G * 2 < 1l << 31) G *= 2;   // a launch's threads
  const long L = 256 / G;
  if (N % 4 == 0)
    hipLaunchKernelGGL(splitk_reduce_kernel<4>, dim3((unsigned)((n / 4 + L - 1) / L)), dim3(256),
                       0, st, S, M, N, G, work, out, ldo, csum);
  else
    hipLaunchKernelGGL(splitk_reduce_kernel<1>, dim3((unsigned)((n + L - 1) / L)), dim3(256), 0,
                       st, S, M, N, G, work, out, ldo, csum);
}

// partial column sums of a bf16 matrix: block (x, y) sums rows of split y for
// 64 columns; 4 row lanes per column are combined in a fixed order
__global__ __launch_bounds__(256) void colsum_bf16_kernel(int M, int N, const uint16_t* G,
                                                         long ldg, int S, float* work)
{
  __shared__ float part[4][64];
  const int cx = threadIdx.x & 63, ry = threadIdx.x >> 6;
  const int c = blockIdx.x * 64 + cx;
  const long r0 = (long)M * blockIdx.y / S, r1 = (long)M * (blockIdx.y + 1) / S;
  float s = 0.f;
  if (c < N)
    for (long r = r0 + ry; r < r1; r += 4) s = s + bf2f(G[r * ldg + c]);
  part[ry][cx] = s;
  __syncthreads();
  if (ry == 0 && c < N)
    work[(long)blockIdx.y * N + c] = ((part[0][cx] + part[1][cx]) + part[2][cx]) + part[3][cx];
}

// per-sample relative squared misfit and its gradient, one block per sample:
// loss[b] = |Y_b - T_b|^2 / (tn2[b] + eps);  G_b = bf16(2 (Y_b - T_b) / (nsamp (tn2[b] + eps)))
__global__ __launch_bounds__(256) void loss_grad_kernel(long n, const float* Y, const float* T,
                                                       const float* tn2, float eps, int nsamp,
                                                       uint16_t* G, float* loss)
{
  __shared__ float red[256];
  const int b = blockIdx.x;
  const float den = tn2[b] + eps;
  const float scale = 2.0f / ((float)nsamp * den);
  const long o = (long)b * n;
  float s = 0.f;
  for (long i = threadIdx.x; i < n; i += 256) {
    const float d = Y[o + i] - T[o + i];
    s = s + d * d;
    if (G) G[o + i] = f2bf(d * scale);
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (threadIdx.x < h) red[threadIdx.x] = red[threadIdx.x] + red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) loss[b] = red[0] / den;
}

// Adam on FP32 master values; w16 (optional) receives the bf16 copy
__device__ __forceinline__ void adam_one(long i, float* w, float* m, float* v, const float* g,
                                         uint16_t* w16, float lr, float b1, float b2, float c1,
                                         float c2, float bc1, float bc2, float eps)
{
  const float gi = g[i];
  const float mi = b1 * m[i] + c1 * gi;
  const float vi = b2 * v[i] + c2 * (gi * gi);
  const float mh = mi / bc1, vh = vi / bc2;
  const float wi = w[i] - lr * (mh / (sqrtf(vh) + eps));
  m[i] = mi;
  v[i] = vi;
  w[i] = wi;
  if (w16) w16[i] = f2bf(wi);
}

__global__ void adam_kernel(long n, float* w, float* m, float* v, const float* g, uint16_t* w16,
                            float lr, float b1, float b2, float c1, float c2, float bc1, float bc2,
                            float eps)
{
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  adam_one(i, w, m, v, g, w16, lr, b1, b2, c1, c2, bc1, bc2, eps);
}

// the same for several tensors in one launch, 1024 values a block: a network's
// 16 launches, most of them a few blocks, took 56 us and the gaps between them,
// one takes 18
constexpr int ADAM_MAX = 32;
struct AdamList {
  int count;
  unsigned start[ADAM_MAX + 1];   // first block of each tensor
  long n[ADAM_MAX];
  float *w[ADAM_MAX], *m[ADAM_MAX], *v[ADAM_MAX];
  const float* g[ADAM_MAX];
  uint16_t* w16[ADAM_MAX];
};

__global__ __launch_bounds__(256) void adam_multi_kernel(AdamList a, float lr, float b1, float b2,
                                                        float c1, float c2, float bc1, float bc2,
                                                        float eps)
{
  int q = 0;
  while (q + 1 < a.count && blockIdx.x >= a.start[q + 1]) ++q;
  const long i0 = (long)(blockIdx.x - a.start[q]) * 1024 + threadIdx.x;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (i0 + e * 256 < a.n[q])
      adam_one(i0 + e * 256, a.w[q], a.m[q], a.v[q], a.g[q], a.w16[q], lr, b1, b2, c1, c2, bc1,
               bc2, eps);
}

// moment-tensor contraction of basis waveforms, one block per sample:
// y[b][t][c] = sum_k m[b][k] g[b][t][k][c] (k in increasing order).  NK terms,
// known when compiled: their loads leave together, not one latency after
// another; U indexes a sample, 32 bits wide where they suffice, for which a
// division is a few instructions.  2048 samples of 1024 x 3 x 6 values with
// misfit and gradient 112 us, 84 so.
template <int NK, typename U>
__global__ __launch_bounds__(256) void mt_contract_kernel(U nt, U nc,
                                                         const float* __restrict__ m,
                                                         const float* __restrict__ g,
                                                         float* __restrict__ y)
{
  const long b = blockIdx.x;
  float mk[NK];
#pragma unroll
  for (int k = 0; k < NK; ++k) mk[k] = m[b * NK + k];
  const U n = nt * nc;
  const float* gb = g + b * n * NK;
#pragma unroll 2
  for (U e = threadIdx.x; e < n; e += 256) {
    const U t = e / nc;
    const float* q = gb + (t * (NK - 1) * nc + e);
    float v = mk[0] * q[0];
#pragma unroll
    for (int k = 1; k < NK; ++k) v = v + mk[k] * q[k * nc];
    y[b * n + e] = v;
  }
}

// the contraction fused with the per-sample relative misfit and its gradient
// with respect to the basis waveforms: dg[b][t][k][c] = bf16(m[b][k] dy[b][t][c]),
// dy = 2 (y - T) / (nsamp (tn2[b] + eps))
template <int NK, typename U>
__global__ __launch_bounds__(256) void mt_loss_grad_kernel(
    U nt, U nc, const float* __restrict__ m, const float* __restrict__ g,
    const float* __restrict__ T, const float* __restrict__ tn2, float eps, int nsamp,
    uint16_t* __restrict__ dg, float* __restrict__ loss)
{
  __shared__ float red[256];
  const long b = blockIdx.x;
  float mk[NK];
#pragma unroll
  for (int k = 0; k < NK; ++k) mk[k] = m[b * NK + k];
  const float den = tn2[b] + eps;
  const float scale = 2.0f / ((float)nsamp * den);
  const U n = nt * nc;
  const float* gb = g + b * n * NK;
  uint16_t* db = dg ? dg + b * n * NK : nullptr;
  float s = 0.f;
#pragma unroll 2
  for (U e = threadIdx.x; e < n; e += 256) {
    const U o = e / nc * (NK - 1) * nc + e;
    float v = mk[0] * gb[o];
#pragma unroll
    for (int k = 1; k < NK; ++k) v = v + mk[k] * gb[o + k * nc];
    const float d = v - T[b * n + e];
    s = s + d * d;
    if (db) {
      const float dy = d * scale;
#pragma unroll
      for (int k = 0; k < NK; ++k) db[o + k * nc] = f2bf(mk[k] * dy);
    }
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (threadIdx.x < h) red[threadIdx.x] = red[threadIdx.x] + red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) loss[b] = red[0] / den;
}

// a kernel of the number of terms
#define CGFDS_TERMS(nk, F) \
  switch (nk) {            \
  case 1: F(1); break;     \
  case 2: F(2); break;     \
  case 3: F(3); break;     \
  case 4: F(4); break;     \
  case 5: F(5); break;     \
  case 6: F(6); break;     \
  case 7: F(7); break;     \
  default: F(8); break;    \
  }

__global__ void to_bf16_kernel(long n, const float* src, uint16_t* dst)
{
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = f2bf(src[i]);
}

static bool al16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

static int launch_check(const char* what)
{
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) return 0;
  char buf[256];
  snprintf(buf, sizeof buf, "%s: launch failed: %s", what, hipGetErrorString(e));
  return sfail(CGFDH_EDEVICE, buf);
}

}  // namespace cgfds

using namespace cgfds;

// what the products have in common: the checks, the split of the contraction,
// the tile, the order of the blocks, the launches
static int gemm_launch(const char* name, GemmArgs g, int transA, int transB, int splitk,
                       float* work, hipStream_t st)
{
  auto bad = [&](const char* why) {
    char buf[256];
    snprintf(buf, sizeof buf, "%s: %s", name, why);
    return sfail(CGFDH_EINVAL, buf);
  };
  const int M = g.M, N = g.N, K = g.K;
  if (M <= 0 || N <= 0 || K <= 0 || !g.A || !g.B || (!g.C32 && !g.C16))
    return bad("empty shape or null operand");
  if (M % 8 || N % 8 || K % 8 || g.lda % 8 || g.ldb % 8 || !al16(g.A) || !al16(g.B))
    return bad("M, N, K and the A/B leading dimensions must be multiples "
               "of 8 and A, B 16-byte aligned");
  if (g.lda < (transA ? M : K) || g.ldb < (transB ? K : N) || (g.C32 && g.ldc32 < N) ||
      (g.C16 && g.ldc16 < N))
    return bad("leading dimension below the row length");
  if (g.epi < EPI_NONE || g.epi > EPI_MASK || (g.epi == EPI_MASK && (!g.mask || g.ldm < N)))
    return bad("bad epilogue or missing mask");
  if (splitk < 1 || splitk > 1024) return bad("splitk outside 1..1024");
  if ((N + 63) / 64 > 65535) return bad("N above 65535*64 columns");
  g.kchunk = ((K + splitk - 1) / splitk + 31) / 32 * 32;
  const int S = g.S = (K + g.kchunk - 1) / g.kchunk;
  if (S > 1 && (!work || !g.C32 || g.C16 || g.bias || g.epi != EPI_NONE))
    return bad("split-K needs a work buffer, FP32 output and no epilogue");
  g.work = S > 1 ? work : nullptr;
  auto vec = [](const void* p, long ld) { return !p || (al16(p) && ld % 8 == 0); };
  g.vec16 = vec(g.mask, g.ldm) && vec(g.C16, g.ldc16);
  const int form = (transA ? 2 : 0) + (transB ? 1 : 0);
  // Whole groups of blocks go to an XCD where there are enough of them: the
  // tiles of one range of the contraction read the same rows of A and B, the
  // column tiles of a row tile the same rows of A.
  auto shape = [&](int BM, int BN) {
    g.mt = (M + BM - 1) / BM;
    g.nt = (N + BN - 1) / BN;
    g.order = S >= 8 ? ORD_SPLIT : (S == 1 && g.nt > 1 && g.mt >= 64 ? ORD_ROWS : ORD_PLAIN);
    if (g.order == ORD_ROWS) return (long)((g.mt + 7) / 8 * 8) * g.nt;
    return (long)g.mt * g.nt * (g.order == ORD_SPLIT ? (S + 7) / 8 * 8 : S);
  };
  long blocks = 0;
  // whether an operand's rows are too far apart for a tile's 32-bit offsets
  auto too_wide = [&](auto bm, auto bn, auto bk) {
    constexpr int BM = decltype(bm)::value, BN = decltype(bn)::value, BK = decltype(bk)::value;
    return (transA ? Operand<false, BM, BK, 256, false>::too_wide(g.lda)
                   : Operand<true, BM, BK, 256, false>::too_wide(g.lda)) ||
           (transB ? Operand<true, BN, BK, 256, false>::too_wide(g.ldb)
                   : Operand<false, BN, BK, 256, false>::too_wide(g.ldb));
  };
  bool wide = false;
  auto launch = [&](auto bm, auto bn, auto bk, auto ns, auto wm) {
    constexpr int BM = decltype(bm)::value, BN = decltype(bn)::value, BK = decltype(bk)::value,
                  NS = decltype(ns)::value, WM = decltype(wm)::value;
    wide = too_wide(bm, bn, bk);
    if (wide) return;
    blocks = shape(BM, BN);
    if (blocks > 0x7fffffffl) return;
    const dim3 grid = gemm_grid(blocks), blk(128 * WM);
    switch (form) {
    case 0: hipLaunchKernelGGL((gemm_bf16_kernel<0, 0, BM, BN, BK, NS, WM, 2>), grid, blk, 0, st, g); break;
    case 1: hipLaunchKernelGGL((gemm_bf16_kernel<0, 1, BM, BN, BK, NS, WM, 2>), grid, blk, 0, st, g); break;
    case 2: hipLaunchKernelGGL((gemm_bf16_kernel<1, 0, BM, BN, BK, NS, WM, 2>), grid, blk, 0, st, g); break;
    default: hipLaunchKernelGGL((gemm_bf16_kernel<1, 1, BM, BN, BK, NS, WM, 2>), grid, blk, 0, st, g); break;
    }
  };
#define CGFDS_I(n) std::integral_constant<int, n>{}
  // The largest tile that still leaves a block for each of the 256 compute
  // units: fewer bytes through LDS a product.  us, 128 x 128 and 64 x 64:
  // 2048 x 4096 x 512 (512 large tiles) 22, 31; 2048 x 512 x 512 (64) 13, 9.
  // Short contractions are bound by the latency of a block's loads and stores,
  // so the large tile has 8 waves: 1048576 x 512 x 128 493 us (2.7 TB/s), with 4
  // waves 595, in 64 x 128 tiles 582; 16384 x 4096 x 512 130, 144, 154.
  // Where even 64 x 64 leaves units idle the contraction is a serial chain, so
  // fewer, deeper stages and twice the tiles: 64 x 512 x 4096 28, 37; 512 x 512
  // x 4096 29, 51; level with 64 x 64 at K = 512 and below.
  const long big = (long)((M + 127) / 128) * ((N + 127) / 128) * S;
  const long mid = (long)((M + 63) / 64) * ((N + 63) / 64) * S;
  if (big >= 256) {
    launch(CGFDS_I(128), CGFDS_I(128), CGFDS_I(64), CGFDS_I(2), CGFDS_I(4));
  } else if (g.y) {
    // the contraction needs whole rows in a block
    wide = too_wide(CGFDS_I(64), CGFDS_I(128), CGFDS_I(64));
    if (!wide) {
      blocks = shape(64, 128);
      if (blocks > 0x7fffffffl) return bad("more than 2^31 - 1 tiles");
      hipLaunchKernelGGL((gemm_bf16_kernel<0, 0, 64, 128, 64, 3, 2, 2>), gemm_grid(blocks),
                         dim3(256), 0, st, g);
    }
  } else if (mid >= 256) {
    launch(CGFDS_I(64), CGFDS_I(64), CGFDS_I(64), CGFDS_I(3), CGFDS_I(2));
  } else {
    launch(CGFDS_I(64), CGFDS_I(32), CGFDS_I(128), CGFDS_I(4), CGFDS_I(2));
  }
  if (wide) {
    // one tile serves them: matrices of gigabytes of which few values are read
    blocks = g.y ? shape(64, 128) : shape(64, 32);
    const dim3 grid = gemm_grid(blocks), blk(256);
#define CGFDS_W(TA, TB) \
  hipLaunchKernelGGL((gemm_bf16_kernel<TA, TB, 64, 32, 128, 4, 2, 2, true>), grid, blk, 0, st, g)
    if (blocks > 0x7fffffffl) return bad("more than 2^31 - 1 tiles");
    if (g.y)
      hipLaunchKernelGGL((gemm_bf16_kernel<0, 0, 64, 128, 64, 3, 2, 2, true>), grid, blk, 0, st, g);
    else if (form == 0) CGFDS_W(0, 0);
    else if (form == 1) CGFDS_W(0, 1);
    else if (form == 2) CGFDS_W(1, 0);
    else CGFDS_W(1, 1);
#undef CGFDS_W
  }
#undef CGFDS_I
  if (blocks > 0x7fffffffl) return bad("more than 2^31 - 1 tiles");
  if (int rc = launch_check(name)) return rc;
  if (S > 1) {
    launch_reduce(st, S, M, N, work, g.C32, g.ldc32, g.csum);
    return launch_check(name);
  }
  return 0;
}

extern "C" int cgfds_gemm_bf16(int M, int N, int K, const void* A, long lda, int transA,
                               const void* B, long ldb, int transB, const float* bias,
                               int epilogue, const void* mask, long ldm, float* C32, long ldc32,
                               void* C16, long ldc16, int splitk, float* work, void* stream)
{
  GemmArgs g = {};
  g.M = M; g.N = N; g.K = K;
  g.A = (const uint16_t*)A; g.lda = lda;
  g.B = (const uint16_t*)B; g.ldb = ldb;
  g.bias = bias; g.epi = epilogue;
  g.mask = (const uint16_t*)mask; g.ldm = ldm;
  g.C32 = C32; g.ldc32 = ldc32;
  g.C16 = (uint16_t*)C16; g.ldc16 = ldc16;
  return gemm_launch("cgfds_gemm_bf16", g, transA, transB, splitk, work, (hipStream_t)stream);
}

extern "C" int cgfds_gemm_bf16_colsum(int M, int N, int K, const void* A, long lda, const void* G,
                                      long ldg, float* C32, long ldc32, float* csum, int splitk,
                                      float* work, void* stream)
{
  if (!C32 || !csum) return sfail(CGFDH_EINVAL, "cgfds_gemm_bf16_colsum: null output");
  GemmArgs g = {};
  g.M = M; g.N = N; g.K = K;
  g.A = (const uint16_t*)A; g.lda = lda;
  g.B = (const uint16_t*)G; g.ldb = ldg;
  g.C32 = C32; g.ldc32 = ldc32;
  g.csum = csum;
  return gemm_launch("cgfds_gemm_bf16_colsum", g, 1, 0, splitk, work, (hipStream_t)stream);
}

extern "C" int cgfds_gemm_bf16_mt(int M, int N, int K, const void* A, long lda, const void* B,
                                  long ldb, const float* bias, float* C32, long ldc32, int nk,
                                  int nc, int rps, const float* m, float* y, void* stream)
{
  if (!C32 || !m || !y || nk < 1 || nk > MT_MAX || nc < 1 || rps < 1 || N > 128 ||
      (long)N % ((long)nk * nc))
    return sfail(CGFDH_EINVAL, "cgfds_gemm_bf16_mt: bad argument (N must be a multiple of "
                               "nk * nc of at most 128, nk 1..8)");
  GemmArgs g = {};
  g.M = M; g.N = N; g.K = K;
  g.A = (const uint16_t*)A; g.lda = lda;
  g.B = (const uint16_t*)B; g.ldb = ldb;
  g.bias = bias;
  g.C32 = C32; g.ldc32 = ldc32;
  g.mten = m; g.y = y; g.nk = nk; g.nc = nc; g.rps = rps;
  return gemm_launch("cgfds_gemm_bf16_mt", g, 0, 0, 1, nullptr, (hipStream_t)stream);
}

extern "C" int cgfds_colsum_bf16(int M, int N, const void* G, long ldg, float* out, int splits,
                                 float* work, void* stream)
{
  if (M <= 0 || N <= 0 || !G || !out || !work || ldg < N || splits < 1 || splits > 65535)
    return sfail(CGFDH_EINVAL, "cgfds_colsum_bf16: bad argument");
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(colsum_bf16_kernel, dim3((N + 63) / 64, splits), dim3(256), 0, st, M, N,
                     (const uint16_t*)G, ldg, splits, work);
  if (int rc = launch_check("cgfds_colsum_bf16")) return rc;
  launch_reduce(st, splits, 1, N, work, out, N, nullptr);
  return launch_check("cgfds_colsum_bf16 (reduce)");
}

extern "C" int cgfds_loss_grad(int nsamp, long n, const float* Y, const float* T,
                               const float* tnorm2, float eps, void* G16, float* loss,
                               void* stream)
{
  if (nsamp <= 0 || n <= 0 || !Y || !T || !tnorm2 || !loss)
    return sfail(CGFDH_EINVAL, "cgfds_loss_grad: bad argument");
  hipLaunchKernelGGL(loss_grad_kernel, dim3(nsamp), dim3(256), 0, (hipStream_t)stream, n, Y, T,
                     tnorm2, eps, nsamp, (uint16_t*)G16, loss);
  return launch_check("cgfds_loss_grad");
}

extern "C" int cgfds_adam(long n, float* w, float* m, float* v, const float* g, void* w16,
                          float lr, float b1, float b2, float c1, float c2, float bc1, float bc2,
                          float eps, void* stream)
{
  if (n <= 0 || !w || !m || !v || !g) return sfail(CGFDH_EINVAL, "cgfds_adam: bad argument");
  hipLaunchKernelGGL(adam_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, n, w, m, v, g, (uint16_t*)w16, lr, b1, b2, c1, c2, bc1,
                     bc2, eps);
  return launch_check("cgfds_adam");
}

extern "C" int cgfds_adam_multi(int count, const long* n, float* const* w, float* const* m,
                                float* const* v, const float* const* g, void* const* w16, float lr,
                                float b1, float b2, float c1, float c2, float bc1, float bc2,
                                float eps, void* stream)
{
  if (count <= 0 || !n || !w || !m || !v || !g || !w16)
    return sfail(CGFDH_EINVAL, "cgfds_adam_multi: bad argument");
  for (int q = 0; q < count; ++q)
    if (n[q] <= 0 || n[q] > 1l << 40 || !w[q] || !m[q] || !v[q] || !g[q])
      return sfail(CGFDH_EINVAL, "cgfds_adam_multi: bad tensor");
  for (int q0 = 0; q0 < count; q0 += ADAM_MAX) {
    AdamList a = {};
    a.count = std::min(ADAM_MAX, count - q0);
    for (int q = 0; q < a.count; ++q) {
      a.n[q] = n[q0 + q];
      a.w[q] = w[q0 + q]; a.m[q] = m[q0 + q]; a.v[q] = v[q0 + q]; a.g[q] = g[q0 + q];
      a.w16[q] = (uint16_t*)w16[q0 + q];
      const long end = a.start[q] + (a.n[q] + 1023) / 1024;
      if (end > 0x7fffffffl) return sfail(CGFDH_EINVAL, "cgfds_adam_multi: too many values");
      a.start[q + 1] = (unsigned)end;
    }
    hipLaunchKernelGGL(adam_multi_kernel, dim3(a.start[a.count]), dim3(256), 0,
                       (hipStream_t)stream, a, lr, b1, b2, c1, c2, bc1, bc2, eps);
    if (int rc = launch_check("cgfds_adam_multi")) return rc;
  }
  return 0;
}

extern "C" int cgfds_mt_contract(int nsamp, int nt, int nc, int nk, const float* m,
                                 const float* g, float* y, void* stream)
{
  if (nsamp <= 0 || nt <= 0 || nc <= 0 || nk < 1 || nk > MT_MAX || !m || !g || !y)
    return sfail(CGFDH_EINVAL, "cgfds_mt_contract: bad argument (nk must be 1..8)");
  auto launch = [&](auto u) {
    typedef decltype(u) U;
#define CGFDS_F(n)                                                                       \
  hipLaunchKernelGGL((mt_contract_kernel<n, U>), dim3(nsamp), dim3(256), 0,              \
                     (hipStream_t)stream, (U)nt, (U)nc, m, g, y)
    CGFDS_TERMS(nk, CGFDS_F)
#undef CGFDS_F
  };
  if ((double)nt * nc * nk < 2147483648.0) launch(0u);
  else launch(0ul);
  return launch_check("cgfds_mt_contract");
}

extern "C" int cgfds_mt_loss_grad(int nsamp, int nt, int nc, int nk, const float* m,
                                  const float* g, const float* T, const float* tnorm2, float eps,
                                  void* dg16, float* loss, void* stream)
{
  if (nsamp <= 0 || nt <= 0 || nc <= 0 || nk < 1 || nk > MT_MAX || !m || !g || !T || !tnorm2 ||
      !loss)
    return sfail(CGFDH_EINVAL, "cgfds_mt_loss_grad: bad argument (nk must be 1..8)");
  auto launch = [&](auto u) {
    typedef decltype(u) U;
#define CGFDS_F(n)                                                                       \
  hipLaunchKernelGGL((mt_loss_grad_kernel<n, U>), dim3(nsamp), dim3(256), 0,             \
                     (hipStream_t)stream, (U)nt, (U)nc, m, g, T, tnorm2, eps, nsamp,     \
                     (uint16_t*)dg16, loss)
    CGFDS_TERMS(nk, CGFDS_F)
#undef CGFDS_F
  };
  if ((double)nt * nc * nk < 2147483648.0) launch(0u);
  else launch(0ul);
  return launch_check("cgfds_mt_loss_grad");
}

extern "C" int cgfds_f32_to_bf16(long n, const float* src, void* dst, void* stream)
{
  if (n <= 0 || !src || !dst) return sfail(CGFDH_EINVAL, "cgfds_f32_to_bf16: bad argument");
  hipLaunchKernelGGL(to_bf16_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, n, src, (uint16_t*)dst);
  return launch_check("cgfds_f32_to_bf16");
}
