// Surrogate network kernels: BF16 MFMA GEMMs with FP32 accumulation and the
// small elementwise/reduction kernels that training needs (loss gradient,
// column sums, Adam).  Every layer of the network (the MLP and the 1-D
// transposed convolutions with kernel = stride, whose channels-last layout
// makes them plain GEMMs) runs through cgfds_gemm_bf16.
//
// Storage: bf16 values are raw 16-bit words (upper half of an IEEE binary32,
// round-to-nearest-even on conversion); matrices are row-major with explicit
// leading dimensions in elements.
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
  int vec16;              // mask and C16 rows allow 8-byte accesses
};

enum { EPI_NONE = 0, EPI_RELU = 1, EPI_MASK = 2 };

// ---------------------------------------------------------------------------
// GEMM
// ---------------------------------------------------------------------------

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));

constexpr unsigned OUT = ~15u;   // an offset past every operand: loads zeros

// One operand's tile, loaded straight to LDS 16 bytes a lane.  KC: the
// contraction index is the contiguous one, R rows of BK; otherwise BK rows of R.
// Inside a row the 16-byte chunks are exchanged by an exclusive or with bits of
// the row, so that the 16 rows (KC) or the 4 x 2 rows (not KC) a fragment reads
// at one chunk lie in different banks.
template <bool KC, int R, int BK, int NT> struct Operand {
  static constexpr int ROWS = KC ? R : BK, COLS = KC ? BK : R;
  static constexpr int CH = COLS / 8;             // chunks of a row
  static constexpr int N = ROWS * CH / NT;        // loads of a thread
  static_assert(ROWS * CH % NT == 0 && (CH & (CH - 1)) == 0, "");
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
      const __amdgpu_buffer_rsrc_t q = __builtin_amdgcn_make_buffer_rsrc(
          (void*)(p + rw * ld), 0, (int)0xfffffff0, 0x00020000);
      const bool ok = KC ? (r0 + r < nr && k + 8 * c < ke) : (k + r < ke && r0 + 8 * c < nr);
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
template <int TA, int TB, int BM, int BN, int BK, int NS, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN) void gemm_bf16_kernel(GemmArgs g)
{
  constexpr int NT = 64 * WM * WN;
  using OA = Operand<!TA, BM, BK, NT>;
  using OB = Operand<TB, BN, BK, NT>;
  constexpr int FM = BM / WM / 16, FN = BN / WN / 16;
  __shared__ __attribute__((aligned(16))) uint16_t As[NS][BM * BK];
  __shared__ __attribute__((aligned(16))) uint16_t Bs[NS][BN * BK];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m0 = blockIdx.x * BM, n0 = blockIdx.y * BN;
  const int kb = blockIdx.z * g.kchunk;
  const int ke = min(g.K, kb + g.kchunk);
  const int wm = w / WN * (BM / WM), wn = w % WN * (BN / WN);
  // columns of 16 this wave has to form
  const int nj = min(FN, (g.N - n0 - wn + 15) / 16);

  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

  const int nk = (ke - kb + BK - 1) / BK;
  auto load = [&](int s) {
    // past the end the loads bring zeros, so that every turn waits for as many
    OA::load(g.A, g.lda, m0, g.M, kb + s * BK, s < nk ? ke : 0, As[s % NS]);
    OB::load(g.B, g.ldb, n0, g.N, kb + s * BK, s < nk ? ke : 0, Bs[s % NS]);
  };
#pragma unroll
  for (int s = 0; s < NS - 1; ++s) load(s);
  for (int s = 0; s < nk; ++s) {
    load(s + NS - 1);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NS - 1) * (OA::N + OB::N)) : "memory");
    const uint16_t *pa = As[s % NS], *pb = Bs[s % NS];
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
    }
    // the stage is read before it is loaded again
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  }

  // D layout of a 16x16 MFMA tile: lane l holds rows (here columns of C)
  // 4*(l/16)+e, column (row of C) l%16
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int c = n0 + wn + 16 * j + 4 * (lane >> 4);
    if (c >= g.N) continue;          // N is a multiple of 8: all four or none
    f32x4 bias = {0.f, 0.f, 0.f, 0.f};
    if (g.bias && !g.work) bias = *(const f32x4u*)(g.bias + c);
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int r = m0 + wm + 16 * i + (lane & 15);
      if (r >= g.M) continue;
      f32x4 v = acc[i][j];
      if (g.work) {
        *(f32x4u*)(g.work + ((long)blockIdx.z * g.M + r) * g.N + c) = v;
        continue;
      }
      if (g.bias) v = v + bias;
      if (g.epi == EPI_RELU) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = v[e] > 0.f ? v[e] : 0.f;
      }
      if (g.epi == EPI_MASK) {
        u16x4 h;
        const uint16_t* q = g.mask + (long)r * g.ldm + c;
        if (g.vec16) h = *(const u16x4*)q;
        else
          for (int e = 0; e < 4; ++e) h[e] = q[e];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = bf_pos(h[e]) ? v[e] : 0.f;
      }
      if (g.C32) *(f32x4u*)(g.C32 + (long)r * g.ldc32 + c) = v;
      if (g.C16) {
        u16x4 h;
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = f2bf(v[e]);
        uint16_t* q = g.C16 + (long)r * g.ldc16 + c;
        if (g.vec16) *(u16x4*)q = h;
        else
          for (int e = 0; e < 4; ++e) q[e] = h[e];
      }
    }
  }
}

// out[r][c] = sum over s of work[s][r][c], s in increasing order (deterministic)
__global__ void splitk_reduce_kernel(int S, int M, int N, const float* work, float* out, long ldo)
{
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long)M * N) return;
  const long r = i / N, c = i % N;
  float s = 0.f;
  for (int z = 0; z < S; ++z) s = s + work[(long)z * M * N + i];
  out[r * ldo + c] = s;
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
__global__ void adam_kernel(long n, float* w, float* m, float* v, const float* g, uint16_t* w16,
                            float lr, float b1, float b2, float c1, float c2, float bc1, float bc2,
                            float eps)
{
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
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

// moment-tensor contraction of basis waveforms, one block per sample:
// y[b][t][c] = sum_k m[b][k] g[b][t][k][c] (k in increasing order)
constexpr int MT_MAX = 8;

__global__ __launch_bounds__(256) void mt_contract_kernel(int nt, int nc, int nk, const float* m,
                                                         const float* g, float* y)
{
  const int b = blockIdx.x;
  float mk[MT_MAX];
  for (int k = 0; k < nk; ++k) mk[k] = m[b * nk + k];
  const long n = (long)nt * nc;
  const float* gb = g + (long)b * n * nk;
  for (long e = threadIdx.x; e < n; e += 256) {
    const long t = e / nc, c = e - t * nc;
    const float* q = gb + t * nk * nc + c;
    float v = mk[0] * q[0];
    for (int k = 1; k < nk; ++k) v = v + mk[k] * q[(long)k * nc];
    y[(long)b * n + e] = v;
  }
}

// the contraction fused with the per-sample relative misfit and its gradient
// with respect to the basis waveforms: dg[b][t][k][c] = bf16(m[b][k] dy[b][t][c]),
// dy = 2 (y - T) / (nsamp (tn2[b] + eps))
__global__ __launch_bounds__(256) void mt_loss_grad_kernel(int nt, int nc, int nk, const float* m,
                                                          const float* g, const float* T,
                                                          const float* tn2, float eps, int nsamp,
                                                          uint16_t* dg, float* loss)
{
  __shared__ float red[256];
  const int b = blockIdx.x;
  float mk[MT_MAX];
  for (int k = 0; k < nk; ++k) mk[k] = m[b * nk + k];
  const float den = tn2[b] + eps;
  const float scale = 2.0f / ((float)nsamp * den);
  const long n = (long)nt * nc;
  const float* gb = g + (long)b * n * nk;
  uint16_t* db = dg ? dg + (long)b * n * nk : nullptr;
  float s = 0.f;
  for (long e = threadIdx.x; e < n; e += 256) {
    const long t = e / nc, c = e - t * nc;
    const long o = t * nk * nc + c;
    float v = mk[0] * gb[o];
    for (int k = 1; k < nk; ++k) v = v + mk[k] * gb[o + (long)k * nc];
    const float d = v - T[(long)b * n + e];
    s = s + d * d;
    if (db) {
      const float dy = d * scale;
      for (int k = 0; k < nk; ++k) db[o + (long)k * nc] = f2bf(mk[k] * dy);
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

extern "C" int cgfds_gemm_bf16(int M, int N, int K, const void* A, long lda, int transA,
                               const void* B, long ldb, int transB, const float* bias,
                               int epilogue, const void* mask, long ldm, float* C32, long ldc32,
                               void* C16, long ldc16, int splitk, float* work, void* stream)
{
  if (M <= 0 || N <= 0 || K <= 0 || !A || !B || (!C32 && !C16))
    return sfail(CGFDH_EINVAL, "cgfds_gemm_bf16: empty shape or null operand");
  if (M % 8 || N % 8 || K % 8 || lda % 8 || ldb % 8 || !al16(A) || !al16(B))
    return sfail(CGFDH_EINVAL,
                 "cgfds_gemm_bf16: M, N, K and the A/B leading dimensions must be multiples "
                 "of 8 and A, B 16-byte aligned");
  if (lda < (transA ? M : K) || ldb < (transB ? K : N) || (C32 && ldc32 < N) ||
      (C16 && ldc16 < N))
    return sfail(CGFDH_EINVAL, "cgfds_gemm_bf16: leading dimension below the row length");
  if (epilogue < EPI_NONE || epilogue > EPI_MASK || (epilogue == EPI_MASK && (!mask || ldm < N)))
    return sfail(CGFDH_EINVAL, "cgfds_gemm_bf16: bad epilogue or missing mask");
  if (splitk < 1 || splitk > 1024)
    return sfail(CGFDH_EINVAL, "cgfds_gemm_bf16: splitk outside 1..1024");
  int kchunk = ((K + splitk - 1) / splitk + 31) / 32 * 32;
  int S = (K + kchunk - 1) / kchunk;
  if (S > 1 && (!work || !C32 || C16 || bias || epilogue != EPI_NONE))
    return sfail(CGFDH_EINVAL,
                 "cgfds_gemm_bf16: split-K needs a work buffer, FP32 output and no epilogue");
  auto al8 = [](const void* p, long ld) { return !p || (((uintptr_t)p & 7u) == 0 && ld % 4 == 0); };
  GemmArgs g{M, N, K, (const uint16_t*)A, lda, (const uint16_t*)B, ldb, bias, epilogue,
             (const uint16_t*)mask, ldm, C32, ldc32, (uint16_t*)C16, ldc16, kchunk,
             S > 1 ? work : nullptr, al8(mask, ldm) && al8(C16, ldc16)};
  hipStream_t st = (hipStream_t)stream;
  if ((N + 63) / 64 > 65535)
    return sfail(CGFDH_EINVAL, "cgfds_gemm_bf16: N above 65535*64 columns");
  const int form = (transA ? 2 : 0) + (transB ? 1 : 0);
  // row tiles on x (up to 2^31 - 1 blocks), column tiles on y
  auto launch = [&](auto bm, auto bn, auto bk, auto ns, auto wm, auto wn) {
    constexpr int BM = decltype(bm)::value, BN = decltype(bn)::value, BK = decltype(bk)::value,
                  NS = decltype(ns)::value, WM = decltype(wm)::value, WN = decltype(wn)::value;
    const dim3 grid((M + BM - 1) / BM, (N + BN - 1) / BN, S), blk(64 * WM * WN);
    switch (form) {
    case 0: hipLaunchKernelGGL((gemm_bf16_kernel<0, 0, BM, BN, BK, NS, WM, WN>), grid, blk, 0, st, g); break;
    case 1: hipLaunchKernelGGL((gemm_bf16_kernel<0, 1, BM, BN, BK, NS, WM, WN>), grid, blk, 0, st, g); break;
    case 2: hipLaunchKernelGGL((gemm_bf16_kernel<1, 0, BM, BN, BK, NS, WM, WN>), grid, blk, 0, st, g); break;
    default: hipLaunchKernelGGL((gemm_bf16_kernel<1, 1, BM, BN, BK, NS, WM, WN>), grid, blk, 0, st, g); break;
    }
  };
#define CGFDS_I(n) std::integral_constant<int, n>{}
  // The largest tile that still leaves a block for each of the 256 compute
  // units: fewer bytes through LDS a product.  us, 128 x 128 and 64 x 64:
  // 2048 x 4096 x 512 (512 large tiles) 23, 31; 2048 x 512 x 512 (64) 16, 9.
  // Where even 64 x 64 leaves units idle the contraction is a serial chain, so
  // fewer, deeper stages and twice the tiles: 64 x 512 x 4096 28, 37; 512 x 512
  // x 4096 34, 51; level with 64 x 64 at K = 512 and below.
  const long big = (long)((M + 127) / 128) * ((N + 127) / 128) * S;
  const long mid = (long)((M + 63) / 64) * ((N + 63) / 64) * S;
  if (big >= 256)
    launch(CGFDS_I(128), CGFDS_I(128), CGFDS_I(64), CGFDS_I(2), CGFDS_I(2), CGFDS_I(2));
  else if (mid >= 256)
    launch(CGFDS_I(64), CGFDS_I(64), CGFDS_I(64), CGFDS_I(3), CGFDS_I(2), CGFDS_I(2));
  else
    launch(CGFDS_I(64), CGFDS_I(32), CGFDS_I(128), CGFDS_I(4), CGFDS_I(2), CGFDS_I(2));
#undef CGFDS_I
  if (int rc = launch_check("cgfds_gemm_bf16")) return rc;
  if (S > 1) {
    long n = (long)M * N;
    hipLaunchKernelGGL(splitk_reduce_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
                       S, M, N, (const float*)work, C32, ldc32);
    return launch_check("cgfds_gemm_bf16 (split-K reduce)");
  }
  return 0;
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
  hipLaunchKernelGGL(splitk_reduce_kernel, dim3((N + 255) / 256), dim3(256), 0, st, splits, 1, N,
                     (const float*)work, out, (long)N);
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

extern "C" int cgfds_mt_contract(int nsamp, int nt, int nc, int nk, const float* m,
                                 const float* g, float* y, void* stream)
{
  if (nsamp <= 0 || nt <= 0 || nc <= 0 || nk < 1 || nk > MT_MAX || !m || !g || !y)
    return sfail(CGFDH_EINVAL, "cgfds_mt_contract: bad argument (nk must be 1..8)");
  hipLaunchKernelGGL(mt_contract_kernel, dim3(nsamp), dim3(256), 0, (hipStream_t)stream, nt, nc,
                     nk, m, g, y);
  return launch_check("cgfds_mt_contract");
}

extern "C" int cgfds_mt_loss_grad(int nsamp, int nt, int nc, int nk, const float* m,
                                  const float* g, const float* T, const float* tnorm2, float eps,
                                  void* dg16, float* loss, void* stream)
{
  if (nsamp <= 0 || nt <= 0 || nc <= 0 || nk < 1 || nk > MT_MAX || !m || !g || !T || !tnorm2 ||
      !loss)
    return sfail(CGFDH_EINVAL, "cgfds_mt_loss_grad: bad argument (nk must be 1..8)");
  hipLaunchKernelGGL(mt_loss_grad_kernel, dim3(nsamp), dim3(256), 0, (hipStream_t)stream, nt, nc,
                     nk, m, g, T, tnorm2, eps, nsamp, (uint16_t*)dg16, loss);
  return launch_check("cgfds_mt_loss_grad");
}

extern "C" int cgfds_f32_to_bf16(long n, const float* src, void* dst, void* stream)
{
  if (n <= 0 || !src || !dst) return sfail(CGFDH_EINVAL, "cgfds_f32_to_bf16: bad argument");
  hipLaunchKernelGGL(to_bf16_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, n, src, (uint16_t*)dst);
  return launch_check("cgfds_f32_to_bf16");
}
