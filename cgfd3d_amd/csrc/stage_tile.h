// stage_tile.h -- the default stage kernel (variant 16) of every medium, on all but
// small grids: one 64 x 8 tile of one plane per block, over whole rows, the PML
// faces folded in.
//
// What bounded the per-point kernels before it (whole rows, two-phase loads)
// was the vector memory path of the compute units, not HBM: 165 loads and 18
// stores per point, the x operator's on lines still on their way, kept the
// address units busy for 77-80 % of the time at 3.0-4.1 TB/s.  Here
//  * the tile and its halo go straight to LDS (no registers, one load per value
//    instead of up to nine), the x and y operators read them there; the z
//    operator's other planes come to registers, from L2 where the planes beside
//    were just read;
//  * whatever else a point needs is requested before the first arithmetic: the
//    coefficients, the RK levels (the middle stages' to LDS) and the memory
//    variables of the first PML face;
//  * rows start on 128-byte lines, so a wave's load is two lines, not three;
//  * registers are kept to 128, 4 waves a SIMD in two blocks a compute unit,
//    whose loads cover each other's arithmetic (three Maxwell bodies spill one
//    register in the middle stages; four take 94 KB of LDS and up to 139
//    registers: one block a unit, 2 waves a SIMD).
// 95 vector memory instructions a point are left and 1.14 times the algorithmic
// traffic (the two-phase kernel: 1.15), 4.7 TB/s on it.  600x600x300 isotropic, ms
// a step, before and now: 29.7, 23.3; without PML 24.7, 19.4; 400x400x200 VTI
// 10.1, 8.3; anisotropic 11.8, 9.9; visco-elastic (3 bodies) 22.7, 15.9;
// 200x200x100 with one to four bodies 2.29, 2.81, 3.34, 3.85 and 1.76, 2.05, 2.43,
// 2.95.
#pragma once
#include <type_traits>

#include "stage_launch.h"

namespace cgfdh {

// Memory accesses are buffer operations: the base of a plane stays in scalar
// registers, the volumes of up to three components are reached by a scalar
// offset, and a lane holds a 32-bit offset in the plane, so no 64-bit addresses
// occupy vector registers.  A lane whose offset is OUT reads zero and stores
// nothing, so partly filled tiles need no branch.
constexpr unsigned OUT = ~3u;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_of(const float* base)
{
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)0xfffffff0, 0x00020000);
}

// component c of a set of volumes V apart that starts at base
template <int AUX = 0>
__device__ __forceinline__ float buf_load(const float* base, int c, long V, unsigned off)
{
  return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
      rsrc_of(base + (c - c % 3) * V), (int)off, (int)(4u * (unsigned)V * (unsigned)(c % 3)), AUX));
}

template <int AUX = 0>
__device__ __forceinline__ void buf_store(float* base, int c, long V, unsigned off, float v)
{
  __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), rsrc_of(base + (c - c % 3) * V),
                                        (int)off, (int)(4u * (unsigned)V * (unsigned)(c % 3)), AUX);
}

template <int AUX = 0>
__device__ __forceinline__ void buf_load_lds(const float* base, int c, long V, unsigned off,
                                             float* lds)
{
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      rsrc_of(base + (c - c % 3) * V), (__attribute__((address_space(3))) void*)lds, 4, (int)off,
      (int)(4u * (unsigned)V * (unsigned)(c % 3)), 0, AUX);
}

// an entry of a table the kernel never writes, the same for every lane
__device__ __forceinline__ float table_at(const float* t, int n)
{
  return ((const __attribute__((address_space(4))) float*)t)[n];
}

// the LDS copy of a tile: per component TY + 4 rows of 64 and, behind them, the
// 4 columns beside the tile, TY x 4
template <int TY> constexpr int tile_comp = (TY + 4) * 64 + 4 * TY;

// The order of the blocks: a unit is one row of tiles over kchunk planes, its
// blocks tile by tile and plane by plane on one XCD, so the planes the z
// operator shares meet in one L2; units go to the XCDs in turn, so that the
// tiles with PML, twice the work and at the grid's ends, are spread over all
// of them.
__device__ __forceinline__ bool tile_block(const BoxParams& B, int& bx, int& by, int& k)
{
  const int per = B.tiles_x * B.kchunk;
  const int n = blockIdx.x / 8;
  const int ul = n / per, r = n - ul * per;
  const int u = ul * 8 + blockIdx.x % 8;
  const int kc = u / B.tiles_y, kk = r / B.tiles_x;
  bx = r - kk * B.tiles_x;
  by = u - kc * B.tiles_y;
  k = B.k0 + kc * B.kchunk + kk;
  return kc < B.nchunk && k < B.k0 + B.nk;
}

// NB: room for Maxwell bodies (visco-elastic medium).  NT: the cache policy of
// what no other point reads, 2 non-temporal, 0 none.
template <int DX, int DY, int DZ, int KIND, int MT, int TY, int NB, int NT>
__global__ void __launch_bounds__(64 * TY, 4) stage_tile_kernel(StageParams P, BoxParams B)
{
  constexpr int xl = Win<DX>::lo, yl = Win<DY>::lo, zl = Win<DZ>::lo;
  constexpr int xo = -xl, yo = -yl;
  constexpr int NC = Medium<MT>::ncoef;
  constexpr int CS = tile_comp<TY>;
  constexpr bool VIS = MT == MEDIUM_VISCO;
  // coefficients requested once the stencil's registers are free (VTI), or sent
  // to LDS (the anisotropic medium's 21)
  constexpr bool LATE = MT == MEDIUM_VTI;
  constexpr bool CLDS = MT == MEDIUM_ANISO;
  // where registers are left, the PML levels of the RK combine are requested
  // with the memory variables themselves
  constexpr bool EARLY = MT == MEDIUM_ISO;
  // levels at the point itself: the middle stages' go to LDS, so that the
  // loads in flight fit 128 registers and 4 waves a SIMD; the last stage's end
  // level to registers; the first stage starts from the level in the tile
  constexpr int NK = KIND == KIND_MID && !CLDS && !VIS ? 2 : 0;
  constexpr bool LPRE = KIND == KIND_MID && (CLDS || VIS);  // to registers, late
  constexpr bool LEND = LPRE || (KIND == KIND_LAST && (CLDS || VIS));
  constexpr int NJ = 6 * NB;                            // memory variables
  constexpr int NL = NK * 9 + (CLDS ? NC : 0) + 8 * NB; // LDS slots of a wave
  static_assert(TY >= 5, "one wave each for the 4 halo rows and the halo columns");
  __shared__ float S[9 * CS + NL * 64 * TY];
  int bx, by, k;
  if (!tile_block(B, bx, by, k)) return;
  const int tx = threadIdx.x, ty = __builtin_amdgcn_readfirstlane(threadIdx.y);
  const int ti0 = B.i0 + bx * 64, tj0 = B.j0 + by * TY;
  const int i = ti0 + tx, j = tj0 + ty;
  const bool act = i < B.i0 + B.ni && j < B.j0 + B.nj;
  auto level_off = [&](int ii, int jj) {         // inside the array
    return ii <= P.ni2 + 3 && jj <= P.nj2 + 3 ? 4u * (unsigned)(ii + jj * P.nx) : OUT;
  };
  const unsigned vo = level_off(i, j);
  const unsigned so = act ? 4u * (unsigned)(i + j * P.nx) : OUT;
  const long V = P.vol, pl = (long)k * P.ss;
  float* K = S + 9 * CS + ty * 64;               // the wave's slots of the point's levels

  // the tile and its halo straight to LDS: each wave its own row, the first
  // four a halo row, the fifth the columns beside the tile
  {
    const float* a = P.wcur + pl;
    if (ty < 4) {
      const int row = ty < yo ? ty : TY + ty;
      const unsigned ho = level_off(i, tj0 + row - yo);
#pragma unroll
      for (int c = 0; c < 9; c++) buf_load_lds(a, c, V, ho, &S[c * CS + row * 64]);
    } else if (ty == 4) {
      const int q = tx & 3, row = tx >> 2;
      const unsigned ho = level_off(ti0 + (q < xo ? q - xo : 64 + q - xo), tj0 + row);
      if (tx < 4 * TY) {
#pragma unroll
        for (int c = 0; c < 9; c++) buf_load_lds(a, c, V, ho, &S[c * CS + (TY + 4) * 64]);
      }
    }
#pragma unroll
    for (int c = 0; c < 9; c++) buf_load_lds(a, c, V, vo, &S[c * CS + (ty + yo) * 64]);
  }
  // the PML faces this tile meets and the memory variables of the first one
  unsigned faces = 0;
#pragma unroll
  for (int f = 0; f < 6; f++) {
    const int lo = f / 2 == 0 ? ti0 : (f / 2 == 1 ? tj0 : k);
    const int hi = f / 2 == 0 ? ti0 + 63 : (f / 2 == 1 ? tj0 + TY - 1 : k);
    if (P.fslot[f] >= 0 && (f % 2 == 0 ? lo <= P.fedge[f] : hi >= P.fedge[f])) faces |= 1u << f;
  }
  unsigned ao = OUT;
  float pa[9], pp[9], pe[9], cA = 0.0f, cB = 0.0f, cD = 0.0f;
  auto aux_plane = [&](const PmlDev& F, const float* a) {
    return a + (long)(k - F.k1) * F.fnx * F.fny;
  };
  auto request_aux_levels = [&](const PmlDev& F) {
#pragma unroll
    for (int c = 0; c < 9; c++) {
      if (KIND == KIND_MID) pp[c] = buf_load<NT>(aux_plane(F, F.aux_pre), c, F.fn, ao);
      if (KIND != KIND_FIRST) pe[c] = buf_load<NT>(aux_plane(F, F.aux_end), c, F.fn, ao);
    }
  };
  auto request_aux = [&](int f) {
    const PmlDev& F = P.pml[P.fslot[f]];
    const bool in = act && (f >= 4 || (f < 2 ? (f == 0 ? i <= P.fedge[0] : i >= P.fedge[1])
                                             : (f == 2 ? j <= P.fedge[2] : j >= P.fedge[3])));
    ao = in ? 4u * (unsigned)((i - F.i1) + (j - F.j1) * F.fnx) : OUT;
#pragma unroll
    for (int c = 0; c < 9; c++) pa[c] = buf_load<NT>(aux_plane(F, F.aux_cur), c, F.fn, ao);
    if (EARLY) request_aux_levels(F);
    if (f < 2) {
      const unsigned co = in ? 4u * (unsigned)(i - F.i1) : OUT;
      cA = buf_load(F.A, 0, 0, co);
      cB = buf_load(F.B, 0, 0, co);
      cD = buf_load(F.D, 0, 0, co);
    } else {
      // rows past the face's last are inactive: any entry serves them
      const int n = f >= 4 ? k - F.k1 : min(max(j - F.j1, 0), F.j2 - F.j1);
      cA = table_at(F.A, n);
      cB = table_at(F.B, n);
      cD = table_at(F.D, n);
    }
  };
  if (faces) request_aux(__builtin_ctz(faces));
  __builtin_amdgcn_sched_barrier(0);
  // the point's own levels, the other planes of the z operator, the coefficients
  float az[9][5], m[9], mv[NC], pre[9], end[9];
  if (NK) {
#pragma unroll
    for (int c = 0; c < 9; c++) {
      buf_load_lds<NT>(P.wpre + pl, c, V, so, K + c * 64 * TY);
      buf_load_lds<NT>(P.wend + pl, c, V, so, K + (9 + c) * 64 * TY);
    }
  }
  if (CLDS) {
#pragma unroll
    for (int q = 0; q < NC; q++) buf_load_lds<NT>(P.med + pl, q, V, so, K + q * 64 * TY);
  }
  if (VIS) {
#pragma unroll
    for (int c = 0; c < NJ; c++)
      buf_load_lds<NT>(P.wcur + 9 * V + pl, c, V, c < 6 * P.nmax ? so : OUT, K + c * 64 * TY);
#pragma unroll
    for (int c = 0; c < 2 * NB; c++)
      buf_load_lds<NT>(P.ylam + pl, c, V, c < 2 * P.nmax ? so : OUT, K + (NJ + c) * 64 * TY);
  }
#pragma unroll
  for (int n = 0; n < 5; n++) {
    if (zl + n == 0) continue;
#pragma unroll
    for (int c = 0; c < 9; c++)
      az[c][n] = buf_load(P.wcur + pl + (long)(zl + n) * P.ss, c, V, vo);
  }
#pragma unroll
  for (int q = 0; q < 9; q++) m[q] = buf_load<NT>(P.met + V + pl, q, V, so);
  if (!LATE && !CLDS) {
#pragma unroll
    for (int q = 0; q < NC; q++) mv[q] = buf_load<NT>(P.med + pl, q, V, so);
  }
  const float slw = buf_load<NT>(P.slw + pl, 0, V, so);
  if (KIND == KIND_LAST && !LEND) {
#pragma unroll
    for (int c = 0; c < 9; c++) end[c] = buf_load<NT>(P.wend + pl, c, V, so);
  }
  // the tile has landed once no more than the loads after it are in flight
  constexpr int later = NL + 36 + 9 + (LATE || CLDS ? 0 : NC) + 1 + (KIND == KIND_LAST && !LEND ? 9 : 0);
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(later < 63 ? later : 63) : "memory");
  __builtin_amdgcn_sched_barrier(0);

  // LDS positions of the x operator's points
  int xp[5];
#pragma unroll
  for (int n = 0; n < 5; n++) {
    const int col = tx + xl + n;
    xp[n] = col < 0    ? (TY + 4) * 64 + ty * 4 + col + xo
            : col > 63 ? (TY + 4) * 64 + ty * 4 + xo + col - 64
                       : (ty + yo) * 64 + col;
  }
  const int cp = (ty + yo) * 64 + tx;            // the point itself
  auto dx = [&](int c) {
    const float* s = S + c * CS;
    return d5v<DX>(s[xp[0]], s[xp[1]], s[xp[2]], s[xp[3]], s[xp[4]]);
  };
  auto dy = [&](int c) {
    const float* t = S + c * CS + ty * 64 + tx;
    return d5v<DY>(t[0], t[64], t[128], t[192], t[256]);
  };
  float X[9], Y[9], Z[9];
#pragma unroll
  for (int c = 0; c < 9; c++) {
    X[c] = dx(c);
    Y[c] = dy(c);
    // three components' LDS reads at a time: all of them at once would spill
    if (c % 3 == 2) __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int c = 0; c < 9; c++) {
    az[c][-zl] = S[c * CS + cp];
    Z[c] = d5v<DZ>(az[c][0], az[c][1], az[c][2], az[c][3], az[c][4]);
  }
  // everything requested so far has landed, the levels in LDS included
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);

  if (LATE) {
#pragma unroll
    for (int q = 0; q < NC; q++) mv[q] = buf_load<NT>(P.med + pl, q, V, so);
  }
  __builtin_amdgcn_sched_barrier(0);

  Medium<MT> md;
  float r[VIS ? 9 + NJ : 9];
  momentum(r, m, slw, X, Y, Z);
  // (from LDS where they are used: kept in registers they would spill)
  auto stiffness = [&](Medium<MT>& q) {
    if (CLDS) {
#pragma unroll
      for (int c = 0; c < NC; c++) mv[c] = K[c * 64 * TY + tx];
    }
    q.from(mv);
  };
  stiffness(md);
  {
    float Xv[3] = {X[VX], X[VY], X[VZ]}, Yv[3] = {Y[VX], Y[VY], Y[VZ]},
          Zv[3] = {Z[VX], Z[VY], Z[VZ]};
    if constexpr (CLDS) {
      // a row of the stress rates at a time: the 54 products of metric and
      // stiffness at once would spill
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < 6; t++) {
        md.hooke_row(t, r, m, Xv, Yv, Zv);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      md.hooke(r, m, Xv, Yv, Zv);
    }
  }
  auto face = [&](auto dim, int f) {
    constexpr int D = decltype(dim)::value;
    const PmlDev& F = P.pml[P.fslot[f]];
    float ah[9];
    if (VIS) request_aux_levels(F);
    if (ao != OUT) {
      // the x and y derivatives once more from the tile: kept from above, they
      // would not fit the registers beside the memory variables
      float d[9], e[9];
#pragma unroll
      for (int c = 0; c < 9; c++) d[c] = D == 0 ? dx(c) : (D == 1 ? dy(c) : Z[c]);
      // nor would Hooke's products of metric and stiffness: formed anew
#pragma unroll
      for (int q = 0; q < 9; q++) {
        e[q] = m[q];
        asm volatile("" : "+v"(e[q]));
      }
      if (CLDS) stiffness(md);
      pml_face_rates<MT, D>(P, i, j, k, cA, cB, cD, d, md, slw, e, r, pa, ah);
    }
    if (!EARLY && !VIS) request_aux_levels(F);
#pragma unroll
    for (int c = 0; c < 9; c++) {
      if (KIND != KIND_LAST)
        buf_store<NT>((float*)aux_plane(F, F.aux_tmp), c, F.fn, ao,
                      (KIND == KIND_FIRST ? pa[c] : pp[c]) + P.ca * ah[c]);
      buf_store<NT>((float*)aux_plane(F, F.aux_end), c, F.fn, ao,
                    (KIND == KIND_FIRST ? pa[c] : pe[c]) + P.cb * ah[c]);
    }
  };
  // (unrolled: in a loop the compiler would form all three directions' terms
  // ahead of it and spill)
  const int f0 = faces ? __builtin_ctz(faces) : 6;
#define CGFDH_FACE(f)                                     \
  if (faces >> f & 1u) {                                  \
    asm volatile("" ::: "memory");                        \
    if (f != f0) request_aux(f);                          \
    face(std::integral_constant<int, f / 2>{}, f);        \
  }
  CGFDH_FACE(0) CGFDH_FACE(1) CGFDH_FACE(2) CGFDH_FACE(3) CGFDH_FACE(4) CGFDH_FACE(5)
#undef CGFDH_FACE
  const long p = (long)i + (long)j * P.nx + pl;
  if (LEND) {
#pragma unroll
    for (int c = 0; c < 9; c++) {
      if (LPRE) pre[c] = buf_load<NT>(P.wpre + pl, c, V, so);
      end[c] = buf_load<NT>(P.wend + pl, c, V, so);
    }
  }
  constexpr int NJ1 = VIS ? NJ : 1;
  float jp[NJ1], je[NJ1];
  if constexpr (VIS) {
#pragma unroll
    for (int c = 0; c < NJ; c++) {
      const unsigned jo = c < 6 * P.nmax ? so : OUT;
      if (KIND == KIND_MID) jp[c] = buf_load<NT>(P.wpre + 9 * V + pl, c, V, jo);
      if (KIND != KIND_FIRST) je[c] = buf_load<NT>(P.wend + 9 * V + pl, c, V, jo);
    }
    float jy[2 * NB];
#pragma unroll
    for (int c = 0; c < 2 * NB; c++) jy[c] = K[(NJ + c) * 64 * TY + tx];
    atten<NB>(P, [&](int c) { return K[(c - 9) * 64 * TY + tx]; }, jy, md.lam, md.mu, r);
  }
  if (act) {
    if (P.nsrc > 0) add_sources(P, i, j, k, p, r);
    add_dd_for<MT>(P, p, r);
  }
#pragma unroll
  for (int c = 0; c < 9; c++) {
    const float b = KIND == KIND_FIRST ? S[c * CS + cp] : (NK ? K[c * 64 * TY + tx] : pre[c]);
    const float e = KIND == KIND_FIRST ? b : (NK ? K[(9 + c) * 64 * TY + tx] : end[c]);
    if (KIND != KIND_LAST) buf_store<NT>(P.wtmp + pl, c, V, so, b + P.ca * r[c]);
    buf_store<NT>(P.wend + pl, c, V, so, e + P.cb * r[c]);
  }
  if constexpr (VIS) {
    const long q = 9 * V + pl;
#pragma unroll
    for (int c = 0; c < NJ; c++) {
      const unsigned jo = c < 6 * P.nmax ? so : OUT;
      const float b = KIND == KIND_FIRST ? K[c * 64 * TY + tx] : jp[c];
      if (KIND != KIND_LAST) buf_store<NT>(P.wtmp + q, c, V, jo, b + P.ca * r[9 + c]);
      buf_store<NT>(P.wend + q, c, V, jo, (KIND == KIND_FIRST ? b : je[c]) + P.cb * r[9 + c]);
    }
  }
}

template <int KIND, int MT, int NB, int NT>
static void launch_tile(const LaunchCtx& L, const StageParams& P, int code)
{
  constexpr int TY = 8;
  static_assert(TY == TILE_ROWS, "");
  BoxParams B;
  const int grid = 8 * tile_box(L.ni, L.nj, L.free_top ? L.nk - 4 : L.nk, B);
  B.i0 = L.ni1; B.j0 = L.nj1; B.k0 = L.nk1;
  dim3 blk(64, TY, 1);
#define CGFDH_TI(c, DX, DY, DZ)                                                             \
  case c:                                                                                   \
    hipLaunchKernelGGL((stage_tile_kernel<DX, DY, DZ, KIND, MT, TY, NB, NT>), dim3(grid),   \
                       blk, 0, L.stream, P, B);                                             \
    break;
  switch (code) {
    CGFDH_TI(0, 0, 0, 0) CGFDH_TI(1, 0, 0, 1) CGFDH_TI(2, 0, 1, 0) CGFDH_TI(3, 0, 1, 1)
    CGFDH_TI(4, 1, 0, 0) CGFDH_TI(5, 1, 0, 1) CGFDH_TI(6, 1, 1, 0) CGFDH_TI(7, 1, 1, 1)
  }
#undef CGFDH_TI
}

template <int MT, int NB, int NT>
void launch_tile_kind(const LaunchCtx& L, const StageParams& P, int kind, int code)
{
  switch (kind) {
    case KIND_FIRST: launch_tile<KIND_FIRST, MT, NB, NT>(L, P, code); break;
    case KIND_MID: launch_tile<KIND_MID, MT, NB, NT>(L, P, code); break;
    default: launch_tile<KIND_LAST, MT, NB, NT>(L, P, code); break;
  }
}

// A solver whose arrays fit the 256 MB last-level cache finds them there at
// the next stage and keeps to plain accesses (100x100x60: 0.291 ms a step
// against 0.333 non-temporal; the two-phase kernel, chosen there, 0.284); a larger one streams past the caches, which
// keep the planes and halo rows that neighbours share (600x600x300: 23.3
// against 23.7, without PML 19.4 against 20.1).
template <int MT, int NB>
void launch_tile_nt(const LaunchCtx& L, const StageParams& P, int kind, int code)
{
  if (L.bytes > 256l << 20)
    launch_tile_kind<MT, NB, 2>(L, P, kind, code);
  else
    launch_tile_kind<MT, NB, 0>(L, P, kind, code);
}

template <int MT>
void launch_tile_mt(const LaunchCtx& L, const StageParams& P, int kind, int dx, int dy, int dz)
{
  const int code = dx * 4 + dy * 2 + dz;
  if constexpr (MT == MEDIUM_VISCO) {
    // LDS for three bodies leaves room for two blocks a compute unit; fewer pay for
    // three and are still ahead of the two-phase kernel (200x200x100, one body 1.76
    // ms a step, 2.19)
    if (P.nmax <= 3)
      launch_tile_nt<MT, 3>(L, P, kind, code);
    else
      launch_tile_nt<MT, MAXWELL_MAX>(L, P, kind, code);
  } else {
    launch_tile_nt<MT, 0>(L, P, kind, code);
  }
}

}  // namespace cgfdh
