// matmul_f32_split.hip -- fp32 matmul template on the bf16 matrix instructions of gfx950.
//
// C[z][m][n] = epilogue( sum_k A(z,m,k) * B(z,k,n) ), fp32 inputs, fp32 accumulation.  The renderer
// (templates.cc) instantiates it by prepending the configuration block of matmul_mfma.hip
// (POLY_TIN float, POLY_MFMA the 32x32x16 MFMA of bf16, POLY_M/N/K/Z, POLY_BM/BN/BK, POLY_WAVES_M/N,
// POLY_A_KC/B_KC, POLY_A_PTR/B_PTR, poly_a_row/poly_b_row/poly_a_z/poly_b_z/poly_a_k/poly_b_k, no two
// strides along K, POLY_SIGNATURE, the POLY_EP* epilogue macros, POLY_GROUP_M, POLY_GROUP_ALONG_N) plus
//
//   POLY_A_PITCH/B_PITCH   elements from one k of the operand to the next
//   POLY_WG_PER_CU         workgroups meant to share a CU (sets the register budget)
//   POLY_FAR               1: an operand is read further than 4 GiB behind its beginning
//   POLY_KSPLIT            (optional) workgroups that share the depth of a tile, a multiple of POLY_BK each
//
// An fp32 value is the sum of three bf16 values, hi + mid + lo (each the rounding of what the ones before
// leave; the differences are exact), as in G. Henry, P. T. P. Tang, A. Heinecke, "Leveraging the bfloat16 Artificial
// Intelligence Datatype For Higher-Precision Computations" (ARITH 2019).  Products of bf16 values are exact in
// fp32, and of the nine of two such sums all but lo lo are added up, which is 2^-34 of the value at most (mid is up to
// 2^-8 of it, lo 2^-17: without mid lo and lo mid a sum of one term is off by up to 1.8 roundings).  The products of the
// leading planes have sums of their own: one rounding at the size of the result for 16 products, where the fp32 MFMA has
// eight, and one more of each product's 2^-7 for those behind.  Errors against float64: 4096 x 512 x 784 1.6e-7 [fp32
// MFMA 5.0e-7], 2048^3 2.7e-7 [8.1e-7], 1024 x 1024 x 4096 1.9e-7 [4.1e-7]; sums of one term 1.01 x 2^-24 [1.00], one in
// a thousand of them not the nearest value.
//
// That holds for finite values of 2^-110 and more, below which bf16 has no 24 bits left, and zeros.
// Operands are looked over for smaller ones on the way, results for infinities and NaN (an
// infinity leaves NaN behind: inf - inf), and a workgroup that met one computes its tile again
// with the fp32 MFMA from operands in memory.  That takes what the fp32 templates take and some of the time up to
// there: 2048^3 is 117 us without such values, 253 with one in every row, 295 with a single one in the middle of a row
// [fp32 MFMA 200], 4096 x 512 x 784 34, 53 and 60 [45], 128 x 50257 x 768 86, 165 and 207 [120].
//
// Data path: global --16-byte loads--> registers, split there, --> LDS, [plane][row][BK] for an operand
// contiguous along K and [plane][k][rows] for one along its rows, swizzled as in matmul_dma.hip, two
// stages; one barrier per K tile.  The end of the depth is a tile of its own, the first, filled up
// with zeros.  What bounds it: 64x64 tiles the first loads and the split, seven vector instructions per
// element (4096 x 512 x 784 45 -> 34 us), larger ones the matrix pipes, 8 MFMAs of 32 cycles where fp32 has 8 of 64
// (2048^3 200 -> 117 us, 97 without the products mid lo and lo mid).
#ifdef POLY_TEMPLATE_STANDALONE
#include <hip/hip_runtime.h>
#define POLY_TIN float
#define POLY_MFMA(a, b, c) __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0)
#define POLY_M 4095
#define POLY_N 1023
#define POLY_K 787
#define POLY_Z 1
#define POLY_BM 64
#define POLY_BN 64
#define POLY_BK 32
#define POLY_GROUP_M 8
#define POLY_GROUP_ALONG_N 0
#define POLY_WAVES_M 2
#define POLY_WAVES_N 2
#define POLY_WG_PER_CU 2
#define POLY_A_KC 1
#define POLY_B_KC 0
#define POLY_A_PITCH 1ll
#define POLY_B_PITCH 1023ll
#define POLY_FAR 0
#define POLY_A_PTR data1
#define POLY_B_PTR data2
__device__ __forceinline__ int poly_a_row(int m) { return m * POLY_K; }
__device__ __forceinline__ int poly_b_row(int n) { return n; }
__device__ __forceinline__ int poly_a_z(int z) { return 0; }
__device__ __forceinline__ int poly_b_z(int z) { return 0; }
__device__ __forceinline__ int poly_a_k(int k) { return k; }
__device__ __forceinline__ int poly_b_k(int k) { return k * POLY_N; }
#define POLY_SIGNATURE float *data0, const float *__restrict__ data1, const float *__restrict__ data2
#define POLY_EPILOGUE(acc, m, n, z) data0[(m) * POLY_N + (n)] = (acc)
#define POLY_EP_CONTIG 1
#define POLY_EP_TYPE float
#define POLY_EP_VALUE(acc, m, n, z) (acc)
#define POLY_EP_PTR(m, n, z) (data0 + (m) * POLY_N + (n))
#endif

typedef __bf16 poly_in8 __attribute__((ext_vector_type(8)));
typedef __bf16 poly_in2 __attribute__((ext_vector_type(2)));
typedef float poly_acc16 __attribute__((ext_vector_type(16)));
typedef float poly_f32x4 __attribute__((ext_vector_type(4)));
typedef poly_f32x4 poly_f32x4_u __attribute__((aligned(4)));
typedef float poly_f32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int poly_u32x4 __attribute__((ext_vector_type(4)));
typedef short poly_s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) poly_s16x4 poly_lds_s16x4;

#define POLY_NW (POLY_WAVES_M * POLY_WAVES_N)
#define POLY_NTHREADS (64 * POLY_NW)
#define POLY_WM (POLY_BM / POLY_WAVES_M)
#define POLY_WN (POLY_BN / POLY_WAVES_N)
#define POLY_TM (POLY_WM / 32)
#define POLY_TN (POLY_WN / 32)
#ifndef POLY_KSPLIT
#define POLY_KSPLIT 1
#endif
#define POLY_KP (POLY_K / POLY_KSPLIT)                 // depth of a workgroup
#define POLY_NTILES ((POLY_KP + POLY_BK - 1) / POLY_BK)
#define POLY_KT (POLY_NTILES - 1)                      // whole tiles; what is left is tile 0
#define POLY_CH (POLY_BK / 8)
#define POLY_A_PLANE (POLY_BM * POLY_BK * 2)           // bytes of a plane of a tile
#define POLY_B_PLANE (POLY_BN * POLY_BK * 2)
#define POLY_STAGE_BYTES (3 * (POLY_A_PLANE + POLY_B_PLANE))
#define POLY_A_UNITS (POLY_BM * POLY_BK / 8 / POLY_NTHREADS)      // rows of 8 elements that a thread carries
#define POLY_B_UNITS (POLY_BN * POLY_BK / 8 / POLY_NTHREADS)
#define POLY_UNITS (POLY_A_UNITS + POLY_B_UNITS)
#define POLY_STAGE_LD 36
static_assert(POLY_BM * POLY_BK / 8 % POLY_NTHREADS == 0 && POLY_BN * POLY_BK / 8 % POLY_NTHREADS == 0, "every thread carries the same number of rows of 8");
static_assert(POLY_KSPLIT == 1 || POLY_K % (POLY_KSPLIT * POLY_BK) == 0, "whole K tiles for every part");

// (as in matmul_dma.hip)
__device__ __forceinline__ int poly_swz_k(int row) { return POLY_CH == 8 ? ((row ^ (row >> 3)) & 7) : ((row >> 2) & 3); }
template <int ROWS>
__device__ __forceinline__ int poly_swz_x(int k) { return (ROWS % 128 == 0) ? ((k & 3) << 2) : ((k & 3) | ((k & 1) << 2)); }

#ifdef POLY_HOST_ADDRESS_CHECK   // compiled for the host to check its indexing: lanes run one by one, no cross-lane arithmetic
#define __builtin_amdgcn_ds_read_tr16_b64_v4i16(p) (*(p))
#define POLY_MFMA_F32(a, b, c) (c)
#else
#define POLY_MFMA_F32(a, b, c) __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0)
#endif
#if POLY_WG_PER_CU * POLY_NW > 4 && !defined(POLY_HOST_ADDRESS_CHECK)
#define POLY_WAVES_ATTR __attribute__((amdgpu_waves_per_eu(POLY_WG_PER_CU * POLY_NW / 4, POLY_WG_PER_CU * POLY_NW / 4)))
#else
#define POLY_WAVES_ATTR
#endif

struct PolyUnit { float v[8]; };
#if POLY_FAR
typedef unsigned long long poly_bytes;
#else
typedef unsigned int poly_bytes;
#endif

extern "C" __global__ void __launch_bounds__(POLY_NTHREADS) POLY_WAVES_ATTR poly_k(POLY_SIGNATURE) {
  __shared__ __attribute__((aligned(1024))) unsigned char lds_raw[2 * POLY_STAGE_BYTES];
  __shared__ int poly_again;
  static_assert(POLY_NW * 32 * POLY_STAGE_LD * 4 <= 2 * POLY_STAGE_BYTES, "staging area exceeds the operand stages");
  if (threadIdx.x == 0) poly_again = 0;      // (published by the K loop's barriers)

  // tile coordinates: as in matmul_dma.hip
  constexpr int TILES_M = (POLY_M + POLY_BM - 1) / POLY_BM, TILES_N = (POLY_N + POLY_BN - 1) / POLY_BN, NT = TILES_M * TILES_N;
  int bid = blockIdx.x;
  {
    constexpr int PER = NT / 8, REM = NT % 8;
    const int xcd = bid & 7, idx = bid >> 3;
    bid = (xcd < REM ? xcd * (PER + 1) : REM * (PER + 1) + (xcd - REM) * PER) + idx;
  }
  int tile_m, tile_n;
  {
    constexpr int GM = POLY_GROUP_M;
#if POLY_GROUP_ALONG_N
    const int per_group = GM * TILES_M, group = bid / per_group, first_n = group * GM, gsz = TILES_N - first_n < GM ? TILES_N - first_n : GM;
    const int in_group = bid - group * per_group;
    tile_n = first_n + in_group % gsz;
    tile_m = in_group / gsz;
#else
    const int per_group = GM * TILES_N, group = bid / per_group, first_m = group * GM, gsz = TILES_M - first_m < GM ? TILES_M - first_m : GM;
    const int in_group = bid - group * per_group;
    tile_m = first_m + in_group % gsz;
    tile_n = in_group / gsz;
#endif
  }
#if POLY_KSPLIT > 1
  const int z = blockIdx.y / POLY_KSPLIT, poly_ks = blockIdx.y % POLY_KSPLIT, k_base = poly_ks * POLY_KP;
#else
  const int z = blockIdx.y;
  constexpr int k_base = 0;
#endif
  const int m0 = tile_m * POLY_BM, n0 = tile_n * POLY_BN;
  const float *__restrict__ gA = POLY_A_PTR + poly_a_z(z) + poly_a_k(k_base);
  const float *__restrict__ gB = POLY_B_PTR + poly_b_z(z) + poly_b_k(k_base);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;

  // Row of 8 `u` of this thread, A's first: along K 8 of them of one row, else 8 rows at one k.  Rows past the
  // edge repeat others: loaded and multiplied, never stored.
  auto is_a = [](int u) { return u < POLY_A_UNITS; };
  auto along_k = [&](int u) { return is_a(u) ? POLY_A_KC != 0 : POLY_B_KC != 0; };
  auto slot_of = [&](int u) { return (is_a(u) ? u : u - POLY_A_UNITS) * POLY_NTHREADS + (int)threadIdx.x; };
  auto rows_of = [&](int u) { return is_a(u) ? POLY_M : POLY_N; };
  auto chunks_of = [&](int u) { return along_k(u) ? POLY_CH : (is_a(u) ? POLY_BM : POLY_BN) / 8; };
  auto first_row = [&](int u) { return (is_a(u) ? m0 : n0) + (along_k(u) ? slot_of(u) / POLY_CH : slot_of(u) % chunks_of(u) * 8); };
  auto k_of = [&](int u) { return along_k(u) ? slot_of(u) % POLY_CH * 8 : slot_of(u) / chunks_of(u); };
  // (Two halves of 4 elements half a tile apart, which lanes side by side load side by side, change nothing.)
  poly_bytes from[POLY_UNITS];      // bytes to it in the first whole tile
#pragma unroll
  for (int u = 0; u < POLY_UNITS; u++) {
    const int r = first_row(u), row = r < rows_of(u) ? r : rows_of(u) - (along_k(u) ? 1 : 8);
    from[u] = (poly_bytes)4 * (unsigned int)(is_a(u) ? poly_a_row(row) + poly_a_k(k_of(u)) : poly_b_row(row) + poly_b_k(k_of(u)));
  }
  constexpr long long STEP_A = 4ll * POLY_BK * (POLY_A_KC ? 1 : POLY_A_PITCH), STEP_B = 4ll * POLY_BK * (POLY_B_KC ? 1 : POLY_B_PITCH);
  // Tile s > 0 is the depth from (s - 1) POLY_BK on.  (What 8 elements along the rows read past their end is
  // the beginning of the next k's, which is there: the last k is tile 0's.)
  auto load_unit = [&](PolyUnit (&to)[POLY_UNITS], int s, int u) {
    const char *const p = (is_a(u) ? (const char *)gA + (long long)(s - 1) * STEP_A : (const char *)gB + (long long)(s - 1) * STEP_B) + from[u];
    const poly_f32x4 lo = *(const poly_f32x4_u *)p, hi = *(const poly_f32x4_u *)(p + 16);
#pragma unroll
    for (int e = 0; e < 4; e++) { to[u].v[e] = lo[e]; to[u].v[4 + e] = hi[e]; }
  };
  // Tile 0 is the rest, 1 to POLY_BK deep, the missing part zeros: where fewer than 8 elements are left, the
  // last 8 of the row are read and moved down.
  int gone[POLY_UNITS];
  auto load_end = [&](PolyUnit (&to)[POLY_UNITS]) {
    constexpr int K0 = POLY_KT * POLY_BK;
#pragma unroll
    for (int u = 0; u < POLY_UNITS; u++) {
      const int left_k = POLY_KP - K0 - k_of(u), r = first_row(u), left = rows_of(u) - r;
      long long at;
      if (along_k(u)) {
        const int row = left > 0 ? r : rows_of(u) - 1;
        gone[u] = left_k < 8 ? 8 - left_k : 0;
        at = (long long)(is_a(u) ? poly_a_row(row) + poly_a_k(K0 + k_of(u)) : poly_b_row(row) + poly_b_k(K0 + k_of(u))) - gone[u];
      } else {
        const int row = left > 0 ? r : rows_of(u) - 8, k = left_k > 0 ? K0 + k_of(u) : POLY_KP - 1;
        gone[u] = left > 0 && left < 8 ? 8 - left : 0;
        at = (long long)(is_a(u) ? poly_a_row(row) + poly_a_k(k) : poly_b_row(row) + poly_b_k(k)) - gone[u];
        if (left_k <= 0) gone[u] = 8;
      }
      const float *const p = (is_a(u) ? gA : gB) + at;
      const poly_f32x4 lo = *(const poly_f32x4_u *)p, hi = *(const poly_f32x4_u *)(p + 4);
#pragma unroll
      for (int e = 0; e < 4; e++) { to[u].v[e] = lo[e]; to[u].v[4 + e] = hi[e]; }
    }
  };
  // (Each of the two is read whether it is taken or not: a choice between two places keeps the array in scratch memory,
  // which at depths of 9 to 12, 17 to 20 and 25 to 28 modulo 32 took 12.5 us in place of 6.4 for 320x3776x82.)
  auto move_down = [&](PolyUnit &x, int by) {
#pragma unroll
    for (int step = 4; step > 0; step /= 2)
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const unsigned int here = __builtin_bit_cast(unsigned int, x.v[e]), behind = e + step < 8 ? __builtin_bit_cast(unsigned int, x.v[e + step < 8 ? e + step : e]) : 0u;
        const unsigned int taken = 0u - (unsigned int)((by & step) != 0);
        x.v[e] = __builtin_bit_cast(float, (here & ~taken) | (behind & taken));
      }
#pragma unroll
    for (int e = 0; e < 8; e++) x.v[e] = by >= 8 ? 0.0f : x.v[e];
  };
  // elements of a unit along rows of its operand that exist, where not all may: what lies behind a row is nothing
  // that the product is made of
  auto cut = [&](int u) { return !along_k(u) && rows_of(u) % 8 != 0; };
  int exist[POLY_UNITS];
#pragma unroll
  for (int u = 0; u < POLY_UNITS; u++) exist[u] = rows_of(u) - first_row(u) > 0 ? rows_of(u) - first_row(u) : 8;
  // smallest magnitude met that is not 0, as twice the bits of the float less 1
  unsigned int least = 0xffffffffu;
  // elements 2 p and 2 p + 1 of a row of 8, as words p of its three planes
  struct Planes { poly_u32x4 t[3]; };
  auto split_pair = [&](const PolyUnit &x, Planes &to, int p) {
    float a = x.v[2 * p], b = x.v[2 * p + 1];
    const unsigned int sa = (__builtin_bit_cast(unsigned int, a) << 1) - 1u, sb = (__builtin_bit_cast(unsigned int, b) << 1) - 1u;
    least = least < sa ? least : sa;
    least = least < sb ? least : sb;
#pragma unroll
    for (int t = 0; t < 3; t++) {
      const unsigned int bits = __builtin_bit_cast(unsigned int, __builtin_convertvector(poly_f32x2{a, b}, poly_in2));
      to.t[t][p] = bits;
      if (t < 2) {
        a -= __builtin_bit_cast(float, bits << 16);
        b -= __builtin_bit_cast(float, bits & 0xffff0000u);
      }
    }
  };
  auto store_unit = [&](const Planes &x, int stage, int u) {
    const int slot = slot_of(u), row = slot / chunks_of(u), swz = along_k(u) ? poly_swz_k(row) : is_a(u) ? poly_swz_x<POLY_BM>(row) : poly_swz_x<POLY_BN>(row);
    unsigned char *const at = lds_raw + stage * POLY_STAGE_BYTES + (is_a(u) ? 0 : 3 * POLY_A_PLANE) + (row * chunks_of(u) + (slot % chunks_of(u) ^ swz)) * 16;
#pragma unroll
    for (int t = 0; t < 3; t++) *(poly_u32x4 *)(at + t * (is_a(u) ? POLY_A_PLANE : POLY_B_PLANE)) = x.t[t];
  };

  const int wm = (wave % POLY_WAVES_M) * POLY_WM, wn = (wave / POLY_WAVES_M) * POLY_WN;
  // (the products of the leading planes by themselves: one rounding for 16 of them)
  poly_acc16 acc[POLY_TM][POLY_TN], low[POLY_TM][POLY_TN];
#pragma unroll
  for (int i = 0; i < POLY_TM; i++)
#pragma unroll
    for (int j = 0; j < POLY_TN; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = low[i][j][r] = 0.0f;

  // fragment addresses within a plane: as in matmul_dma.hip
  int a_fr[POLY_TM], a_sw[POLY_TM], b_fr[POLY_TN], b_sw[POLY_TN];
  const int frag_col = lane >> 5, kl = 8 * (lane >> 5) + ((lane & 15) >> 2), xl = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
#pragma unroll
  for (int i = 0; i < POLY_TM; i++) {
    const int r = wm + i * 32 + (POLY_A_KC ? (lane & 31) : xl);
    a_fr[i] = POLY_A_KC ? r * (POLY_BK * 2) : kl * (POLY_BM * 2) + (((r >> 3) ^ poly_swz_x<POLY_BM>(kl)) * 16) + (r & 7) * 2;
    a_sw[i] = poly_swz_k(r);
  }
#pragma unroll
  for (int j = 0; j < POLY_TN; j++) {
    const int r = wn + j * 32 + (POLY_B_KC ? (lane & 31) : xl);
    b_fr[j] = POLY_B_KC ? r * (POLY_BK * 2) : kl * (POLY_BN * 2) + (((r >> 3) ^ poly_swz_x<POLY_BN>(kl)) * 16) + (r & 7) * 2;
    b_sw[j] = poly_swz_k(r);
  }
  auto read_tr = [&](const unsigned char *p, int pitch) {
    union { poly_s16x4 h[2]; poly_in8 v; } u;
    u.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((poly_lds_s16x4 *)p);
    u.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((poly_lds_s16x4 *)(p + 4 * pitch));
    return u.v;
  };
  auto read_a = [&](int stage, int ks, int t, int i) {
    const unsigned char *p = lds_raw + stage * POLY_STAGE_BYTES + t * POLY_A_PLANE + a_fr[i];
    return POLY_A_KC ? *(const poly_in8 *)(p + (((ks * 2 + frag_col) ^ a_sw[i]) * 16)) : read_tr(p + ks * 16 * (POLY_BM * 2), POLY_BM * 2);
  };
  auto read_b = [&](int stage, int ks, int t, int j) {
    const unsigned char *p = lds_raw + stage * POLY_STAGE_BYTES + 3 * POLY_A_PLANE + t * POLY_B_PLANE + b_fr[j];
    return POLY_B_KC ? *(const poly_in8 *)(p + (((ks * 2 + frag_col) ^ b_sw[j]) * 16)) : read_tr(p + ks * 16 * (POLY_BN * 2), POLY_BN * 2);
  };

  // Iteration s: tile s is in LDS; the registers of tile s + 1 are split and stored into the other stage, a
  // pair of elements behind each MFMA or so, and refilled from tile s + 3, while it is multiplied.
  constexpr int KS = POLY_BK / 16, SLOTS = KS * 8 * POLY_TM * POLY_TN, PAIRS = 4 * POLY_UNITS;
  PolyUnit ring[2][POLY_UNITS];
  load_end(ring[0]);
  if (POLY_NTILES > 1) {
#pragma unroll
    for (int u = 0; u < POLY_UNITS; u++) load_unit(ring[1], 1, u);
  }
#pragma unroll
  for (int u = 0; u < POLY_UNITS; u++) {
    Planes planes;
    move_down(ring[0][u], gone[u]);
#pragma unroll
    for (int p = 0; p < 4; p++) split_pair(ring[0][u], planes, p);
    store_unit(planes, 0, u);
    if (POLY_NTILES > 2) load_unit(ring[0], 2, u);
  }
  auto iteration = [&](int s, int stage, auto &next, bool st, bool ld) {
    __syncthreads();
    poly_in8 fa[2][3][POLY_TM], fb[2][3][POLY_TN];
    auto read_step = [&](int ks) {
#pragma unroll
      for (int t = 0; t < 3; t++) {
#pragma unroll
        for (int i = 0; i < POLY_TM; i++) fa[ks & 1][t][i] = read_a(stage, ks, t, i);
#pragma unroll
        for (int j = 0; j < POLY_TN; j++) fb[ks & 1][t][j] = read_b(stage, ks, t, j);
      }
    };
    Planes planes;
    read_step(0);
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      if (ks + 1 < KS) read_step(ks + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < 8; c++) {
        constexpr int PA[8] = {0, 0, 1, 1, 0, 2, 1, 2}, PB[8] = {0, 1, 0, 1, 2, 0, 2, 1};
#pragma unroll
        for (int i = 0; i < POLY_TM; i++)
#pragma unroll
          for (int j = 0; j < POLY_TN; j++) {
            poly_acc16 &to = c == 0 ? acc[i][j] : low[i][j];
            to = POLY_MFMA(fa[ks & 1][PA[c]][i], fb[ks & 1][PB[c]][j], to);
            const int slot = ((ks * 8 + c) * POLY_TM + i) * POLY_TN + j;
            if (st) {
#pragma unroll
              for (int q = 0; q < PAIRS; q++)
                if (q * SLOTS / PAIRS == slot) {
                  if (cut(q / 4))
#pragma unroll
                    for (int e = q % 4 * 2; e < q % 4 * 2 + 2; e++) next[q / 4].v[e] = e < exist[q / 4] ? next[q / 4].v[e] : 0.0f;
                  split_pair(next[q / 4], planes, q % 4);
                  if (q % 4 == 3) {
                    store_unit(planes, stage ^ 1, q / 4);
                    if (ld) load_unit(next, s + 3, q / 4);
                  }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
          }
      }
    }
  };
  constexpr int STEADY = POLY_NTILES > 3 ? (POLY_NTILES - 3) / 2 * 2 : 0;
  constexpr unsigned int LEAST = 2u * ((127u - 110u) << 23) - 1u;
  // (a workgroup that has met a value below 2^-110 stops: one iteration's barrier lies between what it writes here and
  // what every wave reads)
  bool stopped = false;
#pragma unroll 1
  for (int s = 0; s < STEADY && !stopped; s += 2) {
    iteration(s, 0, ring[1], true, true);
#ifndef POLY_HOST_ADDRESS_CHECK
    stopped = poly_again != 0;
#endif
    if (!stopped) iteration(s + 1, 1, ring[0], true, true);
    if (least < LEAST) poly_again = 1;
  }
  if (!stopped) {
#pragma unroll
    for (int s = STEADY; s < POLY_NTILES; s++) iteration(s, s & 1, ring[(s + 1) & 1], s + 1 < POLY_NTILES, s + 3 < POLY_NTILES);
  }

#pragma unroll
  for (int i = 0; i < POLY_TM; i++)
#pragma unroll
    for (int j = 0; j < POLY_TN; j++) acc[i][j] += low[i][j];

  // Values that three planes do not hold: the tile again in fp32.
  {
    bool again = least < LEAST;
#pragma unroll
    for (int i = 0; i < POLY_TM; i++)
#pragma unroll
      for (int j = 0; j < POLY_TN; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) again = again || !(__builtin_fabsf(acc[i][j][r]) < __builtin_inff());
    if (again) poly_again = 1;
    __syncthreads();
    if (poly_again) {
      poly_acc16 third[POLY_TM][POLY_TN], fourth[POLY_TM][POLY_TN];
#pragma unroll
      for (int i = 0; i < POLY_TM; i++)
#pragma unroll
        for (int j = 0; j < POLY_TN; j++)
#pragma unroll
          for (int r = 0; r < 16; r++) acc[i][j][r] = low[i][j][r] = third[i][j][r] = fourth[i][j][r] = 0.0f;
      // 16 of the depth at a time, 8 to each half of the lanes, which is read while the 16 before are multiplied, into
      // four sums of each result, as many as the fp32 templates have of products of these sizes
      const float *pa[POLY_TM], *pb[POLY_TN];
#pragma unroll
      for (int i = 0; i < POLY_TM; i++) {
        const int m = m0 + wm + i * 32 + (lane & 31);
        pa[i] = gA + poly_a_row(m < POLY_M ? m : POLY_M - 1);
      }
#pragma unroll
      for (int j = 0; j < POLY_TN; j++) {
        const int n = n0 + wn + j * 32 + (lane & 31);
        pb[j] = gB + poly_b_row(n < POLY_N ? n : POLY_N - 1);
      }
      auto load_16 = [&](PolyUnit (&a)[POLY_TM], PolyUnit (&b)[POLY_TN], int k0) {
        const int k = k0 + 8 * (lane >> 5);
        auto load_8 = [&](PolyUnit &to, const float *row, bool kc, auto &&at) {
          if (kc) {
            const poly_f32x4 lo = *(const poly_f32x4_u *)(row + at(k)), hi = *(const poly_f32x4_u *)(row + at(k) + 4);
#pragma unroll
            for (int e = 0; e < 4; e++) { to.v[e] = lo[e]; to.v[4 + e] = hi[e]; }
          } else {
#pragma unroll
            for (int e = 0; e < 8; e++) to.v[e] = row[at(k + e)];
          }
        };
#pragma unroll
        for (int i = 0; i < POLY_TM; i++) load_8(a[i], pa[i], POLY_A_KC, [](int x) { return poly_a_k(x); });
#pragma unroll
        for (int j = 0; j < POLY_TN; j++) load_8(b[j], pb[j], POLY_B_KC, [](int x) { return poly_b_k(x); });
      };
      auto multiply_16 = [&](const PolyUnit (&a)[POLY_TM], const PolyUnit (&b)[POLY_TN]) {
#pragma unroll
        for (int e = 0; e < 8; e++)
#pragma unroll
          for (int i = 0; i < POLY_TM; i++)
#pragma unroll
            for (int j = 0; j < POLY_TN; j++) {
              poly_acc16 &to = e % 4 == 0 ? acc[i][j] : e % 4 == 1 ? low[i][j] : e % 4 == 2 ? third[i][j] : fourth[i][j];
              to = POLY_MFMA_F32(a[i].v[e], b[j].v[e], to);
            }
      };
      constexpr int WHOLE = POLY_KP / 16 * 16;
      PolyUnit a0[POLY_TM], b0[POLY_TN], a1[POLY_TM], b1[POLY_TN];
      if (WHOLE > 0) load_16(a0, b0, 0);
#pragma unroll 1
      for (int k0 = 0; k0 < WHOLE; k0 += 32) {
        if (k0 + 16 < WHOLE) load_16(a1, b1, k0 + 16);
        __builtin_amdgcn_sched_barrier(0);
        multiply_16(a0, b0);
        if (k0 + 16 < WHOLE) {
          if (k0 + 32 < WHOLE) load_16(a0, b0, k0 + 32);
          __builtin_amdgcn_sched_barrier(0);
          multiply_16(a1, b1);
        }
      }
#pragma unroll 1
      for (int k0 = WHOLE; k0 < POLY_KP; k0 += 2) {
        const int k = k0 + (lane >> 5);
        float fa[POLY_TM], fb[POLY_TN];
#pragma unroll
        for (int i = 0; i < POLY_TM; i++) fa[i] = k < POLY_KP ? pa[i][poly_a_k(k)] : 0.0f;
#pragma unroll
        for (int j = 0; j < POLY_TN; j++) fb[j] = k < POLY_KP ? pb[j][poly_b_k(k)] : 0.0f;
#pragma unroll
        for (int i = 0; i < POLY_TM; i++)
#pragma unroll
          for (int j = 0; j < POLY_TN; j++) acc[i][j] = POLY_MFMA_F32(fa[i], fb[j], acc[i][j]);
      }
#pragma unroll
      for (int i = 0; i < POLY_TM; i++)
#pragma unroll
        for (int j = 0; j < POLY_TN; j++) acc[i][j] = (acc[i][j] + low[i][j]) + (third[i][j] + fourth[i][j]);
    }
  }

  // Epilogue: as in matmul_dma.hip.  (The barrier above: every wave is done reading the operand tiles.)
#if !POLY_EP_CONTIG
#pragma unroll
  for (int i = 0; i < POLY_TM; i++)
#pragma unroll
    for (int j = 0; j < POLY_TN; j++) {
      const int n = n0 + wn + j * 32 + (lane & 31);
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const int m = m0 + wm + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        if (m < POLY_M && n < POLY_N) { POLY_EPILOGUE(acc[i][j][r], m, n, z); }
      }
    }
#else
  float *const stage = (float *)lds_raw + wave * (32 * POLY_STAGE_LD);
#pragma unroll
  for (int i = 0; i < POLY_TM; i++)
#pragma unroll
    for (int j = 0; j < POLY_TN; j++) {
#pragma unroll
      for (int r = 0; r < 16; r++) stage[(8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * POLY_STAGE_LD + (lane & 31)] = acc[i][j][r];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
      for (int h = 0; h < 4; h++) {
        const int row = (lane >> 3) + 8 * h, c0 = (lane & 7) * 4;
        const poly_f32x4 v = *(const poly_f32x4 *)(stage + row * POLY_STAGE_LD + c0);
        const int m = m0 + wm + i * 32 + row, n = n0 + wn + j * 32 + c0;
        if (m >= POLY_M || n >= POLY_N) continue;
        typedef POLY_EP_TYPE poly_out4 __attribute__((ext_vector_type(4)));
        typedef poly_out4 poly_out4_u __attribute__((aligned(sizeof(POLY_EP_TYPE))));
        poly_out4 o;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int ne = (POLY_N % 4 == 0 || n + e < POLY_N) ? n + e : n;
          o[e] = POLY_EP_VALUE(v[e], m, ne, z);
        }
        if (POLY_N % 4 == 0 || n + 3 < POLY_N) *(poly_out4_u *)POLY_EP_PTR(m, n, z) = o;
        else
#pragma unroll
          for (int e = 0; e < 4; e++)
            if (n + e < POLY_N) *POLY_EP_PTR(m, n + e, z) = o[e];
#ifdef POLY_EP_MID_VALUE
        {
          // a value on the way to the stored one that other kernels read as well: stored too
          typedef POLY_EP_MID_TYPE poly_mid4 __attribute__((ext_vector_type(4)));
          typedef poly_mid4 poly_mid4_u __attribute__((aligned(sizeof(POLY_EP_MID_TYPE))));
          poly_mid4 mv;
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const int ne = (POLY_N % 4 == 0 || n + e < POLY_N) ? n + e : n;
            mv[e] = POLY_EP_MID_VALUE(v[e], m, ne, z);
          }
          if (POLY_N % 4 == 0 || n + 3 < POLY_N) *(poly_mid4_u *)POLY_EP_MID_PTR(m, n, z) = mv;
          else
#pragma unroll
            for (int e = 0; e < 4; e++)
              if (n + e < POLY_N) *POLY_EP_MID_PTR(m, n + e, z) = mv[e];
        }
#endif
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
#endif
}
