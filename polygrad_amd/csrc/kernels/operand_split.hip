// operand_split.hip -- writes computed matmul operands as 16-bit planes the 16-bit MFMA
// template can stream: OUT[z][row][part][k], rows of PARTS * POLY_SP_KP elements,
// k-contiguous, zero for k >= POLY_SP_K.
//
// An fp32 value x is cut into three bf16 pieces hi + mid + lo (each the bf16 rounding of
// what the previous ones left over; the two residuals are exact in fp32 and the last
// rounding is below 2^-25 |x|), or into the first two of them (what is left is below
// 2^-17 |x|) for a product whose result is stored as a 16-bit float.  A bf16 x bf16 product is exact in fp32, so
//     sum_k x[k] * b[k]  =  sum over the 3 K_p-long planes of  piece[k'] * b[k' mod K_p]
// on the bf16 MFMA with fp32 accumulation carries the same information as the fp32
// product at about a third of the bf16 rate (the fp32 MFMA runs at a sixteenth).  An
// operand that is a 16-bit value cast to fp32 is written as the single plane it is (fp16
// only where the other operand is one, too).
//
// Configuration (prepended by templates.cc):
//   POLY_SP_T                              element type of the planes (fp16: one part each)
//   POLY_SP_K / POLY_SP_Z                  depth and batch
//   POLY_SP_KP                             K rounded up to the K tile of the matmul
//   POLY_SP_A, POLY_SP_B                   1: the launch writes this operand.  Its workgroups
//                                          are blockIdx.x = 0 .. tiles - 1, B's behind A's
//   per operand X = A, B, where written:
//   POLY_SP_X_ROWS                         its extent (M or N)
//   POLY_SP_X_PARTS                        3 or 2 (fp32 value) or 1 (already a 16-bit value)
//   POLY_SP_X_WALK_K                       1: the source is contiguous along k, 0: along rows
//   POLY_SP_X_NRAW, POLY_SP_X_LOAD(row, k, z, raw), POLY_SP_X_MATH(row, k, z, raw)
//                                          the operand as the computed-operand matmul has it
//   POLY_SP_X_OUT                          where its planes go
//   POLY_SIGNATURE
//
// One workgroup of 256 threads handles a 64 (rows) x 64 (k) tile, 16 values per thread: two
// groups of 8 neighbours along k when the source is contiguous in k and K a multiple of 8;
// otherwise with lanes along the source's contiguous axis and through LDS, to leave with
// lanes along k.
//
// Where the operands are a few megabytes what it takes is latency, of the launch and of the
// loads: hence both operands in one launch, and for an operand of a single load all 16 of a
// thread's loads in flight (four otherwise: the registers of what computes the value).
// Measured, whole plan: bf16 1111x999x1501 27.3 us with a launch per operand and four loads in
// flight, 21.3 so, 17.8 without launches that read the operands ahead; 3001x2999x1003 53 -> 46.  fp16 operands as fp16 planes where they were one
// computed-operand product on the fp32 MFMA: 1111x999x1501 105 -> 25, 3001x2999x1003 411 -> 48.
#ifdef POLY_TEMPLATE_STANDALONE
#include <hip/hip_runtime.h>
#define POLY_SP_T __bf16
#define POLY_SP_K 1000
#define POLY_SP_KP 1024
#define POLY_SP_Z 1
#define POLY_SP_A 1
#define POLY_SP_B 1
#define POLY_SP_A_ROWS 4096
#define POLY_SP_A_PARTS 3
#define POLY_SP_A_WALK_K 1
#define POLY_SP_A_NRAW 1
#define POLY_SP_A_LOAD(row, k, z, raw) raw[0] = __builtin_bit_cast(unsigned int, data1[(row) * POLY_SP_K + (k)])
#define POLY_SP_A_MATH(row, k, z, raw) __builtin_bit_cast(float, raw[0])
#define POLY_SP_A_OUT poly_planes
#define POLY_SP_B_ROWS 1001
#define POLY_SP_B_PARTS 1
#define POLY_SP_B_WALK_K 0
#define POLY_SP_B_NRAW 1
#define POLY_SP_B_LOAD(row, k, z, raw) raw[0] = (unsigned int)__builtin_bit_cast(unsigned short, data2[(k) * POLY_SP_B_ROWS + (row)])
#define POLY_SP_B_MATH(row, k, z, raw) (float)__builtin_bit_cast(__bf16, (unsigned short)raw[0])
#define POLY_SP_B_OUT (poly_planes + 4096 * 3 * 1024)
#define POLY_SIGNATURE float *data0, const float *__restrict__ data1, const __bf16 *__restrict__ data2, __bf16 *poly_planes
#endif

typedef POLY_SP_T sp_out8 __attribute__((ext_vector_type(8)));

// Tile `block` of one operand of ROWS rows whose value at (row, k) is `value`.
template <int ROWS, int PARTS, bool WALK_K, int NRAW, class V>
__device__ __forceinline__ void poly_split_tile(int block, int z, POLY_SP_T *planes, float (&tile)[64][65], V value) {
  constexpr int TILES_K = POLY_SP_KP / 64;
  const int row0 = block / TILES_K * 64, k0 = block % TILES_K * 64;
  POLY_SP_T *const out = planes + (size_t)z * ROWS * (PARTS * POLY_SP_KP);
  // 8 consecutive k of one row leave as one 16-byte store per plane (rows of the planes
  // start on multiples of 64 elements from a 256-byte aligned base)
  auto write_planes = [&](int row, int lk, const float (&x)[8]) {
    POLY_SP_T *const dst = out + (size_t)row * (PARTS * POLY_SP_KP) + k0 + lk;
    sp_out8 hi, mid, lo;
#pragma unroll
    for (int e = 0; e < 8; e++) {
      hi[e] = (POLY_SP_T)x[e];
      if (PARTS >= 2) {
        // (an infinite or NaN x is all in hi: no inf - inf in the residuals)
        const float r1 = __builtin_isfinite((float)hi[e]) ? x[e] - (float)hi[e] : 0.0f;
        mid[e] = (POLY_SP_T)r1;
        lo[e] = (POLY_SP_T)(r1 - (float)mid[e]);
      }
    }
    *(sp_out8 *)dst = hi;
    if (PARTS >= 2) *(sp_out8 *)(dst + POLY_SP_KP) = mid;
    if (PARTS == 3) *(sp_out8 *)(dst + 2 * POLY_SP_KP) = lo;
  };
  if constexpr (WALK_K && POLY_SP_K % 8 == 0) {
    // along k, rows a multiple of 8 long: a thread takes 8 neighbours, so that what the operand's expression loads for
    // them sits side by side and can be fetched together, and they are a row's piece as the
    // planes store it: no exchange needed
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int g = threadIdx.x + i * 256;
      const int lr = g / 8, lk = (g % 8) * 8;
      const int row = row0 + lr;
      if (row >= ROWS) continue;
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const int k = k0 + lk + e;
        x[e] = k < POLY_SP_K ? value(row, k) : 0.0f;
      }
      write_planes(row, lk, x);
    }
  } else {
    // along the rows, or along rows of k of any length: lanes along that axis (64 neighbours
    // per load), through LDS, to leave with lanes along k
    constexpr int FLIGHT = NRAW == 1 ? 16 : 4;
#pragma unroll 1
    for (int j = 0; j < 16; j += FLIGHT) {
      float v[FLIGHT];
#pragma unroll
      for (int i = 0; i < FLIGHT; i++) {
        const int c = threadIdx.x + (j + i) * 256;
        const int row = row0 + (WALK_K ? c / 64 : c % 64), k = k0 + (WALK_K ? c % 64 : c / 64);
        v[i] = row < ROWS && k < POLY_SP_K ? value(row, k) : 0.0f;
      }
#pragma unroll
      for (int i = 0; i < FLIGHT; i++) {
        const int c = threadIdx.x + (j + i) * 256;
        tile[WALK_K ? c / 64 : c % 64][WALK_K ? c % 64 : c / 64] = v[i];
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int g = threadIdx.x + i * 256;
      const int lr = g / 8, lk = (g % 8) * 8;
      const int row = row0 + lr;
      if (row >= ROWS) continue;
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; e++) x[e] = tile[lr][lk + e];
      write_planes(row, lk, x);
    }
  }
}

extern "C" __global__ void __launch_bounds__(256) poly_k(POLY_SIGNATURE) {
  __shared__ float tile[64][65];
  const int z = blockIdx.y;
  int block = blockIdx.x;
#if POLY_SP_A
  constexpr int BLOCKS_A = (POLY_SP_A_ROWS + 63) / 64 * (POLY_SP_KP / 64);
  if (!POLY_SP_B || block < BLOCKS_A) {
    auto value = [&](int row, int k) {
      unsigned int raw[POLY_SP_A_NRAW];
      POLY_SP_A_LOAD(row, k, z, raw);
      return POLY_SP_A_MATH(row, k, z, raw);
    };
    poly_split_tile<POLY_SP_A_ROWS, POLY_SP_A_PARTS, POLY_SP_A_WALK_K, POLY_SP_A_NRAW>(block, z, POLY_SP_A_OUT, tile, value);
    return;
  }
  block -= BLOCKS_A;
#endif
#if POLY_SP_B
  auto value = [&](int row, int k) {
    unsigned int raw[POLY_SP_B_NRAW];
    POLY_SP_B_LOAD(row, k, z, raw);
    return POLY_SP_B_MATH(row, k, z, raw);
  };
  poly_split_tile<POLY_SP_B_ROWS, POLY_SP_B_PARTS, POLY_SP_B_WALK_K, POLY_SP_B_NRAW>(block, z, POLY_SP_B_OUT, tile, value);
#endif
}
