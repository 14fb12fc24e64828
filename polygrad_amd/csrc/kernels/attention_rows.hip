// attention_rows.hip -- fused attention of any number of queries and keys, the scores of a
// query block held whole in the registers of one workgroup.
//
// The kernel group of attention_mfma.hip (scores, pointwise chain, row max, row sum,
// normalise, P V) where that template's blocks of 128 queries x 64 keys do not divide the
// problem, and for fp32 operands.  Every rounding step of the unfused kernels is kept: the
// score as the chain stores it, the term, the probability cast to the operand type before
// the second product.  What differs is the order of the sums, that a term times the sum's
// reciprocal is divided by the sum, and, for the bf16 shapes that attention_mfma.hip could
// take, that a term below 2^-126 is 0 as it is there.  The renderer prepends:
//
//   POLY_TIN, POLY_F32                 operand type, and 1 when it is float
//   POLY_MFMA(a, b, c)                 the 16x16x32 MFMA of a 16-bit type (fp32: 16x16x4)
//   POLY_FA_M, POLY_FA_N, POLY_FA_Z    queries, keys, batch*heads; multiples of nothing
//   POLY_FA_WAVES, POLY_FA_QT          waves of a workgroup; its blocks of 16 queries
//   POLY_FA_PASS_ZEROS                 1: a unit of keys whose probabilities are exact zeros for
//                                      all the queries of a wave is not multiplied (a
//                                      non-finite V under them does not propagate, as in the
//                                      single-pass form of attention_mfma.hip, whose shapes
//                                      these are); 0: it is, as in the unfused kernels
//   POLY_FA_NEAR                       1: no byte of Q, K and V is 2^32 or more from its start
//   POLY_FA_C                          POLY_FA_TERM(x, mx, ..) is exp2((x - mx) * C), C > 0
//   POLY_Q_PTR, POLY_K_PTR, POLY_V_PTR, poly_q_off(z, m), poly_k_off(z, n), poly_v_off(z, n),
//   POLY_FA_SCORE(acc, m, n, z), POLY_FA_MAXV(x, m, n, z), POLY_FA_TERM(x, mx, m, n, z),
//   POLY_FA_OUT(acc, m, d, z), POLY_SIGNATURE: as in attention_mfma.hip
// and the probability is cast(term / sum).
//
// A scheduler's eight launches per layer (three copies of q, k, v, scores, maximum, sum,
// probabilities, product) each wait for the one before, a few microseconds a time whatever
// the size, and write the scores to memory three times.  Here a workgroup takes 16 or 32
// queries, its waves deal the keys among themselves, and nothing but the row statistics and
// the partial outputs goes through LDS: S^T = K Q^T leaves a lane with one query and four
// consecutive keys per 16-key block, which is where the second MFMA wants its A operand
// (the order of keys inside a step is free as long as V is read in the same one).  K and V
// are read from the L2 by every query block.  One launch against the launches it replaces
// (bf16, us): 12 heads of 12 queries and keys 4.1 against eight of 3 to 4 each, 36 of 345 16.3
// [34.2 in three], 36 of 839 61.2 [146 in three]; GPT-2 small on 12 tokens 655 -> 502 us as a
// whole.  What bounds it where rows are long is the arithmetic on the scores (some thirty
// vector instructions each) and what it keeps in registers: two to four waves a SIMD.  The
// scores of masked keys are computed, but not the terms and quotients of units that have no
// other: with that, divisions that a wave decides on together and 32-bit addresses, 36 heads of 345
// keys take 16.0 us inside GPT-2 small where they took 17.4.
#ifdef POLY_TEMPLATE_STANDALONE
#include <hip/hip_runtime.h>
#define POLY_TIN __bf16
#define POLY_F32 0
#define POLY_MFMA(a, b, c) __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0)
#define POLY_FA_M 345
#define POLY_FA_N 345
#define POLY_FA_Z 36
#define POLY_FA_WAVES 8
#define POLY_FA_QT 2
#define POLY_FA_PASS_ZEROS 0
#define POLY_Q_PTR data1
#define POLY_K_PTR data1
#define POLY_V_PTR data1
__device__ __forceinline__ int poly_q_off(int z, int m) { return (z / 12) * 794880 + (z % 12) * 64 + m * 2304; }
__device__ __forceinline__ int poly_k_off(int z, int n) { return (z / 12) * 794880 + (z % 12) * 64 + n * 2304 + 768; }
__device__ __forceinline__ int poly_v_off(int z, int n) { return (z / 12) * 794880 + (z % 12) * 64 + n * 2304 + 1536; }
#define POLY_SIGNATURE __bf16 *data0, const __bf16 *__restrict__ data1, const __bf16 *__restrict__ data2
#define POLY_FA_SCORE(acc, m, n, z) ((__bf16)((float)(__bf16)(acc) * 0.125f + (float)data2[(m) * 345 + (n)]))
#define POLY_FA_MAXV(x, m, n, z) ((float)(x))
#define POLY_FA_TERM(x, mx, m, n, z) __builtin_amdgcn_exp2f(((float)(x) - (mx)) * 0x1.715476p+0f)
#define POLY_FA_C 0x1.715476p+0f
#define POLY_FA_NEAR 1
__device__ __forceinline__ float poly_div_shared(float x, float d, float r, bool ok) { return x / d; }
__device__ __forceinline__ float poly_div_sure(float x, float d, float r) { return x * r; }
#define POLY_FA_OUT(acc, m, d, z) data0[((z) / 12) * 264960 + ((z) % 12) * 22080 + (m) * 64 + (d)] = (__bf16)(acc)
#endif

#ifdef POLY_HOST_ADDRESS_CHECK   // compiled for the host to check its indexing: lanes run one by one, no cross-lane arithmetic
#undef POLY_MFMA
#define POLY_MFMA(a, b, c) (c)
#define POLY_MFMA_F32(a, b, c) (c)
#else
#define POLY_MFMA_F32(a, b, c) __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0)
#endif

typedef float fr_f32x4 __attribute__((ext_vector_type(4)));
typedef POLY_TIN fr_in8 __attribute__((ext_vector_type(8)));
typedef unsigned int fr_u32x4 __attribute__((ext_vector_type(4)));

#define FR_KV (POLY_F32 ? 4 : 8)                  // features per lane and step of the first product
#define FR_STEPS (64 / (4 * FR_KV))               // its steps
#define FR_BU (POLY_F32 ? 1 : 2)                  // 16-key blocks of a unit: one step of the second product
#define FR_UNITS ((POLY_FA_N + 16 * FR_BU - 1) / (16 * FR_BU))
#define FR_UW ((FR_UNITS + POLY_FA_WAVES - 1) / POLY_FA_WAVES)   // units of a wave: unit u of wave w is u * WAVES + w
#define FR_DEPTH (FR_UW < 4 ? FR_UW : 4)          // units whose loads are in flight at a time
#define FR_BM (16 * POLY_FA_QT)

// Element `off` of a buffer: 32-bit byte offsets from its start where they reach all of it, which
// the load instructions add to a scalar base themselves.
#if POLY_FA_NEAR
#define FR_AT(p, off) ((const POLY_TIN *)((const char *)(p) + (size_t)((unsigned)(off) * (unsigned)sizeof(POLY_TIN))))
#else
#define FR_AT(p, off) ((p) + (off))
#endif

// T consecutive elements of any alignment.
template <int T> struct __attribute__((aligned(sizeof(POLY_TIN)))) FrRow { POLY_TIN v[T]; };

__device__ __forceinline__ float fr_lane_xor(float v, int mask) {
  return __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((int)((threadIdx.x & 63) ^ mask) * 4, __builtin_bit_cast(int, v)));
}

#ifdef POLY_FA_OCC   // waves per SIMD the register budget is set for (a tuning candidate: no effect on the values)
#define FR_BUDGET __attribute__((amdgpu_waves_per_eu(POLY_FA_OCC, POLY_FA_OCC)))
#else
#define FR_BUDGET
#endif

extern "C" __global__ void __launch_bounds__(64 * POLY_FA_WAVES) FR_BUDGET poly_k(POLY_SIGNATURE) {
  // Workgroup ids congruent mod 8 run on one XCD (own L2): each XCD gets a contiguous run of
  // query blocks, those of one z side by side, which read the same K and V.
  constexpr int MB = (POLY_FA_M + FR_BM - 1) / FR_BM, NT = MB * POLY_FA_Z;
  int bid = blockIdx.x;
  {
    constexpr int PER = NT / 8, REM = NT % 8;
    const int xcd = bid & 7, idx = bid >> 3;
    bid = (xcd < REM ? xcd * (PER + 1) : REM * (PER + 1) + (xcd - REM) * PER) + idx;
  }
  const int z = bid / MB, m0 = (bid % MB) * FR_BM;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int col = lane & 15, grp = lane >> 4;

  // Rows past the last query and keys past the last one repeat it: their scores are computed
  // and left out.
  int mq[POLY_FA_QT];
  FrRow<FR_KV> q[POLY_FA_QT][FR_STEPS];
#pragma unroll
  for (int i = 0; i < POLY_FA_QT; i++) {
    const int m = m0 + 16 * i + col;
    mq[i] = m < POLY_FA_M ? m : POLY_FA_M - 1;
    const POLY_TIN *p = FR_AT(POLY_Q_PTR, poly_q_off(z, mq[i]) + FR_KV * grp);
#pragma unroll
    for (int s = 0; s < FR_STEPS; s++) q[i][s] = *(const FrRow<FR_KV> *)(p + 4 * FR_KV * s);
  }
  // first key of block b of a wave's unit u
  auto block_at = [&](int u, int b) { return ((u * POLY_FA_WAVES + wave) * FR_BU + b) * 16; };
  auto has_unit = [&](int u) { return u < FR_UW - 1 || u * POLY_FA_WAVES + wave < FR_UNITS; };
  // the last unit of a wave may be the ragged one: is key n there, and the key to read for it
  auto has_key = [&](int u, int n) { return u < FR_UW - 1 || POLY_FA_N % (16 * FR_BU) == 0 || n < POLY_FA_N; };
  auto key_for = [&](int u, int n) { return has_key(u, n) ? n : POLY_FA_N - 1; };

  // ── scores ──────────────────────────────────────────────────────────────────
  float x[POLY_FA_QT][FR_UW][FR_BU][4];    // score of query mq[i] and key block_at(u, b) + 4 grp + r, later its term
  float top[POLY_FA_QT];
#pragma unroll
  for (int i = 0; i < POLY_FA_QT; i++) top[i] = -__builtin_inff();
#pragma unroll
  for (int u0 = 0; u0 < FR_UW; u0 += FR_DEPTH) {
    FrRow<FR_KV> k[FR_DEPTH][FR_BU][FR_STEPS];
#pragma unroll
    for (int d = 0; d < FR_DEPTH; d++) {
      if (u0 + d >= FR_UW || !has_unit(u0 + d)) continue;
#pragma unroll
      for (int b = 0; b < FR_BU; b++) {
        const int n = block_at(u0 + d, b) + col;
        const POLY_TIN *p = FR_AT(POLY_K_PTR, poly_k_off(z, key_for(u0 + d, n)) + FR_KV * grp);
#pragma unroll
        for (int s = 0; s < FR_STEPS; s++) k[d][b][s] = *(const FrRow<FR_KV> *)(p + 4 * FR_KV * s);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int d = 0; d < FR_DEPTH; d++) {
      const int u = u0 + d;
      if (u >= FR_UW || !has_unit(u)) continue;
#pragma unroll
      for (int b = 0; b < FR_BU; b++)
#pragma unroll
        for (int i = 0; i < POLY_FA_QT; i++) {
          fr_f32x4 st = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
          for (int s = 0; s < FR_STEPS; s++) {
#if POLY_F32
#pragma unroll
            for (int e = 0; e < 4; e++) st = POLY_MFMA_F32(k[d][b][s].v[e], q[i][s].v[e], st);
#else
            st = POLY_MFMA(__builtin_bit_cast(fr_in8, k[d][b][s]), __builtin_bit_cast(fr_in8, q[i][s]), st);
#endif
          }
#pragma unroll
          for (int r = 0; r < 4; r++) {
            const int n = block_at(u, b) + 4 * grp + r, nc = key_for(u, n);
            const POLY_TIN v = POLY_FA_SCORE(st[r], mq[i], nc, z);
            x[i][u][b][r] = (float)v;
            if (has_key(u, n)) top[i] = __builtin_fmaxf(top[i], POLY_FA_MAXV(v, mq[i], nc, z));   // like (a < v) ? v : a, a NaN v is ignored
          }
        }
    }
  }
  // V of the first units, on its way while the rows are normalised: 8 (fp32: 4) keys of a
  // lane, the features 4 col .. 4 col + 3 of each; keys past the last one are zeros
  FrRow<4> v[FR_DEPTH][4 * FR_BU];
  auto load_v = [&](int u0) {
#pragma unroll
    for (int d = 0; d < FR_DEPTH; d++) {
      if (u0 + d >= FR_UW || !has_unit(u0 + d)) continue;
#pragma unroll
      for (int e = 0; e < 4 * FR_BU; e++) {
        const int n = block_at(u0 + d, e / 4) + 4 * grp + e % 4;
        v[d][e] = *(const FrRow<4> *)FR_AT(POLY_V_PTR, poly_v_off(z, key_for(u0 + d, n)) + 4 * col);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  load_v(0);

  // ── row maximum and sum of terms: over a lane's keys, the four lanes of a query, the waves ──
  __shared__ float row_top[POLY_FA_WAVES][FR_BM], row_sum[POLY_FA_WAVES][FR_BM];
#pragma unroll
  for (int i = 0; i < POLY_FA_QT; i++) {
    top[i] = __builtin_fmaxf(top[i], fr_lane_xor(top[i], 16));
    top[i] = __builtin_fmaxf(top[i], fr_lane_xor(top[i], 32));
    if (grp == 0) row_top[wave][16 * i + col] = top[i];
  }
  __syncthreads();
  float sum[POLY_FA_QT], rcp[POLY_FA_QT];
  bool rcp_ok[POLY_FA_QT], all_ok[POLY_FA_QT];
  // units (a bit each) whose terms are 0 for all queries of the wave, which masked keys' are, and
  // units whose terms are all small enough for poly_div_sure
  unsigned long long dead[POLY_FA_QT], small[POLY_FA_QT];
#pragma unroll
  for (int i = 0; i < POLY_FA_QT; i++) {
    float t = row_top[0][16 * i + col];
#pragma unroll
    for (int w = 1; w < POLY_FA_WAVES; w++) t = __builtin_fmaxf(t, row_top[w][16 * i + col]);
    float acc = 0.0f;
    dead[i] = small[i] = 0;
#pragma unroll
    for (int u = 0; u < FR_UW; u++) {
      if (!has_unit(u)) continue;
      // the unit's largest score, NaN if one is, bounds its terms; 2^-151 rounds to 0
      float most = x[i][u][0][0];
#pragma unroll
      for (int e = 1; e < 4 * FR_BU; e++) most = __builtin_elementwise_maximum(most, x[i][u][e / 4][e % 4]);
      const float power = (most - t) * POLY_FA_C;
      if (__builtin_amdgcn_ballot_w64(!(power < -151.0f)) == 0) {
        dead[i] |= 1ull << u;
#pragma unroll
        for (int e = 0; e < 4 * FR_BU; e++) x[i][u][e / 4][e % 4] = 0.0f;
        continue;
      }
      if (__builtin_amdgcn_ballot_w64(!(power < 25.0f)) == 0) small[i] |= 1ull << u;
#pragma unroll
      for (int b = 0; b < FR_BU; b++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int n = block_at(u, b) + 4 * grp + r, nc = key_for(u, n);
          const float term = POLY_FA_TERM((POLY_TIN)x[i][u][b][r], t, mq[i], nc, z);
          x[i][u][b][r] = has_key(u, n) ? term : 0.0f;
          acc += x[i][u][b][r];
        }
    }
    acc += fr_lane_xor(acc, 16);
    acc += fr_lane_xor(acc, 32);
    if (grp == 0) row_sum[wave][16 * i + col] = acc;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < POLY_FA_QT; i++) {
    sum[i] = row_sum[0][16 * i + col];
#pragma unroll
    for (int w = 1; w < POLY_FA_WAVES; w++) sum[i] += row_sum[w][16 * i + col];
    rcp[i] = 1.0f / sum[i];
    rcp_ok[i] = __builtin_fabsf(sum[i]) >= 0x1p-100f && __builtin_fabsf(sum[i]) <= 0x1p+100f;
    all_ok[i] = __builtin_amdgcn_ballot_w64(!rcp_ok[i]) == 0;
  }

  // ── P V over the wave's keys: tile t of the output has the features 4 col + t ────────────
  fr_f32x4 o[POLY_FA_QT][4];
#pragma unroll
  for (int i = 0; i < POLY_FA_QT; i++)
#pragma unroll
    for (int t = 0; t < 4; t++) o[i][t] = fr_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int u0 = 0; u0 < FR_UW; u0 += FR_DEPTH) {
    if (u0) load_v(u0);
#pragma unroll
    for (int d = 0; d < FR_DEPTH; d++) {
      const int u = u0 + d;
      if (u >= FR_UW || !has_unit(u)) continue;
#if POLY_FA_PASS_ZEROS
      {
        bool some = false;
#pragma unroll
        for (int i = 0; i < POLY_FA_QT; i++)
#pragma unroll
          for (int e = 0; e < 4 * FR_BU; e++) some = some || !(x[i][u][e / 4][e % 4] == 0.0f);
        if (__builtin_amdgcn_ballot_w64(some) == 0) continue;
      }
#endif
      if (POLY_FA_N % (16 * FR_BU) != 0 && u == FR_UW - 1) {
#pragma unroll
        for (int e = 0; e < 4 * FR_BU; e++) {
          const bool in = has_key(u, block_at(u, e / 4) + 4 * grp + e % 4);
#pragma unroll
          for (int t = 0; t < 4; t++) v[d][e].v[t] = in ? v[d][e].v[t] : (POLY_TIN)0.0f;
        }
      }
#if !POLY_F32
      fr_in8 vf[4];
#pragma unroll
      for (int t = 0; t < 4; t++) {
        fr_u32x4 f;
#pragma unroll
        for (int p = 0; p < 4; p++) {
          const unsigned int lo = __builtin_bit_cast(unsigned short, v[d][2 * p].v[t]), hi = __builtin_bit_cast(unsigned short, v[d][2 * p + 1].v[t]);
          f[p] = lo | (hi << 16);
        }
        vf[t] = __builtin_bit_cast(fr_in8, f);
      }
#endif
#pragma unroll
      for (int i = 0; i < POLY_FA_QT; i++) {
        POLY_TIN p[4 * FR_BU];
        if (all_ok[i] && (dead[i] >> u & 1)) {
#pragma unroll
          for (int e = 0; e < 4 * FR_BU; e++) p[e] = (POLY_TIN)0.0f;
        } else if (all_ok[i] && (small[i] >> u & 1)) {      // (a key that is not there has the term 0)
#pragma unroll
          for (int e = 0; e < 4 * FR_BU; e++) p[e] = (POLY_TIN)poly_div_sure(x[i][u][e / 4][e % 4], sum[i], rcp[i]);
        } else {
#pragma unroll
          for (int e = 0; e < 4 * FR_BU; e++) {
            const POLY_TIN prob = (POLY_TIN)poly_div_shared(x[i][u][e / 4][e % 4], sum[i], rcp[i], rcp_ok[i]);
            p[e] = has_key(u, block_at(u, e / 4) + 4 * grp + e % 4) ? prob : (POLY_TIN)0.0f;
          }
        }
#if POLY_F32
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
          for (int t = 0; t < 4; t++) o[i][t] = POLY_MFMA_F32(p[e], v[d][e].v[t], o[i][t]);
#else
        fr_in8 pf;
#pragma unroll
        for (int e = 0; e < 8; e++) pf[e] = p[e];
#pragma unroll
        for (int t = 0; t < 4; t++) o[i][t] = POLY_MFMA(pf, vf[t], o[i][t]);
#endif
      }
    }
  }

  // ── the waves' partial outputs, added in wave order; register r of a lane is query 4 grp + r ──
  __shared__ __attribute__((aligned(16))) float part[POLY_FA_WAVES][16 * 64];
#pragma unroll
  for (int i = 0; i < POLY_FA_QT; i++) {
    if (i) __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; r++)
      *(fr_f32x4 *)(part[wave] + (4 * grp + r) * 64 + 4 * col) = fr_f32x4{o[i][0][r], o[i][1][r], o[i][2][r], o[i][3][r]};
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 16 / POLY_FA_WAVES; j++) {
      const int row = j * POLY_FA_WAVES + wave, m = m0 + 16 * i + row;
      if (m >= POLY_FA_M) continue;
      float acc = part[0][row * 64 + lane];
#pragma unroll
      for (int w = 1; w < POLY_FA_WAVES; w++) acc += part[w][row * 64 + lane];
      POLY_FA_OUT(acc, m, lane, z);
    }
  }
}
