// matmul_wave.hip -- matmul template for products of few or ragged output tiles.
//
// C[z][m][n] = epilogue( sum_k A(z,m,k) * B(z,k,n) ), bf16 / fp16 / fp32 inputs, fp32
// accumulation on the 16x16 MFMAs.  The renderer (templates.cc) prepends:
//
//   POLY_TIN, POLY_F32  input element type, and 1 when it is float
//   POLY_MFMA(a,b,c)    the 16x16x32 MFMA of a 16-bit type (fp32: 16x16x4)
//   POLY_M/N/K/Z        problem sizes; no multiple of anything
//   POLY_BLOCK          (optional) rows and columns of a block: 16, or 32 for fp32 (the 32x32x2 MFMA)
//   POLY_TM, POLY_TN    output tile of a workgroup in blocks
//   POLY_WAVES          waves of a workgroup: each has the whole tile and every
//                       POLY_WAVES-th step of the depth
//   POLY_DEPTH          steps of a wave whose loads are in flight at a time
//   POLY_SUMS           (optional) 2: a wave adds its even and its odd steps up apart, and the
//                       two at the end (POLY_DEPTH is even)
//   POLY_KSPLIT         (optional) workgroups that share the depth of a tile (blockIdx.y =
//                       z * POLY_KSPLIT + part): each leaves its sum where POLY_EPILOGUE puts
//                       it, which may use `poly_ks`, the part
//   POLY_TOUCH_WGS      (optional, one z, no POLY_KSPLIT) that many extra workgroups at the front of
//                       the grid, a multiple of 8, which multiply nothing: they read one element of every
//                       64 bytes of B and leave, each the columns that the tiles of its own XCD have
//   POLY_A_KC/B_KC      1: operand contiguous along K; 0: along M (resp. N)
//   POLY_A_ROWS(row, lane, out)  (optional, one z, A contiguous along K in rows of K
//                       elements) A is no buffer: this stores element f of its row `row` at
//                       position row * K + f of `out`, called by POLY_A_ROW_LANES (32 or 64)
//                       lanes; PolyRowsOut{place, first}, what `out` is: the rows from position
//                       `first` on, in LDS at `place`; and POLY_A_UNREAD, which declares the
//                       pointer A would have had
//   POLY_A_PTR/B_PTR, poly_a_row(m), poly_b_row(n), poly_a_z(z), poly_b_z(z),
//   poly_a_k(k), poly_b_k(k), POLY_SIGNATURE, POLY_EPILOGUE(acc, m, n, z) and
//   optionally POLY_EP_MID_VALUE / POLY_EP_MID_PTR: as in matmul_mfma.hip
//
// What such a product waits for is memory latency: a few dozen workgroups cannot keep
// HBM busy through a pipeline of LDS tiles with a barrier per tile (12 x 768 x 3072 took
// 29.7 us on 64x256 tiles of the register-staged template, of which 3 workgroups exist;
// its 4.7 MB of weights are 1 us of HBM time).  Here the depth is dealt to the waves of a
// workgroup instead.  No two waves need the same operand element, so nothing goes through
// LDS on the way in: a lane loads what the MFMA wants of it straight into registers,
// POLY_DEPTH steps ahead, without a barrier before the end, where the waves' partial tiles
// are added in wave order through LDS.  The order of k inside a step is free as long as
// both operands agree, so a k-contiguous operand is read as 16 bytes per lane (lane group g
// of a step has k = g * KV .. g * KV + KV - 1) and one contiguous along its rows as POLY_T
// rows per lane and k, put together by byte permutes (16-bit) or not at all (fp32).
// Measured against the tile templates (one launch, us): bf16 12 x 768 x 3072 31.0 -> 5.4,
// 64 x 3072 x 768 12.5 -> 3.9, 7473 x 219 x 188 17.7 -> 6.9, 410 x 7104 x 318 39.1 -> 13.5;
// fp32 128 x 3072 x 768 22.3 -> 10.1 (60 TFLOP/s of the 157 of the fp32 MFMAs),
// 33 x 129 x 784 30.6 -> 3.8.  What bounds it where there are
// many rows is the address path: 16 lanes of a load along K read 16 different rows, 64 bytes
// of each (1035 x 768 x 3072 takes 20 us where tiles in LDS take 12).  Where B comes from HBM
// it is its latency: the waves have some 50 KB a CU on their way, which at 2 us is half of what
// they take.  CUs without a tile read ahead then (POLY_TOUCH_WGS: fp32 128 x 768 x 3072
// 17.3 -> 14.1 us, 13.0 with B in the caches; bf16 12 x 768 x 3072 7.6 -> 6.5).
#ifdef POLY_TEMPLATE_STANDALONE
#include <hip/hip_runtime.h>
#define POLY_TIN __bf16
#define POLY_F32 0
#define POLY_MFMA(a, b, c) __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0)
#define POLY_M 1035
#define POLY_N 1001
#define POLY_K 3077
#define POLY_Z 1
#define POLY_TM 4
#define POLY_TN 4
#define POLY_WAVES 8
#define POLY_DEPTH 3
#define POLY_A_KC 1
#define POLY_B_KC 0
#define POLY_A_PTR data1
#define POLY_B_PTR data2
__device__ __forceinline__ int poly_a_row(int m) { return m * POLY_K; }
__device__ __forceinline__ int poly_b_row(int n) { return n; }
__device__ __forceinline__ int poly_a_z(int z) { return 0; }
__device__ __forceinline__ int poly_b_z(int z) { return 0; }
__device__ __forceinline__ int poly_a_k(int k) { return k; }
__device__ __forceinline__ int poly_b_k(int k) { return k * POLY_N; }
#define POLY_SIGNATURE float *data0, const __bf16 *__restrict__ data1, const __bf16 *__restrict__ data2
#define POLY_EPILOGUE(acc, m, n, z) data0[(m) * POLY_N + (n)] = (acc)
#endif

#ifdef POLY_HOST_ADDRESS_CHECK   // compiled for the host to check its indexing: lanes run one by one, no cross-lane arithmetic
#undef POLY_MFMA
#define POLY_MFMA(a, b, c) (c)
#define POLY_MFMA_F32(a, b, c) (c)
#elif defined(POLY_BLOCK) && POLY_BLOCK == 32
#define POLY_MFMA_F32(a, b, c) __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0)
#else
#define POLY_MFMA_F32(a, b, c) __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0)
#endif
#ifndef POLY_BLOCK
#define POLY_BLOCK 16
#endif
#define POLY_GROUPS (64 / POLY_BLOCK)              // of lanes: a group has a block's rows, each group its own k
#define POLY_ACC (POLY_BLOCK * POLY_BLOCK / 64)    // registers of a block's sums

typedef float poly_acc __attribute__((ext_vector_type(POLY_ACC)));
typedef POLY_TIN poly_in8 __attribute__((ext_vector_type(8)));
typedef unsigned int poly_u32x4 __attribute__((ext_vector_type(4)));

#define POLY_NTHREADS (64 * POLY_WAVES)
#define POLY_KV (POLY_F32 ? 4 : 8)          // k per lane and step
#define POLY_KSTEP (POLY_GROUPS * POLY_KV)  // k per step
#ifndef POLY_KSPLIT
#define POLY_KSPLIT 1
#endif
#define POLY_KPART (POLY_K / POLY_KSPLIT)   // depth of one workgroup
#ifndef POLY_SUMS
#define POLY_SUMS 1
#endif
#define POLY_BM (POLY_BLOCK * POLY_TM)
#define POLY_BN (POLY_BLOCK * POLY_TN)

// T consecutive elements of any alignment.
template <int T> struct __attribute__((aligned(sizeof(POLY_TIN)))) PolyRow { POLY_TIN v[T]; };

// One operand's share of a step for one lane.
// Along K: T rows of KV elements.
template <bool KC, int T> struct PolyOp {
  PolyRow<POLY_KV> r[T];
  template <class K> __device__ __forceinline__ void load(const POLY_TIN *__restrict__ base, const int (&row)[T], int k, K kofs) {
    const int o = kofs(k);
#pragma unroll
    for (int t = 0; t < T; t++) r[t] = *(const PolyRow<POLY_KV> *)(base + row[t] + o);
  }
  // the elements from POLY_KPART on as zeros, and not read
  template <class K> __device__ __forceinline__ void load_end(const POLY_TIN *__restrict__ base, const int (&row)[T], int k, K kofs) {
    if (k + POLY_KV <= POLY_KPART) { load(base, row, k, kofs); return; }
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
      for (int e = 0; e < POLY_KV; e++) r[t].v[e] = k + e < POLY_KPART ? base[row[t] + kofs(k + e)] : (POLY_TIN)0.0f;
  }
  __device__ __forceinline__ POLY_TIN at(int t, int e) const { return r[t].v[e]; }
#if !POLY_F32
  __device__ __forceinline__ poly_in8 frag(int t) const { return __builtin_bit_cast(poly_in8, r[t]); }
#endif
};
// Along the rows: KV times T rows of one k.
template <int T> struct PolyOp<false, T> {
  PolyRow<T> r[POLY_KV];
  template <class K> __device__ __forceinline__ void load(const POLY_TIN *__restrict__ base, const int (&row)[1], int k, K kofs) {
#pragma unroll
    for (int e = 0; e < POLY_KV; e++) r[e] = *(const PolyRow<T> *)(base + row[0] + kofs(k + e));
  }
  template <class K> __device__ __forceinline__ void load_end(const POLY_TIN *__restrict__ base, const int (&row)[1], int k, K kofs) {
#pragma unroll
    for (int e = 0; e < POLY_KV; e++) {
      PolyRow<T> x = {};
      if (k + e < POLY_KPART) x = *(const PolyRow<T> *)(base + row[0] + kofs(k + e));
      r[e] = x;
    }
  }
  __device__ __forceinline__ POLY_TIN at(int t, int e) const { return r[e].v[t]; }
#if !POLY_F32
  __device__ __forceinline__ poly_in8 frag(int t) const {
    poly_u32x4 f;
#pragma unroll
    for (int p = 0; p < 4; p++) {
      const unsigned int lo = __builtin_bit_cast(unsigned short, r[2 * p].v[t]), hi = __builtin_bit_cast(unsigned short, r[2 * p + 1].v[t]);
      f[p] = lo | (hi << 16);
    }
    return __builtin_bit_cast(poly_in8, f);
  }
#endif
};

#ifdef POLY_A_ROWS
// Rows in LDS, 16 bytes further apart than they are long: the 16 lanes that read a chunk of 16
// rows meet 16 different 16-byte slots of the banks.  K is a multiple of KV.
#define POLY_ROW_PAD (16 / (int)sizeof(POLY_TIN))
struct PolyOpRows {
  PolyRow<POLY_KV> r[POLY_TM];
  template <class K> __device__ __forceinline__ void load(const POLY_TIN *base, const int (&row)[POLY_TM], int k, K) {
#pragma unroll
    for (int t = 0; t < POLY_TM; t++) r[t] = __builtin_bit_cast(PolyRow<POLY_KV>, *(const poly_u32x4 *)(base + row[t] + k));
  }
  template <class K> __device__ __forceinline__ void load_end(const POLY_TIN *base, const int (&row)[POLY_TM], int k, K kofs) {
    if (k < POLY_KPART) { load(base, row, k, kofs); return; }
#pragma unroll
    for (int t = 0; t < POLY_TM; t++) r[t] = PolyRow<POLY_KV>{};
  }
  __device__ __forceinline__ POLY_TIN at(int t, int e) const { return r[t].v[e]; }
#if !POLY_F32
  __device__ __forceinline__ poly_in8 frag(int t) const { return __builtin_bit_cast(poly_in8, r[t]); }
#endif
};
#endif

extern "C" __global__ void __launch_bounds__(POLY_NTHREADS) poly_k(POLY_SIGNATURE) {
  // Workgroup ids congruent mod 8 run on one XCD (own L2): each XCD gets a contiguous run of
  // tiles, down the rows first, so that the workgroups that read one panel of B share an L2.
  constexpr int TILES_M = (POLY_M + POLY_BM - 1) / POLY_BM, NT = TILES_M * ((POLY_N + POLY_BN - 1) / POLY_BN);
#ifdef POLY_TOUCH_WGS
  static_assert(POLY_TOUCH_WGS % 8 == 0, "the workgroups behind keep their XCDs");
  if (blockIdx.x < POLY_TOUCH_WGS) {
    // this XCD's tiles, and their columns of B: one element of every 64 bytes
    constexpr int PER = NT / 8, REM = NT % 8, EL = 64 / (int)sizeof(POLY_TIN);
    const int xcd = blockIdx.x & 7, first = xcd < REM ? xcd * (PER + 1) : REM * (PER + 1) + (xcd - REM) * PER, last = first + PER + (xcd < REM) - 1;
    const int n_lo = first / TILES_M * POLY_BN, n_end = (last / TILES_M + 1) * POLY_BN, n_hi = n_end < POLY_N ? n_end : POLY_N;
    if (last < first) return;
    const POLY_TIN *__restrict__ const p = POLY_B_PTR + poly_b_z(0);
    constexpr int STEP = POLY_TOUCH_WGS / 8 * POLY_NTHREADS;
    unsigned int seen = 0;
#if POLY_B_KC
    const int per_row = (POLY_K + EL - 1) / EL, lines = (n_hi - n_lo) * per_row;
#else
    const int per_row = (n_hi - n_lo + EL - 1) / EL, lines = POLY_K * per_row;
#endif
#pragma unroll 8
    for (int i = (blockIdx.x >> 3) * POLY_NTHREADS + threadIdx.x; i < lines; i += STEP) {
      const int r = i / per_row, x = (i - r * per_row) * EL;
#if POLY_B_KC
      const POLY_TIN v = p[poly_b_row(n_lo + r) + poly_b_k(x)];
#else
      const POLY_TIN v = p[poly_b_row(n_lo + x) + poly_b_k(r)];
#endif
#if POLY_F32
      seen ^= __builtin_bit_cast(unsigned int, v);
#else
      seen ^= __builtin_bit_cast(unsigned short, v);
#endif
    }
    asm volatile("" ::"v"(seen));
    return;
  }
  int bid = blockIdx.x - POLY_TOUCH_WGS;
#else
  int bid = blockIdx.x;
#endif
  {
    constexpr int PER = NT / 8, REM = NT % 8;
    const int xcd = bid & 7, idx = bid >> 3;
    bid = (xcd < REM ? xcd * (PER + 1) : REM * (PER + 1) + (xcd - REM) * PER) + idx;
  }
  const int m0 = (bid % TILES_M) * POLY_BM, n0 = (bid / TILES_M) * POLY_BN;
#if POLY_KSPLIT > 1
  const int z = blockIdx.y / POLY_KSPLIT, poly_ks = blockIdx.y % POLY_KSPLIT, k_base = poly_ks * POLY_KPART;
#else
  const int z = blockIdx.y;
  constexpr int k_base = 0;
#endif
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int col = lane % POLY_BLOCK, grp = lane / POLY_BLOCK;
#ifdef POLY_A_ROWS
  POLY_A_UNREAD;
  __shared__ __attribute__((aligned(16))) POLY_TIN gA[POLY_BM * (POLY_K + POLY_ROW_PAD)];
  const int n_rows = POLY_M - m0 < POLY_BM ? POLY_M - m0 : POLY_BM;
  static_assert(POLY_BLOCK == 16 && POLY_KSPLIT == 1 && POLY_K % POLY_KV == 0, "a tile of whole rows");
#else
  const POLY_TIN *__restrict__ gA = POLY_A_PTR + poly_a_z(z);
#endif
  const POLY_TIN *__restrict__ gB = POLY_B_PTR + poly_b_z(z);

  // Rows of A (columns of B) of a lane.  Along K: block t has row POLY_BLOCK t + col; rows past the
  // edge repeat the last one and are not stored.  Along the rows: rows T col .. T col + T - 1,
  // one of each block; a lane whose T rows cross the edge starts T rows before it, and its
  // block t then has row T col + t - (shift), which another lane's block has too unless
  // t >= shift: only that one is stored.
#ifdef POLY_A_ROWS
  int a_row[POLY_TM];
#pragma unroll
  for (int t = 0; t < POLY_TM; t++) a_row[t] = (16 * t + col < n_rows ? 16 * t + col : n_rows - 1) * (POLY_K + POLY_ROW_PAD);
#elif POLY_A_KC
  int a_row[POLY_TM];
#pragma unroll
  for (int t = 0; t < POLY_TM; t++) { const int m = m0 + POLY_BLOCK * t + col; a_row[t] = poly_a_row(m < POLY_M ? m : POLY_M - 1); }
#else
  int a_row[1];
  { const int m = m0 + POLY_TM * col; a_row[0] = poly_a_row(m <= POLY_M - POLY_TM ? m : POLY_M - POLY_TM); }
#endif
#if POLY_B_KC
  int b_row[POLY_TN];
#pragma unroll
  for (int t = 0; t < POLY_TN; t++) { const int n = n0 + POLY_BLOCK * t + col; b_row[t] = poly_b_row(n < POLY_N ? n : POLY_N - 1); }
#else
  int b_row[1];
  { const int n = n0 + POLY_TN * col; b_row[0] = poly_b_row(n <= POLY_N - POLY_TN ? n : POLY_N - POLY_TN); }
#endif
#ifdef POLY_A_ROWS
  typedef PolyOpRows OpA;
#else
  typedef PolyOp<POLY_A_KC, POLY_TM> OpA;
#endif
  typedef PolyOp<POLY_B_KC, POLY_TN> OpB;
  auto ka = [&](int k) { return poly_a_k(k_base + k); };
  auto kb = [&](int k) { return poly_b_k(k_base + k); };

  poly_acc sums[POLY_SUMS][POLY_TM][POLY_TN];
#pragma unroll
  for (int s = 0; s < POLY_SUMS; s++)
#pragma unroll
    for (int i = 0; i < POLY_TM; i++)
#pragma unroll
      for (int j = 0; j < POLY_TN; j++)
#pragma unroll
        for (int r = 0; r < POLY_ACC; r++) sums[s][i][j][r] = 0.0f;
  auto multiply = [&](const OpA &a, const OpB &b, poly_acc (&acc)[POLY_TM][POLY_TN]) {
#if POLY_F32
#pragma unroll
    for (int e = 0; e < POLY_KV; e++)
#pragma unroll
      for (int i = 0; i < POLY_TM; i++)
#pragma unroll
        for (int j = 0; j < POLY_TN; j++) acc[i][j] = POLY_MFMA_F32(a.at(i, e), b.at(j, e), acc[i][j]);
#else
    poly_in8 fb[POLY_TN];
#pragma unroll
    for (int j = 0; j < POLY_TN; j++) fb[j] = b.frag(j);
#pragma unroll
    for (int i = 0; i < POLY_TM; i++) {
      const poly_in8 fa = a.frag(i);
#pragma unroll
      for (int j = 0; j < POLY_TN; j++) acc[i][j] = POLY_MFMA(fa, fb[j], acc[i][j]);
    }
#endif
  };

  // Step s of a wave covers k from (s * POLY_WAVES + wave) * POLY_KSTEP on.  STEPS of them
  // are complete for every wave; whatever is left is one more step with the missing part of
  // the depth as zeros, the first to be loaded and multiplied.
  constexpr int STEPS = POLY_KPART / (POLY_KSTEP * POLY_WAVES);
  constexpr int END = POLY_KPART % (POLY_KSTEP * POLY_WAVES) != 0, ALL = STEPS + END;
  constexpr int D = POLY_DEPTH;
  OpA ra[D];
  OpB rb[D];
  const int kl = wave * POLY_KSTEP + grp * POLY_KV;
  // (fenced: the compiler would move every load down to its use)
  auto load = [&](int d, int s, bool a = true, bool b = true) {
    __builtin_amdgcn_sched_barrier(0);
    if (END && s == 0) {
      const int k = kl + STEPS * (POLY_KSTEP * POLY_WAVES);
      if (a) ra[d].load_end(gA, a_row, k, ka);
      if (b) rb[d].load_end(gB, b_row, k, kb);
    } else {
      const int k = kl + (s - END) * (POLY_KSTEP * POLY_WAVES);
      if (a) ra[d].load(gA, a_row, k, ka);
      if (b) rb[d].load(gB, b_row, k, kb);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
#ifdef POLY_A_ROWS
  // A's rows while B's first steps are on their way
#pragma unroll
  for (int s = 0; s < (ALL < D ? ALL : D); s++) load(s, s, false, true);
  for (int row = wave * (64 / POLY_A_ROW_LANES) + lane / POLY_A_ROW_LANES; row < n_rows; row += POLY_WAVES * (64 / POLY_A_ROW_LANES)) {
    const PolyRowsOut to{gA + row * (POLY_K + POLY_ROW_PAD), (m0 + row) * POLY_K};
    POLY_A_ROWS((long long)(m0 + row), lane % POLY_A_ROW_LANES, to);
  }
  __syncthreads();
#pragma unroll
  for (int s = 0; s < (ALL < D ? ALL : D); s++) load(s, s, true, false);
#else
#pragma unroll
  for (int s = 0; s < (ALL < D ? ALL : D); s++) load(s, s);
#endif
  constexpr int STEADY = ALL > 2 * D ? (ALL - D) / D * D : 0;
#pragma unroll 1
  for (int s = 0; s < STEADY; s += D) {
#pragma unroll
    for (int d = 0; d < D; d++) { multiply(ra[d], rb[d], sums[d % POLY_SUMS]); load(d, s + d + D); }
  }
#pragma unroll
  for (int s = STEADY; s < ALL; s++) {
    multiply(ra[s % D], rb[s % D], sums[s % POLY_SUMS]);
    if (s + D < ALL) load(s % D, s + D);
  }
  static_assert(D % POLY_SUMS == 0, "a step of the unrolled loop has its sum");
  poly_acc (&acc)[POLY_TM][POLY_TN] = sums[0];
#if POLY_SUMS == 2
#pragma unroll
  for (int i = 0; i < POLY_TM; i++)
#pragma unroll
    for (int j = 0; j < POLY_TN; j++) acc[i][j] += sums[1][i][j];
#endif

  // The partial tiles of the waves, CH blocks of rows at a time, in LDS as the MFMA leaves
  // them (lane l, register r of a block of 16: row 4 (l / 16) + r, column l % 16; of 32: row
  // 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32): rows 20 (36) floats apart and blocks 336
  // (1168), which keeps both the writes and the reads along n off each other's banks.  Each
  // thread then adds up the elements it finishes, in wave order.
  constexpr int RS = POLY_BLOCK + 4, BS = POLY_BLOCK * RS + 16;
  constexpr int CH = POLY_TM % 2 == 0 && POLY_WAVES * 2 * POLY_TN * BS * 4 <= 65536 ? 2 : 1;
  __shared__ float part[POLY_WAVES * CH * POLY_TN * BS];
#pragma unroll
  for (int c = 0; c < POLY_TM; c += CH) {
    if (c) __syncthreads();
#pragma unroll
    for (int i = 0; i < CH; i++)
#pragma unroll
      for (int j = 0; j < POLY_TN; j++)
#pragma unroll
        for (int r = 0; r < POLY_ACC; r++)
          part[((wave * CH + i) * POLY_TN + j) * BS + (4 * POLY_GROUPS * (r / 4) + 4 * grp + r % 4) * RS + col] = acc[c + i][j][r];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < (CH * POLY_BLOCK * POLY_BN + POLY_NTHREADS - 1) / POLY_NTHREADS; q++) {
      const int id = q * POLY_NTHREADS + (int)threadIdx.x;
      if (CH * POLY_BLOCK * POLY_BN % POLY_NTHREADS != 0 && id >= CH * POLY_BLOCK * POLY_BN) break;
      const int x = id % POLY_BN, y = id / POLY_BN, row = y % POLY_BLOCK, i = y / POLY_BLOCK;
      const int n = n0 + x;
#if POLY_A_KC
      const int m = m0 + POLY_BLOCK * (c + i) + row;
      const bool mine = m < POLY_M;
#else
      const int first = m0 + POLY_TM * row, over = first - (POLY_M - POLY_TM), shift = over > 0 ? over : 0;
      const int m = first - shift + c + i;
      const bool mine = c + i >= shift;
#endif
      if (!mine || n >= POLY_N) continue;
#if POLY_B_KC
      const int j = x / POLY_BLOCK, cc = x % POLY_BLOCK;
#else
      const int cc = x / POLY_TN, nf = n0 + POLY_TN * cc - (POLY_N - POLY_TN), j = x % POLY_TN + (nf > 0 ? nf : 0);
#endif
      const float *p = part + (i * POLY_TN + j) * BS + row * RS + cc;
      float acc_sum = p[0];
#pragma unroll
      for (int w = 1; w < POLY_WAVES; w++) acc_sum += p[w * (CH * POLY_TN * BS)];
#ifdef POLY_EP_MID_VALUE
      *POLY_EP_MID_PTR(m, n, z) = POLY_EP_MID_VALUE(acc_sum, m, n, z);
#endif
      POLY_EPILOGUE(acc_sum, m, n, z);
    }
  }
}
