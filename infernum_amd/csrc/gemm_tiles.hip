// C[M, N] = X[M, K] * W[N, K]^T in bf16 with fp32 accumulation for a prompt's rows, or with the activation,
// C[M, N / 2] = silu(X W_first^T) * (X W_second^T), on v_mfma_f32_16x16x32_bf16 with both operands through LDS.
//
// A workgroup of 2 x 2 waves, one on each SIMD, owns a BM x BN tile of C.  A wave owns BM / 2 x BN / 2 of it as four quadrants:
// its rows of X come in two halves (TX0 and TX1 tiles of 16), its rows of W in two (TW0 and TW1).  K is walked in steps of 64;
// LDS holds two steps (128 KB for the largest tile), and a step's half-tiles are read, and fetched again for the step
// after next, one by one:
//
//   phase  products   read from LDS meanwhile      fetched meanwhile, straight into LDS
//     1    X0 W0      W1 of this step              X0 of the step after next
//     2    X0 W1      X1 of this step              W0 of the step after next
//            barrier: X0 and W0 of the next step have come, W1 and X1 of this one are in registers
//     3    X1 W1      X0 of the next step          W1 of the step after next
//     4    X1 W0      W0 of the next step          X1 of the step after next
//            barrier: W1 and X1 of the next step have come, X0 and W0 of it are in registers
//
// A half-tile's memory is free once its values are in registers, a whole step before its products are done, so that loads
// have a step and a half (3,400 cycles with the largest tile, 2 us) to come, and a wave meets a barrier every 64 matrix
// instructions.
//
// What bounds it: the matrix cores, and the clock that the chip's power leaves them (1.6 to 1.75 GHz with random operands, 2.4
// with zeros).  At 4,096 x 4,096 a step of the 256 x 256 tile takes 2,256 cycles where its matrix instructions need 2,048: a load into
// LDS costs a wave some 10 cycles of issue, an LDS read 3, a barrier 12.  What made the difference, in cycles a step:
// 64 values a row and load in place of 32 (2,430: requests of half a line fill L2's request rate), matrix instructions of 16 x 16 x 32 in
// place of 32 x 32 x 16 (the same cycles, 5 to 10 % more clock for the power), a barrier for two phases in place of one (2,384), one value
// of m0 for all loads of a half-tile (2,314).  Whole products, M x N x K, us (library / this; of 4,096 x 4,096 x 4,096 1.42 PFLOP/s):
//   2,048 x 28,672 x 4,096 374 / 371   2,048 x 4,096 x 14,336 199 / 184   1,934 x 9,472 x 4,096 253 / 110   2,003 x 9,216 x 2,048 85 / 70
//   4,096 x 4,096 x 4,096 95 / 97      8,192 x 28,672 x 4,096 1,276 / 1,312 (with the activation 1,428, a launch of its own / 1,271)
//
// Both matrices have K contiguous.  Lane (r, q) = (lane % 16, lane / 16) of an operand holds the 8 values k = 32 s + 8 q .. + 7 of
// row r, one 16-byte LDS read.  A load instruction of a wave fills 1,024 consecutive bytes of LDS, lane by lane: 8 rows of 128
// bytes without padding.  The 16-byte piece c of row r lies at position c ^ (r % 8), so that the reads of 8 neighbouring rows fall on
// different banks: the lane that fills position p of row r fetches piece p ^ (r % 8).
//
// The sums run over K in its order whatever the tile: a row's result depends neither on the rows beside it nor on
// their number.  K must be a multiple of 64, M and N are arbitrary (rows beyond them are read from the last valid row and not stored).
//
// The matrix instructions are written in assembly with the accumulators tied: given as builtins, the compiler keeps the four quadrants'
// accumulators moving between registers (650 moves a step, a third of the speed).  The assembler's hazards are then this file's to
// keep: operands come from LDS reads, for which the compiler waits, and from nothing else (no vector instruction writes one: tests
// read the loop's assembly for moves), and the accumulators are written before and read after with a wait between.
#include "common.h"
#include <cmath>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

#define GT_BK 64
#define GT_ROW 128                       // bytes of a row of a step
#define GT_LDS (160 * 1024)
#define GT_TWO_COST 500                  // of a second launch, in units of 10 ns
#define GT_TWO_PAYS 30                   // two launches where they are estimated to save one part in so many

#if defined(__HIP_DEVICE_COMPILE__)
typedef __attribute__((address_space(3))) void* gt_lds_ptr;
#define GT_BUFFER(p, bytes) __builtin_amdgcn_make_buffer_rsrc((void*)(p), 0, (int)(bytes), 0x00020000)
#define GT_FETCH_AT(rsrc, lds, at, step, imm) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (gt_lds_ptr)(lds), 16, at, step, imm, 0)
#else
#define GT_BUFFER(p, bytes) 0
#define GT_FETCH_AT(rsrc, lds, at, step, imm) (void)0
#endif
// Load f of a half-tile: the instruction's immediate moves the place in LDS and the place in memory alike, so `at` counts 1,024 f bytes
// less, and the buffers begin GT_AHEAD bytes in front of the matrices so that it stays positive.
#define GT_AHEAD 3072u
#define GT_FETCH(rsrc, lds, at, step, f)                            \
  do {                                                              \
    if ((f) == 0) GT_FETCH_AT(rsrc, lds, at, step, 0);              \
    else if ((f) == 1) GT_FETCH_AT(rsrc, lds, at, step, 1024);      \
    else if ((f) == 2) GT_FETCH_AT(rsrc, lds, at, step, 2048);      \
    else GT_FETCH_AT(rsrc, lds, at, step, 3072);                    \
  } while (0)

enum { GT_PLAIN, GT_GLU, GT_GROUPED };

template <int TX0, int TX1, int TW0, int TW1, int MODE>
struct GemmTile {
  static constexpr bool GLU = MODE == GT_GLU;
  static constexpr int BM = 32 * (TX0 + TX1), BN = 32 * (TW0 + TW1);      // rows of X and of W
  static constexpr int COLS = GLU ? BN / 2 : BN;                          // columns of the result
  static constexpr int STAGE = (BM + BN) * GT_ROW;
  static constexpr int OUT_ROW = COLS / 2 * 2 + 16;                       // a wave's row of the result in LDS, with 16 bytes of padding
  static constexpr int OUT = 4 * (BM / 2) * OUT_ROW;
  static constexpr int LDS = 2 * STAGE > OUT ? 2 * STAGE : OUT;
  static_assert(LDS <= GT_LDS && TX0 <= 4 && TX1 <= 4 && TW0 <= 4 && TW1 <= 4 && TX0 >= TX1 && TW0 >= TW1, "the tile's shape");
  static_assert(!GLU || TW0 == TW1, "the halves of W meet in a wave");
};

// One value of the accumulators: D = A B + D, all of D in accumulation registers.
#define GT_MFMA(d, a, b) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(d) : "v"(a), "v"(b))

// Wait until at most n loads are under way and the LDS reads are through, then a bare barrier (__syncthreads() would wait
// for every load).
#define GT_BARRIER(n)                                                   \
  do {                                                                  \
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(n) : "memory"); \
    __builtin_amdgcn_s_barrier();                                       \
    asm volatile("" ::: "memory");                                      \
    __builtin_amdgcn_sched_barrier(0);                                  \
  } while (0)

// The products of wr [TW] and xr [TX] (two slices of 32 of K) into acc, with READS LDS reads (half of the way through) and
// FETCHES loads between them, in the order as written: nothing moves across a sched_barrier.  The first matrix instruction
// stands in front of the first read, so that the wait for its operands does not wait for that read.
#define GT_PHASE(acc, TW, TX, wr, xr, READS, READ, FETCHES, FETCH)                                             \
  _Pragma("unroll") for (int g = 0; g < (TW) * (TX) * 2; ++g) {                                                \
    constexpr int MF = (TW) * (TX) * 2;                                                                        \
    const int ks = g / ((TW) * (TX)), ti = (g % ((TW) * (TX))) / (TX), tj = g % (TX);                          \
    GT_MFMA(acc[ti][tj], wr[ti][ks], xr[tj][ks]);                                                              \
    __builtin_amdgcn_sched_barrier(0);                                                                         \
    _Pragma("unroll") for (int i = 0; i < (READS); ++i) if ((i * MF) / (2 * (READS)) == g) { READ(i); }        \
    _Pragma("unroll") for (int f = (g * (FETCHES)) / MF; f < ((g + 1) * (FETCHES)) / MF; ++f) { FETCH(f); }    \
    __builtin_amdgcn_sched_barrier(0);                                                                         \
  }

template <int TX0, int TX1, int TW0, int TW1, int MODE>
__global__ __launch_bounds__(256, 1) void gemm_tiles_kernel(const uint16_t* __restrict__ X, const uint16_t* __restrict__ W,
                                                            uint16_t* __restrict__ C, int M, int N, int K, int tiles_m, int tiles_n,
                                                            int n_first, const int* __restrict__ rows_at, int groups) {
  using T = GemmTile<TX0, TX1, TW0, TW1, MODE>;
  constexpr bool GLU = T::GLU, GROUPED = MODE == GT_GROUPED;
  constexpr int BM = T::BM, BN = T::BN, WM = BM / 2, WN = BN / 2, STAGE = T::STAGE;
  constexpr int RX0 = 0, RX1 = 32 * TX0, RW0 = BM, RW1 = BM + 32 * TW0;       // a step's half-tiles, in rows of its stage
  constexpr int ALL = TX0 + TX1 + TW0 + TW1;                                  // a wave's loads a step
  extern __shared__ __attribute__((aligned(1024))) char lds[];

  // workgroups go to the 8 dies in turn (workgroup i to die i % 8), and each die has an L2 of its own: every die gets one
  // contiguous run of tiles, four tiles of M under one tile of N at a time
  if constexpr (GROUPED) {
    // the tiles of rows that the groups have in this step (the launch has one for every case): the dies share those evenly,
    // and the workgroups beyond them leave
    tiles_m = 0;
    for (int g = 0; g < groups; ++g) tiles_m += (rows_at[g + 1] - rows_at[g] + BM - 1) / BM;
  }
  const int total = tiles_m * tiles_n, xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
  if (GROUPED && idx >= (total >> 3) + (xcd < (total & 7) ? 1 : 0)) return;
  const int bid = xcd * (total >> 3) + min(xcd, total & 7) + idx;
  constexpr int GROUP = 4;
  const int group = bid / (GROUP * tiles_n), in_group = bid - group * (GROUP * tiles_n);
  const int group_rows = min(GROUP, tiles_m - group * GROUP);
  const int tm = group * GROUP + in_group % group_rows, tn = in_group / group_rows;
  const int m0 = GROUPED ? 0 : tm * BM;
  const int NO = GLU ? N / 2 : N, n0 = n_first + tn * T::COLS;                // columns of the result

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1, r16 = lane & 15, q4 = lane >> 4;

  // GROUPED: the tile's group, its first row among the sorted ones; from here on M is what the group has from there on
  int rot = 0;
  if constexpr (GROUPED) {
    int g = 0, seen = 0;
    for (; g < groups - 1; ++g) {
      const int t = (rows_at[g + 1] - rows_at[g] + BM - 1) / BM;
      if (tm < seen + t) break;
      seen += t;
    }
    const int first = rows_at[g] + (tm - seen) * BM;
    M = rows_at[g + 1] - first;
    W += ((size_t)g * N + n0) * K;
    X += (size_t)first * K;
    C += (size_t)first * N;
    static_assert(!GROUPED || 512 % BN == 0, "a tile lies in the columns that share a start");
    rot = ia_expert_first_chunk(n0, K) * (IA_EXPERT_CHUNK / GT_BK);
  }

  // ---- loads: load f of a half-tile of 32 T rows fills its rows 8 (T wave + f) .. + 7, this lane position lane % 8 of row
  // lane / 8 of them.  The half-tile's first 16 T rows belong to the waves with wm (wn) 0, the others to those with 1.
  const int x_rows = GROUPED ? min(M, BM) : M, w_rows = GROUPED ? min(N - n0, BN) : N;
  const auto x_all = GT_BUFFER(reinterpret_cast<const char*>(X) - GT_AHEAD, (unsigned)x_rows * (unsigned)K * 2u + GT_AHEAD);
  const auto w_all = GT_BUFFER(reinterpret_cast<const char*>(W) - GT_AHEAD, (unsigned)w_rows * (unsigned)K * 2u + GT_AHEAD);
  auto place = [&](int t, int f, int from, int apart, int rows, int behind) {
    const int row = 8 * (t * wave + f) + (lane >> 3), of = row / (16 * t), in = row - of * (16 * t);
    const uint32_t r = (uint32_t)(min(from + of * apart + in, rows - 1) + behind);
    return GT_AHEAD - 1024u * (uint32_t)f + (r * (uint32_t)K + (uint32_t)(((lane & 7) ^ (row & 7)) * 8)) * 2u;
  };
  uint32_t sx0[TX0], sx1[TX1], sw0[TW0], sw1[TW1];
#pragma unroll
  for (int f = 0; f < TX0; ++f) sx0[f] = place(TX0, f, m0, WM, M, 0);
#pragma unroll
  for (int f = 0; f < TX1; ++f) sx1[f] = place(TX1, f, m0 + 16 * TX0, WM, M, 0);
  // GLU: the first half of a wave's rows of W is of the first half of the matrix, the second of the second, for the same columns
#pragma unroll
  for (int f = 0; f < TW0; ++f) sw0[f] = place(TW0, f, GROUPED ? 0 : n0, GLU ? WN / 2 : WN, GROUPED ? w_rows : NO, 0);
#pragma unroll
  for (int f = 0; f < TW1; ++f)
    sw1[f] = GLU ? place(TW1, f, n0, WN / 2, NO, NO)
                 : place(TW1, f, (GROUPED ? 0 : n0) + 16 * TW0, WN, GROUPED ? w_rows : NO, 0);
  const int steps = K / GT_BK;
  // past the end the last step is fetched again, into memory that is not read any more; GROUPED: the walk begins at step
  // rot and wraps around
  auto step_at = [&](int t) {
    const int k = min(t, steps - 1) + rot;
    return (GROUPED && k >= steps ? k - steps : k) * GT_ROW;
  };
#define GT_X0(t, f) GT_FETCH(x_all, lds + ((t) & 1) * STAGE + RX0 * GT_ROW + 1024 * (TX0 * wave), sx0[f], step_at(t), f)
#define GT_X1(t, f) GT_FETCH(x_all, lds + ((t) & 1) * STAGE + RX1 * GT_ROW + 1024 * (TX1 * wave), sx1[f], step_at(t), f)
#define GT_W0(t, f) GT_FETCH(w_all, lds + ((t) & 1) * STAGE + RW0 * GT_ROW + 1024 * (TW0 * wave), sw0[f], step_at(t), f)
#define GT_W1(t, f) GT_FETCH(w_all, lds + ((t) & 1) * STAGE + RW1 * GT_ROW + 1024 * (TW1 * wave), sw1[f], step_at(t), f)

  // ---- accumulators of the quadrants, W the first operand: register e of lane (r, q) of tile [i][j] is the product for
  // n = 16 i + 4 q + e and m = 16 j + r, four neighbours in a row of C
  f32x4 a00[TW0][TX0], a10[TW1][TX0], a11[TW1][TX1], a01[TW0][TX1];           // [half of W][half of X]
#define GT_ZERO(a, I, J)                                        \
  _Pragma("unroll") for (int i = 0; i < I; ++i)                 \
  _Pragma("unroll") for (int j = 0; j < J; ++j) {               \
    a[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};                      \
    asm volatile("" : "+a"(a[i][j]));                           \
  }
  GT_ZERO(a00, TW0, TX0) GT_ZERO(a10, TW1, TX0) GT_ZERO(a11, TW1, TX1) GT_ZERO(a01, TW0, TX1)
  asm volatile("s_nop 7" ::: "memory");

  bf16x8 x0[TX0][2], x1[TX1][2], wa[TW0][2], wb[TW0][2];
  const int piece[2] = {(q4 ^ (r16 & 7)) * 16, ((4 + q4) ^ (r16 & 7)) * 16};
  const int ox0 = (RX0 + wm * 16 * TX0 + r16) * GT_ROW, ox1 = (RX1 + wm * 16 * TX1 + r16) * GT_ROW;
  const int ow0 = (RW0 + wn * 16 * TW0 + r16) * GT_ROW, ow1 = (RW1 + wn * 16 * TW1 + r16) * GT_ROW;
#define GT_READ(dst, first, t, i) \
  dst[(i) >> 1][(i) & 1] = *reinterpret_cast<const bf16x8*>(lds + ((t) & 1) * STAGE + first + ((i) >> 1) * (16 * GT_ROW) + piece[(i) & 1])

  // two steps under way, X0 and W0 of the first in registers
#pragma unroll
  for (int f = 0; f < TX0; ++f) GT_X0(0, f);
#pragma unroll
  for (int f = 0; f < TW0; ++f) GT_W0(0, f);
#pragma unroll
  for (int f = 0; f < TW1; ++f) GT_W1(0, f);
#pragma unroll
  for (int f = 0; f < TX1; ++f) GT_X1(0, f);
#pragma unroll
  for (int f = 0; f < TX0; ++f) GT_X0(1, f);
#pragma unroll
  for (int f = 0; f < TW0; ++f) GT_W0(1, f);
#pragma unroll
  for (int f = 0; f < TW1; ++f) GT_W1(1, f);
#pragma unroll
  for (int f = 0; f < TX1; ++f) GT_X1(1, f);
  GT_BARRIER(TW1 + TX1 + ALL);
#pragma unroll
  for (int i = 0; i < 2 * TX0; ++i) GT_READ(x0, ox0, 0, i);
#pragma unroll
  for (int i = 0; i < 2 * TW0; ++i) GT_READ(wa, ow0, 0, i);
  GT_BARRIER(ALL);

  // w0 holds W0 of step t, and leaves with W1's place taken by W0 of step t + 1
  auto step = [&](int t, bf16x8 (&w0)[TW0][2], bf16x8 (&w1)[TW0][2]) {
#define GT_READ1(i) GT_READ(w1, ow1, t, i)
#define GT_FETCH1(f) GT_X0(t + 2, f)
    GT_PHASE(a00, TW0, TX0, w0, x0, 2 * TW1, GT_READ1, TX0, GT_FETCH1)
#define GT_READ2(i) GT_READ(x1, ox1, t, i)
#define GT_FETCH2(f) GT_W0(t + 2, f)
    GT_PHASE(a10, TW1, TX0, w1, x0, 2 * TX1, GT_READ2, TW0, GT_FETCH2)
    GT_BARRIER(ALL);
#define GT_READ3(i) GT_READ(x0, ox0, t + 1, i)
#define GT_FETCH3(f) GT_W1(t + 2, f)
    GT_PHASE(a11, TW1, TX1, w1, x1, 2 * TX0, GT_READ3, TW1, GT_FETCH3)
#define GT_READ4(i) GT_READ(w1, ow0, t + 1, i)
#define GT_FETCH4(f) GT_X1(t + 2, f)
    GT_PHASE(a01, TW0, TX1, w0, x1, 2 * TW0, GT_READ4, TX1, GT_FETCH4)
    GT_BARRIER(ALL);
  };
  int t = 0;
  for (; t + 1 < steps; t += 2) {
    step(t, wa, wb);
    step(t + 1, wb, wa);
  }
  if (t < steps) step(t, wa, wb);
  // the loads asked for past the end write LDS too; and the last products are through before an accumulator is read
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#define GT_KEEP(a, I, J)                        \
  _Pragma("unroll") for (int i = 0; i < I; ++i) \
  _Pragma("unroll") for (int j = 0; j < J; ++j) asm volatile("" : "+a"(a[i][j]));
  GT_KEEP(a00, TW0, TX0) GT_KEEP(a10, TW1, TX0) GT_KEEP(a11, TW1, TX1) GT_KEEP(a01, TW0, TX1)

  // ---- C through LDS, a region of its own for every wave, so that rows leave as consecutive 16-byte pieces
  char* const region = lds + wave * (WM * T::OUT_ROW);
  const bool vec8 = (NO & 7) == 0;
  auto put = [&](int i, int j, const float (&v)[4]) {
    uint2 o;
    o.x = two_bf16_bits(v[0], v[1]);
    o.y = two_bf16_bits(v[2], v[3]);
    *reinterpret_cast<uint2*>(region + (j * 16 + r16) * T::OUT_ROW + (i * 16 + 4 * q4) * 2) = o;
  };
  if constexpr (GLU) {
    // silu(g) u with the hardware's exponential and reciprocal (a unit in the last place each; what is kept has 8 bits), on a quarter
    // of 1 + exp(-g): the reciprocal takes a result below the smallest normal number for 0, which the sigmoid's is from -87.4 down.
    auto pair = [&](int i, int j, const f32x4& gate, const f32x4& up) {
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[e] = 0.25f * gate[e] * __builtin_amdgcn_rcpf(0.25f + __builtin_amdgcn_exp2f(fmaf(-1.4426950408889634f, gate[e], -2.0f))) * up[e];
      put(i, j, v);
    };
#pragma unroll
    for (int i = 0; i < TW0; ++i) {
#pragma unroll
      for (int j = 0; j < TX0; ++j) pair(i, j, a00[i][j], a10[i][j]);
#pragma unroll
      for (int j = 0; j < TX1; ++j) pair(i, TX0 + j, a01[i][j], a11[i][j]);
    }
  } else {
    auto one = [&](int i, int j, const f32x4& a) {
      const float v[4] = {a[0], a[1], a[2], a[3]};
      put(i, j, v);
    };
#define GT_LEAVE(a, I, J, i0, j0)               \
  _Pragma("unroll") for (int i = 0; i < I; ++i) \
  _Pragma("unroll") for (int j = 0; j < J; ++j) one(i0 + i, j0 + j, a[i][j]);
    GT_LEAVE(a00, TW0, TX0, 0, 0) GT_LEAVE(a10, TW1, TX0, TW0, 0) GT_LEAVE(a11, TW1, TX1, TW0, TX0) GT_LEAVE(a01, TW0, TX1, 0, TX0)
  }
  // a wave reads back what it wrote itself: no barrier, only the wait for its LDS writes
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  constexpr int WCOLS = T::COLS / 2, PIECES = WCOLS / 8;                      // a wave's columns; 16-byte pieces of its rows
  const int c0 = n0 + wn * WCOLS;
  for (int p = lane; p < WM * PIECES; p += 64) {
    const int row = p / PIECES, c = p - row * PIECES, m = m0 + wm * WM + row, n = c0 + c * 8;
    if (m >= M || n >= NO) continue;
    const uint4 v = *reinterpret_cast<const uint4*>(region + row * T::OUT_ROW + c * 16);
    uint16_t* const dst = C + (size_t)m * NO + n;
    if (vec8) {
      *reinterpret_cast<uint4*>(dst) = v;
    } else {
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (n + e < NO) dst[e] = (uint16_t)(w[e >> 1] >> (16 * (e & 1)));
    }
  }
}

template <int TX0, int TX1, int TW0, int TW1, int MODE>
static int launch_gemm_tiles(const uint16_t* x, const uint16_t* w, uint16_t* c, int M, int N, int K, int n_first, int n_end,
                             const int* rows_at, int groups, hipStream_t stream) {
  using T = GemmTile<TX0, TX1, TW0, TW1, MODE>;
  static bool configured = false;
  if (!configured) {
    const hipError_t e = hipFuncSetAttribute((const void*)gemm_tiles_kernel<TX0, TX1, TW0, TW1, MODE>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, T::LDS);
    if (e != hipSuccess) return (int)e;
    configured = true;
  }
  // grouped: a tile for every way the rows can fall into groups
  const int tiles_m = MODE == GT_GROUPED ? M / T::BM + (M < groups ? M : groups) : (M + T::BM - 1) / T::BM;
  const int tiles_n = (n_end - n_first + T::COLS - 1) / T::COLS;
  if ((long long)tiles_m * tiles_n > 0x7fffffffLL) return IA_ERR_UNSUPPORTED;
  gemm_tiles_kernel<TX0, TX1, TW0, TW1, MODE><<<tiles_m * tiles_n, 256, T::LDS, stream>>>(x, w, c, M, N, K, tiles_m, tiles_n, n_first, rows_at, groups);
  IA_LAUNCH_CHECK();
  return IA_OK;
}

// The tiles: rows of X and of W, and as template arguments.
#define GT_TILES(F)                                                                                                            \
  F(256, 256, 4, 4, 4, 4) F(256, 224, 4, 4, 4, 3) F(256, 192, 4, 4, 3, 3) F(256, 160, 4, 4, 3, 2) F(256, 128, 4, 4, 2, 2)      \
  F(224, 256, 4, 3, 4, 4) F(192, 256, 3, 3, 4, 4) F(192, 192, 3, 3, 3, 3) F(192, 128, 3, 3, 2, 2) F(160, 256, 3, 2, 4, 4)      \
  F(160, 192, 3, 2, 3, 3) F(160, 128, 3, 2, 2, 2) F(128, 256, 2, 2, 4, 4) F(128, 192, 2, 2, 3, 3) F(128, 128, 2, 2, 2, 2)

static bool gemm_tiles_takes(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0 || K % GT_BK != 0) return false;
  // rows are addressed with 32 bits, with GT_AHEAD bytes in front of them
  return (unsigned long long)M * K * 2 <= 0xffffffffULL - GT_AHEAD && (unsigned long long)N * K * 2 <= 0xffffffffULL - GT_AHEAD;
}

// Which tile: the one with the least estimated time, in units of 10 ns.  A workgroup of a BM x BN tile takes K / 64 steps of
// 0.615 us a 256 x 256 tile's products and 0.56 us the loads of its BM + BN rows, and 10 us times the square root of its area around them
// (the first loads, C); the launch takes as many turns as the tiles need with one workgroup a compute unit.  Tiles of at most 192 x 128
// leave room for two, which together take 0.95 of two one after the other.  The constants are a fit to 80 products of 160 to 8,192 rows of
// 768 to 28,672 columns, K of 768 to 14,336, with all fifteen tiles each: what it picks takes 1.2 % longer than the fastest on average.  They date from when a
// value's rounding took ten instructions: since it takes one, the estimate is 17 % above what is measured below 80 us, 10 % up to 200 and right
// beyond, for all tiles alike.  So the picks are as good: of 144 other products 0.8 % longer than the fastest, 0.7 with the constants
// fitted to these anew.
static long tile_cost(int M, int NO, int K, int bm, int bn, int cols) {
  const long tiles = (long)((M + bm - 1) / bm) * ((NO + cols - 1) / cols), steps = K / GT_BK;
  const long one = steps * (62L * bm * bn / 65536 + 56L * (bm + bn) / 512);
  const long around = bm * bn >= 65536 ? 1030 : bm * bn >= 57344 ? 960 : bm * bn >= 49152 ? 890 : bm * bn >= 40960 ? 810
                      : bm * bn >= 36864 ? 770 : bm * bn >= 30720 ? 700 : bm * bn >= 24576 ? 630 : bm * bn >= 20480 ? 570 : 510;
  if (bm * bn > 192 * 128 || (bm + bn) * 256 > GT_LDS / 2) return (tiles + 255) / 256 * (around + one);
  const long pair = around * 13 / 10 + one * 19 / 10, rest = tiles % 512;
  return tiles / 512 * pair + (rest > 256 ? pair : rest > 0 ? around + one : 0);
}

// A product's tiles; with two, the first `split` columns of the result in one and the others in the other.
struct TileChoice {
  int rows, cols, split, rows2, cols2;
};

// Large tiles fill turns of the compute units and leave a part of one.  Where that is estimated to cost more than a second launch does
// and one part in GT_TWO_PAYS of the product, the columns of the whole turns take them, and the others, in a launch of their own, smaller
// tiles.  One tile / two, us, M x rows of W x K, with the activation: 2,048 x 28,672 x 4,096 (3.5 turns of 256 x 256) 371 / 340, 7,680 rows
// (13.1 turns) 1,258 / 1,223, 1,000 rows (1.8) 180 / 169, 2,925 x 11,008 x 2,048 114 / 108; plain: 4,054 x 25,664 x 4,096 627 / 593.  Of 432 products
// of 160 to 8,192 rows it takes 13 in 100, 4.9 % faster on average.  The second launch counts 5 us although it takes some 3: below 80 us,
// where the estimate is high, it is as often wrong (1,755 x 10,304 x 2,048 61 / 66, 1,776 x 11,008 x 2,048 71 / 67).  Of the 144 products above
// it takes 5: 1,559 x 22,234 x 3,904 241 / 222, 4,027 x 26,220 x 2,496 465 / 456, three within 2 % (counted 4 us, as many).
static TileChoice choose_tiles(int M, int N, int K, bool glu) {
  const int NO = glu ? N / 2 : N;
  const auto best = [&](int columns, int& rows, int& cols) {
    long least = -1;
#define GT_COST(BM, BN, TX0, TX1, TW0, TW1)                                                                  \
    if (!glu || TW0 == TW1) {                                                                                \
      const long cost = tile_cost(M, columns, K, BM, BN, glu ? BN / 2 : BN);                                 \
      if (least < 0 || cost < least) { least = cost; rows = BM; cols = BN; }                                 \
    }
    GT_TILES(GT_COST)
#undef GT_COST
    return least;
  };
  TileChoice one{0, 0, 0, 0, 0};
  const long alone = best(NO, one.rows, one.cols);
  long least = alone - alone / GT_TWO_PAYS;
#define GT_COST(BM, BN, TX0, TX1, TW0, TW1)                                                                  \
  if ((!glu || TW0 == TW1) && BM * BN >= 192 * 256) {                                                        \
    const int wide = glu ? BN / 2 : BN, down = (M + BM - 1) / BM;                                            \
    const int split = (int)((long)down * (NO / wide) / 256 * 256 / down) * wide;                             \
    if (split > 0 && split < NO) {                                                                           \
      TileChoice two{BM, BN, split, 0, 0};                                                                   \
      const long cost = tile_cost(M, split, K, BM, BN, wide) + GT_TWO_COST + best(NO - split, two.rows2, two.cols2); \
      if (cost < least) { least = cost; one = two; }                                                         \
    }                                                                                                        \
  }
  GT_TILES(GT_COST)
#undef GT_COST
  return one;
}

// Whether this kernel or the vendor library's takes a whole product of many rows (with the activation there is a rule of its own where the
// routes are planned: 260 products of 129 to 8,192 rows 1.16 times as fast as the library's with a launch for the activation, up to half as fast
// where few tiles walk a long K).  The library's large tile runs
// 5 to 10 % faster than this kernel's (8,192 x 4,096 x 4,096 184 / 205 us, 4,096 x 4,096 x 14,336 313 / 325), so where tiles of 256 x 256
// fill their turns of the compute units it is ahead, and for few tiles it splits K (512 x 4,096 x 14,336 85 / 110, 1,000 x 2,048 x 5,504
// 40 / 50).  Between them, where such tiles leave a fifth of their turns empty and tiles of 128 x 128 occupy 200 units,
// the choice of a tile gains: 2,048 x 4,096 x 14,336 208 / 184, 1,500 x 6,144 x 4,096 77 / 66, 2,300 x 2,048 x 8,192 86 / 74.  With short
// K and more than half a turn of large tiles the library is ahead again (5,700 x 2,048 x 2,048 43 / 48, 3,737 x 3,072 x 2,048 43 / 46); with
// long K and more than a turn it has kernels that take half as long again as their neighbours (4,096 columns, K = 14,336 at
// 4,600 / 5,700 / 6,600 / 7,650 rows 765 / 764 / 847 / 966 us, this one 415 / 515 / 579 / 651), from K = 10,240 on more often than not (with K of
// 8,192 it is ahead, 10,240 columns and 4,600 rows 494 / 548, 9,472 and 3,000 325 / 352, or behind, 9,472 and 4,096 655 / 462).  Over 403 products
// of 400 to 8,192 rows this rule's picks take 0.92 of the library's time, 12 of them more than 3 % longer, at most 11 %.
extern "C" int ia_gemm_tiles_pays(int M, int N, int K) {
  if (!gemm_tiles_takes(M, N, K)) return 0;
  const long large = (long)((M + 255) / 256) * ((N + 255) / 256), small = (long)((M + 127) / 128) * ((N + 127) / 128);
  const long places = (large + 255) / 256 * 256;                          // in the turns that the large tiles need
  if (small < 200 || K < 2048 || (K < 4096 && large > 140)) return 0;
  return places * 100 >= large * (K >= 10240 && large > 256 ? 106 : 120);
}

// Columns of the result that the first of a product's two launches takes (0: it is one launch).
extern "C" int ia_gemm_tiles_split(int M, int N, int K, int glu) {
  return gemm_tiles_takes(M, N, K) && !(glu && (N & 1)) ? choose_tiles(M, N, K, glu != 0).split : 0;
}

// Columns n_first to n_end - 1 of the result.
static int gemm_tiles_columns(const uint16_t* x, const uint16_t* w, uint16_t* c, int M, int N, int K, int glu, int rows, int cols,
                              int n_first, int n_end, hipStream_t stream) {
#define GT_ONE(BM, BN, TX0, TX1, TW0, TW1)                                                                                            \
  if (rows == BM && cols == BN) {                                                                                                     \
    if (!glu) return launch_gemm_tiles<TX0, TX1, TW0, TW1, GT_PLAIN>(x, w, c, M, N, K, n_first, n_end, nullptr, 0, stream);            \
    if constexpr (TW0 == TW1) return launch_gemm_tiles<TX0, TX1, TW0, TW1, GT_GLU>(x, w, c, M, N, K, n_first, n_end, nullptr, 0, stream); \
  }
  GT_TILES(GT_ONE)
#undef GT_ONE
  return IA_ERR_BAD_ARG;
}

// X [M, K], W [N, K], C [M, N] (glu: [M, N / 2], N even), bf16, contiguous, on 16 bytes.  rows, cols: the tile; 0: chosen here; rows < 0:
// the same, where ia_gemm_tiles_pays (else IA_ERR_UNSUPPORTED).
extern "C" int ia_gemm_tiles(const void* X, const void* W, void* C, int M, int N, int K, int glu, int rows, int cols, hipStream_t stream) {
  if (!X || !W || !C || (glu && (N & 1))) return IA_ERR_BAD_ARG;
  if (!gemm_tiles_takes(M, N, K)) return IA_ERR_UNSUPPORTED;
  if (((uintptr_t)X | (uintptr_t)W | (uintptr_t)C) & 15) return IA_ERR_UNSUPPORTED;
  if (rows < 0 && !glu && !ia_gemm_tiles_pays(M, N, K)) return IA_ERR_UNSUPPORTED;
  const uint16_t *x = (const uint16_t*)X, *w = (const uint16_t*)W;
  uint16_t* c = (uint16_t*)C;
  const int NO = glu ? N / 2 : N;
  if (rows > 0) return gemm_tiles_columns(x, w, c, M, N, K, glu, rows, cols, 0, NO, stream);
  const TileChoice t = choose_tiles(M, N, K, glu != 0);
  const int rc = gemm_tiles_columns(x, w, c, M, N, K, glu, t.rows, t.cols, 0, t.split > 0 ? t.split : NO, stream);
  return rc == IA_OK && t.split > 0 ? gemm_tiles_columns(x, w, c, M, N, K, glu, t.rows2, t.cols2, t.split, NO, stream) : rc;
}

// ---- rows in groups, each with a matrix of its own: the routed experts' products of many tokens ----
// Rows rows_at[g] .. rows_at[g + 1] - 1 of X (sorted by group) times matrix g of W [groups, N, K]; rows_at [groups + 1] lies on the device
// and nothing is read back: the launch has a workgroup for every way the rows can fall into groups, and those to spare leave.  The walk
// over K starts where the tiles of few pairs do (ia_expert_first_chunk) and wraps: the same bits from either.  among: how many groups the
// rows are spread over, with those that have no matrix and lie behind the others (the choice of a tile goes by it).
//
// What bounds it: between the stream of the experts' weights and the matrix cores, and the turns of the compute units that tiles fill in
// part.  First / second products, us, with the tiles of 128 x 256 of 32 x 32 x 16 instructions before and now:
//   20 experts of 2,432 x 4,096, 161 rows each 243 -> 219 / 140 -> 111   32 of 1,408 x 2,048, 255 rows 165 -> 136 / 97 -> 73
//   16 of 1,408 x 2,048, 256 rows 79 -> 71 / 53 -> 33                    8 of 2,752 x 2,048 without a gate, 500 rows 66 -> 61 / 81 -> 52

// The tiles: rows of X and of W, and as template arguments.
#define GT_GROUP_TILES(G)                                                                                                    \
  G(96, 128, 2, 1, 2, 2) G(128, 128, 2, 2, 2, 2) G(160, 128, 3, 2, 2, 2) G(192, 128, 3, 3, 2, 2) G(128, 256, 2, 2, 4, 4)     \
  G(192, 256, 3, 3, 4, 4) G(256, 256, 4, 4, 4, 4)

// Which tile: the one with the least estimated time, in us.  A workgroup takes K / 64 steps of 0.61 a 256 x 256 tile's products, 0.43 the
// loads of its bm + bn rows and 0.1 besides, and 15.6 times the square root of its area around them; two that share a compute unit take
// 2.03 of their steps and 0.74 of the rest.  A few tiles beyond a turn of the compute units are a whole turn more, and how many there will be
// is not known on the host: the estimate is the mean over groups whose sizes differ as those of a random choice do and by 0.3 of their
// mean beside that, each with as many tiles more and less as the groups' last ones scatter by.  Tiles that have a unit to themselves count 1.1
// times: a turn of theirs that was not expected costs the most, and they cost the chip its clock (192 x 256 and 256 x 256 3 and 4 % longer over 15 ms
// than over 12 launches; 8 groups of 404 rows of 2,752 x 2,048 and of 2,048 x 2,752 took 53 + 52 us with two of them and 59 + 59 with 160 x 128,
// yet the pass of 2.7 ms that they are in 0.6 % longer).
// The constants are a fit to 478 products of 4 to 128 groups of 49 to 1,024 rows on average (and those of the benchmark's designs, up to
// 2,048), 1,024 to 28,672 columns, K of 768 to 14,336, of sizes that differ in these two ways and by 0.6 of the mean, each of ten tiles for
// 15 ms: what it picks takes 3.9 % longer than the fastest (2 % if the sizes were known).  Against 96 x 128, 160 x 128 or 192 x 128 by the mean
// rows it takes 0.96 of the time, more than 3 % longer in 41 of them, at most 1.25 times (by the mean / now, N x K: 16 groups of 187 rows,
// 1,408 x 2,048 57 / 40 us; 8 of 175, 2,048 x 2,752 50 / 35; 16 of 187, 2,432 x 4,096 116 / 94; but 20 of 102, 4,096 x 2,432 100 / 118, 8 of 2,048,
// 2,752 x 2,048 181 / 221, three tiles beyond three turns).
static double grouped_strips(double mean, double spread, int bm) {           // of rows, a group: sum over k of how likely it has more than k
  const double sd = std::sqrt(mean + spread * spread * mean * mean);
  if (sd > bm) return mean / bm + 0.5;
  const double sure = std::floor((mean - 4.0 * sd) / bm);
  double strips = sure > 0.0 ? sure : 0.0;
  for (double k = strips; k * bm < mean + 4.0 * sd; k += 1.0) strips += 0.5 * std::erfc((k * bm + 0.5 - mean) / (1.4142135623730951 * sd));
  return strips;
}

static double grouped_cost(int groups, int mean, int N, int K, int bm, int bn) {
  const double area = (double)bm * bn / 65536, around = 15.6 * std::sqrt(area);
  const double walk = K / GT_BK * (0.613 * area + 0.431 * (bm + bn) / 512 + 0.104), one = around + walk;
  const bool shared = (bm + bn) * 256 <= GT_LDS / 2;
  const double pair = 0.736 * around + 2.03 * walk, cols = (N + bn - 1) / bn;
  const auto least = [](double a) { return a < 1.0 ? a : 1.0; };
  const auto time = [&](double tiles) {
    const double units = shared ? 512 : 256, turns = std::floor(tiles / units), rest = tiles - units * turns;
    if (!shared) return 1.1 * one * (tiles < 256 ? 1.0 : turns + (rest > 0.0 ? 0.87 + 0.13 * least(rest / 26) : 0.0));
    return turns * pair + (rest > 0.0 ? one : 0.0) + (rest > 256 ? (pair - one) * least((rest - 256) / 12) : 0.0);
  };
  double sum = 0.0;
  for (const double spread : {0.0, 0.3}) {
    const double tiles = grouped_strips(mean > 0 ? mean : 1, spread, bm) * groups * cols, more = cols * std::sqrt(groups * 0.125);
    sum += time(tiles - more > 1.0 ? tiles - more : 1.0) + time(tiles) + time(tiles + more);
  }
  return sum;
}

// The tile for a mean of `mean` rows a group: its rows * 1,024 + its columns.
extern "C" int ia_gemm_tiles_grouped_tile(int groups, int mean, int N, int K) {
  if (groups <= 0 || mean < 0 || N <= 0 || K <= 0) return 0;
  double best = -1.0;
  int tile = 0;
#define GT_GROUP_COST(BM, BN, ...)                                                  \
  {                                                                                 \
    const double cost = grouped_cost(groups, mean, N, K, BM, BN);                   \
    if (best < 0.0 || cost < best) { best = cost; tile = BM * 1024 + BN; }          \
  }
  GT_GROUP_TILES(GT_GROUP_COST)
#undef GT_GROUP_COST
  return tile;
}

extern "C" int ia_gemm_tiles_grouped(const void* X, const void* W, void* C, const int* rows_at, int groups, int among, int rows, int N, int K,
                                     hipStream_t stream) {
  if (groups <= 0 || among < groups || !rows_at) return IA_ERR_BAD_ARG;
  if (rows == 0) return IA_OK;
  if (rows < 0 || N <= 0 || K <= 0 || K % GT_BK != 0) return IA_ERR_UNSUPPORTED;
  // rows are addressed with 32 bits from the tile's first on, whose GT_AHEAD bytes in front are within reach of 256 rows
  if ((unsigned long long)rows * K * 2 > 0xffffffffULL || (unsigned long long)N * K * 2 > 0xffffffffULL) return IA_ERR_UNSUPPORTED;
  if (256ULL * K * 2 > 0xffffffffULL - GT_AHEAD) return IA_ERR_UNSUPPORTED;
  const uint16_t *x = (const uint16_t*)X, *w = (const uint16_t*)W;
  uint16_t* c = (uint16_t*)C;
  const int tile = ia_gemm_tiles_grouped_tile(groups, rows / among, N, K);
#define GT_GROUP_ONE(BM, BN, TX0, TX1, TW0, TW1) \
  if (tile == BM * 1024 + BN) return launch_gemm_tiles<TX0, TX1, TW0, TW1, GT_GROUPED>(x, w, c, rows, N, K, 0, N, rows_at, groups, stream);
  GT_GROUP_TILES(GT_GROUP_ONE)
#undef GT_GROUP_ONE
  return IA_ERR_BAD_ARG;
}

// ---- the launchers of this file as operations of a step's program (see op_call.h) ----
#include "op_call.h"
IA_OP(ia_gemm_tiles)
IA_OP(ia_gemm_tiles_grouped)
