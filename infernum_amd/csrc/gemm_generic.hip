// C[M, N] = A[M, K] * W[N, K]^T for any M, N, K, on the vector ALUs with fp32
// multiply-add only: the matrix product of the true 32-bit path, and the plain
// twin that the MFMA kernels are checked against.  fp32 operands whose rows can be
// read 16 bytes at a time go to the fp32 matrix instructions, further down: the
// same sums in the same order.
//
// Every output element is summed in one fixed order, whatever M, N and the tile
// it falls into: results do not depend on how many rows a step brings.  The order
// is in three levels, so that rounding grows with the square root of K / 256 and
// not of K: a chain of 16 fused multiply-adds from zero (one LDS stage), 16 such
// chains added up (256 values of k), and those sums added in the order of k.
#include "common.h"

#define GT 64   // tile of C: GT x GT
#define GK 16   // depth of one LDS stage

template <typename TA, typename TW, typename TC>
__global__ __launch_bounds__(256) void gemm_nt_kernel(const TA* __restrict__ A, const TW* __restrict__ W,
                                                      TC* __restrict__ C, int M, int N, int K, int lda, int ldw,
                                                      int ldc) {
  __shared__ float As[GK][GT + 4];
  __shared__ float Ws[GK][GT + 4];
  const int tid = threadIdx.x;
  const int tx = tid & 15, ty = tid >> 4;
  const int m0 = blockIdx.y * GT, n0 = blockIdx.x * GT;
  const int lr = tid >> 2;          // row of the tile this thread loads: 0..63
  const int lk = (tid & 3) * 4;     // first of its 4 consecutive k
  float acc[4][4], mid[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = mid[i][j] = 0.f;

  for (int k0 = 0; k0 < K; k0 += GK) {
    {
      const int m = m0 + lr, n = n0 + lr;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int k = k0 + lk + e;
        As[lk + e][lr] = (m < M && k < K) ? to_float(A[(size_t)m * lda + k]) : 0.f;
        Ws[lk + e][lr] = (n < N && k < K) ? to_float(W[(size_t)n * ldw + k]) : 0.f;
      }
    }
    __syncthreads();
    float part[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) part[i][j] = 0.f;
#pragma unroll
    for (int kk = 0; kk < GK; ++kk) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = As[kk][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = Ws[kk][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) part[i][j] = fmaf(a[i], b[j], part[i][j]);
    }
    const bool close = ((k0 / GK) & 15) == 15 || k0 + GK >= K;      // 256 values of k are in, or the last stage
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        mid[i][j] += part[i][j];
        if (close) {
          acc[i][j] += mid[i][j];
          mid[i][j] = 0.f;
        }
      }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + ty * 4 + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx * 4 + j;
      if (n < N) C[(size_t)m * ldc + n] = from_float<TC>(acc[i][j]);
    }
  }
}

// ---- fp32 operands on the fp32 matrix instructions, the same bits ------------------------------------------------
// v_mfma_f32_16x16x4_f32 adds its four products one after the other, each with one rounding, as fmaf does (checked
// bit for bit against a chain of fmaf, subnormal sums included), so a chain of 16 is four of them from zero, and the
// two kernels below leave the bits of the kernel above at twice the vector ALUs' rate and with a sixteenth of their
// instructions.  A lane (r = lane % 16, q = lane / 16) must hold k = 4 t + q of row r for instruction t of a chain; it
// loads k = 4 q .. 4 q + 3 (16 bytes), and four exchanges between the quarters of the wave turn one into the other.
typedef float gf32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void exchange32(float& a, float& b) {      // a's upper half of the wave for b's lower half
  const auto v = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(v[0]);
  b = __uint_as_float(v[1]);
}
__device__ __forceinline__ void exchange16(float& a, float& b) {      // a's odd quarters for b's even ones
  const auto v = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(v[0]);
  b = __uint_as_float(v[1]);
}
__device__ __forceinline__ float4 quarters_turned(float4 v) {
  exchange32(v.x, v.z);
  exchange32(v.y, v.w);
  exchange16(v.x, v.y);
  exchange16(v.z, v.w);
  return v;
}

// one chain of 16: w (rows of W) and x (rows of A) as quarters_turned left them
__device__ __forceinline__ gf32x4 chain_of_16(const float4& w, const float4& x) {
  gf32x4 p = __builtin_amdgcn_mfma_f32_16x16x4f32(w.x, x.x, gf32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
  p = __builtin_amdgcn_mfma_f32_16x16x4f32(w.y, x.y, p, 0, 0, 0);
  p = __builtin_amdgcn_mfma_f32_16x16x4f32(w.z, x.z, p, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x4f32(w.w, x.w, p, 0, 0, 0);
}

__device__ __forceinline__ void store_four(float* __restrict__ C, int m, int n, int M, int N, int ldc, bool wide, gf32x4 v) {
  if (m >= M) return;
  float* o = C + (size_t)m * ldc + n;
  if (wide && n + 3 < N) {
    *reinterpret_cast<gf32x4*>(o) = v;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < N) o[e] = v[e];
  }
}

// Few rows (a decode step, a short prompt): bound by reading W once.  A workgroup takes RT * 16 rows of W, MT * 16 rows of A and
// all of K; a wave takes every WAVES-th stretch of 256 values, straight into registers (each byte of W is used by one wave of a
// row of workgroups), PIECE chains of 16 at a time in two sets of registers: the next piece is asked for before this one is worked
// on, and no load has a condition (what lies beyond K is read from the row's end and cleared), so that the wait for one piece
// leaves the other under way.  The stretches' sums meet in LDS, where they are added in the order of k.
// Cold weights, us: 128,256 x 2,048 at 1 / 4 / 12 rows 178 / 195 / 229 (1.05 GB: 5.9 to 4.6 TB/s); 16,384 x 2,048 27.5 / 29.3 / 33.1;
// 2,048 x 8,192 24.1 / 26.8 / 34.3; 28,672 x 4,096 87.9 / 93.7 / 108; shapes of more rows beside the rule below.
// SHORT: a wave is done where K ends within its stretch.  The branches cost what they leave out where stretches are full (16,384 x
// 1,024 at 8 rows 19.8 us without and 21.1 with them), so only K of few stretches takes it: 2,048 x 64 / 300 / 516 / 900 at 8 rows 4.9 / 5.4 / 5.5 /
// 5.6 without and 2.6 / 4.8 / 5.0 / 5.1 with them.
template <int MT, int RT, int WAVES, int PIECE, bool SHORT>
__global__ __launch_bounds__(WAVES * 64) void gemm_f32_stream_kernel(const float* __restrict__ A,
                                                                     const float* __restrict__ W,
                                                                     float* __restrict__ C, int M, int N, int K,
                                                                     int lda, int ldw, int ldc, bool wide) {
  constexpr int TILES = MT * RT, OWN = (TILES + WAVES - 1) / WAVES;    // tiles whose stretches a wave adds up
  static_assert(16 % (2 * PIECE) == 0, "a stretch is a whole number of pairs of pieces");
  // written out for the smallest tile only: of the others, a whole stretch at once kept twice the registers and more (48 x 32 all
  // 512), one wave a SIMD for two or three (142 rows x 2,048 x 8,192 107 us, as a loop 91; 40 x 6,144 x 4,096 57.8 and 50.4)
  constexpr int ROUNDS = TILES == 1 ? 16 / (2 * PIECE) : 1;
  __shared__ gf32x4 mids[2][WAVES][TILES][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, q = lane >> 4;
  const int n0 = blockIdx.x * (16 * RT), m0 = blockIdx.y * (16 * MT);
  // the workgroup's first rows as scalars, a lane's place behind them in 32 bits (the host looks after that)
  const char* const wbase = (const char*)(W + (size_t)n0 * ldw);
  const char* const abase = (const char*)(A + (size_t)m0 * lda);
  uint32_t wrow[RT], arow[MT];
#pragma unroll
  for (int i = 0; i < RT; ++i) wrow[i] = (uint32_t)min(16 * i + r, N - 1 - n0) * (uint32_t)ldw * 4u;
#pragma unroll
  for (int i = 0; i < MT; ++i) arow[i] = (uint32_t)min(16 * i + r, M - 1 - m0) * (uint32_t)lda * 4u;
  const int stretches = (K + 255) / 256;
  float4 w0[PIECE][RT], x0[PIECE][MT], w1[PIECE][RT], x1[PIECE][MT];
  auto load = [&](int k0, float4 (&w)[PIECE][RT], float4 (&x)[PIECE][MT]) {
#pragma unroll
    for (int c = 0; c < PIECE; ++c) {
      const uint32_t k = (uint32_t)min(k0 + 16 * c + 4 * q, K - 4) * 4u;
#pragma unroll
      for (int i = 0; i < RT; ++i) w[c][i] = *reinterpret_cast<const float4*>(wbase + (wrow[i] + k));
#pragma unroll
      for (int i = 0; i < MT; ++i) x[c][i] = *reinterpret_cast<const float4*>(abase + (arow[i] + k));
    }
  };
  gf32x4 mid[TILES];
  auto work = [&](int k0, float4 (&w)[PIECE][RT], float4 (&x)[PIECE][MT]) {
    if (k0 + 16 * PIECE > K) {                                         // the row's end
#pragma unroll
      for (int c = 0; c < PIECE; ++c)
        if (k0 + 16 * c + 4 * q >= K) {
#pragma unroll
          for (int i = 0; i < RT; ++i) w[c][i] = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
          for (int i = 0; i < MT; ++i) x[c][i] = make_float4(0.f, 0.f, 0.f, 0.f);
        }
    }
#pragma unroll
    for (int c = 0; c < PIECE; ++c) {
#pragma unroll
      for (int i = 0; i < RT; ++i) w[c][i] = quarters_turned(w[c][i]);
#pragma unroll
      for (int j = 0; j < MT; ++j) {
        const float4 xt = quarters_turned(x[c][j]);
#pragma unroll
        for (int i = 0; i < RT; ++i) mid[i * MT + j] += chain_of_16(w[c][i], xt);
      }
    }
  };
  gf32x4 acc[OWN];                                                     // wave t: tiles t, t + WAVES, ...
#pragma unroll
  for (int o = 0; o < OWN; ++o) acc[o] = gf32x4{0.f, 0.f, 0.f, 0.f};
  int buf = 0;
  if (wave < stretches) load(wave * 256, w0, x0);
  for (int s0 = 0; s0 < stretches; s0 += WAVES, buf ^= 1) {
    const int s = s0 + wave, k0 = s * 256;
    if (s < stretches) {
#pragma unroll
      for (int t = 0; t < TILES; ++t) mid[t] = gf32x4{0.f, 0.f, 0.f, 0.f};
      const int next = s + WAVES < stretches ? k0 + WAVES * 256 : k0;  // behind the wave's last stretch anything that can be read
#pragma clang loop unroll_count(ROUNDS)
      for (int c = 0; c < 16 && (!SHORT || k0 + 16 * c < K); c += 2 * PIECE) {
        load(k0 + 16 * (c + PIECE), w1, x1);
        __builtin_amdgcn_sched_barrier(0);                             // all of them in front of the first wait
        work(k0 + 16 * c, w0, x0);
        load(c + 2 * PIECE < 16 ? k0 + 16 * (c + 2 * PIECE) : next, w0, x0);
        __builtin_amdgcn_sched_barrier(0);
        work(k0 + 16 * (c + PIECE), w1, x1);
      }
#pragma unroll
      for (int t = 0; t < TILES; ++t) mids[buf][wave][t][lane] = mid[t];
    }
    __syncthreads();                 // the other buffer is written next, and this one only after the next barrier
    const int have = min(WAVES, stretches - s0);
#pragma unroll
    for (int o = 0; o < OWN; ++o)
      if (wave + o * WAVES < TILES)
        for (int i = 0; i < have; ++i) acc[o] += mids[buf][i][wave + o * WAVES][lane];
  }
#pragma unroll
  for (int o = 0; o < OWN; ++o) {
    const int t = wave + o * WAVES;
    if (t < TILES) store_four(C, m0 + 16 * (t % MT) + r, n0 + 16 * (t / MT) + 4 * q, M, N, ldc, wide, acc[o]);
  }
}

// Many rows: bound by the matrix instructions (157 TFLOP/s): 2,048 rows x 28,672 x 4,096 at 102 TFLOP/s, 4.7 against
// 12.7 ms with the vector kernel.  Tiles of 32 WM rows of A x 32 WN rows of W, four waves, 16 WM x 16 WN of the result each.  K is walked 32
// values (two chains) at a time through two LDS stages, written as the matrix instructions read them; the loads of the
// stage after next are in flight meanwhile.
template <int WM, int WN>
__global__ __launch_bounds__(256) void gemm_f32_tile_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                            float* __restrict__ C, int M, int N, int K, int lda, int ldw,
                                                            int ldc, bool wide, int tiles_m, int tiles_n) {
  constexpr int GA = 2 * WM, GW = 2 * WN, PER = (GA + GW) / 4;         // groups of 16 rows; a wave loads PER of them
  static_assert((GA + GW) % 4 == 0, "the groups of rows are dealt out over four waves");
  __shared__ float4 stage[2][2][GA + GW][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, q = lane >> 4;
  // eight tiles of rows of A in a row share the rows of W that they multiply with while those are in the caches
  const int per_band = 8 * tiles_n, band = blockIdx.x / per_band, in_band = blockIdx.x - band * per_band;
  const int rows = min(8, tiles_m - 8 * band);
  const int m0 = (8 * band + in_band % rows) * (32 * WM), n0 = (in_band / rows) * (32 * WN);
  const int wm = (wave >> 1) * WM, wn = (wave & 1) * WN;               // this wave's first groups
  const float* from[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int g = wave * PER + i;
    from[i] = (g < GA ? A + (size_t)min(m0 + 16 * g + r, M - 1) * lda : W + (size_t)min(n0 + 16 * (g - GA) + r, N - 1) * ldw) + 4 * q;
  }
  float4 reg[PER][2];
  auto load = [&](int k0) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const bool in = k0 + 16 * h + 4 * q < K;
#pragma unroll
      for (int i = 0; i < PER; ++i)
        reg[i][h] = in ? *reinterpret_cast<const float4*>(from[i] + k0 + 16 * h) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  };
  auto put = [&](int buf) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < PER; ++i) stage[buf][h][wave * PER + i][lane] = quarters_turned(reg[i][h]);
  };
  gf32x4 acc[WM][WN], mid[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j) acc[i][j] = mid[i][j] = gf32x4{0.f, 0.f, 0.f, 0.f};
  const int steps = (K + 31) / 32;
  load(0);
  put(0);
  if (steps > 1) load(32);
  __syncthreads();
  for (int s = 0; s < steps; ++s) {
    const int buf = s & 1;
    if (s + 1 < steps) {
      put(buf ^ 1);                                                    // read last before the barrier that ended step s - 1
      if (s + 2 < steps) load((s + 2) * 32);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float4 a[WM], w[WN];
#pragma unroll
      for (int i = 0; i < WM; ++i) a[i] = stage[buf][h][wm + i][lane];
#pragma unroll
      for (int j = 0; j < WN; ++j) w[j] = stage[buf][h][GA + wn + j][lane];
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j) mid[i][j] += chain_of_16(w[j], a[i]);
    }
    if ((s & 7) == 7) {                                                // 256 values of k are in
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j) {
          acc[i][j] += mid[i][j];
          mid[i][j] = gf32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
      store_four(C, m0 + 16 * (wm + i) + r, n0 + 16 * (wn + j) + 4 * q, M, N, ldc, wide, acc[i][j] + mid[i][j]);
}

template <int MT, int RT, int WAVES, int PIECE, bool SHORT = false>
static void launch_f32_stream(const float* A, const float* W, float* C, int M, int N, int K, int lda, int ldw, int ldc,
                              bool wide, hipStream_t stream) {
  gemm_f32_stream_kernel<MT, RT, WAVES, PIECE, SHORT><<<dim3((N + 16 * RT - 1) / (16 * RT), (M + 16 * MT - 1) / (16 * MT)), WAVES * 64,
                                                 0, stream>>>(A, W, C, M, N, K, lda, ldw, ldc, wide);
}

#define GS_MOST_ROWS 32             // rows of A that the streaming kernel takes whatever the shape
#define GS_UNITS 256                // compute units
#define GS_ENOUGH_TILES 512         // the largest tile that still gives so many workgroups
template <int WM, int WN>
static long f32_tiles(int M, int N) { return (long)((M + 32 * WM - 1) / (32 * WM)) * ((N + 32 * WN - 1) / (32 * WN)); }

template <int WM, int WN>
static void launch_f32_tile(const float* A, const float* W, float* C, int M, int N, int K, int lda, int ldw, int ldc,
                            bool wide, hipStream_t stream) {
  const int tm = (M + 32 * WM - 1) / (32 * WM), tn = (N + 32 * WN - 1) / (32 * WN);
  gemm_f32_tile_kernel<WM, WN><<<(unsigned)((long)tm * tn), 256, 0, stream>>>(A, W, C, M, N, K, lda, ldw, ldc, wide, tm, tn);
}

// fp32 with rows that can be read 16 bytes at a time; false: the vector kernel takes the product
static bool gemm_f32(const float* A, const float* W, float* C, int M, int N, int K, int lda, int ldw, int ldc,
                     hipStream_t stream) {
  if (((uintptr_t)A | (uintptr_t)W) & 15 || (K | lda | ldw) & 3) return false;
  // A stretch of 256 a wave leaves seven of eight waves nothing to do with short rows (9,000 x 16 / 32 / 64 at 1 row 10.6 us and with
  // the vector kernel 4.7 / 7.0 / 10.9, at 20 rows 17 / 17 / 18 and 5.2 / 7.8 / 12.5; 1,000 x 16 / 32 at 20 rows 6.9 and 5.0 / 7.5)
  if (M <= GS_MOST_ROWS && (K <= 16 || (N > 4096 && K <= (M > 16 ? 96 : 48)))) return false;
  const bool wide = ((uintptr_t)C & 15) == 0 && (ldc & 3) == 0;
  // Up to 16 rows: 16 rows of W a workgroup, of 16 waves where those are at most one a compute unit and there are more stretches
  // than four waves take at once, although some waves have none until K is 3,841 (4,096 x 4,096 at 1 row 15.7 us, with four waves
  // 21.6; x 1,028 / 2,048 8.4 / 10.0 and 10.4 / 12.6; with eight, where four of sixteen or fewer have one, the same; 6,144 x 4,096, more than one a unit, 26.5 and 25.2), of eight where each has two (28,672 x 4,096
  // at 1 / 4 rows 87.9 / 93.7, with four 94.7 / 98.4; with one each 16,384 x 2,048 29.7, with four 27.5), of four otherwise; from nine
  // rows on, whose reads then weigh as much as W's, 64 rows of W share them (16 rows x 128,256 x 2,048 249 us, with 16 rows
  // of W 295; 8,192 x 2,048, which that leaves 128 workgroups, 28.6 and 20.2).
  const bool near = lda < 1 << 24 && ldw < 1 << 24;                    // 64 rows within 32 bits of the first
  if (M <= 16 && near) {
    if (N <= 16 * GS_UNITS && K > 1024) launch_f32_stream<1, 1, 16, 2>(A, W, C, M, N, K, lda, ldw, ldc, wide, stream);
    else if (M > 8 && N >= 64 * GS_UNITS) launch_f32_stream<1, 4, 4, 2>(A, W, C, M, N, K, lda, ldw, ldc, wide, stream);
    else if (K < 1024 && K % 256 != 0) launch_f32_stream<1, 1, 4, 2, true>(A, W, C, M, N, K, lda, ldw, ldc, wide, stream);
    else if (M <= 8 && K >= 4096) launch_f32_stream<1, 1, 8, 2>(A, W, C, M, N, K, lda, ldw, ldc, wide, stream);
    else launch_f32_stream<1, 1, 4, 2>(A, W, C, M, N, K, lda, ldw, ldc, wide, stream);
    return true;
  }
  // Above: the matrix instructions of a compute unit are what its workgroup has, so a shape costs its workgroups in turns of
  // the compute units, and the tile that wastes least of the last turn and of the last rows wins.  A turn, us with K of 8,192: 16
  // x 16 of the result 35, 32 x 16 50, 32 x 32 69, 48 x 32 84, 64 x 32 100, 48 x 48 112, 48 x 64 155, 64 x 64 198 (from 64 x 32 on 12.4 to 12.9 a
  // tile of 16 x 16; the matrix instructions alone 6.8).  The tiles below share both operands but walk K in step with two barriers
  // every 32 values; several of them on a compute unit make up for that, so they cost by the share of a turn: 128 x 128 of many rows
  // 680, 64 x 64 190, 32 x 32 62 and 166 at the least.  Cold weights, us with 32 x 16, 32 x 32 and 48 x 32 alone and now: 16,384 x 2,048 at 40 / 96 /
  // 142 rows 61.8 / 110 / 157 and 45.1 / 85.4 / 126, 6,144 x 4,096 at 64 / 96 / 142 76.8 / 116 / 155 and 57.4 / 59.2 / 107, 4,096 x 14,336 at
  // 142 / 220 372 / 452 and 264 / 349, 2,048 x 8,192 at 24 / 142 / 300 48.3 / 107 / 219 and 35.2 / 84.0 / 154, 128,256 x 2,048 at 142 1,373 and 1,012.
  // Those turns are of 32 stretches, eight on each of a unit's four matrix units.  Against the tiles several turns cost as many stretches as
  // the fullest one has: K of 1,280 is two stretches for one of them and one for the others (300 x 4,096 x 1,280 72.6 us, in tiles 54.8; 142 x
  // 16,384 x 1,280 118 and 93.9; x 3,072, three on each, 221 and 238).  A single turn is mostly the way there and back and stays as it is (96 x
  // 6,144 x 1,280 29.2 us, in tiles 37.9; 33 x 1,000 x 1,280 7.8 and 27.0; left behind: 200 x 4,096 x 1,280 51.9 and 44.7, 64 x 16,384 x 1,280 53.5 and 47.3).
  // (300 x 128,256 x 2,048, where both cost the same by this rule: 2,053 in tiles, 2,236 in 64 x 64: the tiles unless 2 % are won.)
  // Three stretches of K and fewer leave waves without one (4,099 x 516 at 33 rows 15.2 us, the tiles 12.5; 1,000 x 1,000 7.8 and 18.0).
  typedef void (*Launch)(const float*, const float*, float*, int, int, int, int, int, int, bool, hipStream_t);
  static const struct { int rows, cols, turn; Launch launch; } shapes[] = {
      {16, 16, 35, launch_f32_stream<1, 1, 16, 2>}, {32, 16, 50, launch_f32_stream<2, 1, 4, 2>}, {32, 32, 69, launch_f32_stream<2, 2, 4, 2>},
      {48, 32, 84, launch_f32_stream<3, 2, 8, 1>},  {64, 32, 100, launch_f32_stream<4, 2, 8, 1>}, {48, 48, 112, launch_f32_stream<3, 3, 8, 1>},
      {48, 64, 155, launch_f32_stream<3, 4, 4, 1>}, {64, 64, 198, launch_f32_stream<4, 4, 4, 1>}};
  long best = 0, best_turns = 0;
  Launch launch = nullptr;
  for (const auto& s : shapes) {
    const long groups = (long)((M + s.rows - 1) / s.rows) * ((N + s.cols - 1) / s.cols), turns = (groups + GS_UNITS - 1) / GS_UNITS, cost = s.turn * turns;
    if (!launch || cost < best) { best = cost; best_turns = turns; launch = s.launch; }
  }
  if (best_turns > 1) best = best * ((K + 1023) / 1024 * 1024) / K;
  const long t44 = f32_tiles<4, 4>(M, N), t22 = f32_tiles<2, 2>(M, N), t11 = 62 * f32_tiles<1, 1>(M, N) / GS_UNITS;
  const long tiles = t44 >= GS_ENOUGH_TILES ? 680 * t44 / GS_UNITS : t22 >= GS_ENOUGH_TILES ? 190 * t22 / GS_UNITS : t11 < 166 ? 166 : t11;
  if (near && (M <= GS_MOST_ROWS || (K > 768 && 50 * best < 49 * tiles))) {
    launch(A, W, C, M, N, K, lda, ldw, ldc, wide, stream);
    return true;
  }
  if (t44 >= GS_ENOUGH_TILES) launch_f32_tile<4, 4>(A, W, C, M, N, K, lda, ldw, ldc, wide, stream);
  else if (t22 >= GS_ENOUGH_TILES) launch_f32_tile<2, 2>(A, W, C, M, N, K, lda, ldw, ldc, wide, stream);
  else launch_f32_tile<1, 1>(A, W, C, M, N, K, lda, ldw, ldc, wide, stream);
  return true;
}

// in_dtype: dtype of A and W; out_dtype: dtype of C (fp32 out of bf16 in is allowed).
extern "C" int ia_gemm_generic(const void* A, const void* W, void* C, int in_dtype, int out_dtype, int M, int N,
                               int K, int lda, int ldw, int ldc, hipStream_t stream) {
  if (M < 0 || N <= 0 || K <= 0 || lda < K || ldw < K || ldc < N) return IA_ERR_BAD_ARG;
  if (M == 0) return IA_OK;
  dim3 grid((N + GT - 1) / GT, (M + GT - 1) / GT);
  if (grid.y > 65535u) return IA_ERR_UNSUPPORTED;
  if (in_dtype == IA_F32 && out_dtype == IA_F32 &&
      gemm_f32((const float*)A, (const float*)W, (float*)C, M, N, K, lda, ldw, ldc, stream)) {
    // launched
  } else if (in_dtype == IA_F32 && out_dtype == IA_F32)
    gemm_nt_kernel<float, float, float><<<grid, 256, 0, stream>>>((const float*)A, (const float*)W, (float*)C, M, N,
                                                                  K, lda, ldw, ldc);
  else if (in_dtype == IA_BF16 && out_dtype == IA_BF16)
    gemm_nt_kernel<bf16_t, bf16_t, bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)A, (const bf16_t*)W, (bf16_t*)C,
                                                                     M, N, K, lda, ldw, ldc);
  else if (in_dtype == IA_BF16 && out_dtype == IA_F32)
    gemm_nt_kernel<bf16_t, bf16_t, float><<<grid, 256, 0, stream>>>((const bf16_t*)A, (const bf16_t*)W, (float*)C, M,
                                                                    N, K, lda, ldw, ldc);
  else
    return IA_ERR_UNSUPPORTED;
  IA_LAUNCH_CHECK();
  return IA_OK;
}

// ---- the launchers of this file as operations of a step's program (see op_call.h) ----
#include "op_call.h"
IA_OP(ia_gemm_generic)
