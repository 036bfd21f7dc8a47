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

// Few rows (a decode step): bound by reading W once (3 rows x 128,256 x 2,048: 275 us, 3.8 TB/s, against 1,021 with the
// vector kernel; 4,096 x 14,336 at 1 row 52 against 2,263 us, 4.5 TB/s; 2,048 x 2,048 9 against 298 us).  A workgroup of 8 waves takes RT * 16 rows of W and all of K; a
// wave takes every eighth stretch of 256 values, whose loads are all in flight at once (16 KB of W a wave and 16 rows),
// straight into registers: each byte of W is used by one wave.  The stretches' sums meet in LDS, where they are added
// in the order of k.  A's rows come from the caches (MT * 16 of them, RT * 16 rows of W share a load).
#define GS_WAVES 8
#define GS_MOST_ROWS 32             // rows of A that the streaming kernel takes (3,072 x 2,048: 20 us at 32 rows, the tiles 36 at 33)
#define GS_TWO_GROUPS_FROM 8192     // rows of W from which a workgroup takes 32 of them: one workgroup a compute unit
#define GS_ENOUGH_TILES 512         // the largest tile that still gives so many workgroups

template <int MT, int RT>
__global__ __launch_bounds__(GS_WAVES * 64) void gemm_f32_stream_kernel(const float* __restrict__ A,
                                                                        const float* __restrict__ W,
                                                                        float* __restrict__ C, int M, int N, int K,
                                                                        int lda, int ldw, int ldc, bool wide) {
  constexpr int TILES = MT * RT;
  constexpr int PIECE = TILES >= 4 ? 4 : TILES == 2 ? 8 : 16;          // chains whose loads are in flight together
  __shared__ gf32x4 mids[2][GS_WAVES][TILES][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, q = lane >> 4;
  const int n0 = blockIdx.x * (16 * RT);
  const float* wrow[RT];
  const float* arow[MT];
#pragma unroll
  for (int i = 0; i < RT; ++i) wrow[i] = W + (size_t)min(n0 + 16 * i + r, N - 1) * ldw + 4 * q;
#pragma unroll
  for (int i = 0; i < MT; ++i) arow[i] = A + (size_t)min(16 * i + r, M - 1) * lda + 4 * q;
  const int stretches = (K + 255) / 256;
  gf32x4 acc = {0.f, 0.f, 0.f, 0.f};                                   // wave t: tile t
  float4 w[PIECE][RT], x[PIECE][MT];
  auto load = [&](int k0) {                                            // PIECE chains from k0 on; past K zeros
#pragma unroll
    for (int c = 0; c < PIECE; ++c) {
      const bool in = k0 + 16 * c + 4 * q < K;
#pragma unroll
      for (int i = 0; i < RT; ++i)
        w[c][i] = in ? *reinterpret_cast<const float4*>(wrow[i] + k0 + 16 * c) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int i = 0; i < MT; ++i)
        x[c][i] = in ? *reinterpret_cast<const float4*>(arow[i] + k0 + 16 * c) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  };
  int buf = 0;
  if (wave < stretches) load(wave * 256);
  for (int s0 = 0; s0 < stretches; s0 += GS_WAVES, buf ^= 1) {
    const int s = s0 + wave;
    if (s < stretches) {
      gf32x4 mid[TILES];
#pragma unroll
      for (int t = 0; t < TILES; ++t) mid[t] = gf32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int piece = 0; piece < 16; piece += PIECE) {
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
        // the next chains: of this stretch, or of the wave's next one
        if (piece + PIECE < 16) load(s * 256 + (piece + PIECE) * 16);
        else if (s + GS_WAVES < stretches) load((s + GS_WAVES) * 256);
      }
#pragma unroll
      for (int t = 0; t < TILES; ++t) mids[buf][wave][t][lane] = mid[t];
    }
    __syncthreads();                 // the other buffer is written next, and this one only after the next barrier
    if (wave < TILES) {
      const int have = min(GS_WAVES, stretches - s0);
      for (int i = 0; i < have; ++i) acc += mids[buf][i][wave][lane];
    }
  }
  if (wave < TILES) store_four(C, 16 * (wave % MT) + r, n0 + 16 * (wave / MT) + 4 * q, M, N, ldc, wide, acc);
}

// Many rows: bound by the matrix instructions (157 TFLOP/s): 2,048 rows x 28,672 x 4,096 at 102 TFLOP/s, 4.7 against
// 12.7 ms with the vector kernel; 142 rows x 2,048 x 8,192 178 against 1,315 us (320 workgroups, a chain of K).  Tiles of 32 WM rows of A x 32 WN rows of W, four waves, 16 WM x 16 WN of the result each.  K is walked 32
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

template <int MT>
static void launch_f32_stream(const float* A, const float* W, float* C, int M, int N, int K, int lda, int ldw, int ldc,
                              bool wide, hipStream_t stream) {
  if (MT == 1 && N >= GS_TWO_GROUPS_FROM)                              // two of both would not fit the registers
    gemm_f32_stream_kernel<1, 2><<<(N + 31) / 32, GS_WAVES * 64, 0, stream>>>(A, W, C, M, N, K, lda, ldw, ldc, wide);
  else
    gemm_f32_stream_kernel<MT, 1><<<(N + 15) / 16, GS_WAVES * 64, 0, stream>>>(A, W, C, M, N, K, lda, ldw, ldc, wide);
}

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
  if (M <= 16) launch_f32_stream<1>(A, W, C, M, N, K, lda, ldw, ldc, wide, stream);
  else if (M <= GS_MOST_ROWS) launch_f32_stream<2>(A, W, C, M, N, K, lda, ldw, ldc, wide, stream);
  else if (f32_tiles<4, 4>(M, N) >= GS_ENOUGH_TILES) launch_f32_tile<4, 4>(A, W, C, M, N, K, lda, ldw, ldc, wide, stream);
  else if (f32_tiles<2, 2>(M, N) >= GS_ENOUGH_TILES) launch_f32_tile<2, 2>(A, W, C, M, N, K, lda, ldw, ldc, wide, stream);
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
