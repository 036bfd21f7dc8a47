// Latent attention: keys and values of all heads are functions of one low-rank latent per token, and only the
// latent c [rank] and one rotated key part [rot] shared by all heads are cached.  With
//   score_h(i, j) = q_plain_h(i) . (U_h c_j) + q_rot_h(i) . k_rot(j)  =  (U_h^T q_plain_h(i)) . c_j + q_rot_h(i) . k_rot(j)
//   out_h(i)      = V_h sum_j p_h(i, j) c_j
// every head's query becomes a vector [rot | rank] against the one cached key [k_rot | c], and the value is the
// cached latent itself: attention with one key/value head of size rot + rank, which the attention kernels of this
// library serve as they are.  What is here is what stands around them:
//   ia_latent_prepare  from the projections' row [q heads (plain | rot) | latent | k_rot | ...] the row
//                      [H query heads (rot | .) | key (k_rot | c) | value (0 | c)] with c = RMSNorm(latent) * w;
//   ia_gemm_heads      a matrix product per head, out[n, h, :] = x[n, h, :] W_h^T (optionally times
//                      sigmoid(gate[n, h, :])): U_h^T on the plain query parts, V_h on the attended latents.
#include "common.h"
#include "tile_fma.h"

// One workgroup a token.  src row: [H * (dn + dr) | rank | dr | ...]; dst row: (H + 2) heads of d = dr + rank.
template <typename T>
__global__ __launch_bounds__(256) void latent_prepare_kernel(const T* __restrict__ src, int src_stride,
                                                             const T* __restrict__ lat_src, int lat_stride,
                                                             T* __restrict__ dst, int dst_stride,
                                                             const void* __restrict__ w, int w_dtype, int H, int dn,
                                                             int dr, int rank, float eps) {
  __shared__ float red[4];
  const int n = blockIdx.x, d = dr + rank;
  const T* s = src + (size_t)n * src_stride;
  T* o = dst + (size_t)n * dst_stride;
  for (int i = threadIdx.x; i < H * dr; i += 256) {          // the rotated query parts move to the heads' fronts
    const int h = i / dr, r = i - h * dr;
    o[(size_t)h * d + r] = s[(size_t)h * (dn + dr) + dn + r];
  }
  // the latent and the key's rotated part: behind the queries in their row, or rows of their own
  const T* lat = lat_src ? lat_src + (size_t)n * lat_stride : s + (size_t)H * (dn + dr);
  float ss = 0.f;
  for (int i = threadIdx.x; i < rank; i += 256) {
    const float v = to_float(lat[i]);
    ss = fmaf(v, v, ss);
  }
  ss = block_sum<256>(ss, red);
  const float inv = 1.0f / sqrtf(ss / (float)rank + eps);
  T* key = o + (size_t)H * d;
  T* val = key + d;
  for (int i = threadIdx.x; i < rank; i += 256) {
    const T c = from_float<T>(to_float(lat[i]) * inv * load_as_float(w, w_dtype, i));
    key[dr + i] = c;
    val[dr + i] = c;
  }
  for (int i = threadIdx.x; i < dr; i += 256) {
    key[i] = lat[rank + i];
    val[i] = from_float<T>(0.f);
  }
}

extern "C" int ia_latent_prepare(const void* src, int src_stride, const void* lat, int lat_stride, void* dst,
                                 int dst_stride, int dtype, const void* w, int w_dtype, int N, int H, int dn, int dr,
                                 int rank, float eps, hipStream_t stream) {
  if (N < 0 || H <= 0 || dn < 0 || dr < 0 || rank <= 0 || !(eps > 0.f) ||
      src_stride < H * (dn + dr) + (lat ? 0 : rank + dr) || (lat && lat_stride < rank + dr) ||
      dst_stride < (H + 2) * (dr + rank))
    return IA_ERR_BAD_ARG;
  if (N == 0) return IA_OK;
  if (dtype == IA_F32)
    latent_prepare_kernel<float><<<N, 256, 0, stream>>>((const float*)src, src_stride, (const float*)lat, lat_stride, (float*)dst, dst_stride, w,
                                                        w_dtype, H, dn, dr, rank, eps);
  else if (dtype == IA_BF16)
    latent_prepare_kernel<bf16_t><<<N, 256, 0, stream>>>((const bf16_t*)src, src_stride, (const bf16_t*)lat, lat_stride, (bf16_t*)dst, dst_stride, w,
                                                         w_dtype, H, dn, dr, rank, eps);
  else
    return IA_ERR_BAD_ARG;
  IA_LAUNCH_CHECK();
  return IA_OK;
}

// out[n, h, j] = (sum_k x[n, h, k] W[h, j, k]) * (gate ? sigmoid(gate[n, h * Nout + j]) : 1).
// grid: (tiles of Nout, tiles of N, H).  On the vector ALUs in fp32: the 32-bit path, and bfloat16 rows that
// cannot be read 16 bytes at a time.
template <typename T>
__global__ __launch_bounds__(256) void gemm_heads_kernel(const T* __restrict__ x, int x_row, int x_head,
                                                         const T* __restrict__ W, T* __restrict__ out, int o_row,
                                                         int o_head, const T* __restrict__ gate, int g_row, int N,
                                                         int Nout, int K) {
  __shared__ TileFmaLds lds;
  const int h = blockIdx.z;
  const int m0 = blockIdx.y * TF_T, n0 = blockIdx.x * TF_T;
  const int lr = threadIdx.x >> 2;
  const T* a_row = (m0 + lr < N) ? x + (size_t)(m0 + lr) * x_row + (size_t)h * x_head : nullptr;
  const T* w_row = (n0 + lr < Nout) ? W + ((size_t)h * Nout + n0 + lr) * K : nullptr;
  tile_64(a_row, w_row, K, lds, [&](int i, int j0, const float* v) {
    const int m = m0 + i;
    if (m >= N) return;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = n0 + j0 + j;
      if (c >= Nout) continue;
      float y = v[j];
      if (gate) {
        const float g = to_float(gate[(size_t)m * g_row + (size_t)h * Nout + c]);
        y = to_float(from_float<T>(y)) * (1.0f / (1.0f + expf(-g)));    // the product is stored first, as a tensor would be
      }
      out[(size_t)m * o_row + (size_t)h * o_head + c] = from_float<T>(y);
    }
  });
}

// The same on tiles of BM x 128 (tile_mfma_big): grid (tiles of 128 of Nout, tiles of BM of N, H).  With 2,048 rows
// tiles of 32 rows take 185 us where tiles of 128 take 248 (128 heads of 224 x 512); of 48 products of K from 320 to 2,048 with 17 to 4,000
// rows tiles of 128 gain with the longest K and thousands of rows of many heads alone (200 rows of 128 heads of 128 x 2,048 88 / 44).
template <int BM>
__global__ __launch_bounds__(256) void gemm_heads_big_kernel(const bf16_t* __restrict__ x, int x_row, int x_head,
                                                             const bf16_t* __restrict__ W, bf16_t* __restrict__ out,
                                                             int o_row, int o_head, const bf16_t* __restrict__ gate,
                                                             int g_row, int N, int Nout, int K) {
  __shared__ TileBigLds<BM> lds;
  const int h = blockIdx.z;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * TB_N;
  tile_mfma_big<BM>(
      [&](int r) { return x + (size_t)(m0 + r) * x_row + (size_t)h * x_head; },
      [&](int r) { return W + ((size_t)h * Nout + n0 + r) * K; }, N - m0, Nout - n0, K, lds,
      [&](int i, int j0, const float* v) {
        const int m = m0 + i;
        if (m >= N) return;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int c = n0 + j0 + j;
          if (c >= Nout) continue;
          float y = v[j];
          if (gate) {
            const float g = to_float(gate[(size_t)m * g_row + (size_t)h * Nout + c]);
            y = to_float(from_float<bf16_t>(y)) * (1.0f / (1.0f + expf(-g)));
          }
          out[(size_t)m * o_row + (size_t)h * o_head + c] = from_float<bf16_t>(y);
        }
      });
}

// The same for few rows (decoding) and K beyond a head's size, without LDS: bound by one trip to memory.  A wave takes 16 columns of one head for
// up to 16 rows of x and asks for eight steps of 32 values of K of both at once, none under a condition (pieces beyond K are read
// from the last place and cleared); the sums are those of the tiles above, step by step in the same order.  Grid (tiles of
// 64 of Nout, 1, H).
// The reads of x, once for every 16 columns of W, make it lose with long rows and many workgroups.  Its time over that of the
// tiles at 1 / 8 / 16 rows, by K and workgroups: 512 x 128 0.89 / 0.97 / 1.04, 512 x 256 (16 heads of
// 1,024) 1.03 / 1.13 / 1.16; 1,024 x 64 0.98 / 1.07 / 1.14, x 128 1.16 / 1.33 / 1.39.
#define GH_FEW_ROWS 16
static bool heads_few_pays(int N, int H, int Nout, int K) {
  return N <= GH_FEW_ROWS && (long)K * H * ((Nout + 63) / 64) <= (K <= 512 && N <= 8 ? 65536 : 16384);
}

__global__ __launch_bounds__(256) void gemm_heads_few_kernel(const bf16_t* __restrict__ x, int x_row, int x_head,
                                                             const bf16_t* __restrict__ W, bf16_t* __restrict__ out,
                                                             int o_row, int o_head, const bf16_t* __restrict__ gate,
                                                             int g_row, int N, int Nout, int K) {
  constexpr int PIECE = 8;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, q = lane >> 4;
  const int h = blockIdx.z, n0 = (blockIdx.x * 4 + wave) * 16, m = r, mc = min(m, N - 1);
  if (n0 >= Nout) return;
  const bf16_t* w_row = W + ((size_t)h * Nout + min(n0 + r, Nout - 1)) * K;
  const bf16_t* x_row_ = x + (size_t)mc * x_row + (size_t)h * x_head;
  const int c = n0 + 4 * q;
  bf16_t g[4];
  if (gate) {
#pragma unroll
    for (int j = 0; j < 4; ++j) g[j] = gate[(size_t)mc * g_row + (size_t)h * Nout + min(c + j, Nout - 1)];
  }
  tm_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < K; k0 += 32 * PIECE) {
    uint4 wv[PIECE], xv[PIECE];
#pragma unroll
    for (int j = 0; j < PIECE; ++j) {
      const int k = min(k0 + 32 * j + 8 * q, K - 8);
      wv[j] = *reinterpret_cast<const uint4*>(w_row + k);
      xv[j] = *reinterpret_cast<const uint4*>(x_row_ + k);
    }
#pragma unroll
    for (int j = 0; j < PIECE; ++j) {
      if (k0 + 32 * j >= K) break;
      const uint32_t keep = k0 + 32 * j + 8 * q < K ? 0xffffffffu : 0u;
      const uint4 wt = make_uint4(wv[j].x & keep, wv[j].y & keep, wv[j].z & keep, wv[j].w & keep);
      const uint4 xt = make_uint4(xv[j].x & keep, xv[j].y & keep, xv[j].z & keep, xv[j].w & keep);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(tm_bf16x8, wt), __builtin_bit_cast(tm_bf16x8, xt),
                                                    acc, 0, 0, 0);
    }
  }
  if (m >= N) return;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (c + j >= Nout) continue;
    float y = acc[j];
    if (gate) y = to_float(from_float<bf16_t>(y)) * (1.0f / (1.0f + expf(-to_float(g[j]))));
    out[(size_t)m * o_row + (size_t)h * o_head + c + j] = from_float<bf16_t>(y);
  }
}

// The same for short K (a head's size), without LDS: a wave keeps 16 rows of x in registers and walks over its columns of the
// head, 16 at a time, the next ones' rows of W under way (they come from the caches: a head's matrix is some tens of KB, read by every wave).
// Bound by the reads of x and the writes of out; in tiles through LDS a step of K of 64 is a trip to memory and two barriers for 32 rows, and values
// left one by one.  The same sums in the same order.  us, in tiles / so (at 6 TB/s): 2,000 rows of 16 heads of 224 x 64 23.8 / 9.9 (3.0), of
// 64 x 224 with a gate 15.9 / 9.5 (3.7), of 32 heads of 224 x 64 43.0 / 16.7 (6.1).
// A wave may take 32 rows, which share the reads of W; a workgroup's one, two or four waves stand over the rows, so that none is without any.
#define GH_ROWS_K 256
template <int KP, int MT>                                // steps of 32 of K, at most; groups of 16 rows a wave
__global__ __launch_bounds__(256) void gemm_heads_rows_kernel(const bf16_t* __restrict__ x, int x_row, int x_head,
                                                              const bf16_t* __restrict__ W, bf16_t* __restrict__ out, int o_row,
                                                              int o_head, const bf16_t* __restrict__ gate, int g_row, int N, int Nout,
                                                              int K, int tiles, bool fours) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, q = lane >> 4;
  const int h = blockIdx.z, m0 = (blockIdx.y * (blockDim.x >> 6) + wave) * (16 * MT);
  if (m0 >= N) return;
  const int first = blockIdx.x * tiles, last = min(first + tiles, (Nout + 15) / 16);
  int row[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) row[i] = min(m0 + 16 * i + r, N - 1);
  int kc[KP];
  uint32_t keep[KP];                                     // pieces beyond K are read from the last place and cleared
#pragma unroll
  for (int j = 0; j < KP; ++j) {
    kc[j] = min(32 * j + 8 * q, K - 8);
    keep[j] = 32 * j + 8 * q < K ? 0xffffffffu : 0u;
  }
  const auto kept = [](const uint4& v, uint32_t k) { return make_uint4(v.x & k, v.y & k, v.z & k, v.w & k); };
  uint4 xv[MT][KP], w0[KP], w1[KP];
  uint2 g0[MT], g1[MT];
  const auto load = [&](int t, uint4 (&w)[KP], uint2 (&g)[MT]) {
    const bf16_t* w_row = W + ((size_t)h * Nout + min(16 * t + r, Nout - 1)) * K;
#pragma unroll
    for (int j = 0; j < KP; ++j) w[j] = *reinterpret_cast<const uint4*>(w_row + kc[j]);
    if (gate) {
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const bf16_t* g_at = gate + (size_t)row[i] * g_row + (size_t)h * Nout;
        if (fours) {
          g[i] = *reinterpret_cast<const uint2*>(g_at + min(16 * t + 4 * q, Nout - 4));
        } else {
          const int c = 16 * t + 4 * q, end = Nout - 1;
          g[i].x = g_at[min(c, end)].bits | ((uint32_t)g_at[min(c + 1, end)].bits << 16);
          g[i].y = g_at[min(c + 2, end)].bits | ((uint32_t)g_at[min(c + 3, end)].bits << 16);
        }
      }
    }
  };
  const auto work = [&](int t, const uint4 (&w)[KP], const uint2 (&g)[MT]) {
    tm_f32x4 acc[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[i] = tm_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < KP; ++j) {
      if (32 * j >= K) break;
      const uint4 wt = kept(w[j], keep[j]);
#pragma unroll
      for (int i = 0; i < MT; ++i)
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(tm_bf16x8, wt), __builtin_bit_cast(tm_bf16x8, xv[i][j]),
                                                         acc[i], 0, 0, 0);
    }
    const int c = 16 * t + 4 * q;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      float y[4] = {acc[i][0], acc[i][1], acc[i][2], acc[i][3]};
      if (gate) {
        const float z[4] = {__uint_as_float(g[i].x << 16), __uint_as_float(g[i].x & 0xffff0000u), __uint_as_float(g[i].y << 16),
                            __uint_as_float(g[i].y & 0xffff0000u)};
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = to_float(from_float<bf16_t>(y[e])) * (1.0f / (1.0f + expf(-z[e])));
      }
      if (m0 + 16 * i + r >= N || c >= Nout) continue;
      bf16_t* o_at = out + (size_t)row[i] * o_row + (size_t)h * o_head + c;
      if (fours) {
        *reinterpret_cast<uint2*>(o_at) = make_uint2(two_bf16_bits(y[0], y[1]), two_bf16_bits(y[2], y[3]));
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (c + e < Nout) o_at[e] = from_float<bf16_t>(y[e]);
      }
    }
  };
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const bf16_t* x_at = x + (size_t)row[i] * x_row + (size_t)h * x_head;
    g0[i] = g1[i] = make_uint2(0u, 0u);
#pragma unroll
    for (int j = 0; j < KP; ++j) xv[i][j] = *reinterpret_cast<const uint4*>(x_at + kc[j]);
  }
  load(first, w0, g0);
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < KP; ++j) xv[i][j] = kept(xv[i][j], keep[j]);
  int t = first;
  for (; t + 1 < last; t += 2) {
    load(t + 1, w1, g1);
    __builtin_amdgcn_sched_barrier(0);
    work(t, w0, g0);
    load(min(t + 2, last - 1), w0, g0);
    __builtin_amdgcn_sched_barrier(0);
    work(t + 1, w1, g1);
  }
  if (t < last) work(t, w0, g0);
}

// How a launch of the kernel above deals out N rows and `tiles` groups of 16 columns of H heads.
struct HeadsShape {
  int wide, waves, rows, per;            // groups of 16 rows a wave; waves a workgroup; workgroups over the rows; groups of columns a wave
};

// The shape with the least estimated time: the trips of a wave's walk one after the other, and what all waves of the compute unit that has the
// most of them move: their rows of x, and for every group of columns the rows of W and the result (and gate).  The numbers are a fit to
// 763 products of 1 to 2,047 rows of 1 to 128 heads, Nout of 16 to 1,024, K of 16 to 256, each with up to 40 shapes: what it picks takes 3 %
// longer than the fastest on average.  us, in tiles / by some 2,048 waves in workgroups of four over the rows / so: 16 rows of 128 heads of
// 512 x 128 with a gate 7.6 / 9.5 / 5.7, 333 rows of 4 heads of 1,024 x 256 8.7 / 11.2 / 6.7, 100 rows of 16 9.0 / 10.8 / 7.5, 600 rows of 32 heads of
// 64 x 224 9.1 / 9.8 / 6.0.  Few rows too: 1 / 2 / 16 rows of 16 heads of 64 x 224 take 3.4 / 4.7 / 3.7 in the kernel for few rows above (two
// with a gate) and 2.5 / 2.7 / 2.6 so.  Of 1,578 products of 1 to 2,000 rows none takes more than 1.06 of its time in tiles or in that kernel,
// 0.67 in the mean.
static HeadsShape heads_shape(int N, int H, int tiles, int K, bool gate) {
  HeadsShape best{0, 0, 0, 0};
  long least = 0;
  const int kp = K <= 64 ? 2 : K <= 128 ? 4 : 8;
  for (int wide = 1; wide <= (N > 16 ? 2 : 1); ++wide) {
    const int blocks = (N + 16 * wide - 1) / (16 * wide);
    for (int waves = 1; waves <= 4 && (waves == 1 || waves < 2 * blocks); waves *= 2) {
      const int rows = (blocks + waves - 1) / waves;
      if (rows > 65535) continue;                        // (the launch's grid)
      for (int pieces = 1; pieces <= tiles;) {           // of as equal a length as can be
        const int per = (tiles + pieces - 1) / pieces;
        const long workgroups = (long)pieces * rows * H;
        const long unit = (workgroups + 255) / 256 * (waves < blocks ? waves : blocks);
        const long cost = 32 * per + unit * (4 * wide * kp + per * (2 * kp + wide * (gate ? 2 : 1)));
        if (least == 0 || cost < least) {
          least = cost;
          best = HeadsShape{wide, waves, rows, per};
        }
        if (per == 1) break;
        pieces = (tiles + per - 2) / (per - 1);          // the fewest that are shorter
      }
    }
  }
  return best;
}

extern "C" int ia_gemm_heads(const void* x, int x_row, int x_head, const void* W, void* out, int o_row, int o_head,
                             const void* gate, int g_row, int dtype, int N, int H, int Nout, int K,
                             hipStream_t stream) {
  if (N < 0 || H <= 0 || Nout <= 0 || K <= 0 || x_head < 0 || o_head < 0 || x_row < (H - 1) * x_head + K ||
      o_row < (H - 1) * o_head + Nout || (gate && g_row < H * Nout))
    return IA_ERR_BAD_ARG;
  if (N == 0) return IA_OK;
  dim3 grid((Nout + TF_T - 1) / TF_T, (N + TF_T - 1) / TF_T, H);
  if (grid.y > 65535u || grid.z > 65535u) return IA_ERR_UNSUPPORTED;
  if (dtype == IA_F32)
    gemm_heads_kernel<float><<<grid, 256, 0, stream>>>((const float*)x, x_row, x_head, (const float*)W,
                                                              (float*)out, o_row, o_head, (const float*)gate, g_row,
                                                              N, Nout, K);
  else if (dtype == IA_BF16 && (K & 7) == 0 && tile_rows_aligned(x, x_row, x_head) && tile_rows_aligned(W, K)) {
    if (K <= GH_ROWS_K) {
      const int tiles = (Nout + 15) / 16;
      const HeadsShape shape = heads_shape(N, H, tiles, K, gate != nullptr);
      if (shape.waves == 0) return IA_ERR_UNSUPPORTED;
      const bool fours = ((Nout | o_row | o_head) & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 7) == 0 &&
                         (!gate || ((g_row & 3) == 0 && (reinterpret_cast<uintptr_t>(gate) & 7) == 0));
      const dim3 pieces((tiles + shape.per - 1) / shape.per, shape.rows, H);
#define GH_ROWS(KP, MT)                                                                                                              \
  gemm_heads_rows_kernel<KP, MT><<<pieces, 64 * shape.waves, 0, stream>>>((const bf16_t*)x, x_row, x_head, (const bf16_t*)W, (bf16_t*)out, \
                                                                          o_row, o_head, (const bf16_t*)gate, g_row, N, Nout, K, shape.per, fours)
#define GH_ROWS_BY(MT)               \
  do {                               \
    if (K <= 64) GH_ROWS(2, MT);     \
    else if (K <= 128) GH_ROWS(4, MT); \
    else GH_ROWS(8, MT);             \
  } while (0)
      if (shape.wide == 2) GH_ROWS_BY(2);
      else GH_ROWS_BY(1);
#undef GH_ROWS_BY
#undef GH_ROWS
      IA_LAUNCH_CHECK();
      return IA_OK;
    }
    if (heads_few_pays(N, H, Nout, K)) {
      gemm_heads_few_kernel<<<dim3((Nout + 63) / 64, 1, H), 256, 0, stream>>>((const bf16_t*)x, x_row, x_head, (const bf16_t*)W,
                                                                              (bf16_t*)out, o_row, o_head, (const bf16_t*)gate,
                                                                              g_row, N, Nout, K);
      IA_LAUNCH_CHECK();
      return IA_OK;
    }
    const int bm = 32;      // many small workgroups hide each other's steps better than few large ones
    dim3 big((Nout + TB_N - 1) / TB_N, (N + bm - 1) / bm, H);
    if (big.y > 65535u) return IA_ERR_UNSUPPORTED;
    gemm_heads_big_kernel<32><<<big, 256, 0, stream>>>((const bf16_t*)x, x_row, x_head, (const bf16_t*)W,
                                                       (bf16_t*)out, o_row, o_head, (const bf16_t*)gate, g_row, N,
                                                       Nout, K);
  }
  else if (dtype == IA_BF16)
    gemm_heads_kernel<bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)x, x_row, x_head, (const bf16_t*)W,
                                                               (bf16_t*)out, o_row, o_head, (const bf16_t*)gate, g_row,
                                                               N, Nout, K);
  else
    return IA_ERR_BAD_ARG;
  IA_LAUNCH_CHECK();
  return IA_OK;
}

#include "op_call.h"
IA_OP(ia_latent_prepare)
IA_OP(ia_gemm_heads)
