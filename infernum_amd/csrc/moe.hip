// Routed experts: a token's feed-forward is the weighted sum of `top` small gated feed-forwards chosen among E.
//   ia_router_topk   z = logits + bias (fp32); the `top` largest (the lowest index among equals) and the softmax
//                    over those alone;
//   ia_moe_sort      the (token, choice) pairs grouped by expert: offsets[E + 1], perm[P];
//   ia_moe_gate_up   per expert, over its pairs' tokens: g = min(Wg x, limit), u = clamp(Wu x, -limit, limit),
//                    y = g sigmoid(alpha g) (u + shift); the rows of Wg and Wu alternate in the expert's matrix (limit
//                    infinity, alpha 1, shift 0: y = silu(Wg x) (Wu x));
//   ia_moe_down      per expert: Wd y times the pair's routing weight, as fp32 into parts[choice, token, :], which
//                    the kernel that takes the feed-forward's result next adds in the order of the choices.
// A routing weight can stand on the expert's INPUT instead: ia_moe_gate_up (and ia_moe_glu) given the weights multiply
// both products with it, in fp32 (G (w x) = w (G x)), and ia_moe_down (and ia_moe_scatter) given none leave theirs as it is.
// Only the chosen experts' weights are read.  A pair's result is one chain of operations over its own token and
// its expert's weights, whatever else the step holds and wherever the sort has put it.
#include "common.h"
#include "tile_fma.h"

// One wave a token: lane l holds the logits of experts l, l + 64, ...; `top` rounds of "the largest not taken yet"
// (the lowest index among equals), each a maximum over the wave.
#define RT_PER_LANE 16        // experts a lane holds: E <= 64 * RT_PER_LANE
// A wave's choices wait in its lanes, choice k in lane k % 64, and leave with their final weights: written and read back for
// the last factor they cost a trip to memory (one token to 4 of 32: 6.9 us, so 4.4).  Beyond 64 choices the ones
// before are written out on the way and read again at the end.
__device__ __forceinline__ void router_keep(int& mine_e, float& mine_w, int k, int lane, int e, float w, int* ids, float* weights) {
  if (k >= 64 && (k & 63) == lane) {                       // this lane's choice k - 64
    ids[k - 64] = mine_e;
    weights[k - 64] = mine_w;
  }
  mine_e = (k & 63) == lane ? e : mine_e;
  mine_w = (k & 63) == lane ? w : mine_w;
}
__device__ __forceinline__ void router_finish(int mine_e, float mine_w, int top, int lane, float factor, int* ids, float* weights) {
  if (lane >= top) return;
  const int last = lane + (top - 1 - lane) / 64 * 64;      // this lane's last choice
  for (int k = lane; k < last; k += 64) weights[k] *= factor;
  ids[last] = mine_e;
  weights[last] = mine_w * factor;
}

// Up to 64 experts, one a lane: the place of this lane's expert among all, largest first and the lowest index among equals (64 for
// an expert that cannot be chosen).  Every lane compares with every expert, whose values come as scalars: no step waits
// for the one before, where `top` rounds of a maximum over the wave are chains of twelve exchanges each (1 / 64 tokens to 4 of 32 with
// join and sort 7.3 / 8.5 us in rounds, 6.2 / 7.3 so; to 8 of 64 10.5 / 12.0 and 9.0 / 9.8).  The comparisons grow with the experts and
// the rounds with the choices, so few choices of many experts stay with the rounds (1 / 512 / 8,192 tokens to 1 of 64 2.3 / 2.8 / 3.9 us in
// rounds and 4.1 / 4.6 / 9.2 by rank, to 2 of 32 2.9 / 3.4 / 5.5 and 3.0 / 3.5 / 5.9, to 4 of 64 4.2 / 4.5 / 8.6 and 4.2 / 4.6 / 9.2, to 4 of 32
// 4.2 / 4.5 / 8.3 and 3.0 / 3.5 / 6.1).
__device__ __forceinline__ bool choose_by_rank(int E, int top) { return 12 * top >= E; }
__device__ __forceinline__ int expert_rank(float x, bool can, int E, int lane) {
  const int b = __float_as_int(x + 0.0f);                  // -0 counts as 0
  const int key = can ? b ^ ((b >> 31) & 0x7fffffff) : (int)0x80000000;      // in the order of the values
  int rank = 0;
#pragma unroll 8
  for (int i = 0; i < E; ++i) {
    const int other = __builtin_amdgcn_readlane(key, i);
    rank += (other > key || (other == key && i < lane)) ? 1 : 0;
  }
  return can ? rank : 64;
}
// The value of the lane with rank k, for all lanes.
__device__ __forceinline__ float value_of_rank(float v, int rank, int k) {
  const unsigned long long who = __ballot(rank == k);
  return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), who ? __ffsll(who) - 1 : 0));
}

// PL: experts a lane holds (32 experts, one token: 4.4 us with one a lane, 9.0 with sixteen).  v: this lane's logits with their
// biases; leaves the token's choices and weights at ids and weights, and with one expert a lane its place among them in mine_rank.
template <int PL>
__device__ __forceinline__ void choose_then_softmax(const float (&v)[PL], int E, int top, int lane, int* ids, float* weights, int& mine_rank) {
  if (PL == 1 && choose_by_rank(E, top)) {
    // a value that compares with nothing (NaN) counts as the smallest
    const float x = (v[0] == v[0]) ? v[0] : -INFINITY;
    const int rank = expert_rank(x, lane < E, E, lane);
    const float w = expf(x - value_of_rank(x, rank, 0));
    float sum = 0.f;
    for (int k = 0; k < top; ++k) sum += value_of_rank(w, rank, k);
    if (rank < top) {
      ids[rank] = lane;
      weights[rank] = w * (1.0f / sum);
    }
    mine_rank = rank;
    return;
  }
  mine_rank = 64;
  unsigned taken = 0u;
#pragma unroll
  for (int c = 0; c < PL; ++c)
    if (lane + 64 * c >= E) taken |= 1u << c;
  float first_v = 0.f, sum = 0.f, mine_w = 0.f;
  int mine_e = 0;
  for (int k = 0; k < top; ++k) {
    float best_v = -INFINITY;
    int best_e = 0x7fffffff;
#pragma unroll
    for (int c = 0; c < PL; ++c) {
      const bool free_ = !((taken >> c) & 1u);
      // a value that compares with nothing (NaN) counts as the smallest
      const float x = (v[c] == v[c]) ? v[c] : -INFINITY;
      if (free_ && (best_e == 0x7fffffff || x > best_v)) { best_v = x; best_e = lane + 64 * c; }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float ov = __shfl_xor(best_v, o, IA_WAVE);
      const int oe = __shfl_xor(best_e, o, IA_WAVE);
      if (oe != 0x7fffffff && (best_e == 0x7fffffff || ov > best_v || (ov == best_v && oe < best_e))) {
        best_v = ov;
        best_e = oe;
      }
    }
    if ((best_e & 63) == lane) {
      taken |= 1u << (best_e >> 6);
      if (PL == 1) mine_rank = k;
    }
    if (k == 0) first_v = best_v;
    const float w = expf(best_v - first_v);
    sum += w;
    router_keep(mine_e, mine_w, k, lane, best_e, w, ids, weights);
  }
  router_finish(mine_e, mine_w, top, lane, 1.0f / sum, ids, weights);
}

template <int PL>
__global__ __launch_bounds__(256) void router_topk_kernel(const float* __restrict__ logits,
                                                          const void* __restrict__ bias, int bias_dtype,
                                                          int* __restrict__ ids, float* __restrict__ weights, int N,
                                                          int E, int top) {
  const int n = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (n >= N) return;
  const float* z = logits + (size_t)n * E;
  float v[PL];
#pragma unroll
  for (int c = 0; c < PL; ++c) {
    const int e = lane + 64 * c;
    v[c] = e < E ? z[e] + (bias ? load_as_float(bias, bias_dtype, e) : 0.f) : -INFINITY;
  }
  int rank;
  choose_then_softmax<PL>(v, E, top, lane, ids + (size_t)n * top, weights + (size_t)n * top, rank);
}

extern "C" int ia_router_topk(const float* logits, const void* bias, int bias_dtype, int* ids, float* weights, int N,
                              int E, int top, hipStream_t stream) {
  if (N < 0 || E <= 0 || top <= 0 || top > E) return IA_ERR_BAD_ARG;
  if (E > 64 * RT_PER_LANE) return IA_ERR_UNSUPPORTED;
  if (N == 0) return IA_OK;
  if (E <= 64) router_topk_kernel<1><<<(N + 3) / 4, 256, 0, stream>>>(logits, bias, bias_dtype, ids, weights, N, E, top);
  else if (E <= 256) router_topk_kernel<4><<<(N + 3) / 4, 256, 0, stream>>>(logits, bias, bias_dtype, ids, weights, N, E, top);
  else router_topk_kernel<RT_PER_LANE><<<(N + 3) / 4, 256, 0, stream>>>(logits, bias, bias_dtype, ids, weights, N, E, top);
  IA_LAUNCH_CHECK();
  return IA_OK;
}

#define MOE_MAX_E 1024
// One workgroup.  offsets[e] .. offsets[e + 1] - 1 are the places in perm of expert e's pairs; the order of an
// expert's pairs is whatever the atomics give (no result depends on it).
__global__ __launch_bounds__(1024) void moe_sort_kernel(const int* __restrict__ ids, int* __restrict__ offsets,
                                                        int* __restrict__ perm, int P, int E) {
  __shared__ int cnt[MOE_MAX_E];
  __shared__ int cur[MOE_MAX_E];
  for (int e = threadIdx.x; e < E; e += 1024) cnt[e] = 0;
  __syncthreads();
  for (int p = threadIdx.x; p < P; p += 1024) {
    const int e = ids[p];
    if ((unsigned)e < (unsigned)E) atomicAdd(&cnt[e], 1);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int at = 0;
    for (int e = 0; e < E; ++e) {
      offsets[e] = at;
      cur[e] = at;
      at += cnt[e];
    }
    offsets[E] = at;
  }
  __syncthreads();
  for (int p = threadIdx.x; p < P; p += 1024) {
    const int e = ids[p];
    if ((unsigned)e < (unsigned)E) perm[atomicAdd(&cur[e], 1)] = p;
  }
}

extern "C" int ia_moe_sort(const int* ids, int* offsets, int* perm, int P, int E, hipStream_t stream) {
  if (P < 0 || E <= 0) return IA_ERR_BAD_ARG;
  if (E > MOE_MAX_E) return IA_ERR_UNSUPPORTED;
  moe_sort_kernel<<<1, 1024, 0, stream>>>(ids, offsets, perm, P, E);
  IA_LAUNCH_CHECK();
  return IA_OK;
}

// Tile t of the launch (`rows` pairs a tile, expert by expert): its expert and its first place in perm; false when
// the launch has more tiles than the step needs.  A wave's lanes take an expert each and a prefix sum says whose tile it is:
// walking the experts one after the other took 2 us for 32 of them, in front of every workgroup's first load.
__device__ __forceinline__ bool moe_tile(const int* __restrict__ offsets, int E, int t, int& expert, int& first,
                                         int& last, int rows = TF_T) {
  const int lane = threadIdx.x & 63;
  int seen = 0;
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int e = e0 + lane;
    const int lo = offsets[min(e, E)], hi = offsets[min(e + 1, E)];
    const int tiles = (hi - lo + rows - 1) / rows;           // none beyond the last expert
    int upto = tiles;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(upto, o, IA_WAVE);
      upto += lane >= o ? v : 0;
    }
    const unsigned long long reach = __ballot(t < seen + upto);
    if (reach) {
      const int l = __ffsll(reach) - 1;
      expert = e0 + l;
      first = __builtin_amdgcn_readlane(lo, l) + (t - seen - __builtin_amdgcn_readlane(upto - tiles, l)) * rows;
      last = __builtin_amdgcn_readlane(hi, l);
      return true;
    }
    seen += __builtin_amdgcn_readlane(upto, 63);
  }
  return false;
}
// Tiles of `rows` pairs that P pairs of E experts can need: an expert that has any starts one, and every further `rows` of its
// pairs another.
static inline long moe_most_tiles(int P, int E, int rows) {
  const int some = P < E ? P : E;
  return some + (P - some) / rows;
}

// grid: (tiles of 2 * ff columns, moe_most_tiles).  Wgu [E, 2 ff, W]: row 2 j the gate's row j, row 2 j + 1 up's.
// On the vector ALUs in fp32: the 32-bit path, and bfloat16 rows that cannot be read 16 bytes at a time.
template <typename T>
__global__ __launch_bounds__(256) void moe_gate_up_kernel(const T* __restrict__ x, const T* __restrict__ Wgu,
                                                          T* __restrict__ y, const int* __restrict__ offsets,
                                                          const int* __restrict__ perm, int E, int top, int W,
                                                          int ff, float limit, float alpha, float shift,
                                                          const float* __restrict__ in_w) {
  __shared__ TileFmaLds lds;
  int e, first, last;
  if (!moe_tile(offsets, E, blockIdx.y, e, first, last)) return;
  const int n0 = blockIdx.x * TF_T;
  const int lr = threadIdx.x >> 2;
  const T* a_row = (first + lr < last) ? x + (size_t)(perm[first + lr] / top) * W : nullptr;
  const T* w_row = (n0 + lr < 2 * ff) ? Wgu + ((size_t)e * 2 * ff + n0 + lr) * W : nullptr;
  tile_64(a_row, w_row, W, lds, [&](int i, int j0, const float* v) {
    const int p = first + i;
    if (p >= last) return;
    const float wt = in_w ? in_w[perm[p]] : 1.0f;
#pragma unroll
    for (int j = 0; j < 4; j += 2) {
      const int c = n0 + j0 + j;
      if (c + 1 >= 2 * ff) continue;
      // both products are rounded as a stored tensor would be, then the activation in fp32
      const float g = fminf(wt * to_float(from_float<T>(v[j])), limit);
      const float u = fminf(fmaxf(wt * to_float(from_float<T>(v[j + 1])), -limit), limit);
      y[(size_t)p * ff + (c >> 1)] = from_float<T>(g * (1.0f / (1.0f + expf(-alpha * g))) * (u + shift));
    }
  });
}

// ---- tiles of up to 64 pairs ------------------------------------------------------------------------------------------
// What bounds a step of few pairs is the stream of the chosen experts' weights.  A workgroup of WAVES waves takes 16 rows of
// W a wave and walks K in chunks of 256: W straight from memory to registers, one chunk ahead (each byte of it is used by one
// wave only), the chunk of the pairs' rows through LDS, two stages.  No load stands under a condition; chunks are written
// out in pairs so that no register of a load under way is copied; what lies beyond K is read from the row's end and cleared.
// v_mfma_f32_16x16x32_bf16 with W's rows as its first operand: lane (r = lane % 16, q = lane / 16) ends with four
// consecutive columns 4 q .. 4 q + 3 of row r of the result.
// All workgroups walking K in step read places one row's length apart at the same moment, and where that length is a power
// of two those lie on few memory channels, so every 512 columns start their walk at a chunk of their own (ia_expert_first_chunk) and
// wrap around.  The tile of 128 pairs and the grouped product of gemm_tiles.hip start there too: an element is one chain over K in
// an order that depends on K and its column alone.
// Before, tiles of 32 x 128 in steps of 64 through one LDS stage and all walks from the same start (cold weights,
// gate and up / down, microseconds before and now): 4 of 32 experts of 1,408 x 2,048 22.0 / 15.9 and 12.4 / 7.2; 16 of 16, 32
// tokens, 44.7 / 20.3 and 35.3 / 19.3 (184 MB: 5.2 TB/s); 16 of 20 of 2,432 x 4,096 136 / 56.6 and 108.6 / 56.4 (5.9 and 5.7 TB/s).
#define MS_KC IA_EXPERT_CHUNK
#define MS_LD (MS_KC + 8)     // bf16 of a row in LDS (the padding spreads the banks)

// `x_row(r)`: row r of the tile's pairs, 0 <= r < rows; Wm: the expert's matrix [w_rows, K]; this workgroup's columns
// of the result begin at n0.  Rows of 16-byte alignment, K a multiple of 8.
template <int MT, int ROWS, int WAVES, typename XRow, typename Emit>
__device__ __forceinline__ void moe_stream_tile(const bf16_t* __restrict__ Wm, int w_rows, int n0, int K, int rows,
                                                XRow x_row, uint16_t (*xs)[ROWS][MS_LD], Emit emit) {
  constexpr int T = WAVES * 64, NLD = MS_KC / 32, PIECES = MS_KC / 8;
  constexpr int XPT = MT * 16 * PIECES / T;                  // 16-byte pieces of the pairs' rows a thread brings in
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, q = lane >> 4;
  const int n = n0 + (tid >> 6) * 16;
  const bf16_t* wrow = Wm + (size_t)min(n + r, w_rows - 1) * K;
  const int chunks = (K + MS_KC - 1) / MS_KC, rot = ia_expert_first_chunk(n0, K);
  auto at = [&](int c) {                                     // where chunk c of the walk begins
    const int k = c + rot;
    return (k >= chunks ? k - chunks : k) * MS_KC;
  };
  const bf16_t* xp[XPT];
#pragma unroll
  for (int i = 0; i < XPT; ++i) xp[i] = x_row(min((tid + i * T) / PIECES, rows - 1));
  const int xk = (tid % PIECES) * 8;                         // T is a multiple of PIECES: the same place of every row
  uint4 xr[XPT], w0[NLD], w1[NLD];
  tm_f32x4 acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = tm_f32x4{0.f, 0.f, 0.f, 0.f};
  auto load_x = [&](int c) {
    const int k = min(at(c) + xk, K - 8);
#pragma unroll
    for (int i = 0; i < XPT; ++i) xr[i] = *reinterpret_cast<const uint4*>(xp[i] + k);
  };
  auto store_x = [&](int c) {
    const bool in = at(c) + xk < K;
#pragma unroll
    for (int i = 0; i < XPT; ++i)
      *reinterpret_cast<uint4*>(&xs[c & 1][(tid + i * T) / PIECES][xk]) =
          make_uint4(in ? xr[i].x : 0u, in ? xr[i].y : 0u, in ? xr[i].z : 0u, in ? xr[i].w : 0u);
  };
  auto load_w = [&](int c, uint4 (&w)[NLD]) {
    const int k0 = at(c) + 8 * q;
#pragma unroll
    for (int j = 0; j < NLD; ++j) w[j] = *reinterpret_cast<const uint4*>(wrow + min(k0 + 32 * j, K - 8));
  };
  auto products = [&](int c, uint4 (&w)[NLD]) {
    if (K % MS_KC != 0 && at(c) + MS_KC > K) {
#pragma unroll
      for (int j = 0; j < NLD; ++j)
        if (at(c) + 32 * j + 8 * q >= K) w[j] = make_uint4(0u, 0u, 0u, 0u);
    }
#pragma unroll
    for (int j = 0; j < NLD; ++j)
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const uint4 xv = *reinterpret_cast<const uint4*>(&xs[c & 1][16 * m + r][32 * j + 8 * q]);
        acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(tm_bf16x8, w[j]),
                                                         __builtin_bit_cast(tm_bf16x8, xv), acc[m], 0, 0, 0);
      }
  };
  auto round = [&](int c, uint4 (&w)[NLD], uint4 (&next)[NLD]) {
    load_x(c + 1);
    load_w(c + 1, next);
    __builtin_amdgcn_sched_barrier(0);                       // all of them in front of the first wait for this chunk's W
    products(c, w);
    store_x(c + 1);
    __syncthreads();
  };
  load_x(0);
  load_w(0, w0);
  store_x(0);
  __syncthreads();
  int c = 0;
  for (; c + 2 < chunks; c += 2) {
    round(c, w0, w1);
    round(c + 1, w1, w0);
  }
  if (c + 1 < chunks) {
    round(c, w0, w1);
    products(c + 1, w1);
  } else {
    products(c, w0);
  }
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const float v[4] = {acc[m][0], acc[m][1], acc[m][2], acc[m][3]};
    emit(16 * m + r, n + 4 * q, v);
  }
}

// The tile with as many groups of 16 rows as it has pairs.
template <int ROWS, int WAVES, typename XRow, typename Emit>
__device__ __forceinline__ void moe_stream(const bf16_t* __restrict__ Wm, int w_rows, int n0, int K, int rows, XRow x_row,
                                           uint16_t (*xs)[ROWS][MS_LD], Emit emit) {
  if (rows <= 16) return moe_stream_tile<1, ROWS, WAVES>(Wm, w_rows, n0, K, rows, x_row, xs, emit);
  if (rows <= 32) return moe_stream_tile<2, ROWS, WAVES>(Wm, w_rows, n0, K, rows, x_row, xs, emit);
  if constexpr (ROWS > 32) {
    if (rows <= 48) return moe_stream_tile<3, ROWS, WAVES>(Wm, w_rows, n0, K, rows, x_row, xs, emit);
    moe_stream_tile<4, ROWS, WAVES>(Wm, w_rows, n0, K, rows, x_row, xs, emit);
  }
}

// Which tiles (pairs x columns) take a launch.  Measured with cold weights at 1 to 400 pairs an expert on average, microseconds
// of gate and up / down:
// - up to 10 pairs an expert, tiles of 32: with 64 columns, or with 32 where those make few workgroups, so that more compute
//   units read (4 of 32 experts of 1,408 x 2,048 12.4 / 9.3 with 64 columns and 12.7 / 7.2 with 32, 7 of 32 22.2 / 10.5
//   and 18.4 / 10.5; 16 of 16 with 64 pairs 35.3 / 19.4 and 40.0 / 19.1; 20 of 2,432 x 4,096 with 128 pairs 135 / 73 and 137 / 79);
// - above, tiles of 64, so that an expert's weights are read once again (32 experts of 1,408 x 2,048 at 12 pairs 67.4 / 41.0
//   with 32 and 67.1 / 37.0 with 64);
// - from 24 pairs on with 128 columns, which read the pairs' rows half as often, unless that leaves compute units idle (20 experts of
//   2,432 x 4,096 at 37 pairs 160 / 106 with 64 columns and 148 / 97 with 128; 8 of 2,752 x 2,048 at 47 pairs, 286 and 208
//   workgroups, 31.7 / 26.4 and 29.1 / 37.3);
// - from 56 on tiles of 128 x 256 that share both operands, if they fill the chip (32 experts of 1,408 x 2,048 at 64 pairs
//   109 / 67 with 64 x 128 and 108 / 53 with these; 8 of 2,752 x 2,048, at most 100 workgroups, 35 / 42 and 54 / 66).
enum MoeTile { MOE_32_32, MOE_32_64, MOE_64_64, MOE_64_128, MOE_128_256 };
static inline int moe_tile_rows(MoeTile t) { return t == MOE_128_256 ? 128 : t >= MOE_64_64 ? 64 : 32; }
static inline MoeTile moe_tile_for(int P, int E, int columns) {
  auto groups = [&](int rows, int width) { return (columns + width - 1) / width * moe_most_tiles(P, E, rows); };
  if (P >= 56L * E && groups(128, 256) >= 224) return MOE_128_256;
  if (P >= 24L * E && groups(64, 128) >= 224) return MOE_64_128;
  if (P >= 10L * E) return MOE_64_64;
  return groups(32, 64) > 512 ? MOE_32_64 : MOE_32_32;
}

// Gate and up of one row of the result: four consecutive columns are two of each.  Both products are rounded as a stored tensor
// would be, then the activation in fp32.
__device__ __forceinline__ void moe_gate_up_store(bf16_t* __restrict__ y, int ff, int p, int c0, const float* v, float wt, float limit,
                                                  float alpha, float shift) {
#pragma unroll
  for (int j = 0; j < 4; j += 2) {
    const int c = c0 + j;
    if (c + 1 >= 2 * ff) continue;
    const float g = fminf(wt * to_float(from_float<bf16_t>(v[j])), limit);
    const float u = fminf(fmaxf(wt * to_float(from_float<bf16_t>(v[j + 1])), -limit), limit);
    y[(size_t)p * ff + (c >> 1)] = from_float<bf16_t>(g * (1.0f / (1.0f + expf(-alpha * g))) * (u + shift));
  }
}

// Tiles of 128 pairs x 256 columns (tile_mfma_big): grid (tiles of the 2 ff columns, moe_most_tiles).
__global__ __launch_bounds__(512) void moe_gate_up_big_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ Wgu,
                                                              bf16_t* __restrict__ y, const int* __restrict__ offsets,
                                                              const int* __restrict__ perm, int E, int top, int W,
                                                              int ff, float limit, float alpha, float shift,
                                                              const float* __restrict__ in_w) {
  __shared__ TileBigLds<128, 256> lds;
  int e, first, last;
  if (!moe_tile(offsets, E, blockIdx.y, e, first, last, 128)) return;
  const int n0 = blockIdx.x * 256;
  tile_mfma_big<128, 256>(
      [&](int r) { return x + (size_t)(perm[first + r] / top) * W; },
      [&](int r) { return Wgu + ((size_t)e * 2 * ff + n0 + r) * W; }, last - first, 2 * ff - n0, W, lds,
      [&](int i, int j0, const float* v) {
        const int p = first + i;
        if (p < last) moe_gate_up_store(y, ff, p, n0 + j0, v, in_w ? in_w[perm[p]] : 1.0f, limit, alpha, shift);
      }, ia_expert_first_chunk(n0, W) * (MS_KC / TB_KS));
}

// Tiles of up to ROWS pairs x 16 columns a wave (moe_stream_tile): grid (tiles of the 2 ff columns, moe_most_tiles).
template <int ROWS, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void moe_gate_up_stream_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ Wgu,
                                                                        bf16_t* __restrict__ y, const int* __restrict__ offsets,
                                                                        const int* __restrict__ perm, int E, int top, int W,
                                                                        int ff, float limit, float alpha, float shift,
                                                                        const float* __restrict__ in_w) {
  __shared__ __attribute__((aligned(16))) uint16_t xs[2][ROWS][MS_LD];
  int e, first, last;
  if (!moe_tile(offsets, E, blockIdx.y, e, first, last, ROWS)) return;
  const int rows = min(last - first, ROWS), n0 = blockIdx.x * WAVES * 16;
  const bf16_t* Wm = Wgu + (size_t)e * 2 * ff * W;
  auto x_row = [&](int r) { return x + (size_t)(perm[first + r] / top) * W; };
  auto emit = [&](int i, int c0, const float* v) {
    if (i < rows) moe_gate_up_store(y, ff, first + i, c0, v, in_w ? in_w[perm[first + i]] : 1.0f, limit, alpha, shift);
  };
  moe_stream<ROWS, WAVES>(Wm, 2 * ff, n0, W, rows, x_row, xs, emit);
}

extern "C" int ia_moe_gate_up(const void* x, const void* Wgu, void* y, const int* offsets, const int* perm, int dtype,
                              int P, int E, int top, int W, int ff, float limit, float alpha, float shift,
                              const float* in_weights, hipStream_t stream) {
  if (P < 0 || E <= 0 || top <= 0 || W <= 0 || ff <= 0) return IA_ERR_BAD_ARG;
  if (P == 0) return IA_OK;
  const long tiles = moe_most_tiles(P, E, TF_T);
  const dim3 grid((2 * ff + TF_T - 1) / TF_T, (unsigned)tiles);
  if (tiles > 65535) return IA_ERR_UNSUPPORTED;
  if (dtype == IA_F32)
    moe_gate_up_kernel<float><<<grid, 256, 0, stream>>>((const float*)x, (const float*)Wgu, (float*)y, offsets,
                                                               perm, E, top, W, ff, limit, alpha, shift, in_weights);
  else if (dtype == IA_BF16 && tile_rows_aligned(x, W) && tile_rows_aligned(Wgu, W)) {
    const MoeTile tile = moe_tile_for(P, E, 2 * ff);
    const long most = moe_most_tiles(P, E, moe_tile_rows(tile));
    if (most > 65535) return IA_ERR_UNSUPPORTED;
#define IA_GU(kernel, columns, threads)                                                                                \
  kernel<<<dim3((2 * ff + (columns) - 1) / (columns), (unsigned)most), threads, 0, stream>>>(                          \
      (const bf16_t*)x, (const bf16_t*)Wgu, (bf16_t*)y, offsets, perm, E, top, W, ff, limit, alpha, shift, in_weights)
    switch (tile) {
      case MOE_32_32: IA_GU((moe_gate_up_stream_kernel<32, 2>), 32, 128); break;
      case MOE_32_64: IA_GU((moe_gate_up_stream_kernel<32, 4>), 64, 256); break;
      case MOE_64_64: IA_GU((moe_gate_up_stream_kernel<64, 4>), 64, 256); break;
      case MOE_64_128: IA_GU((moe_gate_up_stream_kernel<64, 8>), 128, 512); break;
      case MOE_128_256: IA_GU(moe_gate_up_big_kernel, 256, 512); break;
    }
#undef IA_GU
  }
  else if (dtype == IA_BF16)
    moe_gate_up_kernel<bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)x, (const bf16_t*)Wgu, (bf16_t*)y,
                                                                offsets, perm, E, top, W, ff, limit, alpha, shift, in_weights);
  else
    return IA_ERR_BAD_ARG;
  IA_LAUNCH_CHECK();
  return IA_OK;
}

// grid: (tiles of W columns, moe_most_tiles).  Wd [E, W, ff]; parts [top, N, W] fp32.
template <typename T>
__global__ __launch_bounds__(256) void moe_down_kernel(const T* __restrict__ y, const T* __restrict__ Wd,
                                                       float* __restrict__ parts, const float* __restrict__ weights,
                                                       const int* __restrict__ offsets, const int* __restrict__ perm,
                                                       int E, int top, int N, int W, int ff) {
  __shared__ TileFmaLds lds;
  int e, first, last;
  if (!moe_tile(offsets, E, blockIdx.y, e, first, last)) return;
  const int n0 = blockIdx.x * TF_T;
  const int lr = threadIdx.x >> 2;
  const T* a_row = (first + lr < last) ? y + (size_t)(first + lr) * ff : nullptr;
  const T* w_row = (n0 + lr < W) ? Wd + ((size_t)e * W + n0 + lr) * ff : nullptr;
  tile_64(a_row, w_row, ff, lds, [&](int i, int j0, const float* v) {
    const int p = first + i;
    if (p >= last) return;
    const int pair = perm[p];
    const int token = pair / top, choice = pair - token * top;
    const float wt = weights ? weights[pair] : 1.0f;
    float* o = parts + ((size_t)choice * N + token) * W;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = n0 + j0 + j;
      if (c < W) o[c] = to_float(from_float<T>(v[j])) * wt;
    }
  });
}

// One row of the result times the pair's weight, the product rounded as a stored tensor would be.
__device__ __forceinline__ void moe_down_store(float* __restrict__ parts, const float* __restrict__ weights, int pair, int top, int N,
                                               int W, int c0, const float* v) {
  const int token = pair / top, choice = pair - token * top;
  const float wt = weights ? weights[pair] : 1.0f;
  float* o = parts + ((size_t)choice * N + token) * W;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (c0 + j < W) o[c0 + j] = to_float(from_float<bf16_t>(v[j])) * wt;
}

__global__ __launch_bounds__(512) void moe_down_big_kernel(const bf16_t* __restrict__ y, const bf16_t* __restrict__ Wd,
                                                           float* __restrict__ parts, const float* __restrict__ weights,
                                                           const int* __restrict__ offsets, const int* __restrict__ perm,
                                                           int E, int top, int N, int W, int ff) {
  __shared__ TileBigLds<128, 256> lds;
  int e, first, last;
  if (!moe_tile(offsets, E, blockIdx.y, e, first, last, 128)) return;
  const int n0 = blockIdx.x * 256;
  tile_mfma_big<128, 256>(
      [&](int r) { return y + (size_t)(first + r) * ff; },
      [&](int r) { return Wd + ((size_t)e * W + n0 + r) * ff; }, last - first, W - n0, ff, lds,
      [&](int i, int j0, const float* v) {
        if (first + i < last) moe_down_store(parts, weights, perm[first + i], top, N, W, n0 + j0, v);
      }, ia_expert_first_chunk(n0, ff) * (MS_KC / TB_KS));
}

template <int ROWS, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void moe_down_stream_kernel(const bf16_t* __restrict__ y, const bf16_t* __restrict__ Wd,
                                                                     float* __restrict__ parts, const float* __restrict__ weights,
                                                                     const int* __restrict__ offsets, const int* __restrict__ perm,
                                                                     int E, int top, int N, int W, int ff) {
  __shared__ __attribute__((aligned(16))) uint16_t xs[2][ROWS][MS_LD];
  int e, first, last;
  if (!moe_tile(offsets, E, blockIdx.y, e, first, last, ROWS)) return;
  const int rows = min(last - first, ROWS), n0 = blockIdx.x * WAVES * 16;
  const bf16_t* Wm = Wd + (size_t)e * W * ff;
  auto y_row = [&](int r) { return y + (size_t)(first + r) * ff; };
  auto emit = [&](int i, int c0, const float* v) {
    if (i < rows) moe_down_store(parts, weights, perm[first + i], top, N, W, c0, v);
  };
  moe_stream<ROWS, WAVES>(Wm, W, n0, ff, rows, y_row, xs, emit);
}

extern "C" int ia_moe_down(const void* y, const void* Wd, float* parts, const float* weights, const int* offsets,
                           const int* perm, int dtype, int N, int E, int top, int W, int ff, hipStream_t stream) {
  if (N < 0 || E <= 0 || top <= 0 || W <= 0 || ff <= 0) return IA_ERR_BAD_ARG;
  if (N == 0) return IA_OK;
  const int P = N * top;
  const long tiles = moe_most_tiles(P, E, TF_T);
  const dim3 grid((W + TF_T - 1) / TF_T, (unsigned)tiles);
  if (tiles > 65535) return IA_ERR_UNSUPPORTED;
  if (dtype == IA_F32)
    moe_down_kernel<float><<<grid, 256, 0, stream>>>((const float*)y, (const float*)Wd, parts, weights, offsets,
                                                            perm, E, top, N, W, ff);
  else if (dtype == IA_BF16 && tile_rows_aligned(y, ff) && tile_rows_aligned(Wd, ff)) {
    const MoeTile tile = moe_tile_for(P, E, W);
    const long most = moe_most_tiles(P, E, moe_tile_rows(tile));
    if (most > 65535) return IA_ERR_UNSUPPORTED;
#define IA_DN(kernel, columns, threads)                                                                                     \
  kernel<<<dim3((W + (columns) - 1) / (columns), (unsigned)most), threads, 0, stream>>>(                                    \
      (const bf16_t*)y, (const bf16_t*)Wd, parts, weights, offsets, perm, E, top, N, W, ff)
    switch (tile) {
      case MOE_32_32: IA_DN((moe_down_stream_kernel<32, 2>), 32, 128); break;
      case MOE_32_64: IA_DN((moe_down_stream_kernel<32, 4>), 64, 256); break;
      case MOE_64_64: IA_DN((moe_down_stream_kernel<64, 4>), 64, 256); break;
      case MOE_64_128: IA_DN((moe_down_stream_kernel<64, 8>), 128, 512); break;
      case MOE_128_256: IA_DN(moe_down_big_kernel, 256, 512); break;
    }
#undef IA_DN
  }
  else if (dtype == IA_BF16)
    moe_down_kernel<bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)y, (const bf16_t*)Wd, parts, weights,
                                                             offsets, perm, E, top, N, W, ff);
  else
    return IA_ERR_BAD_ARG;
  IA_LAUNCH_CHECK();
  return IA_OK;
}

// ---- the experts of a step of many rows by the grouped form of the LDS-tiled product (ia_gemm_tiles_grouped) ----------
// The tokens' rows are first brought into the order of the sort (an expert's rows one after the other), the two
// products run expert by expert over those rows, and the activation and the routing weight are passes of their own:
//   ia_moe_gather   xs[p, :] = x[perm[p] / top, :]
//   ia_moe_glu      y[p, j] = g sigmoid(alpha g) (u + shift), g = min(gu[p, 2 j], limit), u = clamp(gu[p, 2 j + 1], +-limit)
//   ia_moe_scatter  parts[choice, token, :] = float(o[p, :]) * weights[perm[p]], for the places p below *last (nullable:
//                   all of them)
// All three in bfloat16 with rows that are read 16 bytes at a time.
__global__ __launch_bounds__(256) void moe_gather_kernel(const uint4* __restrict__ x, const int* __restrict__ perm,
                                                         uint4* __restrict__ xs, int top, int pieces) {
  const int p = blockIdx.x;
  const uint4* src = x + (size_t)(perm[p] / top) * pieces;
  uint4* dst = xs + (size_t)p * pieces;
  for (int i = threadIdx.x; i < pieces; i += 256) dst[i] = src[i];
}

extern "C" int ia_moe_gather(const void* x, const int* perm, void* xs, int P, int top, int W, hipStream_t stream) {
  if (P < 0 || top <= 0 || W <= 0) return IA_ERR_BAD_ARG;
  if ((W & 7) || ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(xs)) & 15)) return IA_ERR_UNSUPPORTED;
  if (P == 0) return IA_OK;
  moe_gather_kernel<<<P, 256, 0, stream>>>((const uint4*)x, perm, (uint4*)xs, top, W / 8);
  IA_LAUNCH_CHECK();
  return IA_OK;
}

__global__ __launch_bounds__(256) void moe_glu_kernel(const uint4* __restrict__ gu, uint2* __restrict__ y, size_t n4,
                                                      float limit, float alpha, float shift, const int* __restrict__ perm,
                                                      const float* __restrict__ in_w, int quads) {
  const size_t stride = (size_t)gridDim.x * 256;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += stride) {
    const uint4 v = gu[i];
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    float o[4];
    const float wt = in_w ? in_w[perm[i / quads]] : 1.0f;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float g = fminf(wt * __uint_as_float(w[k] << 16), limit);
      const float u = fminf(fmaxf(wt * __uint_as_float(w[k] & 0xffff0000u), -limit), limit);
      o[k] = g * (1.0f / (1.0f + expf(-alpha * g))) * (u + shift);
    }
    uint2 r;
    r.x = two_bf16_bits(o[0], o[1]);
    r.y = two_bf16_bits(o[2], o[3]);
    y[i] = r;
  }
}

extern "C" int ia_moe_glu(const void* gu, void* y, int P, int ff, float limit, float alpha, float shift, const int* perm,
                          const float* in_weights, hipStream_t stream) {
  if (P < 0 || ff <= 0 || (in_weights && !perm)) return IA_ERR_BAD_ARG;
  if ((ff & 3) || ((reinterpret_cast<uintptr_t>(gu) | reinterpret_cast<uintptr_t>(y)) & 15)) return IA_ERR_UNSUPPORTED;
  const size_t n4 = (size_t)P * ff / 4;
  if (n4 == 0) return IA_OK;
  const unsigned grid = (unsigned)((n4 + 255) / 256 < 65536 ? (n4 + 255) / 256 : 65536);
  moe_glu_kernel<<<grid, 256, 0, stream>>>((const uint4*)gu, (uint2*)y, n4, limit, alpha, shift, perm, in_weights, ff / 4);
  IA_LAUNCH_CHECK();
  return IA_OK;
}

__global__ __launch_bounds__(256) void moe_scatter_kernel(const uint4* __restrict__ o, const int* __restrict__ perm,
                                                          const float* __restrict__ weights, float* __restrict__ parts,
                                                          const int* __restrict__ last, int N, int top, int W) {
  const int p = blockIdx.x;
  if (last && p >= *last) return;                  // a pair that went to no expert with tensors
  const int pair = perm[p];
  const int token = pair / top, choice = pair - token * top;
  const float wt = weights ? weights[pair] : 1.0f;
  const uint4* src = o + (size_t)p * (W / 8);
  float4* dst = reinterpret_cast<float4*>(parts + ((size_t)choice * N + token) * W);
  for (int i = threadIdx.x; i < W / 8; i += 256) {
    const uint4 v = src[i];
    dst[2 * i] = make_float4(__uint_as_float(v.x << 16) * wt, __uint_as_float(v.x & 0xffff0000u) * wt,
                             __uint_as_float(v.y << 16) * wt, __uint_as_float(v.y & 0xffff0000u) * wt);
    dst[2 * i + 1] = make_float4(__uint_as_float(v.z << 16) * wt, __uint_as_float(v.z & 0xffff0000u) * wt,
                                 __uint_as_float(v.w << 16) * wt, __uint_as_float(v.w & 0xffff0000u) * wt);
  }
}

extern "C" int ia_moe_scatter(const void* o, const int* perm, const float* weights, float* parts, const int* last, int N,
                              int top, int W, hipStream_t stream) {
  if (N < 0 || top <= 0 || W <= 0) return IA_ERR_BAD_ARG;
  if ((W & 7) || ((reinterpret_cast<uintptr_t>(o) | reinterpret_cast<uintptr_t>(parts)) & 15)) return IA_ERR_UNSUPPORTED;
  if (N == 0) return IA_OK;
  moe_scatter_kernel<<<N * top, 256, 0, stream>>>((const uint4*)o, perm, weights, parts, last, N, top, W);
  IA_LAUNCH_CHECK();
  return IA_OK;
}

// ---- experts without a gate, and a router whose choice and weights go by different numbers ----
//   ia_router_softmax_topk   s = softmax(z) over all experts; the `top` largest of s + correction are chosen (the
//                            lowest index among equals); the weights are the chosen s, with `renorm` over their sum
//                            (+ 1e-20).  With `sigmoid` s = sigmoid(z) instead, and without a correction the choice goes
//                            by z itself (large z have equal s in fp32).  With `groups` > 1 the experts form that many groups of neighbours, a group's
//                            score is its largest s + correction, and only experts of the `keep` best groups (the
//                            lowest index among equals) can be chosen;
//   ia_moe_up                per expert, over its pairs' tokens: y = act(Wu x), Wu [E, ff, W]; act by the codes of
//                            ia_activation (2: the erf GELU, 3: the square of relu).
// PL: experts a lane holds (lane, lane + 64, ...).  zv: this lane's logits; scores: 64 PL floats of LDS, this wave's own (read
// with groups only); the rest as for choose_then_softmax.
template <int PL>
__device__ __forceinline__ void softmax_then_choose(const float (&zv)[PL], const void* __restrict__ corr, int corr_dtype, int E, int top,
                                                    int groups, int keep, int renorm, int sigmoid, int lane, float* scores,
                                                    int* ids, float* weights, int& mine_rank) {
  float s[PL], v[PL];
  unsigned taken = 0u;
  float zmax = -INFINITY;
#pragma unroll
  for (int c = 0; c < PL; ++c) {
    const int e = lane + 64 * c;
    s[c] = e < E ? zv[c] : -INFINITY;
    zmax = fmaxf(zmax, s[c]);
    if (e >= E) taken |= 1u << c;
  }
  zmax = wave_max(zmax);
  float total = 0.f;
#pragma unroll
  for (int c = 0; c < PL; ++c) {
    s[c] = (lane + 64 * c) < E ? expf(s[c] - zmax) : 0.f;
    total += s[c];
  }
  total = wave_sum(total);
  const float inv_total = 1.0f / total;
#pragma unroll
  for (int c = 0; c < PL; ++c) {
    const int e = lane + 64 * c;
    if (sigmoid) {
      const float x = e < E ? zv[c] : -INFINITY;
      s[c] = 1.0f / (1.0f + expf(-x));
      v[c] = e < E ? (corr ? s[c] + load_as_float(corr, corr_dtype, e) : x) : -INFINITY;
    } else {
      s[c] *= inv_total;
      v[c] = e < E ? s[c] + (corr ? load_as_float(corr, corr_dtype, e) : 0.f) : -INFINITY;
    }
  }
  if (groups > 1) {
    // each wave works on its own part of LDS: a wave's accesses are in order, no barrier is needed between them
    volatile float* mine = scores;
    const int size = E / groups;
#pragma unroll
    for (int c = 0; c < PL; ++c)
      if (lane + 64 * c < E) mine[lane + 64 * c] = (v[c] == v[c]) ? v[c] : -INFINITY;
    float gs[PL];                        // this lane's groups: lane, lane + 64, ...
#pragma unroll
    for (int c = 0; c < PL; ++c) {
      gs[c] = -INFINITY;
      const int g = lane + 64 * c;
      if (g < groups)
        for (int i = 0; i < size; ++i) gs[c] = fmaxf(gs[c], mine[g * size + i]);
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int c = 0; c < PL; ++c)
      if (lane + 64 * c < groups) mine[lane + 64 * c] = gs[c];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int c = 0; c < PL; ++c) {
      const int e = lane + 64 * c;
      if (e >= E) continue;
      const int g = e / size;
      const float own = mine[g];
      int better = 0;
      for (int i = 0; i < groups; ++i) better += mine[i] > own || (mine[i] == own && i < g);
      if (better >= keep) taken |= 1u << c;
    }
  }
  if (PL == 1 && choose_by_rank(E, top)) {
    const int rank = expert_rank((v[0] == v[0]) ? v[0] : -INFINITY, !(taken & 1u), E, lane);
    float chosen = 0.f;
    for (int k = 0; k < top; ++k) chosen += value_of_rank(s[0], rank, k);
    if (rank < top) {
      ids[rank] = lane;
      weights[rank] = s[0] * (renorm ? 1.0f / (chosen + 1e-20f) : 1.0f);
    }
    mine_rank = rank;
    return;
  }
  mine_rank = 64;
  float sum = 0.f, mine_w = 0.f;
  int mine_e = 0;
  for (int k = 0; k < top; ++k) {
    float best_v = -INFINITY, best_s = 0.f;
    int best_e = 0x7fffffff;
#pragma unroll
    for (int c = 0; c < PL; ++c) {
      const bool free_ = !((taken >> c) & 1u);
      const float x = (v[c] == v[c]) ? v[c] : -INFINITY;
      if (free_ && (best_e == 0x7fffffff || x > best_v)) { best_v = x; best_e = lane + 64 * c; best_s = s[c]; }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float ov = __shfl_xor(best_v, o, IA_WAVE), os = __shfl_xor(best_s, o, IA_WAVE);
      const int oe = __shfl_xor(best_e, o, IA_WAVE);
      if (oe != 0x7fffffff && (best_e == 0x7fffffff || ov > best_v || (ov == best_v && oe < best_e))) {
        best_v = ov;
        best_e = oe;
        best_s = os;
      }
    }
    if ((best_e & 63) == lane) {
      taken |= 1u << (best_e >> 6);
      if (PL == 1) mine_rank = k;
    }
    sum += best_s;
    router_keep(mine_e, mine_w, k, lane, best_e, best_s, ids, weights);
  }
  router_finish(mine_e, mine_w, top, lane, renorm ? 1.0f / (sum + 1e-20f) : 1.0f, ids, weights);
}

template <int PL>
__global__ __launch_bounds__(256) void router_softmax_topk_kernel(const float* __restrict__ logits,
                                                                  const void* __restrict__ corr, int corr_dtype,
                                                                  int* __restrict__ ids, float* __restrict__ weights,
                                                                  int N, int E, int top, int z_stride, int groups,
                                                                  int keep, int renorm, int sigmoid) {
  __shared__ float s_v[4][64 * PL];       // a wave's choice scores, then (in place) its groups' scores
  const int n = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (n >= N) return;
  const float* z = logits + (size_t)n * z_stride;
  float zv[PL];
#pragma unroll
  for (int c = 0; c < PL; ++c) zv[c] = lane + 64 * c < E ? z[lane + 64 * c] : -INFINITY;
  int rank;
  softmax_then_choose<PL>(zv, corr, corr_dtype, E, top, groups, keep, renorm, sigmoid, lane, s_v[threadIdx.x >> 6],
                          ids + (size_t)n * top, weights + (size_t)n * top, rank);
}

extern "C" int ia_router_softmax_topk(const float* logits, const void* corr, int corr_dtype, int* ids, float* weights,
                                      int N, int E, int top, int z_stride, int groups, int keep, int renorm,
                                      int sigmoid, hipStream_t stream) {
  if (N < 0 || E <= 0 || top <= 0 || top > E || z_stride < E || groups < 1 || E % groups || keep < 1 || keep > groups ||
      top > keep * (E / groups) || !logits || !ids || !weights) return IA_ERR_BAD_ARG;
  if (E > 64 * RT_PER_LANE) return IA_ERR_UNSUPPORTED;
  if (N == 0) return IA_OK;
#define IA_RT(PL)                                                                                                        \
  router_softmax_topk_kernel<PL><<<(N + 3) / 4, 256, 0, stream>>>(logits, corr, corr_dtype, ids, weights, N, E, top, z_stride, \
                                                                  groups, keep, renorm, sigmoid)
  if (E <= 64) IA_RT(1);
  else if (E <= 256) IA_RT(4);
  else IA_RT(RT_PER_LANE);
#undef IA_RT
  IA_LAUNCH_CHECK();
  return IA_OK;
}

// ---- a step of few tokens: the parts of the router's product joined, the choices and the sort ---------------------------
// The join of the logits' parts, ia_router_topk or ia_router_softmax_topk and ia_moe_sort are three launches and a few trips to
// memory for some kilobytes.  Up to 16 tokens one workgroup does the lot: all threads join the logits into LDS (the
// parts in the order of their index), a wave a token chooses, and the ids go into the sort from LDS.  With more tokens one compute unit
// takes longer than the launches it saves, and the parts are joined where a wave a token chooses, the sort behind it.  The same
// ids, weights and offsets.  Behind the product's parts, us with a launch each and so: 1 / 16 / 32 / 64 / 128 tokens to 4 of 32 experts
// 6.2 / 6.9 / 7.1 / 7.3 / 7.5 and 3.9 / 5.1 / 5.5 / 5.6 / 5.7 (one workgroup for all of 32 / 64 / 128: 8.4 / 14.5 / 26.4).
#define ROUTE_ONE 16
#define ROUTE_TOKENS 128
#define ROUTE_EXPERTS 64
#define ROUTE_TOP 16
struct RouteArgs {
  const float* parts;        // [splits, N, row]: the logits of the experts (and, with gate, one more per token)
  int splits, row;
  const void* bias;          // the choice's bias or correction (nullable)
  int bias_dtype;
  int* ids;                  // [N, top]
  float* weights;            // [N, top]
  int* offsets;              // [E + 1]
  int* perm;                 // [N * top]
  float* gate;               // nullable: gate[n] = the logit behind the experts'
  int N, E, top, softmax_first, groups, keep, renorm, sigmoid;
};

// Value i of [N, row], its parts added in the order of their index, eight asked for together.
__device__ __forceinline__ float route_logit(const RouteArgs& A, int i) {
  const int values = A.N * A.row;
  float sum = 0.f;
  for (int s0 = 0; s0 < A.splits; s0 += 8) {
    float p[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) p[u] = A.parts[(size_t)min(s0 + u, A.splits - 1) * values + i];
#pragma unroll
    for (int u = 0; u < 8; ++u) sum = s0 + u < A.splits ? sum + p[u] : sum;
  }
  return sum;
}

// Token n's choices; z: this lane's logit (any number beyond the experts).  Returns this lane's expert's place among them.
__device__ __forceinline__ int route_token(const RouteArgs& A, int n, float z, int lane, float* scores) {
  int* ids = A.ids + (size_t)n * A.top;
  float* weights = A.weights + (size_t)n * A.top;
  int rank;
  if (A.softmax_first) {
    const float zv[1] = {lane < A.E ? z : -INFINITY};
    softmax_then_choose<1>(zv, A.bias, A.bias_dtype, A.E, A.top, A.groups, A.keep, A.renorm, A.sigmoid, lane, scores, ids, weights, rank);
  } else {
    const float v[1] = {lane < A.E ? z + (A.bias ? load_as_float(A.bias, A.bias_dtype, lane) : 0.f) : -INFINITY};
    choose_then_softmax<1>(v, A.E, A.top, lane, ids, weights, rank);
  }
  return rank;
}

__global__ __launch_bounds__(1024) void moe_route_kernel(RouteArgs A) {
  __shared__ float z[ROUTE_ONE * (ROUTE_EXPERTS + 1)];
  __shared__ float scores[ROUTE_ONE][ROUTE_EXPERTS];
  __shared__ int chosen[ROUTE_ONE * ROUTE_TOP];
  __shared__ int cnt[ROUTE_EXPERTS], cur[ROUTE_EXPERTS];
  const int tid = threadIdx.x, lane = tid & 63, n = tid >> 6;
  if (tid < A.E) cnt[tid] = 0;
  for (int i = tid; i < A.N * A.row; i += 1024) z[i] = route_logit(A, i);
  __syncthreads();
  if (n < A.N) {
    const float* zn = z + n * A.row;
    const int rank = route_token(A, n, zn[min(lane, A.E - 1)], lane, scores[n]);
    if (rank < A.top) {
      chosen[n * A.top + rank] = lane;
      atomicAdd(&cnt[lane], 1);
    }
    if (A.gate && lane == 0) A.gate[n] = zn[A.E];
  }
  __syncthreads();
  if (n == 0) {
    const int own = lane < A.E ? cnt[lane] : 0;
    int upto = own;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(upto, o, IA_WAVE);
      upto += lane >= o ? v : 0;
    }
    if (lane < A.E) {
      cur[lane] = upto - own;
      A.offsets[lane] = upto - own;
    }
    if (lane == A.E - 1) A.offsets[A.E] = upto;
  }
  __syncthreads();
  for (int p = tid; p < A.N * A.top; p += 1024) A.perm[atomicAdd(&cur[chosen[p]], 1)] = p;
}

__global__ __launch_bounds__(256) void moe_choose_kernel(RouteArgs A) {
  __shared__ float scores[4][ROUTE_EXPERTS];
  const int lane = threadIdx.x & 63, n = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (n >= A.N) return;
  const float z = route_logit(A, n * A.row + min(lane, A.row - 1));
  route_token(A, n, z, lane, scores[threadIdx.x >> 6]);
  if (A.gate && A.E < 64 && lane == A.E) A.gate[n] = z;
  if (A.gate && A.E == 64 && lane == 0) A.gate[n] = route_logit(A, n * A.row + 64);
}

// Whether ia_moe_route takes a step of N tokens.
extern "C" int ia_moe_route_takes(int N, int E, int top) {
  return N >= 1 && N <= ROUTE_TOKENS && E >= 1 && E <= ROUTE_EXPERTS && top >= 1 && top <= ROUTE_TOP && top <= E;
}

// parts: fp32 [splits, N, row], row E, or E + 1 with gate (fp32 [N], nullable): the logit behind the experts' goes there.
// softmax_first != 0: as ia_router_softmax_topk chooses, with bias its correction (nullable); else as ia_router_topk (groups
// 1, keep 1).  ids, weights [N, top], offsets [E + 1], perm [N * top].
extern "C" int ia_moe_route(const float* parts, int splits, int row, const void* bias, int bias_dtype, int* ids, float* weights,
                            int* offsets, int* perm, float* gate, int N, int E, int top, int softmax_first, int groups, int keep,
                            int renorm, int sigmoid, hipStream_t stream) {
  if (N < 0 || E <= 0 || top <= 0 || top > E || splits < 1 || row != E + (gate ? 1 : 0) || groups < 1 || E % groups || keep < 1 ||
      keep > groups || top > keep * (E / groups) || !parts || !ids || !weights || !offsets || !perm) return IA_ERR_BAD_ARG;
  if (N == 0) return IA_OK;
  if (!ia_moe_route_takes(N, E, top)) return IA_ERR_UNSUPPORTED;
  const RouteArgs A{parts, splits, row, bias, bias_dtype, ids, weights, offsets, perm, gate, N, E, top, softmax_first, groups,
                    keep, renorm, sigmoid};
  if (N <= ROUTE_ONE) moe_route_kernel<<<1, 1024, 0, stream>>>(A);
  else moe_choose_kernel<<<(N + 3) / 4, 256, 0, stream>>>(A);
  IA_LAUNCH_CHECK();
  return N <= ROUTE_ONE ? IA_OK : ia_moe_sort(ids, offsets, perm, N * top, E, stream);
}

template <typename T>
__global__ __launch_bounds__(256) void moe_up_kernel(const T* __restrict__ x, const T* __restrict__ Wu, T* __restrict__ y,
                                                     const int* __restrict__ offsets, const int* __restrict__ perm,
                                                     int E, int top, int W, int ff, int act) {
  __shared__ TileFmaLds lds;
  int e, first, last;
  if (!moe_tile(offsets, E, blockIdx.y, e, first, last)) return;
  const int n0 = blockIdx.x * TF_T;
  const int lr = threadIdx.x >> 2;
  const T* a_row = (first + lr < last) ? x + (size_t)(perm[first + lr] / top) * W : nullptr;
  const T* w_row = (n0 + lr < ff) ? Wu + ((size_t)e * ff + n0 + lr) * W : nullptr;
  tile_64(a_row, w_row, W, lds, [&](int i, int j0, const float* v) {
    const int p = first + i;
    if (p >= last) return;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = n0 + j0 + j;
      // the product is rounded as a stored tensor would be, then the activation in fp32
      if (c < ff) y[(size_t)p * ff + c] = from_float<T>(ia_activate(to_float(from_float<T>(v[j])), act));
    }
  });
}

__device__ __forceinline__ void moe_up_store(bf16_t* __restrict__ y, int ff, int p, int c0, const float* v, int act) {
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (c0 + j < ff) y[(size_t)p * ff + c0 + j] = from_float<bf16_t>(ia_activate(to_float(from_float<bf16_t>(v[j])), act));
}

__global__ __launch_bounds__(512) void moe_up_big_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ Wu,
                                                         bf16_t* __restrict__ y, const int* __restrict__ offsets,
                                                         const int* __restrict__ perm, int E, int top, int W, int ff, int act) {
  __shared__ TileBigLds<128, 256> lds;
  int e, first, last;
  if (!moe_tile(offsets, E, blockIdx.y, e, first, last, 128)) return;
  const int n0 = blockIdx.x * 256;
  tile_mfma_big<128, 256>(
      [&](int r) { return x + (size_t)(perm[first + r] / top) * W; },
      [&](int r) { return Wu + ((size_t)e * ff + n0 + r) * W; }, last - first, ff - n0, W, lds,
      [&](int i, int j0, const float* v) {
        if (first + i < last) moe_up_store(y, ff, first + i, n0 + j0, v, act);
      }, ia_expert_first_chunk(n0, W) * (MS_KC / TB_KS));
}

template <int ROWS, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void moe_up_stream_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ Wu,
                                                                   bf16_t* __restrict__ y, const int* __restrict__ offsets,
                                                                   const int* __restrict__ perm, int E, int top, int W, int ff,
                                                                   int act) {
  __shared__ __attribute__((aligned(16))) uint16_t xs[2][ROWS][MS_LD];
  int e, first, last;
  if (!moe_tile(offsets, E, blockIdx.y, e, first, last, ROWS)) return;
  const int rows = min(last - first, ROWS), n0 = blockIdx.x * WAVES * 16;
  const bf16_t* Wm = Wu + (size_t)e * ff * W;
  auto x_row = [&](int r) { return x + (size_t)(perm[first + r] / top) * W; };
  auto emit = [&](int i, int c0, const float* v) {
    if (i < rows) moe_up_store(y, ff, first + i, c0, v, act);
  };
  moe_stream<ROWS, WAVES>(Wm, ff, n0, W, rows, x_row, xs, emit);
}

extern "C" int ia_moe_up(const void* x, const void* Wu, void* y, const int* offsets, const int* perm, int dtype, int P,
                         int E, int top, int W, int ff, int act, hipStream_t stream) {
  if (P < 0 || E <= 0 || top <= 0 || W <= 0 || ff <= 0 || act < 0 || act > 3) return IA_ERR_BAD_ARG;
  if (P == 0) return IA_OK;
  const long tiles = moe_most_tiles(P, E, TF_T);
  const dim3 grid((ff + TF_T - 1) / TF_T, (unsigned)tiles);
  if (tiles > 65535) return IA_ERR_UNSUPPORTED;
  if (dtype == IA_F32)
    moe_up_kernel<float><<<grid, 256, 0, stream>>>((const float*)x, (const float*)Wu, (float*)y, offsets, perm, E, top,
                                                   W, ff, act);
  else if (dtype == IA_BF16 && tile_rows_aligned(x, W) && tile_rows_aligned(Wu, W)) {
    const MoeTile tile = moe_tile_for(P, E, ff);
    const long most = moe_most_tiles(P, E, moe_tile_rows(tile));
    if (most > 65535) return IA_ERR_UNSUPPORTED;
#define IA_UP(kernel, columns, threads)                                                                                     \
  kernel<<<dim3((ff + (columns) - 1) / (columns), (unsigned)most), threads, 0, stream>>>(                                   \
      (const bf16_t*)x, (const bf16_t*)Wu, (bf16_t*)y, offsets, perm, E, top, W, ff, act)
    switch (tile) {
      case MOE_32_32: IA_UP((moe_up_stream_kernel<32, 2>), 32, 128); break;
      case MOE_32_64: IA_UP((moe_up_stream_kernel<32, 4>), 64, 256); break;
      case MOE_64_64: IA_UP((moe_up_stream_kernel<64, 4>), 64, 256); break;
      case MOE_64_128: IA_UP((moe_up_stream_kernel<64, 8>), 128, 512); break;
      case MOE_128_256: IA_UP(moe_up_big_kernel, 256, 512); break;
    }
#undef IA_UP
  } else if (dtype == IA_BF16)
    moe_up_kernel<bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)x, (const bf16_t*)Wu, (bf16_t*)y, offsets, perm, E,
                                                    top, W, ff, act);
  else
    return IA_ERR_BAD_ARG;
  IA_LAUNCH_CHECK();
  return IA_OK;
}

// ---- what a step adds beside its experts' products ----
//   ia_moe_extras   for every pair whose expert is one of the last, without tensors (ids >= E: an expert whose result is
//                   its input): parts[choice, token, :] = weight * x[token, :]; and for every token, with `shared`: its
//                   result ([splits, shared_rows, W], added in the order of the parts) times sigmoid(gate[token]) into
//                   parts[top, token, :], the part after the choices'.
// grid (N, top (+ 1), pieces of 256 V values of a row); V 4: rows of a multiple of four values, 16 (or 8) bytes an access.
__device__ __forceinline__ void mx_load(const float* p, float (&v)[1]) { v[0] = p[0]; }
__device__ __forceinline__ void mx_load(const bf16_t* p, float (&v)[1]) { v[0] = to_float(p[0]); }
__device__ __forceinline__ void mx_load(const float* p, float (&v)[4]) {
  const float4 t = *reinterpret_cast<const float4*>(p);
  v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
}
__device__ __forceinline__ void mx_load(const bf16_t* p, float (&v)[4]) {
  const uint2 t = *reinterpret_cast<const uint2*>(p);
  v[0] = __uint_as_float(t.x << 16); v[1] = __uint_as_float(t.x & 0xffff0000u);
  v[2] = __uint_as_float(t.y << 16); v[3] = __uint_as_float(t.y & 0xffff0000u);
}
__device__ __forceinline__ void mx_store(float* p, const float (&v)[1], float f) { p[0] = f * v[0]; }
__device__ __forceinline__ void mx_store(float* p, const float (&v)[4], float f) {
  *reinterpret_cast<float4*>(p) = make_float4(f * v[0], f * v[1], f * v[2], f * v[3]);
}

template <typename T, typename TS, int V>
__global__ __launch_bounds__(256) void moe_extras_kernel(const T* __restrict__ x, const int* __restrict__ ids,
                                                         const float* __restrict__ weights, float* __restrict__ parts,
                                                         const TS* __restrict__ shared, int splits, size_t split_stride,
                                                         const float* __restrict__ gate, int gate_stride, int N, int E,
                                                         int top, int W) {
  const int n = blockIdx.x, choice = blockIdx.y, i = (blockIdx.z * 256 + threadIdx.x) * V;
  float* o = parts + ((size_t)choice * N + n) * W + i;
  float v[V];
  if (choice == top) {
    if (i >= W) return;
    const TS* s = shared + (size_t)n * W + i;
    mx_load(s, v);
#pragma unroll 4
    for (int k = 1; k < splits; ++k) {                 // the parts in the order of their index
      float p[V];
      mx_load(s + k * split_stride, p);
#pragma unroll
      for (int e = 0; e < V; ++e) v[e] += p[e];
    }
    mx_store(o, v, gate ? 1.0f / (1.0f + expf(-gate[(size_t)n * gate_stride])) : 1.0f);
    return;
  }
  if (ids[(size_t)n * top + choice] < E || i >= W) return;
  mx_load(x + (size_t)n * W + i, v);
  mx_store(o, v, weights[(size_t)n * top + choice]);
}

// parts: fp32 [top (+ 1 with shared), N, W]; shared (nullable) of shared_dtype; gate (nullable): fp32, token n's logit
// at gate[n gate_stride].
extern "C" int ia_moe_extras(const void* x, int dtype, const int* ids, const float* weights, float* parts, const void* shared,
                             int shared_dtype, int splits, int shared_rows, const float* gate, int gate_stride, int N, int E,
                             int top, int W, hipStream_t stream) {
  if (N < 0 || E < 0 || top <= 0 || W <= 0 || !x || !ids || !weights || !parts || top > 65534 ||
      (shared && (splits < 1 || shared_rows < N)) || (dtype != IA_F32 && dtype != IA_BF16) ||
      (shared && shared_dtype != IA_F32 && shared_dtype != IA_BF16))
    return IA_ERR_BAD_ARG;
  if (N == 0) return IA_OK;
  const bool vec = (W & 3) == 0 && (((uintptr_t)x | (uintptr_t)parts | (uintptr_t)shared) & 15) == 0;
  const dim3 grid(N, top + (shared ? 1 : 0), (W + (vec ? 1024 : 256) - 1) / (vec ? 1024 : 256));
  const size_t stride = (size_t)shared_rows * W;
#define IA_MX_V(T, TS, V)                                                                                                    \
  moe_extras_kernel<T, TS, V><<<grid, 256, 0, stream>>>((const T*)x, ids, weights, parts, (const TS*)shared, splits, stride, \
                                                        gate, gate_stride, N, E, top, W)
#define IA_MX(T, TS)                \
  do {                              \
    if (vec) IA_MX_V(T, TS, 4);     \
    else IA_MX_V(T, TS, 1);         \
  } while (0)
  const bool sf = !shared || shared_dtype == IA_F32;
  if (dtype == IA_F32) {
    if (sf) IA_MX(float, float);
    else return IA_ERR_BAD_ARG;
  } else if (sf) IA_MX(bf16_t, float);
  else IA_MX(bf16_t, bf16_t);
#undef IA_MX
#undef IA_MX_V
  IA_LAUNCH_CHECK();
  return IA_OK;
}

#include "op_call.h"
IA_OP(ia_moe_extras)
IA_OP(ia_router_topk)
IA_OP(ia_moe_sort)
IA_OP(ia_moe_route)
IA_OP(ia_moe_gate_up)
IA_OP(ia_moe_down)
IA_OP(ia_moe_gather)
IA_OP(ia_moe_glu)
IA_OP(ia_moe_scatter)
IA_OP(ia_router_softmax_topk)
IA_OP(ia_moe_up)
