// C[M, N] = X[M, K] * W[N, K]^T in bf16 with fp32 accumulation, for M <= 128: the
// matrix product of a decode step.  The weight is read once from HBM, which is
// what bounds the step.
//
// A workgroup of 4 waves owns 64 rows of W (16 per wave) and a range of K.  K is
// walked in chunks of 256.  The chunk of X (all M rows) is staged in LDS once per
// workgroup and shared by its waves (above 64 rows of X the chunks are 128 long, so that
// two stages of X still leave room for two workgroups on a compute unit); every wave reads its own 16 rows of W
// straight from global memory into registers (each byte of W is used by one wave
// only, so LDS would gain nothing), one chunk ahead of the matrix cores, with
// plain 16-byte loads.  What bounds it is how much of W is under way: the rounds are
// written out in pairs and no load has a condition, for with one the compiler waits for
// everything in every round (the 1B shape's gate+up product, 16,384 x 2,048 at 1 to 16
// rows, 18.6 us that way and 14.0 so, 11.1 at the rate of a large read; 10,240 x 8,192 at
// 1 / 64 rows 37.4 / 50.8 and 34.1 / 41.9; a product that fills the chip several times
// over gains 1 to 7 %).  Products run on v_mfma_f32_16x16x32_bf16 with W as the A
// operand and X^T as the B operand.  Lane (r, q) = (lane % 16, lane / 16) holds,
// for load i of a chunk, the 8 values k = chunk*256 + (4 i + q) * 8 .. +7 of row
// r: the four lanes of a row read 64 contiguous bytes.  X uses the same k for the
// same lane, and a sum over k does not care in which order the matrix core takes
// them.
//
// To fill the GPU when N is small, K is split over blockIdx.y; every split
// writes its fp32 partial tile to a workspace [splits, M, N], and a second kernel
// adds the splits in the order of their index (no atomics: the result does not
// depend on timing), optionally applies SwiGLU to [gate | up] halves, and stores.
// The number of splits depends on N and K only, never on M, so a row's result
// does not depend on what else is in the batch.
//
// K must be a multiple of 8 (16-byte loads); N and M are arbitrary (rows beyond
// them are read from the last valid row and not stored).
#include "common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

#define SK_WAVES 4
#define SK_KC 256               // k per chunk
#define SK_XPAD 8               // bf16 elements of padding per LDS row (spreads the banks)
#define SK_BN (SK_WAVES * 16)   // rows of W per workgroup
#define SK_TARGET_BLOCKS 512    // K is split until the grid has about this many workgroups ...
#define SK_ENOUGH_BLOCKS 256    // ... unless the rows of W alone give one workgroup per compute unit

enum { SK_EPI_NONE = 0, SK_EPI_SWIGLU = 1 };

// Plain loads: non-temporal ones measured 5 to 15 % slower for this access pattern on gfx950.
__device__ __forceinline__ uint4 load_stream_16(const uint16_t* p) { return *reinterpret_cast<const uint4*>(p); }

template <typename TO> __device__ __forceinline__ void store_out(TO* p, float v);
template <> __device__ __forceinline__ void store_out<float>(float* p, float v) { *p = v; }
template <> __device__ __forceinline__ void store_out<uint16_t>(uint16_t* p, float v) { *p = float_to_bf16_bits(v); }

// What becomes of a product's values on their way to memory in place of a launch of its own behind it, 2 us each in a step:
// bf16 results get a bias (fp32, by column) and an activation (ia_activate), fp32 results a factor and a softcap c > 0,
// c tanh(v / c).  Every one of them rounds as the launch that stores in between would.
struct SkFinish {
  const float* bias;
  int act;
  float scale, cap;
};
__device__ __forceinline__ void store_finished(uint16_t* p, float v, int n, const SkFinish& f) {
  float x = bf16_bits_to_float(float_to_bf16_bits(v));
  if (f.bias) x = bf16_bits_to_float(float_to_bf16_bits(x + f.bias[n]));
  *p = float_to_bf16_bits(ia_activate(x, f.act));
}
__device__ __forceinline__ void store_finished(float* p, float v, int, const SkFinish& f) {
  if (f.scale != 1.0f) v *= f.scale;
  if (f.cap > 0.f) v = f.cap * tanhf(v * (1.0f / f.cap));
  *p = v;
}

// part != nullptr: fp32 partial tiles go to part[split, m, n]; else the result goes to C (one split only).
// GLU (one split only): a workgroup takes 32 columns n of the result; waves 0 and 1 multiply with the rows n
// of the first half of W, waves 2 and 3 with the rows N/2 + n of the second half; the halves meet in LDS and
// silu(first) * second goes to C[m, n], n < N/2.
// TILED: W is the copy that tile_weight_kernel lays out, in which the 64 rows x 256 values that a workgroup
// multiplies with in one chunk are 32 KB of consecutive memory, chunk after chunk: every workgroup then reads one
// stretch of memory front to back, where the rows of the matrix as the file holds it lie K values apart.
// PAIRS: the rounds written out in pairs (see the top of the file); else one after the other, with the next chunk's W copied
// over this one's (rounds_alone says where).  The sums and their order are the same.
// FIN: without GLU the values are finished on their way to C (SkFinish).  With it, for a weight whose K is split elsewhere (glu_whole),
// the sums join a total after every sum_chunks chunks of SK_KC and begin again, so that they are no longer chains than the parts that
// they stand in for: one chain over K is twice as far from 64 bits (9,600 x 2,048 4.1e-7 of the result, the parts and so 2.0e-7).
template <int MT, bool GLU, typename TO, int KC, bool TILED, bool PAIRS, bool FIN>
__global__ __launch_bounds__(SK_WAVES * 64) void gemm_skinny_kernel(const uint16_t* __restrict__ X,
                                                                    const uint16_t* __restrict__ W,
                                                                    TO* __restrict__ C, float* __restrict__ part,
                                                                    int M, int N, int K, int chunks_per_split,
                                                                    int sum_chunks, SkFinish finish) {
  // chunks_per_split counts chunks of SK_KC; the kernel walks them in pieces of KC (the sums are the same in
  // the same order either way: a piece is a run of the chunk's matrix instructions)
  constexpr int XROW = KC + SK_XPAD;
  constexpr int NLD = KC / 32;                         // 16-byte loads of W per lane and piece
  constexpr int PER_CHUNK = SK_KC / KC;
  constexpr bool SUMS = GLU && FIN;
  extern __shared__ __attribute__((aligned(16))) char skinny_lds[];
  uint16_t (*xs)[MT * 16][XROW] = reinterpret_cast<uint16_t (*)[MT * 16][XROW]>(skinny_lds);      // two stages
  // the second halves' sums meet the first halves' in the same memory, once the last stage has been read
  f32x4 (*glu_up)[MT][64] = reinterpret_cast<f32x4 (*)[MT][64]>(skinny_lds);
  static_assert(2 * MT * 16 * XROW * 2 >= 2 * MT * 64 * 16, "the stages of X hold the halves' sums");
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, q = lane >> 4;
  const int half = GLU ? wave >> 1 : 0;                // which half of W this wave multiplies with
  const int n_base = GLU ? blockIdx.x * (SK_BN / 2) + (wave & 1) * 16 : blockIdx.x * SK_BN + wave * 16;
  const int split = blockIdx.y;
  const int nchunks = (K + KC - 1) / KC;
  const int c0 = split * chunks_per_split * PER_CHUNK;
  const int c1 = min(nchunks, c0 + chunks_per_split * PER_CHUNK);
  const int NO = GLU ? N / 2 : N;                      // columns of the result

  const int n_row = (n_base + r < NO) ? n_base + r : NO - 1;
  const uint16_t* wrow = W + ((size_t)n_row + (size_t)half * NO) * K;
  // TILED: this lane's row within the workgroup's tiles, which follow each other chunk by chunk
  const int chunks256 = (K + SK_KC - 1) / SK_KC;
  const uint16_t* wtile = W + ((size_t)blockIdx.x * chunks256 * SK_BN + (size_t)(wave * 16 + r)) * SK_KC;
  f32x4 acc[MT], total[SUMS ? MT : 1];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) acc[mt] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int mt = 0; mt < (SUMS ? MT : 1); ++mt) total[mt] = (f32x4){0.f, 0.f, 0.f, 0.f};
  int until_total = sum_chunks;

  // the chunk of X is MT*16 rows of KC values = MT*2*KC/16 pieces of 16 bytes, spread over the 256 threads
  constexpr int XPIECES = MT * 16 * (KC / 8);
  constexpr int XPT = XPIECES / (SK_WAVES * 64);
  static_assert(XPIECES % (SK_WAVES * 64) == 0, "pieces of X must divide over the threads");
  // With PAIRS no load stands under a condition: behind one that some lanes, or some rounds, skip the compiler can no longer count
  // which loads are still under way and waits for all of them.  Pieces beyond K are read from the last valid place and
  // cleared: X on its way to LDS, W in front of the products of that chunk.
  uint4 xreg[XPT];
  auto load_x = [&](int c) {
#pragma unroll
    for (int i = 0; i < XPT; ++i) {
      const int pc = tid + i * SK_WAVES * 64;
      const int row = pc / (KC / 8), kk = (pc % (KC / 8)) * 8;
      const int k = c * KC + kk;
      const uint16_t* x_row = X + (size_t)min(row, M - 1) * K;
      if (PAIRS) xreg[i] = *reinterpret_cast<const uint4*>(x_row + min(k, K - 8));
      else xreg[i] = k < K ? *reinterpret_cast<const uint4*>(x_row + k) : make_uint4(0u, 0u, 0u, 0u);
    }
  };
  auto store_x = [&](int buf, int c) {
#pragma unroll
    for (int i = 0; i < XPT; ++i) {
      const int pc = tid + i * SK_WAVES * 64;
      const int row = pc / (KC / 8), kk = (pc % (KC / 8)) * 8;
      const bool in = !PAIRS || c * KC + kk < K;
      *reinterpret_cast<uint4*>(&xs[buf][row][kk]) =
          make_uint4(in ? xreg[i].x : 0u, in ? xreg[i].y : 0u, in ? xreg[i].z : 0u, in ? xreg[i].w : 0u);
    }
  };
  auto load_w = [&](int c, uint4 (&dst)[NLD]) {
    if (TILED) {
      // piece c of KC values lies in chunk c / PER_CHUNK of 256; the copy is padded with zeros to whole chunks
      const uint16_t* src = wtile + (size_t)(c / PER_CHUNK) * (SK_BN * SK_KC) + (c % PER_CHUNK) * KC;
#pragma unroll
      for (int i = 0; i < NLD; ++i) dst[i] = load_stream_16(src + (i * 4 + q) * 8);
      return;
    }
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      const int k = c * KC + (i * 4 + q) * 8;
      if (PAIRS) dst[i] = load_stream_16(wrow + min(k, K - 8));
      else dst[i] = k < K ? load_stream_16(wrow + k) : make_uint4(0u, 0u, 0u, 0u);
    }
  };

  // Workgroups that walk K in step read rows of W one row's length apart at the same moment, and such addresses
  // crowd on few memory channels where that length is a power of two.  Every tile of rows therefore starts its walk
  // over its chunks at a chunk of its own (a hash of the tile's number) and wraps: the 70B shape's output projection
  // (K = 8,192) 26.3 against 36.1 us at 1 to 16 rows, its QKV product 31.7 against 34.2, the 8B shape's gate+up product
  // from the file's layout 43.4 against 47.5 (41.8 from the copy laid out for this kernel), its head 187 either way;
  // a weight whose rows are no power of two long neither gains nor loses.  The start depends on the tile of rows of W
  // alone, and is counted in chunks of SK_KC, so that the order of the sums does not depend on the length of the pieces.
  const int span = c1 - c0, span_chunks = (span + PER_CHUNK - 1) / PER_CHUNK;
  const int rot = (span_chunks > 1)
                      ? (int)((((unsigned)blockIdx.x * 0x9E3779B1u) >> 8) % (unsigned)span_chunks) * PER_CHUNK : 0;
  auto ce = [&](int c) {
    const int k = c + rot;
    return k >= c1 ? k - span : k;
  };
  const bool ragged = PAIRS && !TILED && K % KC != 0;
  auto products = [&](int c, uint4 (&w)[NLD]) {
    const int buf = (c - c0) & 1;
    if (ragged && ce(c) == nchunks - 1) {
#pragma unroll
      for (int i = 0; i < NLD; ++i)
        if (ce(c) * KC + (i * 4 + q) * 8 >= K) w[i] = make_uint4(0u, 0u, 0u, 0u);
    }
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const uint4 xv = *reinterpret_cast<const uint4*>(&xs[buf][mt * 16 + r][(i * 4 + q) * 8]);
        acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w[i]),
                                                          __builtin_bit_cast(bf16x8, xv), acc[mt], 0, 0, 0);
      }
    }
  };
  // behind everything else that a round does, whose instructions a branch among them would keep from mixing
  auto to_total = [&](int c) {
    if constexpr (SUMS) {
      if ((ce(c) + 1) % PER_CHUNK == 0 || ce(c) == nchunks - 1) --until_total;       // a chunk of SK_KC is done (K may end within one)
      if (until_total == 0) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          total[mt] += acc[mt];
          acc[mt] = (f32x4){0.f, 0.f, 0.f, 0.f};
        }
        until_total = sum_chunks;
      }
    }
  };
  uint4 w0[NLD], w1[NLD];
  // the products of chunk c with its W in `w`, while W of the next chunk comes into `next` and its X to the other stage
  auto round = [&](int c, uint4 (&w)[NLD], uint4 (&next)[NLD]) {
    load_x(ce(c + 1));                                 // X first: the wait for it leaves the loads of W under way
    load_w(ce(c + 1), next);
    __builtin_amdgcn_sched_barrier(0);                 // all of them in front of the first wait for this chunk's W
    products(c, w);
    store_x((c - c0 + 1) & 1, ce(c + 1));
    to_total(c);
    __syncthreads();
  };
  if (!PAIRS && c0 < c1) {
    load_x(ce(c0));
    load_w(ce(c0), w0);
    store_x(0, ce(c0));
    __syncthreads();
    for (int c = c0; c < c1; ++c) {
      const bool more = c + 1 < c1;
      if (more) {
        load_x(ce(c + 1));
        load_w(ce(c + 1), w1);
      }
      products(c, w0);
      if (more) {
        store_x((c - c0 + 1) & 1, ce(c + 1));
#pragma unroll
        for (int i = 0; i < NLD; ++i) w0[i] = w1[i];
      }
      to_total(c);
      __syncthreads();
    }
  }
  if (PAIRS && c0 < c1) {
    load_x(ce(c0));
    load_w(ce(c0), w0);
    store_x(0, ce(c0));
    __syncthreads();
    int c = c0;
    for (; c + 2 < c1; c += 2) {                       // two rounds a turn: no register of a load under way is copied
      round(c, w0, w1);
      round(c + 1, w1, w0);
    }
    if (c + 1 < c1) {
      round(c, w0, w1);
      products(c + 1, w1);
    } else {
      products(c, w0);
    }
  }
  if (GLU) __syncthreads();                            // the halves meet in the memory of the stages
  // lane holds D[i = 4 q + e][j = r]: i counts rows of W in the tile, j rows of X
  const int n = n_base + 4 * q;
  if constexpr (SUMS) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = total[mt] + acc[mt];
  }
  if (GLU) {
    if (half == 1) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) glu_up[wave & 1][mt][lane] = acc[mt];
    }
    __syncthreads();
    if (half == 1) return;
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = mt * 16 + r;
    if (m >= M) continue;
    if (GLU) {
      const f32x4 up = glu_up[wave & 1][mt][lane];
      TO* o = C + (size_t)m * NO + n;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float gt = acc[mt][e];
        if (n + e < NO) store_out<TO>(o + e, gt / (1.0f + expf(-gt)) * up[e]);
      }
    } else if (part) {
      float* o = part + ((size_t)split * M + m) * N + n;
      if (n + 3 < N && (N & 3) == 0) {
        *reinterpret_cast<f32x4*>(o) = acc[mt];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) o[e] = acc[mt][e];
      }
    } else {
      TO* o = C + (size_t)m * N + n;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (n + e >= N) continue;
        if constexpr (FIN) store_finished(o + e, acc[mt][e], n + e, finish);
        else store_out<TO>(o + e, acc[mt][e]);
      }
    }
  }
}

// C[m, n] = sum_s part[s, m, n]                                       (SK_EPI_NONE,   n < N)
// C[m, n] = silu(sum_s part[s, m, n]) * sum_s part[s, m, N/2 + n]      (SK_EPI_SWIGLU, n < N/2)
// PRE parts are asked for together and added in the order of their index (eight loads for two parts cost 128 rows of 15,360 x 5,120
// 1.5 of 58 us).
template <typename TO, int EPI, int PRE>
__global__ __launch_bounds__(256) void gemm_skinny_join_kernel(const float* __restrict__ part, TO* __restrict__ C,
                                                               int M, int N, int splits, SkFinish finish) {
  const int NO = EPI == SK_EPI_SWIGLU ? N / 2 : N;
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (size_t)M * NO) return;
  const int m = (int)(idx / NO), n = (int)(idx - (size_t)m * NO);
  const size_t MN = (size_t)M * N;
  const float* p = part + (size_t)m * N + n;
  float a = 0.f, b = 0.f;
  for (int s0 = 0; s0 < splits; s0 += PRE) {
    float pa[PRE], pb[PRE];
#pragma unroll
    for (int u = 0; u < PRE; ++u) {
      const size_t at = (size_t)min(s0 + u, splits - 1) * MN;
      pa[u] = p[at];
      if (EPI == SK_EPI_SWIGLU) pb[u] = p[at + NO];
    }
#pragma unroll
    for (int u = 0; u < PRE; ++u) {
      a = s0 + u < splits ? a + pa[u] : a;
      if (EPI == SK_EPI_SWIGLU) b = s0 + u < splits ? b + pb[u] : b;
    }
  }
  if (EPI == SK_EPI_SWIGLU) store_out<TO>(C + idx, a / (1.0f + expf(-a)) * b);
  else store_finished(C + idx, a, n, finish);
}

// ---- up to 16 rows, the parts of K in one workgroup ---------------------------------------------------------------
// The same sums as the kernel above and its join, in the same order and so the same bits, in one launch: a workgroup
// takes 16 rows of W (GLU: 16 of each half) and a wave the part of K that a workgroup takes there, chunk after chunk
// from the same start; the parts meet in LDS and are added in the order of their index.  A wave reads its rows of W and
// of X straight into registers, a chunk of 256 values in flight at a time.  X comes from the caches once per 16 rows of
// W instead of once per 64, which is what the rule in whole_k_pays weighs against the join's launch.

template <bool GLU, int WAVES, typename TO>            // WAVES: room for so many, GLU ? 2 * splits : splits are launched
__global__ __launch_bounds__(WAVES * 64) void gemm_skinny_whole_kernel(const uint16_t* __restrict__ X,
                                                                       const uint16_t* __restrict__ W,
                                                                       TO* __restrict__ C, int M, int N, int K,
                                                                       int chunks_per_split, int splits, SkFinish finish) {
  constexpr int NLD = SK_KC / 32;
  __shared__ f32x4 parts[WAVES][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, q = lane >> 4;
  const int half = GLU && wave >= splits ? 1 : 0, split = wave - half * splits;
  const int NO = GLU ? N / 2 : N;
  const int n0 = blockIdx.x * 16;
  const int nchunks = (K + SK_KC - 1) / SK_KC;
  const int c0 = split * chunks_per_split, c1 = min(nchunks, c0 + chunks_per_split), span = c1 - c0;
  const uint16_t* wrow = W + ((size_t)min(n0 + r, NO - 1) + (size_t)half * NO) * K + q * 8;
  const uint16_t* xrow = X + (size_t)min(r, M - 1) * K + q * 8;
  const unsigned tile = (unsigned)(n0 + half * NO) / SK_BN;            // the tile of 64 rows that names the first chunk
  int at = c0 + (span > 1 ? (int)(((tile * 0x9E3779B1u) >> 8) % (unsigned)span) : 0);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int c = 0; c < span; ++c) {
    uint4 w[NLD], x[NLD];
#pragma unroll
    for (int j = 0; j < NLD; ++j) {                    // beyond K the last valid piece is read, and cleared below
      const int k = min(at * SK_KC + 32 * j + 8 * q, K - 8) - 8 * q;
      w[j] = load_stream_16(wrow + k);
      x[j] = *reinterpret_cast<const uint4*>(xrow + k);
    }
    if (K % SK_KC != 0 && at == nchunks - 1) {
#pragma unroll
      for (int j = 0; j < NLD; ++j)
        if (at * SK_KC + 32 * j + 8 * q >= K) w[j] = x[j] = make_uint4(0u, 0u, 0u, 0u);
    }
    if (++at == c1) at = c0;
#pragma unroll
    for (int j = 0; j < NLD; ++j)
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w[j]), __builtin_bit_cast(bf16x8, x[j]),
                                                    acc, 0, 0, 0);
  }
  parts[wave][lane] = acc;
  __syncthreads();
  // the first waves add the parts: value e of the four that a lane of the products holds, wave by wave
  const int n = n0 + 4 * q;
  if (r >= M) return;
  for (int e = wave; e < 4; e += GLU ? 2 * splits : splits) {
    float a = 0.f, b = 0.f;
    for (int v = 0; v < splits; ++v) {
      a += parts[v][lane][e];
      if (GLU) b += parts[splits + v][lane][e];
    }
    if (n + e >= NO) continue;
    if (GLU) store_out<TO>(C + (size_t)r * NO + n + e, a / (1.0f + expf(-a)) * b);
    else store_finished(C + (size_t)r * NO + n + e, a, n + e, finish);
  }
}

// Whether the kernel above takes a split product whose parts are wanted joined.  Measured on an MI355X in a chain of products
// with cold weights over N of 512 to 15,360 and K of 1,024 to 13,824, at 1 to 16 rows: the time of this kernel over that of the
// split product with its join.  It gains a launch (2,048 x 2,048 at 1 / 8 rows 0.88 / 0.96, 4,096 x 4,096 0.85 / 0.96, 12,288 x 4,096
// 0.89 / 0.93) and loses
// - where the last turn of workgroups leaves compute units idle: 5,120 rows of W are 320 workgroups, 1.25 a unit (5,120 x 5,120
//   at 1 / 8 rows 1.12 / 1.31, 5,120 x 13,824 1.38 / 1.63), 10,240 are 2.5 (10,240 x 8,192 1.14 / 1.27, x 4,096 0.89 / 1.05);
// - where the reads of X weigh more than a launch: 4,096 x 8,192 at 4 / 12 rows 0.94 / 1.14, 8,192 x 6,144 at 4 / 8 0.97 / 1.05;
// - with few workgroups and more than a chunk a wave (2,048 x 8,192 1.19 / 1.39), or many rows (512 x 2,048 at 4 / 8 0.97 / 1.03);
// - where the chunks do not deal out evenly over more than four waves, which then wait for the longest;
// - with both halves, whose X it reads twice, from nine rows on, with more than six parts (4,096 x 2,048 in eight 1.05 / 1.14) and
//   with few workgroups (2,048 x 2,048 1.31; 5,632 x 2,048 0.88 / 0.99, 13,824 x 2,048 at 1 / 4 0.92 / 0.97).
static bool whole_k_pays(int M, int N, int K, int splits, bool glu) {
  if (M > 16 || splits > 8) return false;
  const int nchunks = (K + SK_KC - 1) / SK_KC, cps = (nchunks + splits - 1) / splits;
  const int groups = ((glu ? N / 2 : N) + 15) / 16, turns = (groups + 255) / 256;
  const int full = groups <= 256 ? 100 : groups * 100 / (turns * 256);     // how much of the chip the turns fill, in per cent
  if (glu) return N % 32 == 0 && K <= 2048 && M <= 8 && splits <= 6 && groups >= 128 && (long)M * N <= 45056;
  if (N < 512 || (splits > 4 && nchunks % splits != 0) || (long)M * N > 98304) return false;
  if (groups < 160) return cps == 1 && (K <= 1024 || M <= (N >= 2048 ? 12 : splits <= 6 ? 8 : 4));
  if (full < 70 && K > 2048) return false;
  if (full < 99 && ((splits >= 5 && cps >= 4) || (splits == 3 && cps > 8))) return false;
  return (long)M * K <= (full < 70 ? 8192 : full < 99 ? 16384 : groups < 768 ? 32768 : 65536);
}

// ---- up to 32 rows, the parts of K in one workgroup behind X in LDS ---------------------------------------------------
// The same sums in the same order again.  A workgroup takes `groups` times 16 rows of W (GLU: of each half) with a wave for each 16 and
// part of K, so that the matrix's rows fill one turn of the compute units; all of X goes to LDS once, straight from memory, while every
// wave's first two chunks of W are under way, and a chunk's registers are asked for again as soon as they are free.  What bounds it: the
// stream of W behind the launch and the first trip to memory (9,216 x 2,048, 6.2 us at the rate of a large read, at 8 / 16 / 32 rows 12.6 / 13.0 /
// 15.0 us with the kernels above and the join, 10.8 / 11.2 / 13.4 so; 12,288 x 4,096 at 16 rows, 16.6, 25.5 and 21.8; 5,376 x 2,048 with the
// activation at 32 rows, 3.6, 11.2 and 10.1).
typedef __attribute__((address_space(3))) void* sk_lds_ptr;
typedef const __attribute__((address_space(1))) void* sk_global_ptr;
#define SK_STAGED_LDS (160 * 1024)
#define SK_STAGED_WAVES 16

template <bool GLU, int MT, typename TO>
__global__ __launch_bounds__(SK_STAGED_WAVES * 64) void gemm_skinny_staged_kernel(const uint16_t* __restrict__ X,
                                                                                  const uint16_t* __restrict__ W,
                                                                                  TO* __restrict__ C, int M, int N, int K,
                                                                                  int chunks_per_split, int splits, int groups,
                                                                                  SkFinish finish) {
  constexpr int NLD = SK_KC / 32;
  extern __shared__ __attribute__((aligned(16))) char staged_lds[];
  const int tid = threadIdx.x, lane = tid & 63, waves = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q = lane >> 4;
  // strips of 16 rows of W: the groups of the first half, then those of the second
  const int split = wave % splits, strip = wave / splits, half = GLU && strip >= groups ? 1 : 0, group = strip - half * groups;
  const int NO = GLU ? N / 2 : N;
  const int n0 = (blockIdx.x * groups + group) * 16;
  const int nchunks = K / SK_KC;
  const int c0 = split * chunks_per_split, c1 = min(nchunks, c0 + chunks_per_split), span = c1 - c0;
  const uint16_t* wrow = W + ((size_t)min(n0 + r, NO - 1) + (size_t)half * NO) * K + q * 8;
  const unsigned tile = (unsigned)(min(n0, NO - 1) + half * NO) / SK_BN;           // the tile of 64 rows that names the first chunk
  const int rot = span > 1 ? (int)(((tile * 0x9E3779B1u) >> 8) % (unsigned)span) : 0;
  const auto chunk = [&](int c) {
    const int k = c0 + rot + min(c, span - 1);
    return k >= c1 ? k - span : k;
  };
  uint4 w0[NLD], w1[NLD];
  const auto load_w = [&](int c, uint4 (&dst)[NLD]) {
    const uint16_t* src = wrow + chunk(c) * SK_KC;
#pragma unroll
    for (int j = 0; j < NLD; ++j) dst[j] = load_stream_16(src + 32 * j);
  };
  load_w(0, w0);
  load_w(1, w1);
  __builtin_amdgcn_sched_barrier(0);                   // in front of X, whose wait is for all of them
  // rows of X with 16 bytes of padding between them, 1,024 bytes a load of a wave
  const int stride = K * 2 + 16, pieces = K / 512;
  for (int p = wave; p < MT * 16 * pieces; p += waves) {
    const int row = p / pieces, at = p - row * pieces;
    __builtin_amdgcn_global_load_lds((sk_global_ptr)(X + (size_t)min(row, M - 1) * K + at * 512 + lane * 8),
                                     (sk_lds_ptr)(staged_lds + row * stride + at * 1024), 16, 0, 0);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  f32x4 acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) acc[mt] = (f32x4){0.f, 0.f, 0.f, 0.f};
  const auto products = [&](int c, const uint4 (&w)[NLD]) {
    const char* x = staged_lds + r * stride + (chunk(c) * SK_KC + q * 8) * 2;
#pragma unroll
    for (int j = 0; j < NLD; ++j)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const uint4 xv = *reinterpret_cast<const uint4*>(x + mt * 16 * stride + j * 64);
        acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w[j]), __builtin_bit_cast(bf16x8, xv), acc[mt], 0, 0, 0);
      }
  };
  for (int c = 0; c < span; c += 2) {
    products(c, w0);
    if (c + 2 < span) load_w(c + 2, w0);
    if (c + 1 < span) products(c + 1, w1);
    if (c + 3 < span) load_w(c + 3, w1);
  }
  __syncthreads();                                     // the parts meet in the memory of X
  f32x4(*parts)[64] = reinterpret_cast<f32x4(*)[64]>(staged_lds);                  // [wave MT + tile of rows of X]
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) parts[wave * MT + mt][lane] = acc[mt];
  __syncthreads();
  for (int t = wave; t < groups * MT; t += waves) {    // a wave adds the parts of a tile of 16 x 16, in the order of their index
    const int g = t / MT, mt = t - g * MT, m = mt * 16 + r, n = (blockIdx.x * groups + g) * 16 + 4 * q;
    f32x4 a = {0.f, 0.f, 0.f, 0.f}, b = {0.f, 0.f, 0.f, 0.f};
    for (int v = 0; v < splits; ++v) {
      a += parts[(g * splits + v) * MT + mt][lane];
      if (GLU) b += parts[((groups + g) * splits + v) * MT + mt][lane];
    }
    if (m >= M) continue;
    TO* o = C + (size_t)m * NO + n;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (n + e >= NO) continue;
      if (GLU) store_out<TO>(o + e, a[e] / (1.0f + expf(-a[e])) * b[e]);
      else store_finished(o + e, a[e], n + e, finish);
    }
  }
}

static size_t staged_lds_bytes(int M, int K) { return (size_t)((M + 15) / 16) * 16 * (K * 2 + 16); }

// How many groups of 16 rows of W a workgroup of the kernel above takes of a split product whose parts are wanted joined, or 0: not that
// kernel.  As many as fill one turn of the compute units.  Measured with cold weights over N of 2,816 to 15,360 and K of 512 to 4,096 at 1 to 32
// rows, its time over that of the kernels above with their join: it gains where a wave has two chunks and more, so that they are under way
// together, and
// - three groups a workgroup (8,193 to 12,288 rows of W), or four of K up to 2,560: 0.82 to 0.99 from four rows on (9,216 x 2,048 at 1 / 4 / 8 /
//   16 / 32 rows 0.95 / 0.90 / 0.85 / 0.87 / 0.89, 12,288 x 4,096 at 4 / 16 0.97 / 0.85; 15,360 x 4,096 at 4 / 16 1.00 / 0.96);
// - two groups with K up to 2,560: from eight rows on (6,144 x 2,048 at 4 / 8 / 32 0.95 / 0.90 / 0.87, 8,192 x 2,048 at 8 / 12 1.01 / 0.96), while
//   5,120 x 4,096 in six parts takes 1.13 to 1.15 and 8,192 x 3,072 0.98 to 1.09;
// - one group with K from 2,560 on: from twelve rows on (4,096 x 2,560 / 3,072 / 4,096 at 8 1.08 / 1.05 / 0.97, at 16 0.77 / 0.87 / 0.96);
// - with the activation one group and up to five parts, K from 1,536 on: from eight rows on (5,376 x 2,048 at 1 / 4 / 8 / 32 0.99 / 0.92 / 0.88 /
//   0.89, 8,192 x 2,560 0.85 at 8; in six parts 5,376 x 3,072 1.06; two groups 9,472 x 2,048 1.00, x 4,096 1.05).
// A single chunk a wave leaves it 1.0 to 1.4 (4,096 x 2,048 in eight parts 1.31 at 8 rows).
static int staged_groups(int M, int N, int K, int splits, bool glu) {
  if (M > 32 || K % 512 != 0 || staged_lds_bytes(M, K) > SK_STAGED_LDS) return 0;
  const int chunks = (K / SK_KC + splits - 1) / splits, tiles = ((glu ? N / 2 : N) + 15) / 16, groups = (tiles + 255) / 256;
  if (chunks < 2 || (glu ? 2 : 1) * groups * splits > SK_STAGED_WAVES) return 0;
  // (a strip of the second half lies in one tile of 64 rows, whose walk over K has one start, where N is a multiple of 32)
  if (glu) return N % 32 == 0 && groups == 1 && splits <= 5 && tiles > 128 && K >= 1536 && M >= 8 ? 1 : 0;
  if (groups == 3 || (groups == 4 && K <= 2560)) return M >= 4 ? groups : 0;
  if (groups == 2) return K <= 2560 && M >= (N <= 7680 ? 8 : 12) ? 2 : 0;
  return groups == 1 && tiles > 128 && K >= 2560 && M >= 12 ? 1 : 0;
}

template <bool GLU, int MT, typename TO>
static int launch_staged(const uint16_t* x, const uint16_t* w, TO* c, int M, int N, int K, int splits, int groups,
                         const SkFinish& finish, hipStream_t stream) {
  static bool allowed = false;      // more than 64 KB of LDS has to be asked for, once per kernel
  if (!allowed) {
    const hipError_t e = hipFuncSetAttribute((const void*)gemm_skinny_staged_kernel<GLU, MT, TO>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, SK_STAGED_LDS);
    if (e != hipSuccess) return (int)e;
    allowed = true;
  }
  const int waves = (GLU ? 2 : 1) * groups * splits, cps = (K / SK_KC + splits - 1) / splits, NO = GLU ? N / 2 : N;
  const size_t rows = staged_lds_bytes(M, K), parts = (size_t)waves * MT * 64 * sizeof(f32x4);
  gemm_skinny_staged_kernel<GLU, MT, TO><<<(NO + 16 * groups - 1) / (16 * groups), waves * 64, rows > parts ? rows : parts, stream>>>(
      x, w, c, M, N, K, cps, splits, groups, finish);
  IA_LAUNCH_CHECK();
  return IA_OK;
}

// Shapes whose number of splits was measured (ia_gemm_skinny_set_splits, filled from a table when the library is
// loaded): few entries, looked up per launch.
struct KnownSplits { int N, K, splits; };
static KnownSplits g_known_splits[64];
static int g_known_count = 0;

static int split_count(int nchunks, int ks) {
  if (ks > nchunks) ks = nchunks;
  if (ks < 1) ks = 1;
  const int cps = (nchunks + ks - 1) / ks;
  return (nchunks + cps - 1) / cps;
}

static int skinny_splits(int N, int K) {
  const int nb = (N + SK_BN - 1) / SK_BN;
  const int nchunks = (K + SK_KC - 1) / SK_KC;
  for (int i = 0; i < g_known_count; ++i)
    if (g_known_splits[i].N == N && g_known_splits[i].K == K) return split_count(nchunks, g_known_splits[i].splits);
  if (nb >= SK_ENOUGH_BLOCKS) return 1;      // measured: a split costs more than it gains here
  return split_count(nchunks, (SK_TARGET_BLOCKS + nb - 1) / nb);
}

// Whether both halves of [gate | up] take all of K in every workgroup, activation included, although K of a weight [N, K] is split:
// a split product with this use has to be joined in a launch of its own, which is worth more than full compute units from some
// 150 workgroups on, unless the parts fill two turns of the compute units and no more: 150 in three parts (K of 1,025 to 1,536), and, with
// longer K, 160 and 170 in three and four.  From 171 on three parts of each spill into a third turn.  Both sides with cold weights, whole /
// in parts and the join, us at 1, 16, 64 and 128 rows:
//   9,600 x 512 (150 workgroups) 4.9 / 5.4, 4.7 / 6.8, 7.0 / 10.1, 11.4 / 15.2; x 1,024 7.2 / 8.2, 7.4 / 9.1, 10.6 / 14.2, 16.6 / 19.3;
//   x 1,536 10.6 / 11.2, 9.8 / 10.5, 13.7 / 14.5, 20.8 / 19.4 (in parts: 72 and 96 rows lose too); x 2,048 11.3 / 13.1, 11.8 / 13.4, 16.6 / 18.8, 25.5 / 25.3;
//   11,008 x 2,048 12.2 / 13.7, 12.0 / 15.2, 16.8 / 21.2, 25.3 / 27.6; x 4,096 21.0 / 24.3, 23.4 / 25.7, 30.9 / 32.3, 43.6 / 42.8;
//   16,320 x 4,096 26.6 / 28.5, 26.4 / 30.7, 32.7 / 38.5, 47.4 / 52.6; 14,336 x 8,192 46.5 / 49.7, 45.5 / 51.6, 58.0 / 60.9, 83.7 / 81.5.
// Below the line for longer K: 10,752 x 5,120 (168) 28.7 / 26.9, 32.1 / 28.5, 36.5 / 35.3, 51.4 / 47.2; x 14,336 68 / 65, 78 / 67, 97 / 83, 131 / 106.
// What it costs at the line: 171 and 172 workgroups at 128 rows 1.02 to 1.05 of the time in parts (80 rows of 11,008 x 8,192 1.04).
static bool glu_whole(int N, int K) {
  const int nb = (N + SK_BN - 1) / SK_BN, splits = skinny_splits(N, K);
  if (splits == 1) return true;
  for (int i = 0; i < g_known_count; ++i)
    if (g_known_splits[i].N == N && g_known_splits[i].K == K) return false;
  if (K > 2048) return nb >= 171;
  return nb >= 150 && (K <= 1024 || nb * splits > 2 * SK_ENOUGH_BLOCKS);
}

// Says into how many parts (about: the chunks of K are dealt out evenly) the inner dimension of a weight [N, K] is
// split from now on, in place of the rule of sizes.  To be called before the first product of that shape (the
// partial sums' layout follows the number).  Returns 0, or 10001 for bad arguments or a full table.
extern "C" int ia_gemm_skinny_set_splits(int N, int K, int splits) {
  if (N <= 0 || K <= 0 || splits < 1) return IA_ERR_BAD_ARG;
  for (int i = 0; i < g_known_count; ++i)
    if (g_known_splits[i].N == N && g_known_splits[i].K == K) {
      g_known_splits[i].splits = splits;
      return IA_OK;
    }
  if (g_known_count >= 64) return IA_ERR_BAD_ARG;
  g_known_splits[g_known_count++] = KnownSplits{N, K, splits};
  return IA_OK;
}

// Number of K splits the kernel uses for a weight [N, K] (a function of N and K only).
extern "C" int ia_gemm_skinny_splits(int N, int K) { return (N > 0 && K > 0) ? skinny_splits(N, K) : 0; }

template <int MT, bool GLU, typename TO, int KC, bool TILED, bool PAIRS, bool FIN>
static int launch_skinny_one(dim3 grid, const uint16_t* x, const uint16_t* w, TO* c, float* part, int M, int N, int K,
                             int cps, int sums, const SkFinish& finish, hipStream_t stream) {
  constexpr size_t lds = (size_t)2 * MT * 16 * (KC + SK_XPAD) * sizeof(uint16_t);
  static bool allowed = false;      // more than 64 KB of LDS has to be asked for, once per kernel
  if (lds > 65536 && !allowed) {
    hipError_t e = hipFuncSetAttribute((const void*)gemm_skinny_kernel<MT, GLU, TO, KC, TILED, PAIRS, FIN>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return (int)e;
    allowed = true;
  }
  gemm_skinny_kernel<MT, GLU, TO, KC, TILED, PAIRS, FIN><<<grid, SK_WAVES * 64, lds, stream>>>(x, w, c, part, M, N, K, cps, sums, finish);
  IA_LAUNCH_CHECK();
  return IA_OK;
}

// Whether the rounds run one after the other instead of in pairs.  Where one workgroup has a compute unit to itself pairs are 15
// to 30 % faster from 33 rows on, and with many in turn 0 to 13; with two side by side and no third, each covers the other's waits,
// and the registers and selects of the unconditional loads cost more than they give at some numbers of tiles of 16 rows (MT).
// The time one after the other over that in pairs, with 257 to 512 workgroups:
// - K a power of two, without a copy: 32,000 x 2,048 at 40 / 64 rows 0.95 / 0.97, 28,672 x 4,096 with the activation 0.98 / 0.98;
//   not so other K (27,648 x 5,120 1.05 / 1.07, 20,480 x 2,560 1.04);
// - copies at 33 to 64 and 113 to 128 rows (28,672 x 4,096 0.95 / 0.99 and 0.97), not at 65 to 112 (1.09, 0.99, 1.09);
// - rows that do not lie on whole lines of 128 bytes (K % 64): 21,056 x 3,680 at 40 / 72 / 96 / 128 rows 0.96 / 0.96 / 0.94 / 0.93,
//   24,000 x 1,480 0.97 / 0.93 / 0.92 / 0.90; walks of many chunks from 65 rows on only (24,000 x 7,400 1.01 / 0.95 / 0.95 / 0.92);
// - at 97 to 112 rows all without a copy, 0.92 to 0.97.
// With more workgroups: short walks at 49 to 64 rows (50,257 x 592 / 2,048 0.92 / 0.99; 36,864 x 4,608 1.10); and at 81 to 96 rows,
// where the rounds alone leave a compute unit the registers for a third workgroup and pairs do not, up to three workgroups a unit
// of a few chunks each (12,288 / 13,312 / 14,336 x 4,096 in three parts 36.2 / 36.7 / 37.2 us against 38.0 / 39.9 / 40.5; with eight
// chunks and more 0.94 to 0.96 in pairs, with two or three 0.95 to 0.99).
static bool rounds_alone(int MT, bool tiled, int K, unsigned groups, unsigned splits, int chunks) {
  const bool whole_lines = tiled || K % 64 == 0, power_of_two = (K & (K - 1)) == 0;
  if (MT == 4 && splits == 1 && chunks <= 8 && groups > 360) return true;
  if (MT == 6 && splits > 1 && groups > 560 && groups <= 3 * SK_ENOUGH_BLOCKS && chunks >= 4 && chunks <= 6) return true;
  if (groups <= SK_ENOUGH_BLOCKS || groups > 2 * SK_ENOUGH_BLOCKS) return false;
  if (!whole_lines && chunks >= 2 && MT >= 3) return MT >= 5 || chunks <= (MT == 3 ? 20 : 8);
  if (MT == 3) return splits == 1 ? tiled || (power_of_two && groups > 360) : power_of_two && splits >= 4 && chunks >= 8;
  if (MT == 4) return splits == 1 && (tiled || power_of_two) && groups > 360;
  return (MT == 7 && !tiled) || (MT == 8 && tiled);
}

template <bool GLU, typename TO, bool TILED = false, bool FIN = false>
static int launch_skinny(const uint16_t* x, const uint16_t* w, TO* c, float* part, int M, int N, int K, int splits,
                         hipStream_t stream, const SkFinish& finish = SkFinish{nullptr, 0, 1.0f, 0.0f}) {
  const int nchunks = (K + SK_KC - 1) / SK_KC;
  const int cps = (nchunks + splits - 1) / splits;
  const int sum_parts = GLU && FIN ? skinny_splits(N, K) : 1, sums = (nchunks + sum_parts - 1) / sum_parts;
  const int NO = GLU ? N / 2 : N;
  const int cols = GLU ? SK_BN / 2 : SK_BN;           // columns of the result per workgroup
  dim3 grid((NO + cols - 1) / cols, splits);
  // Up to 32 rows and with more than one workgroup a compute unit, pieces of 128: less of W under way in each and the first
  // products sooner (2,048 x 8,192 in 16 parts at 16 / 32 rows 8.4 / 9.4 us with pieces of 256 and 7.9 / 8.7 with 128, the
  // 8B shape's gate+up from its copy 43.9 / 49.0 and 42.4 / 45.1).  One workgroup a compute unit wants the longer pieces
  // (the 1B shape's gate+up 14.5 against 15.4), and so do heads of many workgroups (128,256 x 2,048 91.5 against 92.8).
  // Rows off the lines of 128 bytes want the longer pieces too, once the walk has some chunks (21,056 x 1,480 / 3,680 / 7,400 at 1 row
  // 9 / 3 / 10 % and at 32 rows 11 / 10 / 15 % longer in pieces of 128); a single chunk is done sooner in two (2,176 x 128 with
  // the activation 3.6 us and 3.2; from a copy only if the second holds nothing: 2,848 x 224 3.6 and 3.8).
  const unsigned groups = grid.x * grid.y;
  const bool off_lines = !TILED && K % 64 != 0;
  const bool shorter = (cps == 1 && (!TILED || K <= SK_KC / 2)) || (grid.y > 1 ? !off_lines
                                               : groups > SK_ENOUGH_BLOCKS && groups <= 4 * SK_ENOUGH_BLOCKS &&
                                                     !(off_lines && cps >= 4 && groups > SK_ENOUGH_BLOCKS + 8));
  const bool alone = rounds_alone((M + 15) / 16, TILED, K, groups, grid.y, cps);
  switch ((M + 15) / 16) {
    case 1:
      if (shorter) return launch_skinny_one<1, GLU, TO, SK_KC / 2, TILED, true, FIN>(grid, x, w, c, part, M, N, K, cps, sums, finish, stream);
      return launch_skinny_one<1, GLU, TO, SK_KC, TILED, true, FIN>(grid, x, w, c, part, M, N, K, cps, sums, finish, stream);
    case 2:
      if (shorter) return launch_skinny_one<2, GLU, TO, SK_KC / 2, TILED, true, FIN>(grid, x, w, c, part, M, N, K, cps, sums, finish, stream);
      return launch_skinny_one<2, GLU, TO, SK_KC, TILED, true, FIN>(grid, x, w, c, part, M, N, K, cps, sums, finish, stream);
    case 3:
      if (alone) return launch_skinny_one<3, GLU, TO, SK_KC, TILED, false, FIN>(grid, x, w, c, part, M, N, K, cps, sums, finish, stream);
      return launch_skinny_one<3, GLU, TO, SK_KC, TILED, true, FIN>(grid, x, w, c, part, M, N, K, cps, sums, finish, stream);
    case 4:
      if (alone) return launch_skinny_one<4, GLU, TO, SK_KC, TILED, false, FIN>(grid, x, w, c, part, M, N, K, cps, sums, finish, stream);
      return launch_skinny_one<4, GLU, TO, SK_KC, TILED, true, FIN>(grid, x, w, c, part, M, N, K, cps, sums, finish, stream);
    // above 64 rows: pieces of 128, so that the two stages of X of two workgroups fit a compute unit's LDS
    case 5:
      if (alone) return launch_skinny_one<5, GLU, TO, SK_KC / 2, TILED, false, FIN>(grid, x, w, c, part, M, N, K, cps, sums, finish, stream);
      return launch_skinny_one<5, GLU, TO, SK_KC / 2, TILED, true, FIN>(grid, x, w, c, part, M, N, K, cps, sums, finish, stream);
    case 6:
      if (alone) return launch_skinny_one<6, GLU, TO, SK_KC / 2, TILED, false, FIN>(grid, x, w, c, part, M, N, K, cps, sums, finish, stream);
      return launch_skinny_one<6, GLU, TO, SK_KC / 2, TILED, true, FIN>(grid, x, w, c, part, M, N, K, cps, sums, finish, stream);
    case 7:
      if (alone) return launch_skinny_one<7, GLU, TO, SK_KC / 2, TILED, false, FIN>(grid, x, w, c, part, M, N, K, cps, sums, finish, stream);
      return launch_skinny_one<7, GLU, TO, SK_KC / 2, TILED, true, FIN>(grid, x, w, c, part, M, N, K, cps, sums, finish, stream);
    case 8:
      if (alone) return launch_skinny_one<8, GLU, TO, SK_KC / 2, TILED, false, FIN>(grid, x, w, c, part, M, N, K, cps, sums, finish, stream);
      return launch_skinny_one<8, GLU, TO, SK_KC / 2, TILED, true, FIN>(grid, x, w, c, part, M, N, K, cps, sums, finish, stream);
    default: return IA_ERR_UNSUPPORTED;
  }
}

template <typename TO>
static int launch_join(const float* part, TO* c, int M, int N, int splits, int epilogue, const SkFinish& finish, hipStream_t stream) {
  const int NO = epilogue == SK_EPI_SWIGLU ? N / 2 : N;
  const unsigned grid = (unsigned)(((size_t)M * NO + 255) / 256);
#define SK_JOIN(EPI)                                                                                          \
  do {                                                                                                        \
    if (splits <= 2) gemm_skinny_join_kernel<TO, EPI, 2><<<grid, 256, 0, stream>>>(part, c, M, N, splits, finish);    \
    else if (splits <= 4) gemm_skinny_join_kernel<TO, EPI, 4><<<grid, 256, 0, stream>>>(part, c, M, N, splits, finish); \
    else gemm_skinny_join_kernel<TO, EPI, 8><<<grid, 256, 0, stream>>>(part, c, M, N, splits, finish);                \
  } while (0)
  if (epilogue == SK_EPI_SWIGLU) SK_JOIN(SK_EPI_SWIGLU);
  else SK_JOIN(SK_EPI_NONE);
#undef SK_JOIN
  IA_LAUNCH_CHECK();
  return IA_OK;
}

// X [M, K], W [N, K] bf16, contiguous.  C: bf16 (out_dtype 1) or fp32 (0); [M, N], or [M, N/2] with the SwiGLU
// epilogue.  workspace: fp32, at least ia_gemm_skinny_splits(N, K) * M * N values when that count is above one
// or an epilogue is asked for; may be null otherwise.  C == null: the partial sums are left in the workspace
// as [splits, M, N] for a later kernel to join.
template <bool TILED>
static int skinny_product(const void* X, const void* W, void* C, int out_dtype, int M, int N, int K, int epilogue,
                          float* workspace, size_t workspace_floats, hipStream_t stream,
                          const SkFinish& finish = SkFinish{nullptr, 0, 1.0f, 0.0f}) {
  if (M <= 0 || M > 128 || N <= 0 || K <= 0 || (K % 8) != 0) return IA_ERR_UNSUPPORTED;
  if (epilogue != SK_EPI_NONE && epilogue != SK_EPI_SWIGLU) return IA_ERR_BAD_ARG;
  if (epilogue == SK_EPI_SWIGLU && (N & 1)) return IA_ERR_BAD_ARG;
  if (out_dtype != IA_F32 && out_dtype != IA_BF16) return IA_ERR_BAD_ARG;
  const int splits = skinny_splits(N, K);
  if (splits > 65535) return IA_ERR_UNSUPPORTED;
  const uint16_t* x = (const uint16_t*)X;
  const uint16_t* w = (const uint16_t*)W;
  if (splits > 1 && (!workspace || workspace_floats < (size_t)splits * M * N)) return IA_ERR_BAD_ARG;
  if (epilogue == SK_EPI_SWIGLU && C != nullptr && glu_whole(N, K)) {
    // one pass: both halves of W in the same wave, the activation in the epilogue
    if (splits > 1) {                                  // the sums in as many pieces as K has parts
      if (out_dtype == IA_F32) return launch_skinny<true, float, TILED, true>(x, w, (float*)C, nullptr, M, N, K, 1, stream);
      return launch_skinny<true, uint16_t, TILED, true>(x, w, (uint16_t*)C, nullptr, M, N, K, 1, stream);
    }
    if (out_dtype == IA_F32) return launch_skinny<true, float, TILED>(x, w, (float*)C, nullptr, M, N, K, 1, stream);
    return launch_skinny<true, uint16_t, TILED>(x, w, (uint16_t*)C, nullptr, M, N, K, 1, stream);
  }
  const bool via_workspace = splits > 1 || epilogue != SK_EPI_NONE || C == nullptr;
  if (via_workspace && (!workspace || workspace_floats < (size_t)splits * M * N)) return IA_ERR_BAD_ARG;
  if (!via_workspace) {
    if (out_dtype == IA_F32) return launch_skinny<false, float, TILED>(x, w, (float*)C, nullptr, M, N, K, 1, stream);
    return launch_skinny<false, uint16_t, TILED>(x, w, (uint16_t*)C, nullptr, M, N, K, 1, stream);
  }
  const bool glu = epilogue == SK_EPI_SWIGLU;
  const int groups = !TILED && C != nullptr && splits > 1 ? staged_groups(M, N, K, splits, glu) : 0;
  if (groups > 0) {
#define SK_STAGED(G, TO)                                                                                             \
  (M <= 16 ? launch_staged<G, 1, TO>(x, w, (TO*)C, M, N, K, splits, groups, finish, stream)                          \
           : launch_staged<G, 2, TO>(x, w, (TO*)C, M, N, K, splits, groups, finish, stream))
    if (out_dtype == IA_F32) return glu ? SK_STAGED(true, float) : SK_STAGED(false, float);
    return glu ? SK_STAGED(true, uint16_t) : SK_STAGED(false, uint16_t);
#undef SK_STAGED
  }
  if (!TILED && C != nullptr && splits > 1 && whole_k_pays(M, N, K, splits, glu)) {
    const int nchunks = (K + SK_KC - 1) / SK_KC, cps = (nchunks + splits - 1) / splits, NO = glu ? N / 2 : N;
    const dim3 grid((NO + 15) / 16), block((glu ? 2 : 1) * splits * 64);
#define SK_WHOLE(G, WAVES)                                                                                            \
  do {                                                                                                                \
    if (out_dtype == IA_F32)                                                                                          \
      gemm_skinny_whole_kernel<G, WAVES, float><<<grid, block, 0, stream>>>(x, w, (float*)C, M, N, K, cps, splits, finish);   \
    else                                                                                                              \
      gemm_skinny_whole_kernel<G, WAVES, uint16_t><<<grid, block, 0, stream>>>(x, w, (uint16_t*)C, M, N, K, cps, splits, finish); \
  } while (0)
    if (!glu) SK_WHOLE(false, 8);
    else if (splits <= 4) SK_WHOLE(true, 8);
    else SK_WHOLE(true, 16);
#undef SK_WHOLE
    IA_LAUNCH_CHECK();
    return IA_OK;
  }
  const int rc = launch_skinny<false, float, TILED>(x, w, nullptr, workspace, M, N, K, splits, stream);
  if (rc != IA_OK || C == nullptr) return rc;
  if (out_dtype == IA_F32) return launch_join<float>(workspace, (float*)C, M, N, splits, epilogue, finish, stream);
  return launch_join<uint16_t>(workspace, (uint16_t*)C, M, N, splits, epilogue, finish, stream);
}

extern "C" int ia_gemm_skinny(const void* X, const void* W, void* C, int out_dtype, int M, int N, int K,
                              int epilogue, float* workspace, size_t workspace_floats, hipStream_t stream) {
  return skinny_product<false>(X, W, C, out_dtype, M, N, K, epilogue, workspace, workspace_floats, stream);
}

// ia_gemm_skinny without an epilogue whose values are finished on their way to C (SkFinish): a bf16 result by bias (nullable)
// and act, an fp32 one by scale and cap (0: none).  The same bits as the launches behind it (ia_add_bias, ia_activation, ia_scale,
// ia_softcap); a bf16 product in one part is followed by them.
extern "C" int ia_add_bias(void* y, int code, const float* bias, int N, int C, hipStream_t stream);
extern "C" int ia_activation(const void* in, void* out, int dtype, size_t n, int kind, hipStream_t stream);
extern "C" int ia_gemm_skinny_finished(const void* X, const void* W, void* C, int out_dtype, int M, int N, int K, const float* bias,
                                       int act, float scale, float cap, float* workspace, size_t workspace_floats,
                                       hipStream_t stream) {
  if (C == nullptr || act < 0 || act > 3 || !(cap >= 0.f) || (out_dtype == IA_F32 ? bias != nullptr || act != 0 : scale != 1.0f || cap > 0.f))
    return IA_ERR_BAD_ARG;
  const SkFinish finish{bias, act, scale, cap};
  if (M <= 0 || M > 128 || N <= 0 || K <= 0 || (K % 8) != 0) return IA_ERR_UNSUPPORTED;
  if (skinny_splits(N, K) > 1)
    return skinny_product<false>(X, W, C, out_dtype, M, N, K, SK_EPI_NONE, workspace, workspace_floats, stream, finish);
  if (out_dtype == IA_F32)
    return launch_skinny<false, float, false, true>((const uint16_t*)X, (const uint16_t*)W, (float*)C, nullptr, M, N, K, 1, stream, finish);
  int rc = skinny_product<false>(X, W, C, out_dtype, M, N, K, SK_EPI_NONE, workspace, workspace_floats, stream);
  if (rc == IA_OK && bias) rc = ia_add_bias(C, IA_BF16, bias, M, N, stream);
  if (rc == IA_OK && act) rc = ia_activation(C, C, IA_BF16, (size_t)M * N, act, stream);
  return rc;
}

// ---- the weight laid out for the kernel: every workgroup's 64 rows x 256 values of a chunk consecutive ----------
// Whether the copy for this weight and use is laid out for the kernel that multiplies with both halves of
// [gate | up] at once (a workgroup then takes 32 rows of each half).
static bool tiled_glu(int N, int K, int epilogue) { return epilogue == SK_EPI_SWIGLU && glu_whole(N, K); }

// Elements (bf16) of the copy: rows padded to whole workgroups, K to whole chunks.
extern "C" size_t ia_gemm_skinny_tiled_elements(int N, int K, int epilogue) {
  if (N <= 0 || K <= 0) return 0;
  const int NO = tiled_glu(N, K, epilogue) ? N / 2 : N, cols = tiled_glu(N, K, epilogue) ? SK_BN / 2 : SK_BN;
  const size_t blocks = (size_t)(NO + cols - 1) / cols, chunks = (size_t)(K + SK_KC - 1) / SK_KC;
  return blocks * chunks * SK_BN * SK_KC;
}

__global__ __launch_bounds__(256) void tile_weight_kernel(const uint16_t* __restrict__ W, uint16_t* __restrict__ T,
                                                          int N, int K, int glu, size_t total) {
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;      // one element of the copy
  if (idx >= total) return;
  const int kk = (int)(idx % SK_KC);
  const size_t rowi = idx / SK_KC;
  const int rib = (int)(rowi % SK_BN);                            // row within the workgroup's tile
  const size_t bc = rowi / SK_BN;
  const int chunks = (K + SK_KC - 1) / SK_KC;
  const int chunk = (int)(bc % chunks);
  const size_t block = bc / chunks;
  const int k = chunk * SK_KC + kk;
  int n;
  bool ok;
  if (glu) {
    const int NO = N / 2, col = (int)block * (SK_BN / 2) + (rib & 15) + ((rib >> 4) & 1) * 16, half = rib >> 5;
    ok = col < NO;
    n = half * NO + col;
  } else {
    n = (int)block * SK_BN + rib;
    ok = n < N;
  }
  T[idx] = (ok && k < K) ? W[(size_t)n * K + k] : (uint16_t)0;
}

// T (ia_gemm_skinny_tiled_elements(N, K, epilogue) values) = W [N, K] laid out for ia_gemm_skinny_tiled with the
// same epilogue.
extern "C" int ia_gemm_skinny_tile(const void* W, void* T, int N, int K, int epilogue, hipStream_t stream) {
  if (!W || !T || N <= 0 || K <= 0 || (epilogue != SK_EPI_NONE && epilogue != SK_EPI_SWIGLU)) return IA_ERR_BAD_ARG;
  const size_t total = ia_gemm_skinny_tiled_elements(N, K, epilogue);
  const size_t grid = (total + 255) / 256;
  if (grid > 0x7fffffffu) return IA_ERR_UNSUPPORTED;
  tile_weight_kernel<<<(unsigned)grid, 256, 0, stream>>>((const uint16_t*)W, (uint16_t*)T, N, K,
                                                         tiled_glu(N, K, epilogue) ? 1 : 0, total);
  IA_LAUNCH_CHECK();
  return IA_OK;
}

// ia_gemm_skinny with the weight given as the copy that ia_gemm_skinny_tile made for the same epilogue: the same
// sums in the same order, the same bits.
extern "C" int ia_gemm_skinny_tiled(const void* X, const void* T, void* C, int out_dtype, int M, int N, int K,
                                    int epilogue, float* workspace, size_t workspace_floats, hipStream_t stream) {
  return skinny_product<true>(X, T, C, out_dtype, M, N, K, epilogue, workspace, workspace_floats, stream);
}

// The same product for any number of rows, 128 at a time (a result in fp32 from bf16 operands has no other
// kernel here: the head of a step that wants the logits of many places).  The workspace serves every piece in turn.
// tiled != 0: W is the copy of ia_gemm_skinny_tile (no epilogue).
extern "C" int ia_gemm_skinny_rows(const void* X, const void* W, int tiled, void* C, int out_dtype, int M, int N, int K,
                                   float* workspace, size_t workspace_floats, hipStream_t stream) {
  if (M <= 0 || N <= 0 || K <= 0 || (K % 8) != 0) return IA_ERR_UNSUPPORTED;
  if (out_dtype != IA_F32 && out_dtype != IA_BF16) return IA_ERR_BAD_ARG;
  const size_t out_bytes = out_dtype == IA_F32 ? 4 : 2;
  for (int m0 = 0; m0 < M; m0 += 128) {
    const int m = M - m0 < 128 ? M - m0 : 128;
    const void* x = (const char*)X + (size_t)m0 * K * 2;
    void* c = (char*)C + (size_t)m0 * N * out_bytes;
    const int rc = tiled ? ia_gemm_skinny_tiled(x, W, c, out_dtype, m, N, K, SK_EPI_NONE, workspace, workspace_floats, stream)
                         : ia_gemm_skinny(x, W, c, out_dtype, m, N, K, SK_EPI_NONE, workspace, workspace_floats, stream);
    if (rc != IA_OK) return rc;
  }
  return IA_OK;
}

// ---- the same product for callers that cannot allocate: the workspace is an array of this library ----------
#include <mutex>
#include "no_alloc.h"

#define IA_MAX_DEVICES 64

// Partial sums of a split product.  In host code this name only stands for the array (it is no device address);
// hipGetSymbolAddress gives the address on the current device, and host code uses that and nothing else.
static __device__ __align__(256) float scratch[IA_SKINNY_SCRATCH_FLOATS];
static float* scratch_on_device[IA_MAX_DEVICES];      // each GPU has its own copy of the array at its own address
static std::mutex scratch_lock;

static int scratch_of_current_device(float** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= IA_MAX_DEVICES) return IA_ERR_UNSUPPORTED;
  std::lock_guard<std::mutex> hold(scratch_lock);
  if (scratch_on_device[dev] == nullptr) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    if (p == nullptr) return IA_ERR_BAD_ARG;
    scratch_on_device[dev] = static_cast<float*>(p);
  }
  *out = scratch_on_device[dev];
  return IA_OK;
}

extern "C" size_t ia_gemm_skinny_no_alloc_capacity(void) { return IA_SKINNY_SCRATCH_FLOATS; }

extern "C" size_t ia_gemm_skinny_no_alloc_needs(int M, int N, int K, int epilogue) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const int splits = skinny_splits(N, K);
  (void)epilogue;      // with one part the activation is done in the product's own epilogue, without a workspace
  return splits > 1 ? (size_t)splits * (size_t)M * (size_t)N : 0;
}

extern "C" int ia_gemm_skinny_no_alloc(const void* X, const void* W, void* C, int out_dtype, int M, int N, int K,
                                       int epilogue, hipStream_t stream) {
  if (X == nullptr || W == nullptr || C == nullptr) return IA_ERR_BAD_ARG;
  if (M <= 0 || M > 128 || N <= 0 || K <= 0 || (K % 8) != 0) return IA_ERR_UNSUPPORTED;
  const size_t needs = ia_gemm_skinny_no_alloc_needs(M, N, K, epilogue);
  if (needs > IA_SKINNY_SCRATCH_FLOATS) return IA_ERR_SCRATCH_TOO_SMALL;
  float* ws = nullptr;
  const int rc = scratch_of_current_device(&ws);
  if (rc != IA_OK) return rc;
  return ia_gemm_skinny(X, W, C, out_dtype, M, N, K, epilogue, ws, IA_SKINNY_SCRATCH_FLOATS, stream);
}

// ---- the launchers of this file as operations of a step's program (see op_call.h) ----
#include "op_call.h"
IA_OP(ia_gemm_skinny)
IA_OP(ia_gemm_skinny_finished)
IA_OP(ia_gemm_skinny_tiled)
IA_OP(ia_gemm_skinny_rows)
