// Causal attention of a ragged batch over paged keys and values, one wave per
// (query token, query head), in fp32 throughout.  It serves the true 32-bit
// path, and is the plain twin of the MFMA kernels.  Any head size up to 640,
// any page size, any grouping of query heads over key/value heads, an optional
// window.  Keys are summed in the order of their positions, 64 at a time, so the
// result at a position does not depend on what else the batch holds.
//
// Key pages are [num_pages, nkv, page_size, d], value pages [num_pages, nkv, d,
// page_size]; block_tables[s, j / page_size] is the page of key j of sequence s.  The query of token n stands at positions[n] and
// sees keys max(0, pos - window + 1) .. pos  (window 0: all keys from 0; window < 0: the keys of its own
// chunk of -window positions, see ia_first_visible_key).  sinks (nullable, fp32 [nh]): exp(sinks[h]) is added to
// the softmax's denominator of head h; it has no key and no value.  Value heads may have another size, dv, than
// query and key heads (value pages [num_pages, nkv, dv, page_size], out rows of nh dv values).  Under a window the
// request's first `keep` keys stay visible; a softcap c > 0 turns a scaled score s into c tanh(s / c).  bias (nullable,
// fp32 [nh, span + 2 pad], the layout of attention_mfma.hip): a number added to the score by the key's distance; gate
// (nullable, rows of gate_stride values): what a head leaves, times sigmoid(gate), value by value.
#include "common.h"

#define AG_MAX_D 640
#define AG_BIAS_PAD 64

// 64 keys of a request are a few trips to memory long for a wave: the keys' rows, 16 bytes a load and 64 values of each asked for
// together where they can be read so (VEC), then the values, eight keys' together.  NC: 64 channels of the values a piece.
// Every sum is in the same order whatever is asked for together.  fp32, 32 heads of 64 on 8, 3 tokens with 45, 60 and 75 keys 27.3 us
// before and 15.0 so, three prompts of 45, 60 and 37 tokens 34.4 and 25.5, 2 tokens with 1,000 and 2,000 keys 654 and 321 (a value and a key at a time, ten pieces of channels with a condition each, a
// division a key before).  Values four keys a load where they lie side by side: steps and prompts of such a pass 18.2 us on average and 12.3 so.
template <typename T>
__device__ __forceinline__ void load_four(const T* p, float (&v)[4]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = to_float(p[e]);
}
template <>
__device__ __forceinline__ void load_four<float>(const float* p, float (&v)[4]) {
  const float4 t = *reinterpret_cast<const float4*>(p);
  v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
}

template <typename T, int NC, bool VEC>
__global__ __launch_bounds__(64) void attn_generic_kernel(const T* __restrict__ q, int q_row_stride,
                                                          const T* __restrict__ k_pages,
                                                          const T* __restrict__ v_pages, T* __restrict__ out,
                                                          int out_row_stride, const int* __restrict__ token_seq,
                                                          const int* __restrict__ positions,
                                                          const int* __restrict__ block_tables, int bt_stride, int nh,
                                                          int nkv, int d, int dv, int page_size, int num_pages,
                                                          float scale, int window, const float* __restrict__ sinks,
                                                          int keep, float softcap, const float* __restrict__ bias,
                                                          int span, const T* __restrict__ gate, int gate_stride) {
  __shared__ float qs[AG_MAX_D];
  __shared__ float ps[64];
  __shared__ size_t vs[64];          // where a key's values begin, channel after channel page_size apart
  const int n = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  const int s = token_seq[n];
  const int pos = positions[n];
  const int g = h / (nh / nkv);
  const int* bt = block_tables + (size_t)s * bt_stride;
  const T* qr = q + (size_t)n * q_row_stride + (size_t)h * d;
  for (int i = lane; i < d; i += 64) qs[i] = to_float(qr[i]);
  __syncthreads();

  const int j_hi = pos;
  const int j_lo = ia_first_visible_key(pos, window);
  float m = -INFINITY, l = 0.f;
  float acc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[c] = 0.f;

  // the keys in the order of their positions: the kept ones before the window, then the window's
  const int kept = window > 0 ? (keep < j_lo ? keep : j_lo) : 0;
  const int count = kept + (j_hi - j_lo + 1);
  // pieces of 64 keys begin on a multiple of four positions, and so does a page: whole quads of keys in one page, beyond the last key too
  const bool quads = kept == 0 && ((j_lo | page_size) & 3) == 0 && (reinterpret_cast<uintptr_t>(v_pages) & 15) == 0;
  for (int j0 = 0; j0 < count; j0 += 64) {
    const int j = j0 + lane < kept ? j0 + lane : j0 + lane - kept + j_lo;
    const bool valid = j <= j_hi;
    float sc = -INFINITY;
    size_t value_at = 0;
    if (valid) {
      const int page = bt[j / page_size];
      if ((unsigned)page < (unsigned)num_pages) {
        const size_t head_page = (size_t)page * nkv + g;
        const int off = j % page_size;
        value_at = head_page * dv * page_size + off;
        const T* kr = k_pages + (head_page * page_size + off) * d;
        float dot = 0.f;
        if (VEC) {
          for (int i0 = 0; i0 < d; i0 += 64) {
            float k4[16][4];
#pragma unroll
            for (int u = 0; u < 16; ++u) load_four(kr + min(i0 + 4 * u, d - 4), k4[u]);
#pragma unroll
            for (int u = 0; u < 16; ++u) {
              if (i0 + 4 * u < d) {
#pragma unroll
                for (int e = 0; e < 4; ++e) dot = fmaf(qs[i0 + 4 * u + e], k4[u][e], dot);
              }
            }
          }
        } else {
          for (int i = 0; i < d; ++i) dot = fmaf(qs[i], to_float(kr[i]), dot);
        }
        sc = dot * scale;
        if (softcap > 0.f) sc = softcap * tanhf(sc / softcap);
        if (bias) {
          const int back = pos - j < span - 1 ? pos - j : span - 1;
          sc += bias[(size_t)h * (span + 2 * AG_BIAS_PAD) + AG_BIAS_PAD + span - 1 - back];
        }
      } else {
        sc = __uint_as_float(0x7fc00000u);  // a block table without a page here: poison, never a stray read
      }
    }
    const float m_new = fmaxf(m, wave_max(sc));
    const float p = valid ? expf(sc - m_new) : 0.f;
    const float corr = expf(m - m_new);
    l = l * corr + wave_sum(p);
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[c] *= corr;
    ps[lane] = p;
    vs[lane] = value_at;
    __syncthreads();
    const int cnt = (count - j0) < 64 ? (count - j0) : 64;
    if (VEC && quads) {
      // four keys' values of a channel lie side by side
      constexpr int QUADS = NC <= 4 ? 16 / NC : 1;                     // of keys, whose values are asked for together
      for (int j4 = 0; j4 < cnt; j4 += 4 * QUADS) {
        float v[QUADS][NC][4];
#pragma unroll
        for (int u = 0; u < QUADS; ++u) {
          const T* vr = v_pages + vs[min(j4 + 4 * u, (cnt - 1) & ~3)];
#pragma unroll
          for (int c = 0; c < NC; ++c) load_four(vr + (size_t)min(lane + 64 * c, dv - 1) * page_size, v[u][c]);
        }
#pragma unroll
        for (int u = 0; u < 4 * QUADS; ++u) {
          if (j4 + u >= cnt) break;
          const float pj = ps[j4 + u];
#pragma unroll
          for (int c = 0; c < NC; ++c) acc[c] = fmaf(pj, v[u >> 2][c][u & 3], acc[c]);
        }
      }
    } else {
      constexpr int AHEAD = 8;        // keys whose values are asked for together
      for (int jj = 0; jj < cnt; jj += AHEAD) {
        float v[AHEAD][NC];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
          const T* vr = v_pages + vs[min(jj + u, cnt - 1)];
#pragma unroll
          for (int c = 0; c < NC; ++c) v[u][c] = to_float(vr[(size_t)min(lane + 64 * c, dv - 1) * page_size]);
        }
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
          if (jj + u >= cnt) break;
          const float pj = ps[jj + u];
#pragma unroll
          for (int c = 0; c < NC; ++c) acc[c] = fmaf(pj, v[u][c], acc[c]);
        }
      }
    }
    __syncthreads();
    m = m_new;
  }
  if (sinks) {          // a sink: exp(sink) more in the denominator, nothing in the sum
    const float sk = sinks[h];
    const float m_new = fmaxf(m, sk);
    const float corr = expf(m - m_new);
    l = l * corr + expf(sk - m_new);
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[c] *= corr;
  }
  T* o = out + (size_t)n * out_row_stride + (size_t)h * dv;
  const float inv_l = 1.0f / l;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int dim = lane + 64 * c;
    if (dim >= dv) continue;
    float v = acc[c] * inv_l;
    if (gate) v *= 1.0f / (1.0f + expf(-to_float(gate[(size_t)n * gate_stride + (size_t)h * dv + dim])));
    o[dim] = from_float<T>(v);
  }
}

extern "C" int ia_attention_generic(const void* q, int q_row_stride, const void* k_pages, const void* v_pages,
                                    void* out, int out_row_stride, int dtype, const int* token_seq,
                                    const int* positions, const int* block_tables, int bt_stride, int N, int nh,
                                    int nkv, int d, int dv, int page_size, int num_pages, float scale, int window,
                                    const float* sinks, int keep, float softcap, const float* bias, int span,
                                    const void* gate, int gate_stride, hipStream_t stream) {
  if (N < 0 || nh <= 0 || nkv <= 0 || nh % nkv != 0 || d <= 0 || d > AG_MAX_D || dv <= 0 || dv > AG_MAX_D || keep < 0 ||
      !(softcap >= 0.f) || q_row_stride < nh * d || out_row_stride < nh * dv || page_size <= 0 || num_pages <= 0 ||
      bt_stride <= 0 || (bias && span < 1) || (gate && gate_stride < nh * dv))
    return IA_ERR_BAD_ARG;
  if (nh > 65535) return IA_ERR_UNSUPPORTED;
  if (N == 0) return IA_OK;
  if (dtype != IA_F32 && dtype != IA_BF16) return IA_ERR_BAD_ARG;
  dim3 grid(N, nh);
#define AG_LAUNCH(T, NC, VEC)                                                                                              \
  attn_generic_kernel<T, NC, VEC><<<grid, 64, 0, stream>>>((const T*)q, q_row_stride, (const T*)k_pages, (const T*)v_pages, \
                                                           (T*)out, out_row_stride, token_seq, positions, block_tables,    \
                                                           bt_stride, nh, nkv, d, dv, page_size, num_pages, scale, window, \
                                                           sinks, keep, softcap, bias, span, (const T*)gate, gate_stride)
#define AG_PIECES(T, VEC)                       \
  do {                                          \
    if (dv <= 64) AG_LAUNCH(T, 1, VEC);         \
    else if (dv <= 128) AG_LAUNCH(T, 2, VEC);   \
    else if (dv <= 256) AG_LAUNCH(T, 4, VEC);   \
    else AG_LAUNCH(T, AG_MAX_D / 64, VEC);      \
  } while (0)
  if (dtype == IA_BF16) AG_PIECES(bf16_t, false);
  else if ((d & 3) == 0 && (reinterpret_cast<uintptr_t>(k_pages) & 15) == 0) AG_PIECES(float, true);
  else AG_PIECES(float, false);
#undef AG_PIECES
#undef AG_LAUNCH
  IA_LAUNCH_CHECK();
  return IA_OK;
}

// ---- the launchers of this file as operations of a step's program (see op_call.h) ----
#include "op_call.h"
IA_OP(ia_attention_generic)
