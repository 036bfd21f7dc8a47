// Attention whose weights are sigmoids, not a softmax: for the query of head h at position i and the key at j <= i,
//     w_ij = sigmoid( scale q_i.k_j - r1_h ln(1 + r2_h (i - j)) + b_h ),      o_i = g_ih sum_j w_ij v_j,
// nothing normalised over the keys, g = sigmoid(gate logit) one number per token and head.  Query heads share
// key/value heads in groups; keys have `dim` values, values `vdim`.
//
//   ia_sigattn_prepare   from a token's projected row [q | k | v | ...]: biases, the root mean square over ALL of a
//                        row's queries (and over all of its keys) with a weight per value, the query's factor
//                        1 + coef ln(floor((p + 1) / every) + 1), queries into their own rows, keys and values into
//                        their pages;
//   ia_sigattn_generic   one wave per (token, head), fp32 throughout, keys 64 at a time in the order of their
//                        positions: the 32-bit path and the plain twin of the matrix-core kernels;
//   ia_sigattn_mfma      bf16 on the matrix cores: single tokens (the query heads of a key/value head side by side,
//                        the keys in parts over workgroups and waves, joined in a fixed order) and portions of
//                        prompts (a wave per 16 rows of a head).
//
// Pages: keys [num_pages, nkv, page_size, dim], values transposed [num_pages, nkv, vdim, page_size] (four keys of
// one value channel are 8 contiguous bytes, the operand of the second product); block_tables[s, j / page_size]
// is the page of key j of request s.  A sum of weights has no reference point to move, so parts of the keys add up.
#include "common.h"

#define SA_MAX_D 640

// Bound by trips to memory where tokens are few: grid (N, 2), the queries' norm and the keys' and values' side by side, and
// up to 8 values a thread (rows of 2,048; KEEP: as many as the row has, what is asked for twice costs) with their bias and
// weight asked for together and kept for the second use (one token of 16 heads of 128: 13.4 us with the loads one after the
// other, twice, so 7.2; 3,000 tokens of 4 heads of 64 12.1 one after the other, 13.8 with eight kept).
template <typename T>
__device__ __forceinline__ float sq_value(const T* __restrict__ row, const float* __restrict__ b, int i) {
  return to_float(row[i]) + (b ? b[i] : 0.f);
}

// emit(i, value over the root mean square times factor and w[i]) for every value of one norm of `n` values
template <int KEEP, typename T, typename Factor, typename Emit>
__device__ __forceinline__ void sq_norm(const T* __restrict__ row, const float* __restrict__ b, const float* __restrict__ w,
                                        int n, float eps, float* red, Factor factor, Emit emit) {
  const int tid = threadIdx.x;
  float x[KEEP], wx[KEEP], ss = 0.f;
#pragma unroll
  for (int u = 0; u < KEEP; ++u) {
    const int i = min(tid + 256 * u, n - 1);
    x[u] = sq_value(row, b, i);
    wx[u] = w[i];
  }
#pragma unroll
  for (int u = 0; u < KEEP; ++u) ss = tid + 256 * u < n ? fmaf(x[u], x[u], ss) : ss;
  for (int i = tid + 256 * KEEP; i < n; i += 256) {
    const float v = sq_value(row, b, i);
    ss = fmaf(v, v, ss);
  }
  ss = block_sum<256>(ss, red);
  const float f = factor(1.0f / sqrtf(ss / (float)n + eps));
#pragma unroll
  for (int u = 0; u < KEEP; ++u)
    if (tid + 256 * u < n) emit(tid + 256 * u, x[u] * f * wx[u]);
  for (int i = tid + 256 * KEEP; i < n; i += 256) emit(i, sq_value(row, b, i) * f * w[i]);
}

template <typename T, int KEEP>
__global__ __launch_bounds__(256) void sigattn_prepare_kernel(
    const T* __restrict__ proj, int proj_stride, const float* __restrict__ bq, const float* __restrict__ bk,
    const float* __restrict__ bv, const float* __restrict__ wq, const float* __restrict__ wk, float eps, float temp_coef,
    int temp_every, const int* __restrict__ positions, const int* __restrict__ slots, T* __restrict__ q_out,
    T* __restrict__ k_pages, T* __restrict__ v_pages, int nh, int nkv, int dim, int vdim, int page_size, int num_pages) {
  __shared__ float red[4];
  const int n = blockIdx.x, tid = threadIdx.x;
  const T* row = proj + (size_t)n * proj_stride;
  const int nq = nh * dim, nk = nkv * dim, nv = nkv * vdim;
  if (blockIdx.y == 0) {
    const int p = temp_every > 0 ? positions[n] : 0;
    sq_norm<KEEP>(row, bq, wq, nq, eps, red,
            [&](float f) { return temp_every > 0 ? f * (1.0f + temp_coef * logf((float)((p + 1) / temp_every) + 1.0f)) : f; },
            [&](int i, float v) { q_out[(size_t)n * nq + i] = from_float<T>(v); });
    return;
  }
  const int slot = slots[n];
  const int page = slot / page_size, off = slot - page * page_size;
  if (slot < 0 || page >= num_pages) return;                  // a token without a place: nothing is written
  sq_norm<KEEP>(row + nq, bk, wk, nk, eps, red, [](float f) { return f; },
          [&](int i, float v) {
            const int g = i / dim, c = i - g * dim;
            k_pages[(((size_t)page * nkv + g) * page_size + off) * dim + c] = from_float<T>(v);
          });
  for (int i = tid; i < nv; i += 256) {
    const int g = i / vdim, c = i - g * vdim;
    v_pages[(((size_t)page * nkv + g) * vdim + c) * page_size + off] = from_float<T>(sq_value(row + nq + nk, bv, i));
  }
}

// proj rows [nh dim | nkv dim | nkv vdim | ...] of proj_stride values; biases and norm weights fp32 (biases nullable);
// temp_every 0: no factor on the queries; slots null: queries only (the pages are another run's).
extern "C" int ia_sigattn_prepare(const void* proj, int code, int proj_stride, const float* bq, const float* bk,
                                  const float* bv, const float* wq, const float* wk, float eps, float temp_coef,
                                  int temp_every, const int* positions, const int* slots, void* q_out, void* k_pages,
                                  void* v_pages, int N, int nh, int nkv, int dim, int vdim, int page_size, int num_pages,
                                  hipStream_t stream) {
  if (N < 0 || nh <= 0 || nkv <= 0 || dim <= 0 || vdim <= 0 || !(eps > 0.f) || temp_every < 0 ||
      proj_stride < nh * dim + (slots ? nkv * (dim + vdim) : 0))
    return IA_ERR_BAD_ARG;
  if (N == 0) return IA_OK;
  if (!proj || !wq || !q_out || !positions || (slots && (!wk || !k_pages || !v_pages || page_size <= 0 || num_pages <= 0)))
    return IA_ERR_BAD_ARG;
  if (code != IA_F32 && code != IA_BF16) return IA_ERR_BAD_ARG;
#define IA_SQ(T, KEEP)                                                                                                 \
  sigattn_prepare_kernel<T, KEEP><<<dim3(N, slots ? 2 : 1), 256, 0, stream>>>(                                        \
      (const T*)proj, proj_stride, bq, bk, bv, wq, wk, eps, temp_coef, temp_every, positions, slots, (T*)q_out,       \
      (T*)k_pages, (T*)v_pages, nh, nkv, dim, vdim, page_size, num_pages)
#define IA_SQ_KEEP(T)                        \
  do {                                       \
    if (widest <= 256) IA_SQ(T, 1);          \
    else if (widest <= 512) IA_SQ(T, 2);     \
    else if (widest <= 1024) IA_SQ(T, 4);    \
    else IA_SQ(T, 8);                        \
  } while (0)
  const int widest = (slots && nkv > nh ? nkv : nh) * dim;
  if (code == IA_F32) IA_SQ_KEEP(float);
  else IA_SQ_KEEP(bf16_t);
#undef IA_SQ_KEEP
#undef IA_SQ
  IA_LAUNCH_CHECK();
  return IA_OK;
}

template <typename T>
__global__ __launch_bounds__(64) void sigattn_generic_kernel(
    const T* __restrict__ q, int q_stride, const T* __restrict__ k_pages, const T* __restrict__ v_pages,
    const T* __restrict__ gate, int gate_stride, T* __restrict__ out, const int* __restrict__ token_seq,
    const int* __restrict__ positions, const int* __restrict__ block_tables, int bt_stride, const float* __restrict__ r1,
    const float* __restrict__ r2, const float* __restrict__ pb, int nh, int nkv, int dim, int vdim, int page_size,
    int num_pages, float scale) {
  __shared__ float qs[SA_MAX_D];
  __shared__ float ps[64];
  __shared__ int rs[64];
  __shared__ size_t vs[64];
  const int n = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  const int s = token_seq[n];
  const int pos = positions[n];
  const int g = h / (nh / nkv);
  const int* bt = block_tables + (size_t)s * bt_stride;
  const T* qr = q + (size_t)n * q_stride + (size_t)h * dim;
  for (int i = lane; i < dim; i += 64) qs[i] = to_float(qr[i]);
  __syncthreads();
  const float a1 = r1 ? r1[h] : 0.f, a2 = r2 ? r2[h] : 0.f, b = pb ? pb[h] : 0.f;
  float acc[SA_MAX_D / 64];
#pragma unroll
  for (int c = 0; c < SA_MAX_D / 64; ++c) acc[c] = 0.f;
  for (int j0 = 0; j0 <= pos; j0 += 64) {
    const int j = j0 + lane;
    float p = 0.f;
    int row = 0;
    size_t vat = 0;
    if (j <= pos) {
      const int page = bt[j / page_size];
      if ((unsigned)page < (unsigned)num_pages) {
        row = (page * nkv + g) * page_size + (j % page_size);
        vat = ((size_t)page * nkv + g) * vdim * page_size + (j % page_size);
        const T* kr = k_pages + (size_t)row * dim;
        float dot = 0.f;
        for (int i = 0; i < dim; ++i) dot = fmaf(qs[i], to_float(kr[i]), dot);
        const float sc = dot * scale - a1 * log1pf(a2 * (float)(pos - j)) + b;
        p = 1.0f / (1.0f + expf(-sc));
      } else {
        p = __uint_as_float(0x7fc00000u);     // a block table without a page here: poison, never a stray read
      }
    }
    ps[lane] = p;
    rs[lane] = row;
    vs[lane] = vat;
    __syncthreads();
    const int cnt = (pos - j0 + 1) < 64 ? (pos - j0 + 1) : 64;
    for (int jj = 0; jj < cnt; ++jj) {
      const T* vr = v_pages + vs[jj];
      const float pj = ps[jj];
#pragma unroll
      for (int c = 0; c < SA_MAX_D / 64; ++c) {
        const int i = lane + 64 * c;
        if (i < vdim) acc[c] = fmaf(pj, to_float(vr[(size_t)i * page_size]), acc[c]);
      }
    }
    __syncthreads();
  }
  float gt = 1.0f;
  if (gate) gt = 1.0f / (1.0f + expf(-to_float(gate[(size_t)n * gate_stride + h])));
  T* o = out + ((size_t)n * nh + h) * vdim;
#pragma unroll
  for (int c = 0; c < SA_MAX_D / 64; ++c) {
    const int i = lane + 64 * c;
    if (i < vdim) o[i] = from_float<T>(acc[c] * gt);
  }
}

// q rows of q_stride values (head h's dim values from h * dim); gate (nullable): rows of gate_stride values, head h's
// logit at [h]; r1, r2, pb (nullable) fp32 [nh]; out [N, nh vdim].
extern "C" int ia_sigattn_generic(const void* q, int q_stride, const void* k_pages, const void* v_pages, const void* gate,
                                  int gate_stride, void* out, int dtype, const int* token_seq, const int* positions,
                                  const int* block_tables, int bt_stride, const float* r1, const float* r2,
                                  const float* pb, int N, int nh, int nkv, int dim, int vdim, int page_size,
                                  int num_pages, float scale, hipStream_t stream) {
  if (N < 0 || nh <= 0 || nkv <= 0 || nh % nkv != 0 || dim <= 0 || dim > SA_MAX_D || vdim <= 0 || vdim > SA_MAX_D ||
      page_size <= 0 || num_pages <= 0 || bt_stride <= 0 || q_stride < nh * dim || (gate && gate_stride < nh))
    return IA_ERR_BAD_ARG;
  if (nh > 65535) return IA_ERR_UNSUPPORTED;
  if (N == 0) return IA_OK;
  dim3 grid(N, nh);
  if (dtype == IA_F32)
    sigattn_generic_kernel<float><<<grid, 64, 0, stream>>>((const float*)q, q_stride, (const float*)k_pages,
                                                           (const float*)v_pages, (const float*)gate, gate_stride,
                                                           (float*)out, token_seq, positions, block_tables, bt_stride,
                                                           r1, r2, pb, nh, nkv, dim, vdim, page_size, num_pages, scale);
  else if (dtype == IA_BF16)
    sigattn_generic_kernel<bf16_t><<<grid, 64, 0, stream>>>((const bf16_t*)q, q_stride, (const bf16_t*)k_pages,
                                                            (const bf16_t*)v_pages, (const bf16_t*)gate, gate_stride,
                                                            (bf16_t*)out, token_seq, positions, block_tables, bt_stride,
                                                            r1, r2, pb, nh, nkv, dim, vdim, page_size, num_pages, scale);
  else
    return IA_ERR_BAD_ARG;
  IA_LAUNCH_CHECK();
  return IA_OK;
}

#include "op_call.h"
IA_OP(ia_sigattn_prepare)
IA_OP(ia_sigattn_generic)
