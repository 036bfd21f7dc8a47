// Shared device helpers for the gfx950 kernels: element types, 16-byte vectors,
// wave (64 lanes) and workgroup reductions with a fixed order of summation.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define IA_WAVE 64

// dtype codes of the C interface
enum { IA_F32 = 0, IA_BF16 = 1 };

// Error codes beyond hipError_t (which is returned as is when a launch fails).
enum { IA_OK = 0, IA_ERR_BAD_ARG = 10001, IA_ERR_UNSUPPORTED = 10002 };

struct bf16_t { uint16_t bits; };

__device__ __forceinline__ float bf16_bits_to_float(uint16_t b) {
  return __uint_as_float(((uint32_t)b) << 16);
}
// Round to nearest, ties to even; NaN stays NaN: v_cvt_pk_bf16_f32.
__device__ __forceinline__ uint16_t float_to_bf16_bits(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
// Two values in one instruction, the first in the lower half.
__device__ __forceinline__ uint32_t two_bf16_bits(float a, float b) {
  typedef __bf16 pair_t __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, (pair_t){(__bf16)a, (__bf16)b});
}

__device__ __forceinline__ float to_float(float x) { return x; }
__device__ __forceinline__ float to_float(bf16_t x) { return bf16_bits_to_float(x.bits); }
template <typename T> __device__ __forceinline__ T from_float(float x);
template <> __device__ __forceinline__ float from_float<float>(float x) { return x; }
template <> __device__ __forceinline__ bf16_t from_float<bf16_t>(float x) {
  bf16_t r; r.bits = float_to_bf16_bits(x); return r;
}

// Load one element of a tensor whose dtype is known only at run time.
__device__ __forceinline__ float load_as_float(const void* p, int dtype, size_t i) {
  return dtype == IA_F32 ? ((const float*)p)[i] : bf16_bits_to_float(((const uint16_t*)p)[i]);
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, IA_WAVE);
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, IA_WAVE));
  return v;
}

// Sum over a workgroup of NT threads (NT a multiple of 64, at most 1024).
// Every thread gets the result; `red` holds at least NT/64 floats.
template <int NT>
__device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  float t = 0.f;
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) t += red[w];
  return t;
}
template <int NT>
__device__ __forceinline__ float block_max(float v, float* red) {
  v = wave_max(v);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  float t = red[0];
#pragma unroll
  for (int w = 1; w < NT / 64; ++w) t = fmaxf(t, red[w]);
  return t;
}

// ---- rotation of queries and keys: one arithmetic for every kernel that rotates
// A value that may be a stack of partial sums of a split matrix product: added in the order of their index.
template <typename TS>
__device__ __forceinline__ float load_split_sum(const TS* p, int splits, size_t split_stride) {
  float v = to_float(p[0]);
#pragma unroll 4
  for (int k = 1; k < splits; ++k) v += to_float(p[k * split_stride]);
  return v;
}

// The sums of several values whose parts lie alike: all parts of all of them are asked for before the first addition, and no load
// has a condition (the last part is read again in place of those there are not; more than eight parts: the loop above).  The same order of additions, the same bits.
template <int PRE, int NV, typename TS>
__device__ __forceinline__ void load_split_sums_by(const TS* const (&p)[NV], int splits, size_t split_stride, float (&v)[NV]) {
  TS x[NV][PRE];
#pragma unroll
  for (int k = 0; k < PRE; ++k)
#pragma unroll
    for (int i = 0; i < NV; ++i) x[i][k] = p[i][(size_t)min(k, splits - 1) * split_stride];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    v[i] = to_float(x[i][0]);
#pragma unroll
    for (int k = 1; k < PRE; ++k) v[i] = k < splits ? v[i] + to_float(x[i][k]) : v[i];
  }
}
template <int NV, typename TS>
__device__ __forceinline__ void load_split_sums(const TS* const (&p)[NV], int splits, size_t split_stride, float (&v)[NV]) {
  if (splits == 1) {
    load_split_sums_by<1>(p, splits, split_stride, v);
  } else if (splits <= 4) {
    load_split_sums_by<4>(p, splits, split_stride, v);
  } else if (splits <= 8) {
    load_split_sums_by<8>(p, splits, split_stride, v);
  } else {
#pragma unroll
    for (int i = 0; i < NV; ++i) v[i] = load_split_sum(p[i], splits, split_stride);
  }
}

// Four consecutive values as floats.
__device__ __forceinline__ float4 load4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float4 load4(const bf16_t* p) {
  const uint2 u = *reinterpret_cast<const uint2*>(p);
  return make_float4(__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
                     __uint_as_float(u.y & 0xffff0000u));
}

// Four values of every part added in the order of their index.  The loads of up to sixteen parts are asked for together, none
// under a condition of its own: a load that some lanes or some counts skip is waited for before the next (behind the
// product that left them, a norm of one row of 2,048 took 4.4 us with eight parts and 5.1 with eleven that way, so 3.0).
template <int PRE, typename TD>
__device__ __forceinline__ void add_parts4_by(float4& sum, const TD* p, int splits, size_t split_stride) {
  for (int k0 = 0; k0 < splits; k0 += PRE) {
    float4 d[PRE];
#pragma unroll
    for (int u = 0; u < PRE; ++u) d[u] = load4(p + (size_t)min(k0 + u, splits - 1) * split_stride);
#pragma unroll
    for (int u = 0; u < PRE; ++u) {
      const bool on = k0 + u < splits;
      sum.x = on ? sum.x + d[u].x : sum.x;
      sum.y = on ? sum.y + d[u].y : sum.y;
      sum.z = on ? sum.z + d[u].z : sum.z;
      sum.w = on ? sum.w + d[u].w : sum.w;
    }
  }
}
template <typename TD>
__device__ __forceinline__ float4 load_parts4(const TD* p, int splits, size_t split_stride) {
  if (splits == 1) return load4(p);
  float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
  if (splits == 2) add_parts4_by<2>(sum, p, splits, split_stride);
  else if (splits <= 4) add_parts4_by<4>(sum, p, splits, split_stride);
  else if (splits <= 8) add_parts4_by<8>(sum, p, splits, split_stride);
  else if (splits <= 12) add_parts4_by<12>(sum, p, splits, split_stride);
  else add_parts4_by<16>(sum, p, splits, split_stride);
  return sum;
}

// Whether a launch of one workgroup a row leaves the compute units room: then a row's time is its trips to memory, and its
// loads go out together.  From more than 1,024 threads a compute unit on the rows hide each other's trips, and what counts is
// the registers and instructions of all those loads.  Rows of 2,048, together against one after the other, 256 / 384 rows: 4
// parts 0.92 / 1.10 of the time in the norm in front of a sublayer, 0.96 / 1.18 in the one behind it, 0.98 / 1.22 there with a
// gate; one part 0.96 / 1.12, 1.01 / 1.17, 1.01 / 1.25; 4,096 rows with a gate 52 against 34 us.
static inline bool rows_are_few(int rows, int threads) { return (long)rows * threads <= 256L * 1024; }

// Four values of either type as they lie in memory: asked for early, converted where they are used (a conversion next to
// the load, behind the branch on the type, would wait for it).
struct Raw4 { uint4 u; };
__device__ __forceinline__ Raw4 load_raw4(const void* p, int dtype, int i) {
  Raw4 r;
  if (dtype == IA_F32) {
    r.u = *reinterpret_cast<const uint4*>((const float*)p + i);
  } else {
    const uint2 t = *reinterpret_cast<const uint2*>((const uint16_t*)p + i);
    r.u = make_uint4(t.x, t.y, 0u, 0u);
  }
  return r;
}
__device__ __forceinline__ float4 raw4_values(const Raw4& r, int dtype) {
  return dtype == IA_F32 ? make_float4(__uint_as_float(r.u.x), __uint_as_float(r.u.y), __uint_as_float(r.u.z),
                                       __uint_as_float(r.u.w))
                         : make_float4(__uint_as_float(r.u.x << 16), __uint_as_float(r.u.x & 0xffff0000u),
                                       __uint_as_float(r.u.y << 16), __uint_as_float(r.u.y & 0xffff0000u));
}

// Sine and cosine of position * frequency i.  With a table of float64 frequencies the product is formed in
// float64 and brought into [-pi, pi] there before the fp32 sine and cosine, so that the angle is good to
// 3e-7 rad at any position; with a table of fp32 frequencies the product is the fp32 one.
__device__ __forceinline__ void rope_sincos(int position, const void* __restrict__ table, int table_f64, int i,
                                            float& sn, float& cs) {
  if (table_f64) {
    const double a = (double)position * reinterpret_cast<const double*>(table)[i];
    const double turns = rint(a * 0.15915494309189535);                 // a / (2 pi)
    // 2 pi as a double is off by 2.4e-16: times a million turns still far below the fp32 sine's own error
    const double r = __builtin_fma(-turns, 6.283185307179586, a);
    sincosf((float)r, &sn, &cs);
  } else {
    sincosf((float)position * reinterpret_cast<const float*>(table)[i], &sn, &cs);
  }
}

// The rotation of one pair, in one fixed order of roundings (a product, then a fused multiply-add), so that
// every kernel that rotates gives the same bits.
__device__ __forceinline__ void rope_pair(float a, float b, float cs, float sn, float& lo, float& hi) {
  lo = __builtin_fmaf(a, cs, -(b * sn));
  hi = __builtin_fmaf(a, sn, b * cs);
}

// The activations between two products, by code (0: none): 1 the tanh form of GELU, 2 GELU, 3 the square of relu.
__device__ __forceinline__ float ia_activate(float z, int kind) {
  if (kind == 3) { const float r = fmaxf(z, 0.f); return r * r; }
  if (kind == 2) return 0.5f * z * (1.0f + erff(z * 0.7071067811865476f));
  if (kind == 1) return 0.5f * z * (1.0f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
  return z;
}

// Where the routed experts' products begin their walk over K, by the column of the result: every 512 columns at a chunk of 256 values of
// their own (a hash of the columns' number), from which they wrap around (moe.hip says why).  The tiles of few pairs and the grouped
// product of many both start there, so that a pair's result does not depend on how many share the step.
// Neighbouring tiles of the grouped product read the same rows of X, and fewer of those reads meet where their starts differ.  Its
// time against one start for all columns (mean of nine sizes of experts, with a gate and without, at 1,000 to 4,096 tokens): 1.008 at
// a start for every 256 columns, 0.995 at 512, 0.996 at 1,024, 0.999 at 2,048; 2,048 tokens to 2 of 16 experts without a gate of
// 1,408 x 2,048 take 148.6 us at 256, 143.3 at 512, 140.8 at 1,024 and 139.1 with one start.  The tiles (1 to 200 tokens) take 0.995,
// 1.008 and 1.024 of their time at 256 with 512, 1,024 and 2,048.
#define IA_EXPERT_CHUNK 256
__device__ __forceinline__ int ia_expert_first_chunk(int column, int K) {
  const unsigned chunks = (unsigned)(K + IA_EXPERT_CHUNK - 1) / IA_EXPERT_CHUNK;
  return (int)((((unsigned)(column / 512) * 0x9E3779B1u) >> 8) % chunks);
}

// Every lane's 16 bytes at src + AT, straight into LDS from lds + AT on, lane after lane (lds the same for the wave).  Written out: the
// compiler takes the builtin for an access of memory and of LDS at once, and with one under way it waits for all reads of LDS, the newest
// too, where it needs the oldest (prompt attention with heads of 128, two reads in flight over every product: 8,192 tokens of 32
// heads 515 us with the builtin, 504 so).  Nothing comes back in a register, and nobody
// but the caller waits: for vmcnt before a barrier, before LDS is read and before the workgroup ends.
// Two things the caller sees to, as the compiler does not look inside.  m0 is its own (it warns that m0 is not kept over such a statement): the
// builtin, or whatever else wants m0, does not go into one kernel with these.  And where src is the same for the wave it comes from scalar
// instructions: behind a vector instruction that writes it (v_readfirstlane) a load needs five instructions' distance, and has two here
// (the one that has to lie between the write of m0 and the load, and that write).  The distance in every load costs split products of few
// rows up to a seventh: 328 rows of 84 x 11,712 41.2 / 46.8 us, 278 of 612 x 8,448 in 2 17.8 / 19.7.  A test reads both from the assembly.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
template <int AT>
__device__ __forceinline__ void ia_load_to_lds(const char* src, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off offset:%2" ::"s"(lds), "v"(src), "n"(AT) : "memory", "m0");
}
// The same from src + at, src the same for the wave.
__device__ __forceinline__ void ia_load_to_lds(const char* src, uint32_t at, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(at), "s"(src) : "memory", "m0");
}
#pragma clang diagnostic pop
__device__ __forceinline__ uint32_t ia_lds_address(const char* p) {
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)p);
}

// The first key that a query at position p sees, from the mask's code: 0 all keys from 0; w > 0 a sliding
// window, the last w keys (p - w + 1 .. p); w < 0 chunks of -w positions counted from the request's start,
// the keys of the query's own chunk (floor(p / c) c .. p).  Never decreases with p.
__host__ __device__ __forceinline__ int ia_first_visible_key(int p, int window) {
  if (window > 0) return p - window + 1 > 0 ? p - window + 1 : 0;
  if (window < 0) return p < 0 ? 0 : p / (-window) * (-window);
  return 0;
}

#define IA_LAUNCH_CHECK()                          \
  do {                                             \
    hipError_t e__ = hipGetLastError();            \
    if (e__ != hipSuccess) return (int)e__;        \
  } while (0)
