// Prompt attention with 32 rows of a query head a wave (part of attention_mfma.hip, for a head size of 128 or 256 and two or more query
// heads to a key/value head).
//
// A workgroup takes 64 rows (or, paired, 32 from each end of the request's new tokens) of up to HGW query heads of one key/value
// head: two waves a head, 32 rows each as two tiles of 16 columns.  Keys and values come in tiles of 64 keys, by loads straight into LDS,
// into rings of four stages: the keys of tile i + 3 and the values of tile i + 2 are asked for while tile i is worked on, half by
// half, with one bare barrier a tile.  (Heads of 256: up to two query heads, tiles of 32 keys, each its only half, a barrier each: rings of
// four stages fill LDS so.)
//   S^T[key, col] = K[key, :] . Q[col, :]       v_mfma_f32_16x16x32_bf16 over 32 head dims a step
//   O^T[dim, col] += V^T[dim, key] P^T[key, col] the same over 32 keys a step
// Heads of 128: row r of the S^T tile t (of a half's two) stands for the key 8 (r / 4) + r % 4 + 4 t of the half, so that the accumulators leave
// lane (col, q) with the keys 8 q .. 8 q + 7: what the second product wants of the probabilities, and 16 contiguous bytes of a row
// of V^T, as pages hold it.  Heads of 256 keep the order of the kernel with 16 rows a wave, row r of tile t the key 16 t + r: a lane has the keys
// 4 q .. 4 q + 3 and 16 + 4 q .. 16 + 4 q + 3, two reads of 8 bytes of V^T (3,000 tokens of 16 heads over 1 120 us, 116 in the order of
// heads of 128, which is another sum of the same numbers).
//
// What bounds it: with four heads a workgroup a SIMD has two such waves (LDS holds one workgroup a compute unit: one wave a SIMD with two
// heads, every other SIMD has none with one), whose matrix instructions take 2,176 cycles a tile, their exponentials and what goes with them
// some 1,700, and whose reads of LDS (256 KB a tile and compute unit, half of what waves of 16 rows need) 1,024 where 16 lanes find 16
// different places.  These have to run
// beside each other: a piece of a pair of exponentials of 32 keys' scores stands behind every product of the next 32's scores and every one of the
// probabilities of the 32 before, and a product waits for its own two reads, not for those asked for behind them (ia_load_to_lds).  The
// 8B shape's heads (32 over 8), waves of 16 rows / this kernel, us: 2,048 tokens 63 / 52, 4,096
// 164 / 134, 8,192 600 / 485 (1.13 PFLOP/s), 2,048 after 6,144 cached 271 / 217; under a window of 4,096 8,192 tokens 465 / 388.  (Every read
// waited for and keys where only 8 lanes found different places: 54, 141, 515, 227, 407.)  Heads of 256, 16 over 1: 2,047 tokens under a
// window of 1,024 60.5 / 57, 3,000 tokens 145 / 120, 4,096 198 / 178; 16 over 8, 8,192 732 / 645 (0.85 PFLOP/s): one wave a SIMD, whose
// 66 products of
// 32 keys take 1,056 of the 2,500 cycles that a tile takes it; 512 registers hold no more columns.  Short ranges
// of keys are the other kernel's, by the same order of sums (a prompt of 20 tokens 5.9 / 8.9, of 257 13.9 / 15.5: a longer start, and a
// wave's work one after the other); the line is drawn where launches are shaped.  With the products in a row and the exponentials behind them
// 8,192 tokens took 590 where this took 508; with tests for a wave's first and last half inside the loop 587; with a mask in every half of a
// wave that has rows to spare 4,016 tokens of 4 heads took 111, 80 without.
// Heads of 64 gained nothing (2,048 tokens 48 / 54, 8,192 438 / 418), one query head to a key/value head lost (2,000 tokens of 8 heads 53 / 67).
//
// In LDS the 16-byte piece c of row r (a key's values; a dim's keys) lies at position c ^ s(r), s(key) = key % 4 + 4 (key / 8 % 4),
// s(dim) = dim % 8, for heads of 256 s(key) = key % 16, s(dim) = dim / 4 % 4: the 16 lanes that read 16 bytes together find 16 different places,
// the 32 that read 8 bytes together 32.
#pragma once

#define PW_KT (HD <= 128 ? 64 : 32)      // keys a tile
#define PW_STAGES 4
#define PW_INLINE __attribute__((always_inline))
#define PW_BT 4096                      // block-table entries kept in LDS

constexpr bool PW_EIGHTS = IA_PREFILL_EIGHTS;                 // the order of keys in a half, see above
constexpr int PW_HALVES = PW_KT / 32, PW_VP = PW_KT / 8;      // 32 keys each; pieces of a dim's row of V^T
constexpr int PW_K_BYTES = PW_KT * HD * 2, PW_V_BYTES = VD * PW_KT * 2;
constexpr int PW_LDS = PW_STAGES * (PW_K_BYTES + PW_V_BYTES) + PW_BT * 4;

typedef f32x4 pw_scores[2][2];          // of 32 keys: [tile of 16][column]

template <int HGW, bool WINDOW>
__global__ __launch_bounds__(HGW * 128, HD <= 128 ? 2 : 1) void attn_prefill_wide_kernel(
    const uint16_t* __restrict__ q, int q_row_stride, const uint16_t* __restrict__ k_pages, const uint16_t* __restrict__ v_pages,
    uint16_t* __restrict__ out, int out_row_stride, const int* __restrict__ seq_starts, const int* __restrict__ seq_ctx,
    const int* __restrict__ block_tables, int bt_stride, const int* __restrict__ tiles, int nh, int nkv, int ps_shift, int num_pages,
    float scale_log2, int window, int paired, const float* __restrict__ sinks) {
  constexpr int NW = 2 * HGW, THREADS = NW * 64;
  constexpr int KS = HD / 32;                                           // steps of the scores' product
  constexpr int KF = PW_K_BYTES / 1024 / NW, VF = PW_V_BYTES / 1024 / NW, LOADS = KF + VF;      // a wave's loads a tile
  static_assert(HD % 64 == 0 && VD % 64 == 0 && KF >= 1 && VF >= 1, "whole loads for every wave");
  extern __shared__ __attribute__((aligned(1024))) char pw_lds[];
  char* const k_lds = pw_lds;
  char* const v_lds = pw_lds + PW_STAGES * PW_K_BYTES;
  const uint32_t k_first = ia_lds_address(k_lds), v_first = k_first + PW_STAGES * PW_K_BYTES;
  int* const s_bt = reinterpret_cast<int*>(v_lds + PW_STAGES * PW_V_BYTES);
  __shared__ int s_poison;

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), j = lane & 15, qd = lane >> 4;
  // waves go to the SIMDs in turn: the row blocks are turned from the fourth wave on, so that every SIMD has waves of both
  // and those that run out of keys early leave none empty
  const int hgw = wave >> 1, rblock = (wave ^ (wave >> 2)) & 1;
  // all heads of the first tile, then of the next (the host lists the tiles with the most keys first)
  const int lin = blockIdx.y * gridDim.x + blockIdx.x;
  const int tile = lin / gridDim.y, by = lin - tile * gridDim.y;
  const int sidx = tiles[2 * tile], row0 = tiles[2 * tile + 1];
  const int G = nh / nkv, HC = (G + HGW - 1) / HGW;
  const int g = by / HC, h_in = (by - g * HC) * HGW + hgw;
  const int h = g * G + (h_in < G ? h_in : 0);
  const int qstart = seq_starts[sidx], qlen = seq_starts[sidx + 1] - qstart, ctx = seq_ctx[sidx];
  int rb, first_row, last_row;
  bool wave_live;
  if (paired) {
    const int halves = (qlen + 31) >> 5, ha = row0 >> 6, hb = halves - 1 - ha;      // hb >= ha
    rb = (rblock == 0 ? ha : hb) * 32;
    wave_live = rb < qlen && (rblock == 0 || hb > ha);
    first_row = ha * 32;
    last_row = (hb * 32 + 32 < qlen ? hb * 32 + 32 : qlen) - 1;
  } else {
    rb = row0 + rblock * 32;
    wave_live = rb < qlen;
    first_row = row0;
    last_row = (row0 + 64 < qlen ? row0 + 64 : qlen) - 1;
  }
  wave_live = wave_live && h_in < G;
  if (tid == 0) s_poison = 0;

  // ---- keys: those that the workgroup's rows may see, those that this wave's may
  const int key_hi = ctx + last_row, key_lo = ia_first_visible_key(ctx + first_row, window);
  const int wave_last = rb + 31 < qlen ? rb + 31 : qlen - 1;
  const int wave_hi = ctx + wave_last;
  const int wave_lo_last = ia_first_visible_key(wave_hi, window);
  const int t_begin = key_lo / PW_KT, t_end = key_hi / PW_KT;
  // halves of tiles (32 keys): the wave's first and last, the last of its first 16 rows, the first of the others
  const int w_end = wave_live ? wave_hi / 32 : -2, w_begin = wave_live ? ia_first_visible_key(ctx + rb, window) / 32 : 0;
  const int end0 = (ctx + (rb + 15 < qlen ? rb + 15 : qlen - 1)) / 32, begin1 = WINDOW ? ia_first_visible_key(ctx + rb + 16, window) / 32 : 0;
  const int bt_first = key_lo >> ps_shift, ps = 1 << ps_shift;

  // ---- queries as B operands; columns c = 0, 1 are rows rb + j and rb + 16 + j
  bf16x8_t qreg[2][KS];
  float m[2];
  f32x4 o[NSV][2], lacc[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int row = rb + 16 * c + j;
    const bool ok = wave_live && row < qlen;
    const uint16_t* qrow = q + (size_t)(qstart + (ok ? row : first_row)) * q_row_stride + (size_t)h * HD;
#pragma unroll
    for (int st = 0; st < KS; ++st) qreg[c][st] = *reinterpret_cast<const bf16x8_t*>(qrow + st * 32 + qd * 8);
    m[c] = ok ? -INFINITY : 0.f;         // a column without a row never asks for a reference point
    lacc[c] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int n = 0; n < NSV; ++n) o[n][c] = (f32x4){0.f, 0.f, 0.f, 0.f};
  }
  {
    const int* bt = block_tables + (size_t)sidx * bt_stride;
    const int first = key_lo >> ps_shift, count = (key_hi >> ps_shift) - first + 1;
    for (int i = tid; i < count; i += THREADS) s_bt[i] = bt[first + i];
  }
  // the queries are here before the first load into LDS: waiting for them behind it would wait for all of these too
  static_assert(KS % 4 == 0, "all queries of a lane");
#pragma unroll
  for (int st = 0; st < KS; st += 4)
    asm volatile("" : "+v"(qreg[0][st]), "+v"(qreg[0][st + 1]), "+v"(qreg[0][st + 2]), "+v"(qreg[0][st + 3]), "+v"(qreg[1][st]),
                 "+v"(qreg[1][st + 1]), "+v"(qreg[1][st + 2]), "+v"(qreg[1][st + 3]));
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int st = 0; st < KS; ++st)
      if (!(wave_live && rb + 16 * c + j < qlen)) qreg[c][st] = __builtin_bit_cast(bf16x8_t, make_uint4(0u, 0u, 0u, 0u));
  const f32x4 none = {0.f, 0.f, 0.f, 0.f};
  const bf16x8_t ones = __builtin_bit_cast(bf16x8_t, make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u));

  // ---- loads.  A wave brings KG groups of eight keys, KF / KG loads each, and VF loads of a tile's keys of VDIMS dims each, of which a
  // lane has the same eight every time: eight keys lie in one page.  Groups beyond the range come from the page at its end (scores of theirs are
  // masked, values zeroed).
  constexpr int KG = PW_KT / 8 / NW >= 1 ? PW_KT / 8 / NW : 1, KL = KF / KG;
  static_assert(KG * KL == KF && KG * NW == PW_KT / 8, "whole groups");
  const uint32_t k_page = (uint32_t)nkv * (uint32_t)ps * (HD * 2), v_page = (uint32_t)nkv * (uint32_t)ps * (VD * 2);     // bytes
  const char* const k_base = reinterpret_cast<const char*>(k_pages) + (size_t)g * ps * (HD * 2);
  const char* const v_base = reinterpret_cast<const char*>(v_pages) + (size_t)g * VD * (ps * 2);
  const int k_row = lane / (HD / 8);
  // s(key) of the rows of a load: bits 2 and 3 are the group's number's lowest (heads of 256: bits 1 and 2 the load's of the group, bit 3 the
  // group's number's lowest)
  const uint32_t k_lane_at = (uint32_t)(k_row * HD * 2 + (((lane & (HD / 8 - 1)) ^ (k_row & 3)) * 16));
  constexpr int VDIMS = 64 / PW_VP;
  auto v_swizzle = [&](int dim) PW_INLINE { return PW_KT == 64 ? dim & 7 : (dim >> 2) & 3; };
  const int v_key = 8 * ((lane & (PW_VP - 1)) ^ v_swizzle(lane / PW_VP));
  const uint32_t v_lane_at = (uint32_t)(VDIMS * wave * VF + lane / PW_VP) * (uint32_t)(ps * 2), v_step = (uint32_t)(2 * VDIMS * ps);
  const int last_page = (key_hi >> ps_shift) - bt_first;
  bool bad = false;
  int k_pg[KG], v_pg;
  auto page_of = [&](int key) PW_INLINE { return s_bt[min(max((key >> ps_shift) - bt_first, 0), last_page)]; };
  auto pages_of_k = [&](int t) PW_INLINE {
#pragma unroll
    for (int f = 0; f < KG; ++f) k_pg[f] = page_of(t * PW_KT + 8 * (wave * KG + f));
  };
  auto pages_of_v = [&](int t) PW_INLINE { v_pg = page_of(t * PW_KT + v_key); };
  auto load_k = [&](int t, int slot) PW_INLINE {
#pragma unroll
    for (int f = 0; f < KG; ++f) {
      const bool ok = (unsigned)k_pg[f] < (unsigned)num_pages;
      bad |= !ok;
      const uint32_t in_page = (uint32_t)((t * PW_KT + 8 * (wave * KG + f)) & (ps - 1)) * (HD * 2);
      const uint32_t at = k_lane_at ^ (PW_EIGHTS ? ((wave * KG + f) & 3) * 64u : ((wave * KG + f) & 1) * 128u);
      const char* const page = k_base + (uint64_t)(uint32_t)(ok ? k_pg[f] : 0) * k_page;
      const char* src = page + (in_page + at);
      // a group's loads follow each other in the page and in LDS alike: the instruction's offset moves both
      const uint32_t dst = k_first + slot * PW_K_BYTES + 1024 * KL * (wave * KG + f);
      ia_load_to_lds<0>(src, dst);
      if constexpr (KL == 2) ia_load_to_lds<1024>(src, dst);
      if constexpr (KL == 4) {                    // two keys a load, of the group's eight
        ia_load_to_lds<1024>(page + (in_page + (at ^ 32u)), dst);
        ia_load_to_lds<2048>(page + (in_page + (at ^ 64u)), dst);
        ia_load_to_lds<3072>(page + (in_page + (at ^ 96u)), dst);
      }
      static_assert(PW_EIGHTS ? (HD == 128 && KL <= 2) : (HD == 256 && KL == 4), "a group's loads");
    }
  };
  auto load_v = [&](int t, int slot) PW_INLINE {
    const bool ok = (unsigned)v_pg < (unsigned)num_pages;
    bad |= !ok;
    const uint32_t in_page = (uint32_t)((t * PW_KT + v_key) & (ps - 1)) * 2u;
    const char* src = v_base + ((uint64_t)(uint32_t)(ok ? v_pg : 0) * v_page + (v_lane_at + in_page));
#pragma unroll
    for (int f = 0; f < VF; ++f) ia_load_to_lds<0>(src + (uint64_t)(f * v_step), v_first + slot * PW_V_BYTES + 1024 * (wave * VF + f));
  };

  // ---- reads: this lane's row and pieces
  const int k_lane = (PW_EIGHTS ? 8 * (j >> 2) + (j & 3) : j) * (HD * 2), v_lane = j * (PW_KT * 2);
  const int v_piece0 = PW_EIGHTS ? (qd ^ v_swizzle(j)) * 16 : ((qd >> 1) ^ v_swizzle(j)) * 16 + (qd & 1) * 8;
  const int v_piece1 = ((4 + qd) ^ v_swizzle(j)) * 16;                  // (of 64 keys alone)
  const int v_other = (v_piece0 & 32) ? -32 : 32;                       // from the lane's keys of the first 16 to those of the others
  int k_piece[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) k_piece[s] = k_lane + ((4 * s + qd) ^ j) * 16;
  auto read_k = [&](const char* half, int t, int st) PW_INLINE {        // tile t of the half's two, step st of the head dims
    return *reinterpret_cast<const bf16x8_t*>(half + k_piece[st & 3] + t * ((PW_EIGHTS ? 4 : 16) * HD * 2) + (st >> 2) * 256);
  };
  // `values`: the stage of the half's tile, with this lane's place in it
  auto read_v = [&](const char* values, int n) PW_INLINE {
    if constexpr (PW_EIGHTS) {
      return *reinterpret_cast<const bf16x8_t*>(values + n * (16 * PW_KT * 2));
    } else {
      const uint2 a = *reinterpret_cast<const uint2*>(values + n * (16 * PW_KT * 2));
      const uint2 b = *reinterpret_cast<const uint2*>(values + v_other + n * (16 * PW_KT * 2));
      return __builtin_bit_cast(bf16x8_t, make_uint4(a.x, a.y, b.x, b.y));
    }
  };

  typedef uint32_t packed[2][4];        // probabilities as B operands: [column][pairs of keys]
  float emax[2];
  // the two exponentials of pair i (of four) of column c of 32 keys' scores, packed
  auto pair_of = [&](const pw_scores& s, packed& pk, int c, int i, float neg_m) PW_INLINE {
    const int t = i >> 1, r = 2 * (i & 1);
    const f32x2_t e = {__builtin_amdgcn_exp2f(fmaf(s[t][c][r], scale_log2, neg_m)), __builtin_amdgcn_exp2f(fmaf(s[t][c][r + 1], scale_log2, neg_m))};
    emax[c] = fmaxf(emax[c], fmaxf(e[0], e[1]));
    pk[c][i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(e, bf16x2_t));
  };
  // keys that a column does not see
  auto mask = [&](pw_scores& s, int t0) PW_INLINE {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int row = rb + 16 * c + j, last = ctx + row, first = ia_first_visible_key(last, window);
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int key = t0 + (PW_EIGHTS ? 8 * qd + 4 * t : 16 * t + 4 * qd) + r;
          s[t][c][r] = (key <= last && key >= first) ? s[t][c][r] : -INFINITY;
        }
    }
  };
  // The reference point of the exponentials follows the running maximum lazily, as in the kernel above: only when an exponential against
  // it comes out above 2^PF_LAZY, or a column has none yet, it moves, the accumulators are rescaled and the exponentials taken again.
  auto settle = [&](const pw_scores& s, packed& pk) PW_INLINE {
    if (!__any(emax[0] > PF_LAZY_EXP || emax[1] > PF_LAZY_EXP || m[0] == -INFINITY || m[1] == -INFINITY)) return;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      float top = -INFINITY;
#pragma unroll
      for (int t = 0; t < 2; ++t) top = fmaxf(top, fmaxf(fmaxf(s[t][c][0], s[t][c][1]), fmaxf(s[t][c][2], s[t][c][3])));
      top *= scale_log2;                 // (the scale is positive)
      top = fmaxf(top, __shfl_xor(top, 16, IA_WAVE));
      top = fmaxf(top, __shfl_xor(top, 32, IA_WAVE));
      const float m_new = (top > m[c] + PF_LAZY) ? top : m[c];          // never moves to -inf
      const float m_safe = (m_new == -INFINITY) ? 0.f : m_new;
      const float corr = __builtin_amdgcn_exp2f(m[c] - m_safe);         // 1 where nothing moved, 0 at the start
      lacc[c] *= corr;
#pragma unroll
      for (int n = 0; n < NSV; ++n) o[n][c] *= corr;
      m[c] = m_new;
#pragma unroll
      for (int i = 0; i < 4; ++i) pair_of(s, pk, c, i, -m_safe);
    }
  };
  auto scores = [&](pw_scores& s, const char* half) PW_INLINE {
#pragma unroll
    for (int x = 0; x < 2 * KS; ++x) {
      const bf16x8_t a = read_k(half, x & 1, x >> 1);
      s[x & 1][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, qreg[0][x >> 1], x < 2 ? none : s[x & 1][0], 0, 0, 0);
      s[x & 1][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, qreg[1][x >> 1], x < 2 ? none : s[x & 1][1], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);                     // one read's registers at a time
    }
  };

  // half x of the keys: its scores `cur` become probabilities `pk`, while the scores of half x + 1 (keys at `half`) come into `next` and
  // the probabilities `before` of half x - 1 weigh its `values` into the accumulators: three halves' work, none of
  // which waits for another's.  One path for every half: a wave's first has no probabilities before it (zeros, against values that it
  // multiplies with anyway), its last no scores behind it (of keys that are there; nobody looks at them).
  // 16 rows meet the halves that hold a key some of them may see, and no other: 0 times a value that is not finite is NaN.  So what a column
  // has gathered when its first half's scores are weighed (the values of halves in front of its window or chunk, times 0: nothing, or
  // NaN) is cleared, and the last half's values, which can be beyond the first 16 rows, come in behind the loop.
  auto part = [&](int x, pw_scores& cur, pw_scores& next, packed& pk, const packed& before, const char* half, const char* values) PW_INLINE {
    const int t0 = x * 32;
    // (columns without a row need no mask: their queries are zero, and what they gather goes nowhere)
    if ((t0 + 31 > ctx + rb) || (WINDOW && t0 < wave_lo_last)) mask(cur, t0);
    const float neg[2] = {(m[0] == -INFINITY) ? 0.f : -m[0], (m[1] == -INFINITY) ? 0.f : -m[1]};
    emax[0] = emax[1] = 0.f;
    constexpr int NY = NSV;                                  // turns: a read of keys and one of values, two products each
    static_assert(2 * KS == NSV, "as many reads of keys as of values");
    bf16x8_t ak[3], av[3], p[2];
    f32x2_t e;
#pragma unroll
    for (int y = 0; y < 2; ++y) {
      ak[y] = read_k(half, y & 1, y >> 1);
      av[y] = read_v(values, y);
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) p[c] = __builtin_bit_cast(bf16x8_t, make_uint4(before[c][0], before[c][1], before[c][2], before[c][3]));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < 2; ++c) lacc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, p[c], lacc[c], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int y = 0; y < NY; ++y) {
      if (y + 2 < NY) {
        ak[(y + 2) % 3] = read_k(half, (y + 2) & 1, (y + 2) >> 1);
        av[(y + 2) % 3] = read_v(values, y + 2);
      }
      // the turn's pair of exponentials, a piece behind each of its four products (with twice the turns: of two turns' eight)
      constexpr int SLOW = NY / 8;
      static_assert(NY == 8 || NY == 16, "eight pairs of exponentials");
      auto piece = [&](int place) {
        const int stage = SLOW == 1 ? place : (place & 1) ? 2 * (y & 1) + (place >> 1) : 4;
        {
          const int i = y / SLOW, c = i >> 2, t = (i >> 1) & 1, r = 2 * (i & 1);
          if (stage == 0) e = (f32x2_t){fmaf(cur[t][c][r], scale_log2, neg[c]), fmaf(cur[t][c][r + 1], scale_log2, neg[c])};
          if (stage == 1) e[0] = __builtin_amdgcn_exp2f(e[0]);
          if (stage == 2) e[1] = __builtin_amdgcn_exp2f(e[1]);
          if (stage == 3) {
            pk[c][i & 3] = __builtin_bit_cast(uint32_t, __builtin_convertvector(e, bf16x2_t));
            emax[c] = fmaxf(emax[c], fmaxf(e[0], e[1]));
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      };
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        next[y & 1][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ak[y % 3], qreg[c][y >> 1], y < 2 ? none : next[y & 1][c], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        piece(2 * c);
        o[y][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[y % 3], p[c], o[y][c], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        piece(2 * c + 1);
      }
    }
    settle(cur, pk);
    if constexpr (WINDOW) {
      if (x == w_begin) {
#pragma unroll
        for (int n = 0; n < NSV; ++n) o[n][0] = none;
      }
      if (x == begin1) {
#pragma unroll
        for (int n = 0; n < NSV; ++n) o[n][1] = none;
      }
    }
  };
  auto barrier = [&] {                  // behind all loads but those of the round before
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(LOADS) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  // asked for as if by the rounds before: keys of t_begin; keys of the next tile and values of t_begin; keys and values behind those
  __syncthreads();
  pages_of_k(t_begin);
  load_k(t_begin, 0);
  pages_of_k(t_begin + 1);
  pages_of_v(t_begin);
  load_k(t_begin + 1, 1);
  load_v(t_begin, 0);
  barrier();
  pages_of_k(t_begin + 2);
  pages_of_v(t_begin + 1);
  load_k(t_begin + 2, 2);
  load_v(t_begin + 1, 1);
  pages_of_k(t_begin + 3);
  pages_of_v(t_begin + 2);
  pw_scores sa, sb;
  packed pa, pb;
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    sa[0][c] = sa[1][c] = sb[0][c] = sb[1][c] = none;
#pragma unroll
    for (int i = 0; i < 4; ++i) pa[c][i] = pb[c][i] = 0u;
  }
  // A round: everybody's loads and barrier, for every tile of the workgroup's range.  A wave has work in those of its own range.
  auto round = [&](int i) PW_INLINE {
    const int slot = (i - t_begin) & 3;
    barrier();                          // keys up to tile i + 1 and values up to tile i are there; nobody reads keys of tile i - 1 or values of i - 2 any more
    load_k(i + 3, (slot + 3) & 3);      // (past the range: of its last page, for nobody, so that every round has as many loads under way)
    load_v(i + 2, (slot + 2) & 3);
    pages_of_k(i + 4);
    pages_of_v(i + 3);
    // values of keys that no row sees are not the request's: zero them in LDS (the tiles at the ends of the range)
    const int t0 = i * PW_KT;
    if (t0 < key_lo || t0 + PW_KT - 1 > key_hi) {
      for (int at = tid; at < VD * PW_VP; at += THREADS) {
        const int dim = at / PW_VP, key = t0 + 8 * ((at & (PW_VP - 1)) ^ v_swizzle(dim));
        if (key >= key_lo && key + 7 <= key_hi) continue;
        uint16_t* const v = reinterpret_cast<uint16_t*>(v_lds + slot * PW_V_BYTES + at * 16);
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (key + e < key_lo || key + e > key_hi) v[e] = 0;
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    }
  };
  int i = t_begin;
  if (WINDOW) {
    for (; i < w_begin / PW_HALVES; ++i) round(i);
  }
  const int first = i;
  if (wave_live) scores(sa, k_lds + ((i - t_begin) & 3) * PW_K_BYTES);
  bool in_first;                        // the last half was a tile's first, or of tiles of one half an even one
  const char* values;                   // the last half's: of a tile that is there until the next round
  if constexpr (PW_HALVES == 2) {
    auto even = [&]() PW_INLINE {
      const int slot = (i - t_begin) & 3;
      const char* const here = v_lds + slot * PW_V_BYTES + v_lane;
      part(2 * i, sa, sb, pa, pb, k_lds + slot * PW_K_BYTES + 32 * HD * 2,
           i == first ? here + v_piece0 : v_lds + ((slot + 3) & 3) * PW_V_BYTES + v_lane + v_piece1);
      return here;
    };
    for (; 2 * i < w_end; ++i) {
      round(i);
      const char* const here = even();
      part(2 * i + 1, sb, sa, pb, pa, k_lds + (((i - t_begin) + 1) & 3) * PW_K_BYTES, here + v_piece0);
    }
    in_first = 2 * i == w_end;
    if (in_first) {
      round(i);
      even();
      ++i;
    }
    values = v_lds + ((i - 1 - t_begin) & 3) * PW_V_BYTES + v_lane + (in_first ? v_piece0 : v_piece1);
  } else {
    auto keys_of = [&](int x) PW_INLINE { return k_lds + ((x - t_begin) & 3) * PW_K_BYTES; };
    auto values_of = [&](int x) PW_INLINE { return v_lds + ((x - t_begin) & 3) * PW_V_BYTES + v_lane + v_piece0; };
    for (; i < w_end; i += 2) {
      round(i);
      part(i, sa, sb, pa, pb, keys_of(i + 1), values_of(i == first ? i : i - 1));
      round(i + 1);
      part(i + 1, sb, sa, pb, pa, keys_of(i + 2), values_of(i));
    }
    in_first = i == w_end;
    if (in_first) {
      round(i);
      part(i, sa, sb, pa, pb, keys_of(i + 1), values_of(i == first ? i : i - 1));
      ++i;
    }
    values = values_of(i - 1);
  }
  if (wave_live) {
    bf16x8_t p[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const uint4 a = make_uint4(pa[c][0], pa[c][1], pa[c][2], pa[c][3]), b = make_uint4(pb[c][0], pb[c][1], pb[c][2], pb[c][3]);
      p[c] = __builtin_bit_cast(bf16x8_t, in_first ? a : b);
      lacc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, p[c], lacc[c], 0, 0, 0);
    }
#pragma unroll
    for (int n = 0; n < NSV; ++n) {
      const bf16x8_t av = read_v(values, n);
      o[n][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, p[1], o[n][1], 0, 0, 0);
      if (end0 == w_end) o[n][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, p[0], o[n][0], 0, 0, 0);
    }
  }
  for (; i <= t_end; ++i) round(i);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // the loads asked for past the end
  if (bad) s_poison = 1;      // a key that is needed has no page in the block table: the result is NaN
  __syncthreads();
  const bool poison = s_poison != 0;
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    if (!wave_live || rb + 16 * c + j >= qlen) continue;
    float lsum = lacc[c][0];
    if (sinks) lsum += exp2f(sinks[h] * 1.4426950408889634f - m[c]);
    const float inv = poison ? __uint_as_float(0x7fc00000u) : 1.0f / lsum;
    uint16_t* const orow = out + (size_t)(qstart + rb + 16 * c + j) * out_row_stride + (size_t)h * VD + 4 * qd;
#pragma unroll
    for (int n = 0; n < NSV; ++n) {
      uint2 w;
      w.x = two_bf16_bits(o[n][c][0] * inv, o[n][c][1] * inv);
      w.y = two_bf16_bits(o[n][c][2] * inv, o[n][c][3] * inv);
      *reinterpret_cast<uint2*>(orow + n * 16) = w;
    }
  }
}

template <int HGW, bool WINDOW>
static int launch_prefill_wide(dim3 grid, const void* q, int q_row_stride, const void* k_pages, const void* v_pages, void* out,
                               int out_row_stride, const int* seq_starts, const int* seq_ctx, const int* block_tables, int bt_stride,
                               const int* tiles, int nh, int nkv, int ps, int num_pages, float scale_log2, int window, int paired,
                               const float* sinks, hipStream_t stream) {
  static bool configured = false;
  if (!configured) {
    const hipError_t e = hipFuncSetAttribute((const void*)attn_prefill_wide_kernel<HGW, WINDOW>, hipFuncAttributeMaxDynamicSharedMemorySize, PW_LDS);
    if (e != hipSuccess) return (int)e;
    configured = true;
  }
  int shift = 0;
  while ((1 << shift) < ps) ++shift;
  attn_prefill_wide_kernel<HGW, WINDOW><<<grid, HGW * 128, PW_LDS, stream>>>(
      (const uint16_t*)q, q_row_stride, (const uint16_t*)k_pages, (const uint16_t*)v_pages, (uint16_t*)out, out_row_stride, seq_starts,
      seq_ctx, block_tables, bt_stride, tiles, nh, nkv, shift, num_pages, scale_log2, window, paired, sinks);
  IA_LAUNCH_CHECK();
  return IA_OK;
}
