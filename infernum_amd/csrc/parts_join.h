// The parts of a head's keys (attention of single tokens) put together: outputs part_o [.., parts, VD], each against its
// own reference point, and part_ml [.., parts, 2], that point (in powers of two) and the sum of the weights.  One wave
// takes 64 NC channels of one (token, head), a lane every 64th from `dim` on.  Bound by trips to memory: the statistics and the
// first PRE parts' outputs are asked for together, further ones PRE at a time (with sixteen, eleven parts of 256 channels take
// 4.5 us, and 5.4 with one load after the other behind the fourth; for up to four parts four do, the other twelve cost 0.2 us
// there; joined_at_once says how many).  The parts are added in the order of their index.
#pragma once
#include "common.h"

template <int NC>
struct JoinedParts {
  float sum[NC];    // the channels' sums over the parts, against `top`
  float weight;     // the weights' sum, against `top`
  float top;        // the largest reference point
};

template <int PRE, int NC>
__device__ __forceinline__ JoinedParts<NC> join_parts(const float* __restrict__ part_o, const float* __restrict__ part_ml,
                                                      size_t rec0, int parts, int vd, int dim) {
  const int lane = threadIdx.x & 63;
  float v[PRE][NC];
  const auto ask = [&](int first) {
#pragma unroll
    for (int j = 0; j < PRE; ++j)
#pragma unroll
      for (int c = 0; c < NC; ++c) v[j][c] = part_o[(rec0 + min(first + j, parts - 1)) * vd + min(dim + 64 * c, vd - 1)];
  };
  ask(0);
  float M = -INFINITY;
  for (int s = lane; s < parts; s += 64) M = fmaxf(M, part_ml[(rec0 + s) * 2]);
  M = wave_max(M);
  JoinedParts<NC> J;
#pragma unroll
  for (int c = 0; c < NC; ++c) J.sum[c] = 0.f;
  J.weight = 0.f;
  J.top = M;
  for (int s0 = 0; s0 < parts; s0 += 64) {
    const int s = s0 + lane;
    float wgt = 0.f, wl = 0.f;
    if (s < parts) {
      const float ms = part_ml[(rec0 + s) * 2];
      wgt = (ms == -INFINITY) ? 0.f : exp2f(ms - M);
      wl = wgt * part_ml[(rec0 + s) * 2 + 1];
    }
    const int here = min(64, parts - s0);
    for (int j0 = 0; j0 < here; j0 += PRE) {
      if (s0 + j0 > 0) ask(s0 + j0);
#pragma unroll
      for (int j = 0; j < PRE; ++j) {
        if (j0 + j >= here) break;
        J.weight += __shfl(wl, j0 + j, IA_WAVE);
        const float wj = __shfl(wgt, j0 + j, IA_WAVE);
#pragma unroll
        for (int c = 0; c < NC; ++c) J.sum[c] += (wj != 0.f) ? wj * v[j][c] : 0.f;              // an empty part holds zeros
      }
    }
  }
  return J;
}

// How many parts' outputs a launch that joins so many asks for at once.
static inline int joined_at_once(int parts) { return parts <= 2 ? 2 : parts <= 4 ? 4 : 16; }
