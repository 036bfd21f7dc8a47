// The parts of a head's keys (attention of single tokens) put together: outputs part_o [.., parts, VD], each against its
// own reference point, and part_ml [.., parts, 2], that point (in powers of two) and the sum of the weights.  One wave
// takes 64 channels of one (token, head).  Bound by trips to memory: the statistics and the first PRE parts' outputs are
// asked for together, further ones PRE at a time (with sixteen, eleven parts of 256 channels take 4.5 us, and 5.4 with one
// load after the other behind the fourth; for up to four parts four do, the other twelve cost 0.2 us there).  The parts are
// added in the order of their index.
#pragma once
#include "common.h"

struct JoinedParts {
  float sum;        // the channel's sum over the parts, against `top`
  float weight;     // the weights' sum, against `top`
  float top;        // the largest reference point
};

template <int PRE>
__device__ __forceinline__ JoinedParts join_parts_by(const float* __restrict__ part_o, const float* __restrict__ part_ml,
                                                     size_t rec0, int parts, int vd, int dim) {
  const int lane = threadIdx.x & 63, dc = dim < vd ? dim : vd - 1;
  float v[PRE];
#pragma unroll
  for (int j = 0; j < PRE; ++j) v[j] = part_o[(rec0 + (j < parts ? j : 0)) * vd + dc];
  float M = -INFINITY;
  for (int s = lane; s < parts; s += 64) M = fmaxf(M, part_ml[(rec0 + s) * 2]);
  M = wave_max(M);
  float acc = 0.f, L = 0.f;
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
      if (s0 + j0 > 0) {
#pragma unroll
        for (int j = 0; j < PRE; ++j) v[j] = part_o[(rec0 + min(s0 + j0 + j, parts - 1)) * vd + dc];
      }
#pragma unroll
      for (int j = 0; j < PRE; ++j) {
        if (j0 + j >= here) break;
        L += __shfl(wl, j0 + j, IA_WAVE);
        const float wj = __shfl(wgt, j0 + j, IA_WAVE);
        acc += (wj != 0.f) ? wj * v[j] : 0.f;              // an empty part holds zeros
      }
    }
  }
  return JoinedParts{acc, L, M};
}

__device__ __forceinline__ JoinedParts join_parts(const float* __restrict__ part_o, const float* __restrict__ part_ml,
                                                  size_t rec0, int parts, int vd, int dim) {
  return parts <= 4 ? join_parts_by<4>(part_o, part_ml, rec0, parts, vd, dim)
                    : join_parts_by<16>(part_o, part_ml, rec0, parts, vd, dim);
}
