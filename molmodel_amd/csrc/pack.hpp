// pack.hpp -- the pair kernel's packed inputs of one group.
#pragma once
#include "mm_common.hpp"

namespace mmamd {

// FP64 first-site position, FP32 offsets from it with the charges, site count
// and mask/type bytes of the group at sorted slot gs; returns the position
__device__ __forceinline__ double4 pack_group(int gs, int s0, int ns, int info,
                                              const double *__restrict__ r,
                                              const double *__restrict__ q, int N,
                                              double4 *__restrict__ gpos, float4 *__restrict__ spk,
                                              int2 *__restrict__ gmeta) {
  const double x0 = r[s0], y0 = r[N + s0], z0 = r[2 * N + s0];
  const double4 p = make_double4(x0, y0, z0, 0.0);
  gpos[gs] = p;
#pragma unroll
  for (int k = 0; k < MAXS; k++) {
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (k < ns) {
      const int sk = s0 + k;
      v = make_float4((float)(r[sk] - x0), (float)(r[N + sk] - y0), (float)(r[2 * N + sk] - z0),
                      ((info >> (8 * k)) & SITE_HAS_Q) ? (float)q[sk] : 0.f);
    }
    spk[(long)gs * MAXS + k] = v;
  }
  gmeta[gs] = make_int2(ns, info);
  return p;
}

}  // namespace mmamd
