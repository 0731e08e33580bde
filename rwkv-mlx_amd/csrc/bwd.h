// Pieces shared by the backward's kernels (backward.hip, bwd_f32.hip).
#pragma once

#include "common.h"

namespace rwkvmoe {

// The tokens routed to each expert (the counts f_e of the aux loss,
// moe.py:80-83), by the first 256 threads of one workgroup (every thread
// calls it: it holds barriers): 32 loads per thread in flight, LDS integer
// atomics.  h: 64 ints of LDS.
RWKV_DEV void count_selections(const int* __restrict__ inds, int nk, int E, int* h, int* __restrict__ cnt) {
  if (threadIdx.x < 64) h[threadIdx.x] = 0;
  __syncthreads();
  const __amdgpu_buffer_rsrc_t ri = buf_rsrc(inds, (unsigned)nk * 4);
  for (int b0 = 0; threadIdx.x < 256 && b0 < nk; b0 += 256 * 32) {
    unsigned v[32];
#pragma unroll
    for (int u = 0; u < 32; ++u) {
      const int j = b0 + u * 256 + (int)threadIdx.x;
      v[u] = buf_load4(ri, j < nk ? (unsigned)j * 4u : kOOB);
    }
#pragma unroll
    for (int u = 0; u < 32; ++u) {
      const int j = b0 + u * 256 + (int)threadIdx.x, e = (int)v[u];
      if (j < nk && e >= 0 && e < E) atomicAdd(&h[e], 1);
    }
  }
  __syncthreads();
  if ((int)threadIdx.x < E) cnt[threadIdx.x] = h[threadIdx.x];
}

}  // namespace rwkvmoe
