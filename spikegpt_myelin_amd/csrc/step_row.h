// Pieces of the one-token block step's row work (layer norm over a row held by
// a 256-thread workgroup, LIF update), shared by the row kernel and by the
// projections that take the row along.
#pragma once
#include "../../include/wkv_hip.h"
#include "wkv_common.h"

namespace wkv {

constexpr int kStepThreads = 256;

enum StepPre : int {
  kPreEmbed = WKV_STEP_PRE_EMBED,
  kPreLif = WKV_STEP_PRE_LIF,
  kPreGateLif = WKV_STEP_PRE_GATE_LIF,
  kPreNone = WKV_STEP_PRE_NONE
};

using StepRowArgs = ::wkv_step_row_args;

template <int CTRL>
__device__ __forceinline__ float step_dpp(float x) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), CTRL, 0xF, 0xF, true));
}

// Sum over the workgroup's 256 threads, identical in every thread: a DPP
// butterfly over 16 lanes, the wave's four rows by lane reads, the four waves
// through LDS.  red: 4 floats of the caller's own for this sum (so one barrier
// is enough).
__device__ __forceinline__ float step_block_sum(float v, float* red) {
  v += step_dpp<0xB1>(v);   // quad_perm [1,0,3,2]
  v += step_dpp<0x4E>(v);   // quad_perm [2,3,0,1]
  v += step_dpp<0x141>(v);  // row_half_mirror
  v += step_dpp<0x140>(v);  // row_mirror
  const int u = __float_as_int(v);
  const float s = (__int_as_float(__builtin_amdgcn_readlane(u, 0)) +
                   __int_as_float(__builtin_amdgcn_readlane(u, 16))) +
                  (__int_as_float(__builtin_amdgcn_readlane(u, 32)) +
                   __int_as_float(__builtin_amdgcn_readlane(u, 48)));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

// The row's channels of a [C] parameter or a [B][C] row (0 past C).
template <int EPT>
__device__ __forceinline__ void step_load(float (&v)[EPT], const float* p, int C) {
#pragma unroll
  for (int e = 0; e < EPT; ++e) {
    const int c = int(threadIdx.x) + e * kStepThreads;
    v[e] = c < C ? p[c] : 0.f;
  }
}

// x <- layer_norm(x) * weight + bias over the row's C channels (F.layer_norm,
// biased variance); slots past C hold 0 and stay out of the sums.  red: 8
// floats.
template <int EPT>
__device__ __forceinline__ void step_layer_norm(float (&x)[EPT], const float (&w)[EPT],
                                                const float (&bias)[EPT], float eps, int C,
                                                float* red) {
  const int tid = threadIdx.x;
  float s = 0.f;
#pragma unroll
  for (int e = 0; e < EPT; ++e) s += x[e];
  const float mean = step_block_sum(s, red) / float(C);
  float q = 0.f;
#pragma unroll
  for (int e = 0; e < EPT; ++e) {
    const int c = tid + e * kStepThreads;
    const float d = c < C ? x[e] - mean : 0.f;
    q = fmaf(d, d, q);
  }
  const float var = step_block_sum(q, red + 4) / float(C);
  const float rstd = 1.f / sqrtf(var + eps);
#pragma unroll
  for (int e = 0; e < EPT; ++e) {
    const int c = tid + e * kStepThreads;
    if (c < C) x[e] = (x[e] - mean) * rstd * w[e] + bias[e];
  }
}

__device__ __forceinline__ float step_sigmoid(float r) { return 1.f / (1.f + expf(-r)); }

// One LIF step (language.py:833-839) of input v: the value added to the
// residual; mem_new is the membrane kept.  Not spiking: v itself.
__device__ __forceinline__ float step_lif(const StepRowArgs& a, float v, float mem,
                                          float& mem_new) {
  if (!a.spiking) {
    mem_new = mem;
    return v;
  }
  const float h = mem * a.lif_decay + v;
  const float s = a.lif_slope * (h - a.lif_threshold) >= 0.f ? 1.f : 0.f;
  mem_new = h * (1.f - s) + a.lif_reset * s;
  return s;
}

}  // namespace wkv
