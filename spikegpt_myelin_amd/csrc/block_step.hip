// One-token SpikeGPT block step for generation, fused, for gfx950.
//
// The reference advances a block by one token in eager PyTorch
// (SpikeGPTBlock.step, src/spikegpt/language.py:1301-1335, with
// SpikeTimeMix.step :989-1012, SpikeChannelMix.step :1174-1188 and
// SpikingSequenceLIF.step :813-840): ~60 element-wise launches per layer
// around its seven projections.  Here everything between two projections is
// one launch; the projections are step_linear.hip's, which for few rows also
// take the WKV update and relu^2 along (six or seven launches per layer) and for
// one or two rows the row work too (four), the output and value projections
// library GEMMs for many rows:
//
//   row(embed | input | gated LIF) -> LN1 -> token shift (k, v, r) [row kernel]
//   k, v, r projections
//   WKV state update + sigmoid(r) * wkv                             [wkv kernel]
//   output projection
//   row(LIF of the output)  -> LN2 -> token shift (k, r)           [row kernel]
//   key / receptance projections, relu^2, value projection
//
// and the next layer's row kernel (or the final one, which applies ln_out)
// takes the channel mix's sigmoid(r) * value through the second LIF.
//
// Row kernel: one 256-thread workgroup per batch row; thread t owns channels
// t, t + 256, ... (EPT of them, coalesced).  The layer norms reduce the row in
// two passes (mean, then the centred second moment) from registers: a wave
// sum through DPP and lane reads, then four wave partials through LDS in fixed
// order.  All arithmetic is fp32 as in the reference's fp32 step; the state
// (previous-token rows, WKV numerator/denominator/log-scale, LIF membranes)
// is read from *_in and written to *_out, which may alias (each element is
// read and written by the same thread).
#include "../../include/wkv_hip.h"
#include "step_row.h"
#include "wkv_common.h"

namespace wkv {

// Every operand is loaded before the first sum: a row is one workgroup's chain
// of a load and two to four barriers, and loads issued behind a barrier add
// their latency to it (8.4 and 10.5 us per launch at B=1 C=768 before, with
// two barriers per sum).
template <int PRE, int N, int EPT>
__global__ __launch_bounds__(kStepThreads) void block_step_row_kernel(StepRowArgs a, int parts) {
  __shared__ float red[16];
  const int C = int(a.channels);
  const int tid = threadIdx.x;
  const size_t row = size_t(blockIdx.x) * size_t(C);
  const bool norm = a.ln_weight != nullptr;
  float lw[EPT], lb[EPT], mix[N > 0 ? N : 1][EPT], prev[EPT];
  if (norm) {
    step_load<EPT>(lw, a.ln_weight, C);
    step_load<EPT>(lb, a.ln_bias, C);
    if constexpr (N > 0) {
      step_load<EPT>(prev, a.previous_in + row, C);
#pragma unroll
      for (int j = 0; j < N; ++j) step_load<EPT>(mix[j], a.mix[j], C);
    }
  }
  float x[EPT];
  if constexpr (PRE == kPreEmbed || PRE == kPreNone) {
    float w0[EPT], b0[EPT];
    if (a.ln0_weight != nullptr) {
      step_load<EPT>(w0, a.ln0_weight, C);
      step_load<EPT>(b0, a.ln0_bias, C);
    }
    if constexpr (PRE == kPreEmbed) {
      // Spiking embedding (language.py:1386-1394): [slope * e >= 0].
      // An id outside the table reads nothing and poisons the row with NaN.
      const int64_t id = a.ids[blockIdx.x];
      const bool valid = id >= 0 && id < a.vocab;
      const float* e = a.embedding + (valid ? size_t(id) * size_t(C) : 0);
#pragma unroll
      for (int i = 0; i < EPT; ++i) {
        const int c = tid + i * kStepThreads;
        float v = 0.f;
        if (c < C) {
          v = valid ? e[c] : __builtin_nanf("");
          if (a.embedding_spike && valid) v = a.embedding_slope * v >= 0.f ? 1.f : 0.f;
        }
        x[i] = v;
      }
    } else {
      // A block's own input (SpikeGPTBlock.step, language.py:1317).
      step_load<EPT>(x, a.residual + row, C);
    }
    if (a.ln0_weight != nullptr) step_layer_norm<EPT>(x, w0, b0, a.ln_eps, C, red + 8);
  } else {
    // residual + LIF(in), in = the output projection (first LIF) or
    // sigmoid(r) * value (second LIF); language.py:833-839, 1326-1330.
    float in[EPT], mem[EPT], gate[EPT];
    step_load<EPT>(in, a.add + row, C);
    step_load<EPT>(mem, a.membrane_in + row, C);
    if constexpr (PRE == kPreGateLif) step_load<EPT>(gate, a.gate + row, C);
    step_load<EPT>(x, a.residual + row, C);
    for (int p = 1; p < parts; ++p) {
      float more[EPT];
      step_load<EPT>(more, a.add + size_t(p) * size_t(a.batch) * size_t(C) + row, C);
#pragma unroll
      for (int i = 0; i < EPT; ++i) in[i] += more[i];
    }
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      const int c = tid + i * kStepThreads;
      if (c < C) {
        float v = in[i];
        if constexpr (PRE == kPreGateLif) v = step_sigmoid(gate[i]) * v;
        float mem_new;
        v = step_lif(a, v, mem[i], mem_new);
        if (a.spiking || a.membrane_out != a.membrane_in) a.membrane_out[row + c] = mem_new;
        x[i] += v;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < EPT; ++i) {
    const int c = tid + i * kStepThreads;
    if (c < C) a.residual[row + c] = x[i];
  }
  if (!norm) return;  // residual update only (n_mix == 0)
  step_layer_norm<EPT>(x, lw, lb, a.ln_eps, C, red);
#pragma unroll
  for (int i = 0; i < EPT; ++i) {
    const int c = tid + i * kStepThreads;
    if (c >= C) continue;
    if constexpr (N == 0) {
      a.out[0][row + c] = x[i];
    } else {
      // inputs * mu + previous * (1 - mu)  (language.py:996-998, 1181-1182)
#pragma unroll
      for (int j = 0; j < N; ++j)
        a.out[j][row + c] = x[i] * mix[j][i] + prev[i] * (1.f - mix[j][i]);
      a.previous_out[row + c] = x[i];
    }
  }
}

// WKV state update and receptance gate of SpikeTimeMix.step
// (language.py:999-1012): out = sigmoid(r) * wkv, state in natural-log units.
template <int VEC>
__global__ __launch_bounds__(256) void block_step_wkv_kernel(
    const float* __restrict__ key, const float* __restrict__ value,
    const float* __restrict__ receptance, const float* __restrict__ time_decay,
    const float* __restrict__ time_first, const float* num_in, const float* den_in,
    const float* ls_in, float* num_out, float* den_out, float* ls_out, float* __restrict__ out,
    int64_t n, int C) {
  const int64_t i0 = (int64_t(blockIdx.x) * blockDim.x + threadIdx.x) * VEC;
  if (i0 >= n) return;
  const int c0 = int(i0 % C);
  Pack<F32, VEC> kp, vp, rp, np, dp, lp;
  kp.load(key + i0);
  vp.load(value + i0);
  rp.load(receptance + i0);
  np.load(num_in + i0);
  dp.load(den_in + i0);
  lp.load(ls_in + i0);
  float o[VEC], no[VEC], dn[VEC], ls[VEC];
#pragma unroll
  for (int c = 0; c < VEC; ++c) {
    const float k = kp.x[c], v = vp.x[c];
    const float decay = -expf(time_decay[c0 + c]);
    const float first = time_first[c0 + c];
    const float l0 = lp.x[c];
    float nxt = fmaxf(l0, first + k);
    float s_old = expf(l0 - nxt);
    float s_new = expf(first + k - nxt);
    const float mixed = (s_old * np.x[c] + s_new * v) / (s_old * dp.x[c] + s_new);
    o[c] = step_sigmoid(rp.x[c]) * mixed;
    const float decayed = l0 + decay;
    nxt = fmaxf(decayed, k);
    s_old = expf(decayed - nxt);
    s_new = expf(k - nxt);
    no[c] = s_old * np.x[c] + s_new * v;
    dn[c] = s_old * dp.x[c] + s_new;
    ls[c] = nxt;
  }
  store_vec<F32, VEC>(out + i0, o);
  store_vec<F32, VEC>(num_out + i0, no);
  store_vec<F32, VEC>(den_out + i0, dn);
  store_vec<F32, VEC>(ls_out + i0, ls);
}

}  // namespace wkv

// ------------------------------------------------------------ launchers ----
namespace wkv_host {

int decode_vec(int64_t n, int64_t C);

template <int PRE, int N, int EPT>
static int row_launch(const wkv::StepRowArgs& a, int parts, hipStream_t s) {
  launch(wkv::block_step_row_kernel<PRE, N, EPT>, dim3(unsigned(a.batch)), dim3(wkv::kStepThreads),
         s, true, a, parts);
  return check_launch("block_step_row_kernel");
}

template <int PRE, int N>
static int row_ept(const wkv::StepRowArgs& a, int parts, hipStream_t s) {
  const int64_t ept = (a.channels + wkv::kStepThreads - 1) / wkv::kStepThreads;
  if (ept <= 1) return row_launch<PRE, N, 1>(a, parts, s);
  if (ept <= 2) return row_launch<PRE, N, 2>(a, parts, s);
  if (ept <= 3) return row_launch<PRE, N, 3>(a, parts, s);
  if (ept <= 4) return row_launch<PRE, N, 4>(a, parts, s);
  if (ept <= 8) return row_launch<PRE, N, 8>(a, parts, s);
  return row_launch<PRE, N, 16>(a, parts, s);
}

template <int PRE>
static int row_n(const wkv::StepRowArgs& a, int parts, hipStream_t s) {
  switch (a.n_mix) {
    case 0: return row_ept<PRE, 0>(a, parts, s);
    case 2: return row_ept<PRE, 2>(a, parts, s);
    case 3: return row_ept<PRE, 3>(a, parts, s);
    default: return fail(1, "block_step_row: n_mix must be 0, 2 or 3");
  }
}

int block_step_row_impl(int pre, const wkv::StepRowArgs& a, int parts, hipStream_t s) {
  switch (pre) {
    case wkv::kPreEmbed: return row_n<wkv::kPreEmbed>(a, parts, s);
    case wkv::kPreLif: return row_n<wkv::kPreLif>(a, parts, s);
    case wkv::kPreGateLif: return row_n<wkv::kPreGateLif>(a, parts, s);
    case wkv::kPreNone: return row_n<wkv::kPreNone>(a, parts, s);
    default: return fail(1, "block_step_row: unknown pre-op");
  }
}

int block_step_wkv_impl(const float* k, const float* v, const float* r, const float* td,
                        const float* tf, const float* num_in, const float* den_in,
                        const float* ls_in, float* num_out, float* den_out, float* ls_out,
                        float* out, int64_t B, int64_t C, hipStream_t s) {
  const int64_t n = B * C;
  bool vec4 = decode_vec(n, C) == 4;
  for (const void* p : {static_cast<const void*>(k), static_cast<const void*>(v),
                        static_cast<const void*>(r), static_cast<const void*>(num_in),
                        static_cast<const void*>(den_in), static_cast<const void*>(ls_in),
                        static_cast<const void*>(num_out), static_cast<const void*>(den_out),
                        static_cast<const void*>(ls_out), static_cast<const void*>(out)})
    vec4 = vec4 && reinterpret_cast<uintptr_t>(p) % 16 == 0;
  if (vec4) {
    launch(wkv::block_step_wkv_kernel<4>, dim3(unsigned((n / 4 + 255) / 256)), dim3(256), s, true,
           k, v, r, td, tf, num_in, den_in, ls_in, num_out, den_out, ls_out, out, n, int(C));
  } else {
    launch(wkv::block_step_wkv_kernel<1>, dim3(unsigned((n + 255) / 256)), dim3(256), s, true, k,
           v, r, td, tf, num_in, den_in, ls_in, num_out, den_out, ls_out, out, n, int(C));
  }
  return check_launch("block_step_wkv_kernel");
}

}  // namespace wkv_host
