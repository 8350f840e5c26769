// Layer norm fused into the token-shift mix of a SpikeGPT block, for gfx950.
//
// The blocks feed each mixing half through a layer norm
// (src/spikegpt/language.py:1341-1356: self.att(self.ln1(x)),
// self.ffn(self.ln2(x))) and the token-shift mixes (:344-353, 1016-1018,
// 1190-1191).  Per row r = (b, t) of x [B, T, C] (fp32 residual stream):
//   mean_r = sum_c x / C,  rstd_r = 1 / sqrt(sum_c (x - mean)^2 / C + eps)
//   y[r,c] = (x[r,c] - mean_r) rstd_r w[c] + bias[c]                  (F.layer_norm)
//   out_j[b,t,c] = y[b,t,c] mu_j[c] + y[b,t-1,c] (1 - mu_j[c]),  y[b,-1,:] = 0
// rounded once to the output type.  Backward, with g_j the output gradients
// and xhat = (x - mean) rstd:
//   gy[b,t,c] = sum_j g_j[b,t,c] mu_j[c] + g_j[b,t+1,c] (1 - mu_j[c])
//   gmu_j[c]  = sum_{b,t} g_j[b,t,c] (y[b,t,c] - y[b,t-1,c])
//   gw[c] = sum gy xhat,  gbias[c] = sum gy
//   gx = rstd (a - mean_c(a) - xhat mean_c(a xhat)),  a = gy w.
//
// Decomposition: thread c of a workgroup of W = ceil(C / 256) waves owns
// channels 4 c .. 4 c + 3 of every row (C a multiple of 4 up to 1024) and
// walks a chunk of consecutive rows of one sequence, kBatch rows at a time.
// Row sums are formed for the kBatch rows of a batch together: a DPP butterfly
// over 16 lanes and two permlane swaps leave row r's wave sum in lanes 16 r ..,
// the waves' sums meet in LDS (one barrier per sum and batch).  The column sums
// of the parameter gradients need no exchange: a thread keeps its four
// channels' sums and writes them once per chunk; column_sum_kernel adds the
// chunks in fixed order (deterministic).  The forward loads the next batch
// before the current one is summed; the backward has no registers for that
// (256 VGPRs with it) and is covered by the other workgroups of its CU.
//
// Bound by HBM: forward 4 + 2 N bytes per element (N bf16 outputs), backward
// 4 + 2 N + 4 + 4 (x, N gradients, the residual's gradient, grad_x).
// Measured (bf16, kernel trace): B=16 T=1024 C=768 N=3 forward 26.2 us (4.8
// TB/s), backward 45.0 us (5.0 TB/s) + column sums 5.4 us, against 47 + 144 us
// of PyTorch's layer norm, the separate mix kernels and the residual's add.
// B=32 T=1024 C=512: forward 37.8 (N=3) and 33.4 us (N=2), backward 57.0 and
// 53.2 us; with a whole row per wave (all C channels in one wave's registers,
// row by row) they took 42.4, 38.7, 99.0 and 78.0 us.
#include "wkv_common.h"

namespace wkv {

constexpr int kBatch = 4;     // rows per batch
constexpr int kRowsMaxN = 3;
constexpr int kRowsMaxW = 4;  // waves per row: C <= 1024

template <typename RAW>
struct RowPtrs {
  RAW* p[kRowsMaxN];
};

template <int CTRL>
__device__ __forceinline__ float row_dpp(float x) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), CTRL, 0xF, 0xF, true));
}

// Wave sums of four values: lanes 16 r .. 16 r + 15 receive the sum of v[r].
__device__ __forceinline__ float wave_sum4(const float (&v)[4]) {
  float s[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float x = v[r];
    x += row_dpp<0xB1>(x);   // quad_perm [1,0,3,2]
    x += row_dpp<0x4E>(x);   // quad_perm [2,3,0,1]
    x += row_dpp<0x141>(x);  // row_half_mirror
    x += row_dpp<0x140>(x);  // row_mirror
    s[r] = x;
  }
  const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(s[0]), __float_as_uint(s[2]),
                                                  false, false);
  const auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(s[1]), __float_as_uint(s[3]),
                                                  false, false);
  const float a = __uint_as_float(p[0]) + __uint_as_float(p[1]);
  const float b = __uint_as_float(q[0]) + __uint_as_float(q[1]);
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false,
                                                  false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Row sums of a batch over the workgroup's waves, in every thread.  red:
// [kBatch][kRowsMaxW] floats of LDS that no thread still reads.
__device__ __forceinline__ void rows_total(float (&v)[kBatch], float* red, int W, int lane,
                                           int wave) {
  const float s = wave_sum4(v);
  if (W == 1) {
#pragma unroll
    for (int r = 0; r < kBatch; ++r)
      v[r] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s), 16 * r));
    return;
  }
  if ((lane & 15) == 0) red[(lane >> 4) * kRowsMaxW + wave] = s;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kBatch; ++r) {
    const float4 t = *reinterpret_cast<const float4*>(red + r * kRowsMaxW);
    v[r] = t.x + t.y;
    if (W > 2) v[r] += t.z;
    if (W > 3) v[r] += t.w;
  }
}

// x [B,T,C] fp32; w, bias [C]; mix [N][C]; out_j [B,T,C] (EO); mean, rstd
// [B*T].  Grid: B * ceil(T / rows) workgroups of W waves.
template <typename EO, int N>
__global__ __launch_bounds__(256) void ln_rows_fwd_kernel(
    const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias,
    const float* __restrict__ mix, RowPtrs<typename EO::raw> out, float* __restrict__ mean_out,
    float* __restrict__ rstd_out, int T, int C, int rows, float eps) {
  __shared__ __attribute__((aligned(16))) float red[2][kBatch * kRowsMaxW];
  const int W = int(blockDim.x) >> 6;
  const int lane = int(threadIdx.x) & 63;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  const int c = 4 * int(threadIdx.x);
  const bool on = c < C;  // threads past the row's width add zeros
  const int cc = on ? c : 0;
  const int n_tc = (T + rows - 1) / rows;
  const int b = int(blockIdx.x) / n_tc;
  const int t0 = (int(blockIdx.x) - b * n_tc) * rows;
  const int t1 = min(T, t0 + rows);
  const float* xb = x + size_t(b) * T * C + cc;
  const float invC = float(C);

  const float4 w4 = *reinterpret_cast<const float4*>(w + cc);
  const float4 b4 = *reinterpret_cast<const float4*>(bias + cc);
  const float wv[4] = {w4.x, w4.y, w4.z, w4.w}, bv[4] = {b4.x, b4.y, b4.z, b4.w};
  float mu[N][4];
#pragma unroll
  for (int n = 0; n < N; ++n) {
    const float4 m4 = *reinterpret_cast<const float4*>(mix + size_t(n) * C + cc);
    mu[n][0] = m4.x; mu[n][1] = m4.y; mu[n][2] = m4.z; mu[n][3] = m4.w;
  }
  // Row t0 - 1 comes first: its layer-norm output is the previous row of t0
  // (zero before the sequence); it is not stored.
  float prev[4] = {0.f, 0.f, 0.f, 0.f};
  float4 cur[kBatch], nxt[kBatch];
  const int first = t0 > 0 ? t0 - 1 : t0;
  auto load = [&](float4 (&v)[kBatch], int t) {
#pragma unroll
    for (int r = 0; r < kBatch; ++r)
      v[r] = *reinterpret_cast<const float4*>(xb + size_t(min(t + r, T - 1)) * C);
  };
  load(cur, first);
  for (int t = first; t < t1; t += kBatch) {
    load(nxt, t + kBatch);
    float s[kBatch], m[kBatch], q[kBatch];
#pragma unroll
    for (int r = 0; r < kBatch; ++r) s[r] = on ? (cur[r].x + cur[r].y) + (cur[r].z + cur[r].w) : 0.f;
    rows_total(s, red[0], W, lane, wave);
    float d[kBatch][4];
#pragma unroll
    for (int r = 0; r < kBatch; ++r) {
      m[r] = s[r] / invC;
      d[r][0] = cur[r].x - m[r];
      d[r][1] = cur[r].y - m[r];
      d[r][2] = cur[r].z - m[r];
      d[r][3] = cur[r].w - m[r];
      float z = d[r][0] * d[r][0];
#pragma unroll
      for (int e = 1; e < 4; ++e) z = fmaf(d[r][e], d[r][e], z);
      q[r] = on ? z : 0.f;
    }
    rows_total(q, red[1], W, lane, wave);
#pragma unroll
    for (int r = 0; r < kBatch; ++r) {
      const float rs = 1.f / sqrtf(q[r] / invC + eps);
      float y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = d[r][e] * rs * wv[e] + bv[e];
      if (t + r >= t0 && t + r < t1) {
        const size_t row = size_t(b) * T + t + r;
        if (threadIdx.x == 0) {
          mean_out[row] = m[r];
          rstd_out[row] = rs;
        }
        if (on) {
#pragma unroll
          for (int n = 0; n < N; ++n) {
            float o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float a = y[e] * mu[n][e];
              const float p = prev[e] * (1.f - mu[n][e]);
              o[e] = a + p;
            }
            store_vec<EO, 4>(out.p[n] + row * C + c, o);
          }
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) prev[e] = y[e];
    }
#pragma unroll
    for (int r = 0; r < kBatch; ++r) cur[r] = nxt[r];
  }
}

// g_j [B,T,C] (EG); gx [B,T,C] fp32; gadd (optional) [B,T,C] fp32 added to gx;
// partial [N + 2][gridDim.x][C] (rows gmu_0 .. gmu_{N-1}, gw, gbias).
template <typename EG, int N>
__global__ __launch_bounds__(256) void ln_rows_bwd_kernel(
    const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias,
    const float* __restrict__ mix, const float* __restrict__ mean,
    const float* __restrict__ rstd, RowPtrs<const typename EG::raw> g, float* __restrict__ gx,
    const float* __restrict__ gadd, float* __restrict__ partial, int T, int C, int rows) {
  // Two sums per row, two buffers: a batch writes one while slower threads
  // may still read the other.
  __shared__ __attribute__((aligned(16))) float red[2][2][kBatch * kRowsMaxW];
  const int W = int(blockDim.x) >> 6;
  const int lane = int(threadIdx.x) & 63;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  const int c = 4 * int(threadIdx.x);
  const bool on = c < C;
  const int cc = on ? c : 0;
  const int n_tc = (T + rows - 1) / rows;
  const int b = int(blockIdx.x) / n_tc;
  const int t0 = (int(blockIdx.x) - b * n_tc) * rows;
  const int t1 = min(T, t0 + rows);
  const size_t seq = size_t(b) * T;
  const float* xb = x + seq * C + cc;
  const float fC = float(C);

  const float4 w4 = *reinterpret_cast<const float4*>(w + cc);
  const float4 b4 = *reinterpret_cast<const float4*>(bias + cc);
  const float wv[4] = {w4.x, w4.y, w4.z, w4.w}, bv[4] = {b4.x, b4.y, b4.z, b4.w};
  float mu[N][4], acc[N + 2][4];
#pragma unroll
  for (int n = 0; n < N; ++n) {
    const float4 m4 = *reinterpret_cast<const float4*>(mix + size_t(n) * C + cc);
    mu[n][0] = m4.x; mu[n][1] = m4.y; mu[n][2] = m4.z; mu[n][3] = m4.w;
  }
#pragma unroll
  for (int f = 0; f < N + 2; ++f)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[f][e] = 0.f;

  struct Batch {
    float4 x[kBatch];
    float mean[kBatch], rstd[kBatch];
    Pack<EG, 4> g[N][kBatch];  // gradients of rows t + 1 .. t + kBatch
  };
  auto load = [&](Batch& v, int t) {
#pragma unroll
    for (int r = 0; r < kBatch; ++r) {
      const int tr = min(t + r, T - 1);
      v.x[r] = *reinterpret_cast<const float4*>(xb + size_t(tr) * C);
      v.mean[r] = mean[seq + tr];
      v.rstd[r] = rstd[seq + tr];
      const int tn = min(t + r + 1, T - 1);
#pragma unroll
      for (int n = 0; n < N; ++n) v.g[n][r].load(g.p[n] + (seq + tn) * C + cc);
    }
  };
  float prev[4] = {0.f, 0.f, 0.f, 0.f};
  if (t0 > 0) {
    const float4 v = *reinterpret_cast<const float4*>(xb + size_t(t0 - 1) * C);
    const float m = mean[seq + t0 - 1], rs = rstd[seq + t0 - 1];
    prev[0] = (v.x - m) * rs * wv[0] + bv[0];
    prev[1] = (v.y - m) * rs * wv[1] + bv[1];
    prev[2] = (v.z - m) * rs * wv[2] + bv[2];
    prev[3] = (v.w - m) * rs * wv[3] + bv[3];
  }
  float gc[N][4];  // gradients of the row being computed
#pragma unroll
  for (int n = 0; n < N; ++n) {
    Pack<EG, 4> p;
    p.load(g.p[n] + (seq + t0) * C + cc);
#pragma unroll
    for (int e = 0; e < 4; ++e) gc[n][e] = p.get(e);
  }
  int buf = 0;
  for (int t = t0; t < t1; t += kBatch, buf ^= 1) {
    Batch cur;
    load(cur, t);
    float4 ga[kBatch];
    if (gadd) {
#pragma unroll
      for (int r = 0; r < kBatch; ++r)
        ga[r] = *reinterpret_cast<const float4*>(gadd + (seq + min(t + r, T - 1)) * C + cc);
    }
    float a[kBatch][4], xh[kBatch][4], s1[kBatch], s2[kBatch];
#pragma unroll
    for (int r = 0; r < kBatch; ++r) {
      const bool live = t + r < t1;  // rows past the chunk add nothing
      const float xs[4] = {cur.x[r].x, cur.x[r].y, cur.x[r].z, cur.x[r].w};
      const bool next_row = t + r + 1 < T;
      s1[r] = 0.f;
      s2[r] = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        xh[r][e] = (xs[e] - cur.mean[r]) * cur.rstd[r];
        const float y = xh[r][e] * wv[e] + bv[e];
        float gy = 0.f;
#pragma unroll
        for (int n = 0; n < N; ++n) {
          const float gn = next_row ? cur.g[n][r].get(e) : 0.f;
          gy = fmaf(gc[n][e], mu[n][e], gy);
          gy = fmaf(gn, 1.f - mu[n][e], gy);
          if (live) acc[n][e] = fmaf(gc[n][e], y - prev[e], acc[n][e]);
          gc[n][e] = gn;
        }
        prev[e] = y;
        if (live) {
          acc[N][e] = fmaf(gy, xh[r][e], acc[N][e]);
          acc[N + 1][e] += gy;
        }
        a[r][e] = on ? gy * wv[e] : 0.f;
        s1[r] += a[r][e];
        s2[r] = fmaf(a[r][e], xh[r][e], s2[r]);
      }
    }
    // One barrier for both sums.
    if (W == 1) {
      rows_total(s1, red[buf][0], W, lane, wave);
      rows_total(s2, red[buf][1], W, lane, wave);
    } else {
      const float u1 = wave_sum4(s1), u2 = wave_sum4(s2);
      if ((lane & 15) == 0) {
        red[buf][0][(lane >> 4) * kRowsMaxW + wave] = u1;
        red[buf][1][(lane >> 4) * kRowsMaxW + wave] = u2;
      }
      __syncthreads();
#pragma unroll
      for (int r = 0; r < kBatch; ++r) {
        const float4 p = *reinterpret_cast<const float4*>(red[buf][0] + r * kRowsMaxW);
        const float4 q = *reinterpret_cast<const float4*>(red[buf][1] + r * kRowsMaxW);
        s1[r] = p.x + p.y;
        s2[r] = q.x + q.y;
        if (W > 2) { s1[r] += p.z; s2[r] += q.z; }
        if (W > 3) { s1[r] += p.w; s2[r] += q.w; }
      }
    }
#pragma unroll
    for (int r = 0; r < kBatch; ++r) {
      if (t + r < t1 && on) {
        const float m1 = s1[r] / fC, m2 = s2[r] / fC;
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = cur.rstd[r] * (a[r][e] - m1 - xh[r][e] * m2);
        if (gadd) {
          o[0] += ga[r].x; o[1] += ga[r].y; o[2] += ga[r].z; o[3] += ga[r].w;
        }
        store_vec<F32, 4>(gx + (seq + t + r) * C + c, o);
      }
    }
  }
  if (on) {
#pragma unroll
    for (int f = 0; f < N + 2; ++f)
      *reinterpret_cast<float4*>(partial + (size_t(f) * gridDim.x + blockIdx.x) * C + c) =
          make_float4(acc[f][0], acc[f][1], acc[f][2], acc[f][3]);
  }
}

}  // namespace wkv

// ------------------------------------------------------------ launchers ----
namespace wkv_host {

static int rows_waves(int64_t C) { return int((C + 255) / 256); }

// Rows per workgroup: as many as leave 2048 waves (two per SIMD), from
// 16 to 128; a chunk costs one extra row (its predecessor) and, backward, one
// row of partial sums (with 3072 waves the column sums took 9.7 instead of 5.5
// us at B=32 T=1024 C=512, the kernels themselves the same).
static int rows_per_chunk(int64_t B, int64_t T, int64_t C) {
  int rows = 16;
  while (rows < 128 && B * ((T + 2 * rows - 1) / (2 * rows)) * rows_waves(C) >= 2048) rows *= 2;
  return rows;
}

int64_t ln_rows_workgroups(int64_t B, int64_t T, int64_t C) {
  const int rows = rows_per_chunk(B, T, C);
  return B * ((T + rows - 1) / rows);
}

template <typename EO, int N>
static int ln_rows_fwd(const float* x, const float* w, const float* bias, const float* mix,
                       void* const* out, float* mean, float* rstd, int B, int T, int C, float eps,
                       hipStream_t s) {
  wkv::RowPtrs<typename EO::raw> o{};
  for (int n = 0; n < N; ++n) o.p[n] = static_cast<typename EO::raw*>(out[n]);
  launch(wkv::ln_rows_fwd_kernel<EO, N>, dim3(unsigned(ln_rows_workgroups(B, T, C))),
         dim3(unsigned(64 * rows_waves(C))), s, true, x, w, bias, mix, o, mean, rstd, T, C,
         rows_per_chunk(B, T, C), eps);
  return check_launch("ln_rows_fwd_kernel");
}

template <typename EO>
static int ln_rows_fwd_n(int n, const float* x, const float* w, const float* bias,
                         const float* mix, void* const* out, float* mean, float* rstd, int B,
                         int T, int C, float eps, hipStream_t s) {
  return n == 2 ? ln_rows_fwd<EO, 2>(x, w, bias, mix, out, mean, rstd, B, T, C, eps, s)
                : ln_rows_fwd<EO, 3>(x, w, bias, mix, out, mean, rstd, B, T, C, eps, s);
}

int ln_rows_forward_impl(const float* x, const float* w, const float* bias, const float* mix,
                         int n, void* const* out, int out_dtype, float* mean, float* rstd, int B,
                         int T, int C, float eps, hipStream_t s) {
  switch (out_dtype) {
    case 0: return ln_rows_fwd_n<wkv::F32>(n, x, w, bias, mix, out, mean, rstd, B, T, C, eps, s);
    case 1: return ln_rows_fwd_n<wkv::BF16>(n, x, w, bias, mix, out, mean, rstd, B, T, C, eps, s);
    case 2: return ln_rows_fwd_n<wkv::F16>(n, x, w, bias, mix, out, mean, rstd, B, T, C, eps, s);
    default: return fail(1, "layer_norm_shift_mix_rows: unknown output dtype");
  }
}

template <typename EG, int N>
static int ln_rows_bwd(const float* x, const float* w, const float* bias, const float* mix,
                       const float* mean, const float* rstd, const void* const* g, float* gx,
                       const float* gadd, float* partial, float* sums, int B, int T, int C,
                       hipStream_t s) {
  wkv::RowPtrs<const typename EG::raw> gp{};
  for (int n = 0; n < N; ++n) gp.p[n] = static_cast<const typename EG::raw*>(g[n]);
  const int64_t P = ln_rows_workgroups(B, T, C);
  launch(wkv::ln_rows_bwd_kernel<EG, N>, dim3(unsigned(P)), dim3(unsigned(64 * rows_waves(C))), s,
         false, x, w, bias, mix, mean, rstd, gp, gx, gadd, partial, T, C,
         rows_per_chunk(B, T, C));
  int rc = check_launch("ln_rows_bwd_kernel");
  if (rc) return rc;
  launch(wkv::column_sum_kernel<16>, dim3(unsigned((C + 63) / 64), unsigned(N + 2)), dim3(1024), s,
         true, static_cast<const float*>(partial), sums, int(P), C);
  return check_launch("column_sum_kernel");
}

template <typename EG>
static int ln_rows_bwd_n(int n, const float* x, const float* w, const float* bias,
                         const float* mix, const float* mean, const float* rstd,
                         const void* const* g, float* gx, const float* gadd, float* partial,
                         float* sums, int B, int T, int C, hipStream_t s) {
  return n == 2 ? ln_rows_bwd<EG, 2>(x, w, bias, mix, mean, rstd, g, gx, gadd, partial, sums, B, T,
                                     C, s)
                : ln_rows_bwd<EG, 3>(x, w, bias, mix, mean, rstd, g, gx, gadd, partial, sums, B, T,
                                     C, s);
}

int ln_rows_backward_impl(const float* x, const float* w, const float* bias, const float* mix,
                          int n, const float* mean, const float* rstd, const void* const* g,
                          int g_dtype, float* gx, const float* gadd, float* partial, float* sums,
                          int B, int T, int C, hipStream_t s) {
  switch (g_dtype) {
    case 0:
      return ln_rows_bwd_n<wkv::F32>(n, x, w, bias, mix, mean, rstd, g, gx, gadd, partial, sums, B,
                                     T, C, s);
    case 1:
      return ln_rows_bwd_n<wkv::BF16>(n, x, w, bias, mix, mean, rstd, g, gx, gadd, partial, sums,
                                      B, T, C, s);
    case 2:
      return ln_rows_bwd_n<wkv::F16>(n, x, w, bias, mix, mean, rstd, g, gx, gadd, partial, sums, B,
                                     T, C, s);
    default: return fail(1, "layer_norm_shift_mix_rows_backward: unknown gradient dtype");
  }
}

}  // namespace wkv_host
