// The projections of the one-token block step (generation), for gfx950, with
// the element-wise work that follows each of them folded in.
//
// A step multiplies B rows (the batch, 1 to a few hundred) by fp32 weights
// [N][K] with K, N of 128 to 4096: SpikeTimeMix.step's key, value and
// receptance (src/spikegpt/language.py:999-1012), its output projection, and
// SpikeChannelMix.step's three (:1181-1188).  Four modes:
//   PLAIN   out = x W^T, optionally as `parts` partial products over K slices
//           that the next row kernel adds (a long K and few columns leave most
//           CUs without a tile otherwise)
//   KVR     k, v, r = three products over the same columns, then the WKV state
//           update and sigmoid(r) * wkv (the arithmetic of
//           block_step_wkv_kernel)
//   KEY_REC out0 = relu(x0 W0^T)^2, out1 = x1 W1^T
//   THREE   out_j = x_j W_j^T over the same columns (the WKV kernel follows)
//
// Tile: a workgroup of KS waves owns 16 batch rows and 16 TN columns (of each
// of the three matrices in KVR); its waves split K (contiguous 32-deep slices)
// and meet in LDS, where the KS partial sums are added in wave order
// (deterministic).  An operand is read straight from global memory in the
// MFMA's lane layout: lane (m, g) of v_mfma_f32_16x16x4_f32 holds
// row m, columns 8 g .. 8 g + 7 of a 32-deep slice, so each row's 128-byte
// line is one lane group's two 16-byte loads.  All arithmetic is fp32.
//
// Bound by the weights' bytes and the launches for few rows: per layer at
// C = 768, B = 6 the launches take 9.6 (KVR), 4.6 (output), 5.2 (KEY_REC) and
// 4.8 us (value, 4 parts; 9.5 in one part: 48 workgroups cannot draw 9.4 MB
// faster), against 20.1 + 6.6 + 13.6 + 8.3 us of library GEMMs at B = 1 and
// 2 x 5 us for the WKV and relu^2 launches.  One to four rows run one wave per
// dot product instead (below).  Beyond 512
// tiles the operands' 64 bytes per clock and CU become the bound and the
// library's LDS-tiled GEMMs are level or better (the caller's rule).
//
// Workgroups are numbered so that the batch tiles of one column tile run on
// one XCD (round robin over 8): its weights are fetched into one L2.
#include "step_row.h"
#include "wkv_common.h"
#include "wkv_impl.h"

namespace wkv {

typedef float lin_f4 __attribute__((ext_vector_type(4)));

enum StepLinear : int { kLinPlain = 0, kLinKvr = 1, kLinKeyRec = 2, kLinThree = 3 };

// WKV state update and receptance gate of element o (language.py:999-1012,
// natural-log units).
__device__ __forceinline__ void lin_wkv(const wkv_step_linear_args& a, size_t o, float k, float v,
                                        float r, float decay, float first, float num, float den,
                                        float l0) {
  float nxt = fmaxf(l0, first + k);
  float s_old = expf(l0 - nxt);
  float s_new = expf(first + k - nxt);
  const float mixed = (s_old * num + s_new * v) / (s_old * den + s_new);
  a.out[0][o] = step_sigmoid(r) * mixed;
  const float decayed = l0 + decay;
  nxt = fmaxf(decayed, k);
  s_old = expf(decayed - nxt);
  s_new = expf(k - nxt);
  a.num_out[o] = s_old * num + s_new * v;
  a.den_out[o] = s_old * den + s_new;
  a.ls_out[o] = nxt;
}

// Sum over a wave, the same in every lane: 16 lanes by DPP, the four rows of
// lanes by lane reads.
__device__ __forceinline__ float lin_wave_sum(float v) {
  v += step_dpp<0xB1>(v);   // quad_perm [1,0,3,2]
  v += step_dpp<0x4E>(v);   // quad_perm [2,3,0,1]
  v += step_dpp<0x141>(v);  // row_half_mirror
  v += step_dpp<0x140>(v);  // row_mirror
  const int u = __float_as_int(v);
  return (__int_as_float(__builtin_amdgcn_readlane(u, 0)) +
          __int_as_float(__builtin_amdgcn_readlane(u, 16))) +
         (__int_as_float(__builtin_amdgcn_readlane(u, 32)) +
          __int_as_float(__builtin_amdgcn_readlane(u, 48)));
}

// Rows m of a 32-deep slice at column k: two float4 per lane (zero past K).
struct LinFrag {
  float4 v[2];
  __device__ __forceinline__ void load(const float* __restrict__ row, int k, int K) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
      v[h] = k + 4 * h < K ? *reinterpret_cast<const float4*>(row + k + 4 * h)
                           : make_float4(0.f, 0.f, 0.f, 0.f);
  }
};

__device__ __forceinline__ lin_f4 lin_mfma(const LinFrag& a, const LinFrag& b, lin_f4 c) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.v[h].x, b.v[h].x, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.v[h].y, b.v[h].y, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.v[h].z, b.v[h].z, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.v[h].w, b.v[h].w, c, 0, 0, 0);
  }
  return c;
}

// MATS matrices of TN tiles each per workgroup (KVR: 3; otherwise 1).
template <int MODE, int TN, int KS>
__global__ __launch_bounds__(64 * KS) void step_linear_kernel(wkv_step_linear_args a, int n_tiles0,
                                                              int n_tiles, int b_tiles,
                                                              int parts) {
  constexpr int MATS = MODE == kLinKvr ? 3 : 1;
  constexpr int TILES = MATS * TN;
  __shared__ __attribute__((aligned(16))) float part[KS][TILES][16][20];
  const int lane = int(threadIdx.x) & 63;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  const int m = lane & 15, g = lane >> 4;
  // Workgroup -> (column tile, batch tile), batch fastest within an XCD.
  const int xcd = int(blockIdx.x) & 7, idx = int(blockIdx.x) >> 3;
  const int nt = (idx / b_tiles) * 8 + xcd, bt = idx % b_tiles;
  if (nt >= n_tiles) return;
  const int part_id = int(blockIdx.y);
  int mat0 = 0, ntl = nt;
  if constexpr (MODE == kLinThree) {
    mat0 = min(nt / n_tiles0, 2);
    ntl = nt - mat0 * n_tiles0;
  }
  if (MODE == kLinKeyRec && nt >= n_tiles0) {
    mat0 = 1;
    ntl = nt - n_tiles0;
  }
  const int N = int(MODE == kLinKeyRec && mat0 ? a.n1 : a.n0);
  const int K = int(a.k);
  const int B = int(a.batch);
  const int n0 = ntl * 16 * TN;
  const int b0 = bt * 16;
  const float* wrow[MATS][TN];
  const float* xrow[MATS];
#pragma unroll
  for (int q = 0; q < MATS; ++q) {
    const int mi = MODE == kLinKvr ? q : mat0;
    const float* w = mi == 0 ? a.w[0] : mi == 1 ? a.w[1] : a.w[2];
    const float* x = mi == 0 ? a.x[0] : mi == 1 ? a.x[1] : a.x[2];
    xrow[q] = x + size_t(min(b0 + m, B - 1)) * K;
#pragma unroll
    for (int t = 0; t < TN; ++t) wrow[q][t] = w + size_t(min(n0 + 16 * t + m, N - 1)) * K;
  }
  // Slices of 32 columns: a contiguous run for each part, and in it for each
  // wave.
  const int n_all = (K + 31) / 32;
  const int per_part = (n_all + parts - 1) / parts;
  const int p0 = part_id * per_part, p1 = min(n_all, p0 + per_part);
  const int per = (per_part + KS - 1) / KS;
  const int s0 = p0 + wave * per, s1 = min(p1, s0 + per);
  lin_f4 acc[MATS][TN];
#pragma unroll
  for (int q = 0; q < MATS; ++q)
#pragma unroll
    for (int t = 0; t < TN; ++t) acc[q][t] = lin_f4{0.f, 0.f, 0.f, 0.f};
  struct Slice {
    LinFrag w[MATS][TN], x[MATS];
  };
  auto load = [&](Slice& s, int sl) {
    const int k = sl * 32 + 8 * g;
#pragma unroll
    for (int q = 0; q < MATS; ++q) {
      s.x[q].load(xrow[q], k, K);
#pragma unroll
      for (int t = 0; t < TN; ++t) s.w[q][t].load(wrow[q][t], k, K);
    }
  };
  auto compute = [&](const Slice& s) {
#pragma unroll
    for (int q = 0; q < MATS; ++q)
#pragma unroll
      for (int t = 0; t < TN; ++t) acc[q][t] = lin_mfma(s.w[q][t], s.x[q], acc[q][t]);
  };
  if (s0 < s1) {
    Slice even, odd;
    load(even, s0);
    for (int sl = s0; sl < s1; sl += 2) {
      if (sl + 1 < s1) load(odd, sl + 1);
      compute(even);
      if (sl + 1 >= s1) break;
      if (sl + 2 < s1) load(even, sl + 2);
      compute(odd);
    }
  }
  // Tile layout: D row = column n of the output, D column = batch row.
#pragma unroll
  for (int q = 0; q < MATS; ++q)
#pragma unroll
    for (int t = 0; t < TN; ++t)
      *reinterpret_cast<lin_f4*>(&part[wave][q * TN + t][m][4 * g]) = acc[q][t];
  __syncthreads();
  // One thread per (batch row, column) and tile: 256 threads finish a tile.
  constexpr int GROUPS = KS / 4 > 0 ? KS / 4 : 1;  // tiles finished at a time
  const int grp = int(threadIdx.x) >> 8;
  const int bi = (int(threadIdx.x) >> 4) & 15, ni = int(threadIdx.x) & 15;
  for (int t = grp; t < TN; t += GROUPS) {
    const int n = n0 + 16 * t + ni, b = b0 + bi;
    if (n >= N || b >= B) continue;
    float s[MATS];
#pragma unroll
    for (int q = 0; q < MATS; ++q) {
      s[q] = part[0][q * TN + t][bi][ni];
#pragma unroll
      for (int w = 1; w < KS; ++w) s[q] += part[w][q * TN + t][bi][ni];
    }
    const size_t o = size_t(b) * N + n;
    if constexpr (MODE == kLinPlain) {
      a.out[0][size_t(part_id) * B * N + o] = s[0];
    } else if constexpr (MODE == kLinThree) {
      (mat0 == 0 ? a.out[0] : mat0 == 1 ? a.out[1] : a.out[2])[o] = s[0];
    } else if constexpr (MODE == kLinKeyRec) {
      if (mat0 == 0) {
        const float z = fmaxf(s[0], 0.f);  // as relu_square_fwd_kernel
        a.out[0][o] = z * z;
      } else {
        a.out[1][o] = s[0];
      }
    } else {
      lin_wkv(a, o, s[0], s[1], s[2], -expf(a.time_decay[n]), a.time_first[n], a.num_in[o],
              a.den_in[o], a.ls_in[o]);
    }
  }
}

// Workgroups from `first` on copy src [2][n] to the two dst (n = 0: none).
struct StepCopy {
  const float* src;
  float* dst[2];
  int n, first;
};

// ---- a few rows: one wave per dot product ----
// Up to ROWS batch rows.  A wave owns CW columns of each of its matrices; lane
// l reads columns 256 j + 4 l of the weight and x rows, PIECES 16-byte pieces
// of each in flight at once, so a product whose K is at most 1024 (4096 where
// the four waves of a workgroup split K and meet in LDS) waits for memory once.
// The tiles above put 16 columns into a workgroup (48 workgroups at C = 768)
// and take two rounds of loads.  Bound by the launch and one trip to memory:
// at C = 768, B = 1 (us, the tiles before): KVR 4.4 (8.9), output 2.8 (4.5),
// KEY_REC 4.1 (5.0; 11.8 MB, 2.9 TB/s), value 3.9 (4.7); at B = 4: 5.6 (9.3),
// 3.3 (4.6), 5.0 (5.2), 4.6 (4.8).  A lane's sum is K / 64 terms long, a
// tile's K / 8: the error from 64 bits is half the tile's (1.0e-7, 2.0e-7).
// With a branch around each piece the rows' loads wait for one another (B = 4
// KVR 6.5 us); with eight rows 10.0 us either way.
template <int MODE, int ROWS, int CW, int SPLIT, int PIECES>
__global__ __launch_bounds__(256) void step_gemv_kernel(wkv_step_linear_args a, int groups0,
                                                        int groups, StepCopy copy) {
  static_assert(SPLIT == 1 || SPLIT == 4, "one wave or the whole workgroup per column group");
  static_assert(CW * ROWS <= 64, "one lane per output");
  constexpr int MATS = MODE == kLinKvr ? 3 : 1;
  const int lane = int(threadIdx.x) & 63;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  const int group = int(blockIdx.x) * (4 / SPLIT) + (SPLIT == 1 ? wave : 0);
  if (MODE == kLinPlain && int(blockIdx.x) >= copy.first) {
    const int i = (int(blockIdx.x) - copy.first) * 256 + int(threadIdx.x);
    if (i < copy.n)
      copy.dst[0][i] = copy.src[i];
    else if (i < 2 * copy.n)
      copy.dst[1][i - copy.n] = copy.src[i];
    return;
  }
  if (group >= groups) return;  // SPLIT 4: the grid is exact, no wave leaves
  const int mat0 = MODE == kLinKeyRec && group >= groups0 ? 1 : 0;
  const int n0 = (mat0 ? group - groups0 : group) * CW;
  const int N = int(mat0 ? a.n1 : a.n0);
  const int K = int(a.k), B = int(a.batch);
  // The lane's output: column n0 + lane / ROWS of row lane % ROWS.
  const int n = n0 + lane / ROWS, b = lane % ROWS;
  const bool mine = lane < CW * ROWS && n < N && b < B;
  const size_t o = size_t(b) * N + n;
  float decay_in = 0.f, first = 0.f, num = 0.f, den = 0.f, l0 = 0.f;
  if constexpr (MODE == kLinKvr) {
    if (mine) {
      decay_in = a.time_decay[n];
      first = a.time_first[n];
      num = a.num_in[o];
      den = a.den_in[o];
      l0 = a.ls_in[o];
    }
  }
  const int chunks = (K + 255) / 256;
  const int per = (chunks + SPLIT - 1) / SPLIT;
  const int c0 = SPLIT == 1 ? 0 : wave * per;
  const int c1 = min(chunks, c0 + per);
  float acc[MATS][CW][ROWS];
#pragma unroll
  for (int q = 0; q < MATS; ++q)
#pragma unroll
    for (int c = 0; c < CW; ++c)
#pragma unroll
      for (int r = 0; r < ROWS; ++r) acc[q][c][r] = 0.f;
  for (int j = c0; j < c1; j += PIECES) {
    float4 w[MATS][CW][PIECES];
    // Past the end a piece reads the row's start and counts as zero: no branch
    // comes between the loads, so all of them are in flight together.
    bool in[PIECES];
    int at[PIECES];
#pragma unroll
    for (int u = 0; u < PIECES; ++u) {
      const int k = 256 * (j + u) + 4 * lane;
      in[u] = j + u < c1 && k < K;
      at[u] = in[u] ? k : 0;
    }
    auto piece = [&](const float* row, int u) {
      const float4 v = *reinterpret_cast<const float4*>(row + at[u]);
      return make_float4(in[u] ? v.x : 0.f, in[u] ? v.y : 0.f, in[u] ? v.z : 0.f,
                         in[u] ? v.w : 0.f);
    };
#pragma unroll
    for (int q = 0; q < MATS; ++q) {
      const int mi = MODE == kLinKvr ? q : mat0;
      const float* wm = mi == 0 ? a.w[0] : mi == 1 ? a.w[1] : a.w[2];
#pragma unroll
      for (int c = 0; c < CW; ++c)
#pragma unroll
        for (int u = 0; u < PIECES; ++u)
          w[q][c][u] = piece(wm + size_t(min(n0 + c, N - 1)) * K, u);
    }
    float4 v[MATS][ROWS][PIECES];
#pragma unroll
    for (int q = 0; q < MATS; ++q) {
      const int mi = MODE == kLinKvr ? q : mat0;
      const float* x = mi == 0 ? a.x[0] : mi == 1 ? a.x[1] : a.x[2];
#pragma unroll
      for (int r = 0; r < ROWS; ++r)
#pragma unroll
        for (int u = 0; u < PIECES; ++u)
          v[q][r][u] = piece(x + size_t(min(r, B - 1)) * K, u);
    }
#pragma unroll
    for (int q = 0; q < MATS; ++q)
#pragma unroll
      for (int u = 0; u < PIECES; ++u)
#pragma unroll
        for (int r = 0; r < ROWS; ++r)
#pragma unroll
          for (int c = 0; c < CW; ++c) {
            float s = acc[q][c][r];
            s = fmaf(w[q][c][u].x, v[q][r][u].x, s);
            s = fmaf(w[q][c][u].y, v[q][r][u].y, s);
            s = fmaf(w[q][c][u].z, v[q][r][u].z, s);
            acc[q][c][r] = fmaf(w[q][c][u].w, v[q][r][u].w, s);
          }
  }
  // Sum over the wave; lane i keeps the value of output i.
  float s[MATS];
#pragma unroll
  for (int q = 0; q < MATS; ++q) {
    s[q] = 0.f;
#pragma unroll
    for (int c = 0; c < CW; ++c)
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        const float t = lin_wave_sum(acc[q][c][r]);
        if (lane == c * ROWS + r) s[q] = t;
      }
  }
  if constexpr (SPLIT > 1) {
    __shared__ float part[SPLIT][CW * ROWS];
    if (lane < CW * ROWS) part[wave][lane] = s[0];
    __syncthreads();
    if (wave != 0) return;
    if (lane < CW * ROWS) {
      s[0] = part[0][lane];
#pragma unroll
      for (int p = 1; p < SPLIT; ++p) s[0] += part[p][lane];
    }
  }
  if (!mine) return;
  if constexpr (MODE == kLinKvr) {
    lin_wkv(a, o, s[0], s[1], s[2], -expf(decay_in), first, num, den, l0);
  } else if (MODE == kLinKeyRec && mat0 == 0) {
    const float z = fmaxf(s[0], 0.f);  // as relu_square_fwd_kernel
    a.out[0][o] = z * z;
  } else {
    a.out[MODE == kLinKeyRec ? 1 : 0][o] = s[0];
  }
}

// ---- one or two rows: the row work in front of a projection taken along ----
// Every workgroup computes the rows (LIF, residual, layer norm, token shift:
// the row kernel's operations in its order, so the same bits) for itself from
// 40 C bytes a row, while its weights are on their way, and the row kernel's
// launch disappears: KVR behind sigmoid(r) * value and the second LIF, KEY_REC
// behind the first LIF.  Workgroup 0 writes the new rows, to buffers that no
// workgroup of this launch reads: the new residual beside the old one, the
// membrane and the previous row staged for a later launch to copy (StepCopy).
// EPT = 256-column pieces of a row (C <= 1024).  A dependent launch of a few
// microseconds' work costs about 2 us more than the work.  One token, row
// kernels apart -> folded: 18 layers of C = 768, batch 1 528 -> 409 us, batch 2
// 568 -> 473; 6 layers of C = 1024 206 -> 168, 212 -> 193; 4 layers of C = 128
// 73 -> 62, 77 -> 70.  The gain shrinks with each row that every workgroup
// repeats, hence two.
template <int PRE, int MODE, int ROWS, int CW, int EPT>
__global__ __launch_bounds__(kStepThreads) void step_row_gemv_kernel(
    StepRowArgs ra, float* residual_out, wkv_step_linear_args a, int groups0) {
  static_assert(CW * ROWS <= 64, "one lane per output");
  constexpr int MATS = MODE == kLinKvr ? 3 : 1;
  constexpr int MIXES = MODE == kLinKvr ? 3 : 2;
  constexpr int WIDTH = EPT * kStepThreads;
  __shared__ float red[ROWS][8];
  __shared__ __attribute__((aligned(16))) float xs[MIXES][ROWS][WIDTH];
  const int tid = int(threadIdx.x), lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int C = int(a.k), B = int(a.batch);
  // The rows' operands first: loads return in order, and the rows need theirs
  // before the products need the weights.
  float x[ROWS][EPT], in[ROWS][EPT], mem[ROWS][EPT], gate[ROWS][EPT], prev[ROWS][EPT];
  float lw[EPT], lb[EPT], mix[MIXES][EPT];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    const size_t row = size_t(min(r, B - 1)) * size_t(C);
    step_load<EPT>(x[r], ra.residual + row, C);
    step_load<EPT>(in[r], ra.add + row, C);
    step_load<EPT>(mem[r], ra.membrane_in + row, C);
    if constexpr (PRE == kPreGateLif) step_load<EPT>(gate[r], ra.gate + row, C);
    step_load<EPT>(prev[r], ra.previous_in + row, C);
  }
  step_load<EPT>(lw, ra.ln_weight, C);
  step_load<EPT>(lb, ra.ln_bias, C);
#pragma unroll
  for (int j = 0; j < MIXES; ++j) step_load<EPT>(mix[j], ra.mix[j], C);
  // A wave past the last group repeats a column and stores nothing.
  const int group = int(blockIdx.x) * 4 + wave;
  const int mat0 = MODE == kLinKeyRec && group >= groups0 ? 1 : 0;
  const int n0 = (mat0 ? group - groups0 : group) * CW;
  const int N = int(mat0 ? a.n1 : a.n0);
  const int n = n0 + lane / ROWS, b = lane % ROWS;
  const bool mine = lane < CW * ROWS && n < N && b < B;
  const size_t o = size_t(b) * N + n;
  float decay_in = 0.f, first = 0.f, num = 0.f, den = 0.f, l0 = 0.f;
  if constexpr (MODE == kLinKvr) {
    if (mine) {
      decay_in = a.time_decay[n];
      first = a.time_first[n];
      num = a.num_in[o];
      den = a.den_in[o];
      l0 = a.ls_in[o];
    }
  }
  float4 w[MATS][CW][EPT];
#pragma unroll
  for (int q = 0; q < MATS; ++q) {
    const int mi = MODE == kLinKvr ? q : mat0;
    const float* wm = mi == 0 ? a.w[0] : mi == 1 ? a.w[1] : a.w[2];
#pragma unroll
    for (int c = 0; c < CW; ++c)
#pragma unroll
      for (int u = 0; u < EPT; ++u) {
        const int k = 256 * u + 4 * lane;
        const bool ok = k < C;
        const float4 v = *reinterpret_cast<const float4*>(
            wm + size_t(min(n0 + c, N - 1)) * C + (ok ? k : 0));
        w[q][c][u] =
            make_float4(ok ? v.x : 0.f, ok ? v.y : 0.f, ok ? v.z : 0.f, ok ? v.w : 0.f);
      }
  }
  const bool writer = blockIdx.x == 0;
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    const size_t row = size_t(r) * size_t(C);
    const bool keep = writer && r < B;
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      const int c = tid + i * kStepThreads;
      if (c >= C) continue;
      float v = in[r][i], mem_new;
      if constexpr (PRE == kPreGateLif) v = step_sigmoid(gate[r][i]) * v;
      x[r][i] += step_lif(ra, v, mem[r][i], mem_new);
      if (keep) {
        ra.membrane_out[row + c] = mem_new;
        residual_out[row + c] = x[r][i];
      }
    }
    step_layer_norm<EPT>(x[r], lw, lb, ra.ln_eps, C, red[r]);
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      const int c = tid + i * kStepThreads;
      if (keep && c < C) ra.previous_out[row + c] = x[r][i];
#pragma unroll
      for (int j = 0; j < MIXES; ++j)
        xs[j][r][c] =
            c < C ? x[r][i] * mix[j][i] + prev[r][i] * (1.f - mix[j][i]) : 0.f;
    }
  }
  __syncthreads();
  float acc[MATS][CW][ROWS];
#pragma unroll
  for (int q = 0; q < MATS; ++q)
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
#pragma unroll
      for (int c = 0; c < CW; ++c) acc[q][c][r] = 0.f;
#pragma unroll
      for (int u = 0; u < EPT; ++u) {
        const float4 v = *reinterpret_cast<const float4*>(
            &xs[MODE == kLinKvr ? q : mat0][r][256 * u + 4 * lane]);
#pragma unroll
        for (int c = 0; c < CW; ++c) {
          float s = acc[q][c][r];
          s = fmaf(w[q][c][u].x, v.x, s);
          s = fmaf(w[q][c][u].y, v.y, s);
          s = fmaf(w[q][c][u].z, v.z, s);
          acc[q][c][r] = fmaf(w[q][c][u].w, v.w, s);
        }
      }
    }
  float s[MATS];
#pragma unroll
  for (int q = 0; q < MATS; ++q) {
    s[q] = 0.f;
#pragma unroll
    for (int c = 0; c < CW; ++c)
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        const float t = lin_wave_sum(acc[q][c][r]);
        if (lane == c * ROWS + r) s[q] = t;
      }
  }
  if (!mine) return;
  if constexpr (MODE == kLinKvr) {
    lin_wkv(a, o, s[0], s[1], s[2], -expf(decay_in), first, num, den, l0);
  } else if (mat0 == 0) {
    const float z = fmaxf(s[0], 0.f);  // as relu_square_fwd_kernel
    a.out[0][o] = z * z;
  } else {
    a.out[1][o] = s[0];
  }
}

// ---- many rows: LDS-tiled ----
// A workgroup's tile is 16 WN columns by 16 WB rows, one MFMA tile per wave;
// slabs of 32 KD of K are staged in LDS (two buffers, the next slab in
// registers while the current one is multiplied).  Row stride 32 KD + 4 floats:
// the 16 rows of an operand read start on 16 different groups of four banks.
// Two accumulators halve the length of each sum.  Up to three products share a
// launch; the first may end in relu^2.  Measured at B = 256, C = 768: key,
// value and receptance 16.2 us (three library GEMMs 21.9), key + receptance
// with relu^2 20.0 us (24.2 + 5).  MFMA time is 5.9 and 9.8 us: the rest is the
// slab's loads and barriers at two to four workgroups per CU.  Other tiles at
// the same sizes: 32-deep slabs 17.3 / 21.3, 128-deep 18.7 / 21.7, 64 x 64 with
// 4 waves 21.3 / 21.7, with 8 waves 18.8 / 19.1 us (but 18.7 / 18.8 against
// 12.5 / 12.7 us at B = 128).
template <int WN, int WB, int KD>
__global__ __launch_bounds__(64 * WN * WB) void step_gemm_kernel(wkv_step_linear_args a, int mats, int tiles0,
                                                        int n_tiles, int b_tiles, int relu2) {
  constexpr int RN = 16 * WN, RB = 16 * WB;
  constexpr int SLAB = 32 * KD, LD = SLAB + 4;
  constexpr int TPR = SLAB / 4;          // threads per staged row
  constexpr int RPP = 64 * WN * WB / TPR;  // rows per pass
  constexpr int PN = RN / RPP, PB = RB / RPP;
  __shared__ __attribute__((aligned(16))) float lds[2][(RN + RB) * LD];
  const int lane = int(threadIdx.x) & 63;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  const int m = lane & 15, g = lane >> 4;
  const int xcd = int(blockIdx.x) & 7, idx = int(blockIdx.x) >> 3;
  const int nt = (idx / b_tiles) * 8 + xcd, bt = idx % b_tiles;
  if (nt >= n_tiles) return;
  // Matrices of n0 columns each, or a second one of n1 (KEY_REC).
  const int mat = min(nt / tiles0, mats - 1);
  const int N = int(mat == 1 && relu2 ? a.n1 : a.n0);
  const int K = int(a.k), B = int(a.batch);
  const int n0 = (nt - mat * tiles0) * RN, b0 = bt * RB;
  const float* w = mat == 0 ? a.w[0] : mat == 1 ? a.w[1] : a.w[2];
  const float* x = mat == 0 ? a.x[0] : mat == 1 ? a.x[1] : a.x[2];
  float* out = mat == 0 ? a.out[0] : mat == 1 ? a.out[1] : a.out[2];
  const int sr = int(threadIdx.x) / TPR, sc = 4 * (int(threadIdx.x) % TPR);
  const float* wp[PN];
  const float* xp[PB];
#pragma unroll
  for (int i = 0; i < PN; ++i) wp[i] = w + size_t(min(n0 + sr + RPP * i, N - 1)) * K + sc;
#pragma unroll
  for (int i = 0; i < PB; ++i) xp[i] = x + size_t(min(b0 + sr + RPP * i, B - 1)) * K + sc;
  float4 rw[PN], rx[PB];
  auto fetch = [&](int k) {
    const bool in = k + sc < K;
#pragma unroll
    for (int i = 0; i < PN; ++i)
      rw[i] = in ? *reinterpret_cast<const float4*>(wp[i] + k) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int i = 0; i < PB; ++i)
      rx[i] = in ? *reinterpret_cast<const float4*>(xp[i] + k) : make_float4(0.f, 0.f, 0.f, 0.f);
  };
  auto stage = [&](float* l) {
#pragma unroll
    for (int i = 0; i < PN; ++i)
      *reinterpret_cast<float4*>(l + (sr + RPP * i) * LD + sc) = rw[i];
#pragma unroll
    for (int i = 0; i < PB; ++i)
      *reinterpret_cast<float4*>(l + (RN + sr + RPP * i) * LD + sc) = rx[i];
  };
  const int wn = (wave % WN) * 16, wb = (wave / WN) * 16;
  lin_f4 acc[2] = {lin_f4{0.f, 0.f, 0.f, 0.f}, lin_f4{0.f, 0.f, 0.f, 0.f}};
  fetch(0);
  stage(lds[0]);
  __syncthreads();
  int buf = 0;
  for (int k = 0; k < K; k += SLAB, buf ^= 1) {
    const bool more = k + SLAB < K;
    if (more) fetch(k + SLAB);
    const float* l = lds[buf];
#pragma unroll
    for (int d = 0; d < KD; ++d) {
      LinFrag fw, fx;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int c = 32 * d + 8 * g + 4 * h;
        fw.v[h] = *reinterpret_cast<const float4*>(l + (wn + m) * LD + c);
        fx.v[h] = *reinterpret_cast<const float4*>(l + (RN + wb + m) * LD + c);
      }
      acc[d & 1] = lin_mfma(fw, fx, acc[d & 1]);
    }
    // The other buffer was read before the last barrier.
    if (more) {
      stage(lds[buf ^ 1]);
      __syncthreads();
    }
  }
  const int n = n0 + wn + 4 * g, b = b0 + wb + m;
  if (n >= N || b >= B) return;  // N is a multiple of 4
  lin_f4 v = acc[0] + acc[1];
  if (relu2 && mat == 0) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float z = fmaxf(v[r], 0.f);  // as relu_square_fwd_kernel
      v[r] = z * z;
    }
  }
  *reinterpret_cast<lin_f4*>(out + size_t(b) * N + n) = v;
}

}  // namespace wkv

// ------------------------------------------------------------ launchers ----
namespace wkv_host {

template <int MODE, int TN, int KS>
static int step_linear_launch(const wkv_step_linear_args& a, int parts, hipStream_t s) {
  const int tn = 16 * TN;
  const int t0 = int((a.n0 + tn - 1) / tn);
  const int tiles = MODE == wkv::kLinThree    ? 3 * t0
                    : MODE == wkv::kLinKeyRec ? t0 + int((a.n1 + tn - 1) / tn)
                                              : t0;
  const int bt = int((a.batch + 15) / 16);
  launch(wkv::step_linear_kernel<MODE, TN, KS>,
         dim3(unsigned((tiles + 7) / 8 * 8 * bt), unsigned(parts)), dim3(64 * KS), s, true, a, t0,
         tiles, bt, parts);
  return check_launch("step_linear_kernel");
}

// Workgroups that the 256 CUs run one after the other, times the tile's work:
// the measured times of the tile sizes follow it (B=64 C=768 key + receptance,
// 16 / 32 / 48 / 64 / 80 columns: 12.9, 11.0, 14.2, 11.1, 12.9 us for costs 4,
// 4, 6, 4, 5), so the least cost is taken, the widest tile among equals (it
// reads x least often).
static int64_t tile_cost(int mode, const wkv_step_linear_args& a, int tn, int parts) {
  const int64_t c = 16 * tn;
  const int64_t tiles = (mode == wkv::kLinThree ? 3 : 1) * ((a.n0 + c - 1) / c) +
                        (mode == wkv::kLinKeyRec ? (a.n1 + c - 1) / c : 0);
  const int64_t wgs = tiles * ((a.batch + 15) / 16) * parts;
  return (wgs + 255) / 256 * tn * (12 / parts);
}

// Calls that run one wave per dot product.  Against the tiles (us at C = 768,
// 256, 128): PLAIN and KVR gain up to four rows (B = 4 KVR 5.6 / 9.3, 4.3 / 4.6,
// but 4.2 / 3.7 at 128, where a sum over the wave costs more than its loads),
// KEY_REC, which fills the chip with tiles sooner, up to two (B = 2 4.5 / 5.1,
// 2.6 / 2.9, 2.6 / 2.6; B = 3 5.0 / 5.1, 3.0 / 2.9, 3.0 / 2.6).
static bool step_gemv_taken(int mode, int64_t batch, int64_t k) {
  if (mode == wkv::kLinPlain) return batch <= 4;
  if (mode == wkv::kLinKvr) return batch <= 2 || (batch <= 4 && k >= 256);
  return mode == wkv::kLinKeyRec && batch <= 2;
}

template <int MODE, int ROWS, int CW, int SPLIT>
static int step_gemv_launch(const wkv_step_linear_args& a, wkv::StepCopy copy, hipStream_t s) {
  const int64_t g0 = (a.n0 + CW - 1) / CW;
  const int64_t groups = g0 + (MODE == wkv::kLinKeyRec ? (a.n1 + CW - 1) / CW : 0);
  constexpr int64_t per = 4 / SPLIT;
  copy.first = int((groups + per - 1) / per);
  const dim3 grid(unsigned(copy.first + (2 * copy.n + 255) / 256));
  // 256-column pieces of a wave's share of K, at most four at a time.
  switch (((a.k + 255) / 256 + SPLIT - 1) / SPLIT) {
    case 1:
      launch(wkv::step_gemv_kernel<MODE, ROWS, CW, SPLIT, 1>, grid, dim3(256), s, true, a,
             int(g0), int(groups), copy);
      break;
    case 2:
      launch(wkv::step_gemv_kernel<MODE, ROWS, CW, SPLIT, 2>, grid, dim3(256), s, true, a,
             int(g0), int(groups), copy);
      break;
    case 3:
      launch(wkv::step_gemv_kernel<MODE, ROWS, CW, SPLIT, 3>, grid, dim3(256), s, true, a,
             int(g0), int(groups), copy);
      break;
    default:
      launch(wkv::step_gemv_kernel<MODE, ROWS, CW, SPLIT, 4>, grid, dim3(256), s, true, a,
             int(g0), int(groups), copy);
  }
  return check_launch("step_gemv_kernel");
}

template <int ROWS>
static int step_gemv_rows(int mode, const wkv_step_linear_args& a, const wkv::StepCopy& copy,
                          hipStream_t s) {
  if (mode == wkv::kLinKvr) return step_gemv_launch<wkv::kLinKvr, ROWS, 1, 1>(a, copy, s);
  if constexpr (ROWS <= 2) {
    if (mode == wkv::kLinKeyRec)
      return step_gemv_launch<wkv::kLinKeyRec, ROWS, 4, 1>(a, copy, s);
  }
  if (a.k > 1024) return step_gemv_launch<wkv::kLinPlain, ROWS, 2, 4>(a, copy, s);
  return step_gemv_launch<wkv::kLinPlain, ROWS, 1, 1>(a, copy, s);
}

static int step_gemv(int mode, const wkv_step_linear_args& a, const wkv::StepCopy& copy,
                     hipStream_t s) {
  if (a.batch == 1) return step_gemv_rows<1>(mode, a, copy, s);
  if (a.batch == 2) return step_gemv_rows<2>(mode, a, copy, s);
  return step_gemv_rows<4>(mode, a, copy, s);
}

int step_linear_copy_impl(const wkv_step_linear_args& a, const float* src, float* dst0,
                          float* dst1, int64_t n, hipStream_t s) {
  return step_gemv(wkv::kLinPlain, a, wkv::StepCopy{src, {dst0, dst1}, int(n), 0}, s);
}

template <int PRE, int MODE, int ROWS, int CW>
static int step_row_gemv_launch(const wkv_step_row_args& ra, float* residual_out,
                                const wkv_step_linear_args& a, hipStream_t s) {
  const int64_t g0 = (a.n0 + CW - 1) / CW;
  const int64_t groups = g0 + (MODE == wkv::kLinKeyRec ? (a.n1 + CW - 1) / CW : 0);
  const dim3 grid(unsigned((groups + 3) / 4)), block(wkv::kStepThreads);
  switch ((a.k + 255) / 256) {
    case 1:
      launch(wkv::step_row_gemv_kernel<PRE, MODE, ROWS, CW, 1>, grid, block, s, true, ra,
             residual_out, a, int(g0));
      break;
    case 2:
      launch(wkv::step_row_gemv_kernel<PRE, MODE, ROWS, CW, 2>, grid, block, s, true, ra,
             residual_out, a, int(g0));
      break;
    case 3:
      launch(wkv::step_row_gemv_kernel<PRE, MODE, ROWS, CW, 3>, grid, block, s, true, ra,
             residual_out, a, int(g0));
      break;
    case 4:
      launch(wkv::step_row_gemv_kernel<PRE, MODE, ROWS, CW, 4>, grid, block, s, true, ra,
             residual_out, a, int(g0));
      break;
    default:
      return fail(1, "block_step_row_linear: rows of at most 1024 channels");
  }
  return check_launch("step_row_gemv_kernel");
}

int step_row_linear_impl(int mode, const wkv_step_row_args& ra, float* residual_out,
                         const wkv_step_linear_args& a, hipStream_t s) {
  if (mode == wkv::kLinKvr)
    return a.batch == 1
               ? step_row_gemv_launch<wkv::kPreGateLif, wkv::kLinKvr, 1, 1>(ra, residual_out, a, s)
               : step_row_gemv_launch<wkv::kPreGateLif, wkv::kLinKvr, 2, 1>(ra, residual_out, a,
                                                                            s);
  return a.batch == 1
             ? step_row_gemv_launch<wkv::kPreLif, wkv::kLinKeyRec, 1, 4>(ra, residual_out, a, s)
             : step_row_gemv_launch<wkv::kPreLif, wkv::kLinKeyRec, 2, 4>(ra, residual_out, a, s);
}

// Parts of a PLAIN product's K: up to 4, each at least 512 deep.
int step_linear_parts_impl(int64_t batch, int64_t k, int64_t n) {
  wkv_step_linear_args a{};
  a.batch = batch;
  a.k = k;
  a.n0 = n;
  int best = 1;
  if (step_gemv_taken(wkv::kLinPlain, batch, k)) return best;
  int64_t cost = INT64_MAX;
  for (int parts = 1; parts <= 4 && k / parts >= 512; ++parts)
    for (int tn = 1; tn <= 3; ++tn) {
      const int64_t c = tile_cost(wkv::kLinPlain, a, tn, parts);
      if (c < cost) {
        cost = c;
        best = parts;
      }
    }
  return best;
}

static int step_gemm_launch(int mode, const wkv_step_linear_args& a, hipStream_t s) {
  const int mats = mode == wkv::kLinThree ? 3 : 2;
  const int64_t first = (a.n0 + 31) / 32;
  const int64_t tiles = mats == 3 ? 3 * first : first + (a.n1 + 31) / 32;
  const int64_t bt = (a.batch + 31) / 32;
  launch(wkv::step_gemm_kernel<2, 2, 2>, dim3(unsigned((tiles + 7) / 8 * 8 * bt)), dim3(256), s,
         true, a, mats, int(first), int(tiles), int(bt), int(mode == wkv::kLinKeyRec));
  return check_launch("step_gemm_kernel");
}

int step_linear_impl(int mode, const wkv_step_linear_args& a, int parts, hipStream_t s) {
  if (parts == 1 && step_gemv_taken(mode, a.batch, a.k)) return step_gemv(mode, a, wkv::StepCopy{}, s);
  if (mode == wkv::kLinKvr) return step_linear_launch<wkv::kLinKvr, 1, 8>(a, 1, s);
  // THREE: small tiles up to the same line (at C = 768, B = 64, 192 of them, 11.4
  // us with the WKV kernel; from 384 on the LDS tiles, 12.1 and 3.5 us).
  if (mode == wkv::kLinThree && ((a.batch + 15) / 16) * ((a.n0 + 15) / 16) > 256)
    return step_gemm_launch(mode, a, s);
  // KEY_REC beyond 256 16 x 16 tiles of the receptance: at C = 768, B = 128 (384
  // tiles) 12.7 against 18.7 us, at B = 64 (192) about 12 against 11.0.
  if (mode == wkv::kLinKeyRec && a.n0 % 4 == 0 && a.n1 % 4 == 0 &&
      ((a.batch + 15) / 16) * ((a.n1 + 15) / 16) > 256)
    return step_gemm_launch(mode, a, s);
  int tn = 1;
  for (int t = 2; t <= (mode == wkv::kLinKeyRec ? 4 : 3); ++t)
    if (tile_cost(mode, a, t, parts) <= tile_cost(mode, a, tn, parts)) tn = t;
  if (mode == wkv::kLinPlain) {
    switch (tn) {
      case 1: return step_linear_launch<wkv::kLinPlain, 1, 8>(a, parts, s);
      case 2: return step_linear_launch<wkv::kLinPlain, 2, 8>(a, parts, s);
      default: return step_linear_launch<wkv::kLinPlain, 3, 8>(a, parts, s);
    }
  }
  if (mode == wkv::kLinThree) {
    switch (tn) {
      case 1: return step_linear_launch<wkv::kLinThree, 1, 8>(a, 1, s);
      case 2: return step_linear_launch<wkv::kLinThree, 2, 8>(a, 1, s);
      default: return step_linear_launch<wkv::kLinThree, 3, 8>(a, 1, s);
    }
  }
  if (mode == wkv::kLinKeyRec) {
    switch (tn) {
      case 1: return step_linear_launch<wkv::kLinKeyRec, 1, 8>(a, 1, s);
      case 2: return step_linear_launch<wkv::kLinKeyRec, 2, 4>(a, 1, s);
      case 3: return step_linear_launch<wkv::kLinKeyRec, 3, 8>(a, 1, s);
      default: return step_linear_launch<wkv::kLinKeyRec, 4, 4>(a, 1, s);
    }
  }
  return fail(1, "block_step_linear: unknown mode");
}

}  // namespace wkv_host
