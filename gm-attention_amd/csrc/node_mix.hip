// The factored kernel's node-side channel mixing (CDNA4, gfx950): every
// head's node mixes Z_t(j) = W_t v_j for one input frequency as one real
// product over the nodes,
//
//   forward   mix (N, C) = v (N, w) M (w, C)
//   backward  dv (N, w)  = dmix M^T            (the node field's gradient)
//             dM (w, C)  = v^T dmix            (the mixing matrix's gradient)
//
// with v the node field's frequency-n reals (w <= 128, a strided view of the
// flat rows) and M the heads' real mixing matrix (every block's complex
// product and input conjugation encoded as reals; C = H K C_n columns).  The
// reference forms the same numbers as one complex einsum("ja,bat->jtb") per
// node vector and block group (nn/kernels.py:575-603, over _block_weights
// :506-536) and their gradients through autograd.
//
// All three are MFMA products in float32 accuracy: vectors of 17 to 128 reals
// as split bf16 products over 32 contraction indices an instruction
// (node_mix_*_deep), vectors up to 16 over 16 (node_mix_*_split), and under
// GM_SPLIT_PRODUCTS=0 v_mfma_f32_16x16x4f32 (lane l = 16 q + c supplies A[c][q]
// and B[q][c] and holds D[4 q + i][c], i < 4).
//
// * forward: the contraction is short, so each wave keeps its columns of M in
//   registers for the whole launch and streams 64-row tiles of v through LDS;
//   M is the A operand (D = mix^T), so a lane's four D entries are four
//   consecutive columns of one row: one 16-byte store each.
// * input gradient: 128-row tiles, each wave 32 rows over the contraction, M
//   staged per chunk of columns in LDS; the accumulators restart every 256
//   columns into a running total, so no fp32 sum runs sequentially over more.
// * weight gradient: split over row ranges into partial (w, C) matrices; a
//   second pass sums the partials in a fixed order.  No atomics anywhere:
//   results are deterministic.
//
// Bound: the bytes of the mixes, (N, C) written by the forward and read by each
// gradient.  256x512, B = 4 (N = 524,288), w = 64, C = 5,440 (11.4 GB; a plain
// read of them takes 1.85 ms, a plain write 2.0), 16-deep -> 32-deep: forward
// 3.21 -> 2.60 ms, input gradient 3.06 -> 2.61, weight gradient 3.35 -> 2.48;
// w = 32, C = 2,720: 1.25 -> 1.06, 1.12 -> 1.10, 1.14 -> 1.05; w = 128, N =
// 65,536, C = 26,112 (6.8 GB): 3.82 -> 2.57, 3.98 -> 2.50, 5.55 -> 2.75.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "common.hpp"
#include "split.hpp"

// The weight gradient's partials for gm_node_mix_backward_weight_noalloc_f32:
// 2^23 floats (32 MiB) on every GPU the library runs on, held until the process
// ends.  Host code reaches it only through the per-device address below.
static __device__ __align__(256) float scratch[int64_t(1) << 23];

namespace gm {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ floatx4 mfma4(float a, float b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

constexpr int kThreads = 256;
// DPP control: rotate right by 8 lanes within each row of 16 (lane c takes lane c ^ 8's value).
constexpr int kDppRowRor8 = 0x128;
constexpr floatx4 kZero4 = {0.f, 0.f, 0.f, 0.f};

// ---------------------------------------------------------------- forward
//
// Workgroup (x, y): columns [x * 64 CT, (x + 1) * 64 CT), wave wv owning CT
// 16-column tiles from col0 = x * 64 CT + 16 CT wv; row tiles y, y + gridDim.y, ...
// Step s of the contraction pairs slot q with k = q (W / 4) + s, so a lane's
// v operands for consecutive steps are consecutive floats of its row (read
// four at a time from LDS).
template <int W, int CT>
__global__ __launch_bounds__(kThreads) void node_mix_forward_kernel(const float* __restrict__ v, int64_t ldv,
                                                                    const float* __restrict__ M, int64_t N, int w,
                                                                    int64_t C, float* __restrict__ out, int vec_v,
                                                                    int vec_out) {
  constexpr int KS = W / 4;    // contraction steps
  constexpr int LDT = W + 4;   // LDS row stride: a 16-lane b128 read covers all 64 banks once
  constexpr int QUADS = 64 * KS;  // 16-byte pieces of a 64-row tile (KS of them a row)
  __shared__ __align__(16) float vt[64 * LDT];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, c = lane & 15, q = lane >> 4;
  const int64_t col0 = (int64_t)blockIdx.x * (64 * CT) + 16 * CT * wv;
  float mreg[KS][CT];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const int k = q * KS + s;
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const int64_t col = col0 + 16 * j + c;
      mreg[s][j] = (k < w && col < C) ? M[(int64_t)k * C + col] : 0.f;
    }
  }
  const int64_t n_tiles = (N + 63) / 64;
  constexpr int PER = (QUADS + kThreads - 1) / kThreads;
  float4 pre[PER];
  auto fetch = [&](int64_t tile) {
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int idx = threadIdx.x + p * kThreads;
      const int row = idx / KS, kq = idx % KS;
      const int64_t r = tile * 64 + row;
      const int k = 4 * kq;
      float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
      if (idx < QUADS && r < N) {
        const float* src = v + r * ldv + k;
        if (vec_v && k + 3 < w) {
          x = *reinterpret_cast<const float4*>(src);
        } else {
          x.x = k < w ? src[0] : 0.f;
          x.y = k + 1 < w ? src[1] : 0.f;
          x.z = k + 2 < w ? src[2] : 0.f;
          x.w = k + 3 < w ? src[3] : 0.f;
        }
      }
      pre[p] = x;
    }
  };
  if ((int64_t)blockIdx.y < n_tiles) fetch(blockIdx.y);
  for (int64_t tile = blockIdx.y; tile < n_tiles; tile += gridDim.y) {
    __syncthreads();  // the previous tile's LDS reads are done
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int idx = threadIdx.x + p * kThreads;
      if (idx < QUADS) *reinterpret_cast<float4*>(&vt[(idx / KS) * LDT + 4 * (idx % KS)]) = pre[p];
    }
    __syncthreads();
    if (tile + gridDim.y < n_tiles) fetch(tile + gridDim.y);
    const int64_t row0 = tile * 64;
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      float b[KS];
#pragma unroll
      for (int s4 = 0; s4 < KS / 4; ++s4) {
        const float4 x = *reinterpret_cast<const float4*>(&vt[(16 * rt + c) * LDT + q * KS + 4 * s4]);
        b[4 * s4] = x.x;
        b[4 * s4 + 1] = x.y;
        b[4 * s4 + 2] = x.z;
        b[4 * s4 + 3] = x.w;
      }
      floatx4 acc[CT];
#pragma unroll
      for (int j = 0; j < CT; ++j) acc[j] = kZero4;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
#pragma unroll
        for (int j = 0; j < CT; ++j) acc[j] = mfma4(mreg[s][j], b[s], acc[j]);
      }
      const int64_t row = row0 + 16 * rt + c;
      if (row < N) {
        float* dst = out + row * C;
#pragma unroll
        for (int j = 0; j < CT; ++j) {
          const int64_t col = col0 + 16 * j + 4 * q;
          if (vec_out && col + 3 < C) {
            *reinterpret_cast<float4*>(dst + col) = make_float4(acc[j][0], acc[j][1], acc[j][2], acc[j][3]);
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (col + i < C) dst[col + i] = acc[j][i];
          }
        }
      }
    }
  }
}

// ---------------------------------------------------------------- input gradient
//
// Workgroup x: rows [128 x, 128 x + 128); wave wv rows 32 wv + 16 rt + c
// (rt < 2) as the A operand, M's rows (the w columns of dv) as B.  Chunk
// k-slot mapping: step s = 4 t + i of a chunk pairs slot q with column
// c0 + 16 q + s, so both operands read four consecutive floats of an LDS row.
// Two waves a SIMD: the compiler then keeps the accumulators with the operands
// in VGPRs (measured 3.45 vs 3.66 ms at N = 524288, w = 64, C = 5440).
template <int W>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void node_mix_dinput_kernel(const float* __restrict__ dmix,
                                                                   const float* __restrict__ M, int64_t N, int w,
                                                                   int64_t C, float* __restrict__ dv, int64_t lddv) {
  constexpr int KC = 64, LDD = KC + 4, JW = W / 16;
  constexpr int DQ = 128 * KC / 4 / kThreads;  // 16-byte pieces of the dmix tile per thread: 8
  constexpr int MQ = W * KC / 4 / kThreads;    // of the M tile: W / 16
  __shared__ __align__(16) float dt[128 * LDD];
  __shared__ __align__(16) float mt[W * LDD];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, c = lane & 15, q = lane >> 4;
  const int64_t row0 = (int64_t)blockIdx.x * 128;
  const int64_t n_chunks = (C + KC - 1) / KC;
  float4 pd[DQ], pm[MQ];
  auto fetch = [&](int64_t ch) {
    const int64_t c0 = ch * KC;
#pragma unroll
    for (int p = 0; p < DQ; ++p) {
      const int idx = threadIdx.x + p * kThreads, row = idx >> 4, cq = idx & 15;
      const int64_t r = row0 + row, col = c0 + 4 * cq;
      pd[p] = (r < N && col < C) ? *reinterpret_cast<const float4*>(dmix + r * C + col)
                                 : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int p = 0; p < MQ; ++p) {
      const int idx = threadIdx.x + p * kThreads, row = idx >> 4, cq = idx & 15;
      const int64_t col = c0 + 4 * cq;
      pm[p] = (row < w && col < C) ? *reinterpret_cast<const float4*>(M + (int64_t)row * C + col)
                                   : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  };
  floatx4 acc[2][JW], tot[2][JW];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt)
#pragma unroll
    for (int j = 0; j < JW; ++j) acc[rt][j] = tot[rt][j] = kZero4;
  fetch(0);
  for (int64_t ch = 0; ch < n_chunks; ++ch) {
    __syncthreads();
#pragma unroll
    for (int p = 0; p < DQ; ++p) {
      const int idx = threadIdx.x + p * kThreads;
      *reinterpret_cast<float4*>(&dt[(idx >> 4) * LDD + 4 * (idx & 15)]) = pd[p];
    }
#pragma unroll
    for (int p = 0; p < MQ; ++p) {
      const int idx = threadIdx.x + p * kThreads;
      *reinterpret_cast<float4*>(&mt[(idx >> 4) * LDD + 4 * (idx & 15)]) = pm[p];
    }
    __syncthreads();
    if (ch + 1 < n_chunks) fetch(ch + 1);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      float4 a[2], b[JW];
#pragma unroll
      for (int rt = 0; rt < 2; ++rt)
        a[rt] = *reinterpret_cast<const float4*>(&dt[(32 * wv + 16 * rt + c) * LDD + 16 * q + 4 * t]);
#pragma unroll
      for (int j = 0; j < JW; ++j) b[j] = *reinterpret_cast<const float4*>(&mt[(16 * j + c) * LDD + 16 * q + 4 * t]);
#pragma unroll
      for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int j = 0; j < JW; ++j) {
          acc[rt][j] = mfma4(a[rt].x, b[j].x, acc[rt][j]);
          acc[rt][j] = mfma4(a[rt].y, b[j].y, acc[rt][j]);
          acc[rt][j] = mfma4(a[rt].z, b[j].z, acc[rt][j]);
          acc[rt][j] = mfma4(a[rt].w, b[j].w, acc[rt][j]);
        }
    }
    if ((ch & 3) == 3 || ch + 1 == n_chunks) {
#pragma unroll
      for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int j = 0; j < JW; ++j) {
          tot[rt][j] += acc[rt][j];
          acc[rt][j] = kZero4;
        }
    }
  }
  // D[4 q + i][c]: dv row row0 + 32 wv + 16 rt + 4 q + i, column 16 j + c
#pragma unroll
  for (int rt = 0; rt < 2; ++rt)
#pragma unroll
    for (int j = 0; j < JW; ++j) {
      const int col = 16 * j + c;
      if (col >= w) continue;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int64_t r = row0 + 32 * wv + 16 * rt + 4 * q + i;
        if (r < N) dv[r * lddv + col] = tot[rt][j][i];
      }
    }
}

// ---------------------------------------------------------------- weight gradient
//
// Vectors wider than 64 reals: workgroup (x, y) owns columns [128 x, 128 x + 128)
// (wave wv: 32 wv + 16 jc + c, jc < 2) over rows [y rps, min(N, (y + 1) rps));
// v^T as A (w rows in 16-row tiles), dmix as B.  Step s of a 64-row chunk
// pairs slot q with row 4 s + q (so does the kernel below).
template <int W>
constexpr int dweight_ldv() {
  return (W % 64 == 16 || W % 64 == 48) ? W : W + 16;  // rows 4 s + q land 16 banks apart
}

template <int W>
__global__ __launch_bounds__(kThreads) void node_mix_dweight_kernel(const float* __restrict__ v, int64_t ldv,
                                                                    const float* __restrict__ dmix, int64_t N, int w,
                                                                    int64_t C, int64_t rps, float* __restrict__ partial,
                                                                    int vec_v) {
  constexpr int RC = 64, LDV = dweight_ldv<W>(), LDM = 128 + 16, IW = W / 16;
  constexpr int VQ = (RC * W / 4 + kThreads - 1) / kThreads;  // 16-byte pieces of the v tile per thread
  constexpr int DQ = RC * 128 / 4 / kThreads;                  // of the dmix tile: 8
  __shared__ __align__(16) float vt[RC * LDV];
  __shared__ __align__(16) float dt[RC * LDM];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, c = lane & 15, q = lane >> 4;
  const int64_t c0 = (int64_t)blockIdx.x * 128;
  const int64_t first = (int64_t)blockIdx.y * rps, last = first + rps < N ? first + rps : N;
  float4 pv[VQ], pd[DQ];
  auto fetch = [&](int64_t r0) {
#pragma unroll
    for (int p = 0; p < VQ; ++p) {
      const int idx = threadIdx.x + p * kThreads, row = idx / (W / 4), k = 4 * (idx % (W / 4));
      const int64_t r = r0 + row;
      float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
      if (idx < RC * W / 4 && r < last) {
        const float* src = v + r * ldv + k;
        if (vec_v && k + 3 < w) {
          x = *reinterpret_cast<const float4*>(src);
        } else {
          x.x = k < w ? src[0] : 0.f;
          x.y = k + 1 < w ? src[1] : 0.f;
          x.z = k + 2 < w ? src[2] : 0.f;
          x.w = k + 3 < w ? src[3] : 0.f;
        }
      }
      pv[p] = x;
    }
#pragma unroll
    for (int p = 0; p < DQ; ++p) {
      const int idx = threadIdx.x + p * kThreads, row = idx >> 5, cq = idx & 31;
      const int64_t r = r0 + row, col = c0 + 4 * cq;
      pd[p] = (r < last && col < C) ? *reinterpret_cast<const float4*>(dmix + r * C + col)
                                    : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  };
  floatx4 acc[IW][2], tot[IW][2];
#pragma unroll
  for (int i = 0; i < IW; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = tot[i][j] = kZero4;
  int64_t chunk = 0;
  if (first < last) fetch(first);
  for (int64_t r0 = first; r0 < last; r0 += RC, ++chunk) {
    __syncthreads();
#pragma unroll
    for (int p = 0; p < VQ; ++p) {
      const int idx = threadIdx.x + p * kThreads;
      if (idx < RC * W / 4) *reinterpret_cast<float4*>(&vt[(idx / (W / 4)) * LDV + 4 * (idx % (W / 4))]) = pv[p];
    }
#pragma unroll
    for (int p = 0; p < DQ; ++p) {
      const int idx = threadIdx.x + p * kThreads;
      *reinterpret_cast<float4*>(&dt[(idx >> 5) * LDM + 4 * (idx & 31)]) = pd[p];
    }
    __syncthreads();
    if (r0 + RC < last) fetch(r0 + RC);
#pragma unroll 4
    for (int s = 0; s < RC / 4; ++s) {
      const int row = 4 * s + q;
      float a[IW], b[2];
#pragma unroll
      for (int i = 0; i < IW; ++i) a[i] = vt[row * LDV + 16 * i + c];
#pragma unroll
      for (int j = 0; j < 2; ++j) b[j] = dt[row * LDM + 32 * wv + 16 * j + c];
#pragma unroll
      for (int i = 0; i < IW; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mfma4(a[i], b[j], acc[i][j]);
    }
    if ((chunk & 15) == 15) {
#pragma unroll
      for (int i = 0; i < IW; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          tot[i][j] += acc[i][j];
          acc[i][j] = kZero4;
        }
    }
  }
  // D[4 q + ii][c]: dM row 16 i + 4 q + ii, column c0 + 32 wv + 16 j + c
  float* out = partial + (int64_t)blockIdx.y * w * C;
#pragma unroll
  for (int i = 0; i < IW; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int64_t col = c0 + 32 * wv + 16 * j + c;
      if (col >= C) continue;
      const floatx4 sum = tot[i][j] + acc[i][j];
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) {
        const int row = 16 * i + 4 * q + ii;
        if (row < w) out[(int64_t)row * C + col] = sum[ii];
      }
    }
}

// Vectors up to 64 reals wide: workgroup (x, y) owns the whole (w x 64)-column
// tile [64 x, 64 x + 64) over rows [y rps, min(N, (y + 1) rps)); its four waves
// take rows 16 wv .. 16 wv + 15 of each 64-row chunk, each accumulating the whole
// tile (so every operand read feeds four MFMAs), and write one partial each:
// 4 S partial matrices.
template <int W>
__global__ __launch_bounds__(kThreads) void node_mix_dweight_k_kernel(const float* __restrict__ v, int64_t ldv,
                                                                    const float* __restrict__ dmix, int64_t N, int w,
                                                                    int64_t C, int64_t rps, float* __restrict__ partial,
                                                                    int vec_v) {
  constexpr int RC = 64, LDV = dweight_ldv<W>(), LDM = 64 + 16, IW = W / 16;
  constexpr int VQ = (RC * W / 4 + kThreads - 1) / kThreads;
  constexpr int DQ = RC * 64 / 4 / kThreads;  // 4
  __shared__ __align__(16) float vt[RC * LDV];
  __shared__ __align__(16) float dt[RC * LDM];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, c = lane & 15, q = lane >> 4;
  const int64_t c0 = (int64_t)blockIdx.x * 64;
  const int64_t first = (int64_t)blockIdx.y * rps, last = first + rps < N ? first + rps : N;
  float4 pv[VQ], pd[DQ];
  auto fetch = [&](int64_t r0) {
#pragma unroll
    for (int p = 0; p < VQ; ++p) {
      const int idx = threadIdx.x + p * kThreads, row = idx / (W / 4), k = 4 * (idx % (W / 4));
      const int64_t r = r0 + row;
      float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
      if (idx < RC * W / 4 && r < last) {
        const float* src = v + r * ldv + k;
        if (vec_v && k + 3 < w) {
          x = *reinterpret_cast<const float4*>(src);
        } else {
          x.x = k < w ? src[0] : 0.f;
          x.y = k + 1 < w ? src[1] : 0.f;
          x.z = k + 2 < w ? src[2] : 0.f;
          x.w = k + 3 < w ? src[3] : 0.f;
        }
      }
      pv[p] = x;
    }
#pragma unroll
    for (int p = 0; p < DQ; ++p) {
      const int idx = threadIdx.x + p * kThreads, row = idx >> 4, cq = idx & 15;
      const int64_t r = r0 + row, col = c0 + 4 * cq;
      pd[p] = (r < last && col < C) ? *reinterpret_cast<const float4*>(dmix + r * C + col)
                                    : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  };
  floatx4 acc[IW][4];
#pragma unroll
  for (int i = 0; i < IW; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = kZero4;
  if (first < last) fetch(first);
  for (int64_t r0 = first; r0 < last; r0 += RC) {
    __syncthreads();
#pragma unroll
    for (int p = 0; p < VQ; ++p) {
      const int idx = threadIdx.x + p * kThreads;
      if (idx < RC * W / 4) *reinterpret_cast<float4*>(&vt[(idx / (W / 4)) * LDV + 4 * (idx % (W / 4))]) = pv[p];
    }
#pragma unroll
    for (int p = 0; p < DQ; ++p) {
      const int idx = threadIdx.x + p * kThreads;
      *reinterpret_cast<float4*>(&dt[(idx >> 4) * LDM + 4 * (idx & 15)]) = pd[p];
    }
    __syncthreads();
    if (r0 + RC < last) fetch(r0 + RC);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int row = 16 * wv + 4 * s + q;
      float a[IW], b[4];
#pragma unroll
      for (int i = 0; i < IW; ++i) a[i] = vt[row * LDV + 16 * i + c];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = dt[row * LDM + 16 * j + c];
#pragma unroll
      for (int i = 0; i < IW; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = mfma4(a[i], b[j], acc[i][j]);
    }
  }
  float* out = partial + ((int64_t)blockIdx.y * 4 + wv) * w * C;
#pragma unroll
  for (int i = 0; i < IW; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t col = c0 + 16 * j + c;
      if (col >= C) continue;
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) {
        const int row = 16 * i + 4 * q + ii;
        if (row < w) out[(int64_t)row * C + col] = acc[i][j][ii];
      }
    }
}

// ---------------------------------------------------------------- split products
//
// Four consecutive reals k .. k + 3 (< w) of a node vector at src, float32 or
// bfloat16 (widened exactly); vec: 16-byte (8-byte) aligned whole quads.
__device__ __forceinline__ float4 load_v4(const float* src, int k, int w, int vec) {
  if (vec && k + 3 < w) return *reinterpret_cast<const float4*>(src);
  return make_float4(k < w ? src[0] : 0.f, k + 1 < w ? src[1] : 0.f, k + 2 < w ? src[2] : 0.f,
                     k + 3 < w ? src[3] : 0.f);
}
__device__ __forceinline__ float bf16_at(const uint16_t* p) { return __uint_as_float((uint32_t)*p << 16); }
__device__ __forceinline__ float4 load_v4(const uint16_t* src, int k, int w, int vec) {
  if (vec && k + 3 < w) {
    const uint2 u = *reinterpret_cast<const uint2*>(src);
    return make_float4(__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xFFFF0000u), __uint_as_float(u.y << 16),
                       __uint_as_float(u.y & 0xFFFF0000u));
  }
  return make_float4(k < w ? bf16_at(src) : 0.f, k + 1 < w ? bf16_at(src + 1) : 0.f,
                     k + 2 < w ? bf16_at(src + 2) : 0.f, k + 3 < w ? bf16_at(src + 3) : 0.f);
}
// Four consecutive entries of a mix-gradient row, float32 or bfloat16 (widened
// exactly; 8-byte aligned quads).
__device__ __forceinline__ float4 load_dm4(const float* src) { return *reinterpret_cast<const float4*>(src); }
__device__ __forceinline__ float4 load_dm4(const uint16_t* src) {
  const uint2 u = *reinterpret_cast<const uint2*>(src);
  return make_float4(__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xFFFF0000u), __uint_as_float(u.y << 16),
                     __uint_as_float(u.y & 0xFFFF0000u));
}
//
// The same three products for vectors up to 16 reals, with every fp32 product
// formed as six bf16 products on v_mfma_f32_16x16x32_bf16 (three-piece splits,
// fp32 accuracy: split.hpp).  A 16-deep contraction chunk kc gives lane
// (c, q) the indices 16 kc + 4 q + s, s < 4, in both operands.

// A 32-deep operand would be half zeros here; wider vectors take the 32-deep forms
// below.  The forward's two bodies, with and without a check a store, take 112
// registers and four waves a SIMD where one with checks takes 74 and six: N =
// 524,288, w = 16, C = 1,360 836 -> 795 us, C = 5,440 2,368 -> 2,299; a single short
// round of workgroups pays (N = 8,192, C = 2,720 19.4 -> 20.6 us).  The kernels'
// tiling: columns a forward wave owns (16 kSplitCT), rows an input-gradient
// wave owns (16 kSplitRT) and columns a weight-gradient workgroup owns
// (16 kSplitJT).
constexpr int kSplitCT = 2, kSplitRT = 2, kSplitJT = 4;

// A SplitB operand from three bf16 planes (four contraction indices each).
__device__ __forceinline__ SplitB split_b_planes(uint2 hi, uint2 mid, uint2 lo) {
  return SplitB{u32x4{hi.x, hi.y, hi.x, hi.y}, u32x4{mid.x, mid.y, mid.x, mid.y}, u32x4{lo.x, lo.y, hi.x, hi.y}};
}

// Four values' three pieces into three bf16 planes at element `at`.
__device__ __forceinline__ void store_planes(uint16_t* plane0, uint16_t* plane1, uint16_t* plane2, int at,
                                             float4 x) {
  const Split4 sp = split4(x.x, x.y, x.z, x.w);
  *reinterpret_cast<uint2*>(plane0 + at) = make_uint2(sp.hi[0], sp.hi[1]);
  *reinterpret_cast<uint2*>(plane1 + at) = make_uint2(sp.mid[0], sp.mid[1]);
  *reinterpret_cast<uint2*>(plane2 + at) = make_uint2(sp.lo[0], sp.lo[1]);
}

// Four consecutive columns of an output row; FULL: a whole row tile and whole
// aligned columns (no checks, so the stores do not break up the product's
// code: 3.86 -> 2.6 ms for 64 reals at N = 524,288 against a check a store),
// else those below C of the rows below N.
template <bool FULL>
__device__ __forceinline__ void store4(float* out, int64_t row, int64_t col, int64_t N, int64_t C, floatx4 x,
                                       int vec_out) {
  float* dst = out + row * C + col;
  if constexpr (FULL) {
    *reinterpret_cast<floatx4*>(dst) = x;
  } else {
    if (row >= N) return;
    if (vec_out && col + 3 < C) {
      *reinterpret_cast<floatx4*>(dst) = x;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (col + i < C) dst[i] = x[i];
    }
  }
}

// Forward: wave wv of workgroup x owns columns x * 64 CT + 16 CT wv + 16 j + c
// (j < CT); the pieces of M at those columns are split once per wave and held
// in registers; each 64-row tile of v is split once per workgroup into LDS, from
// which every wave takes its B operands: three bf16 planes (row stride W + 4
// halfwords: a 16-lane 8-byte read covers 32 banks once) assembled into
// operands by each wave.
template <int W, typename V = float>
__global__ __launch_bounds__(kThreads) void node_mix_forward_split(const V* __restrict__ v, int64_t ldv,
                                                                   const float* __restrict__ M, int64_t N, int w,
                                                                   int64_t C, float* __restrict__ out, int vec_v,
                                                                   int vec_out) {
  constexpr int KC = W / 16, CT = kSplitCT;
  constexpr int LDP = W + 4;
  constexpr int QUADS = 64 * W / 4;
  constexpr int PER = (QUADS + kThreads - 1) / kThreads;
  __shared__ __align__(16) uint16_t vp[3][64 * LDP];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, c = lane & 15, q = lane >> 4;
  const int64_t col0 = (int64_t)blockIdx.x * (64 * CT) + 16 * CT * wv;
  SplitA ma[KC][CT];
#pragma unroll
  for (int kc = 0; kc < KC; ++kc)
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const int64_t col = col0 + 16 * j + c;
      float x[4];
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) {
        const int k = 16 * kc + 4 * q + s4;
        x[s4] = (k < w && col < C) ? M[(int64_t)k * C + col] : 0.f;
      }
      ma[kc][j] = split_a(x[0], x[1], x[2], x[3]);
    }
  const int64_t n_tiles = (N + 63) / 64;
  float4 pre[PER];
  auto fetch = [&](int64_t tile) {
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int idx = threadIdx.x + p * kThreads;
      const int row = idx / (W / 4), k = 4 * (idx % (W / 4));
      const int64_t r = tile * 64 + row;
      pre[p] = (idx < QUADS && r < N) ? load_v4(v + r * ldv + k, k, w, vec_v) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  };
  if ((int64_t)blockIdx.y < n_tiles) fetch(blockIdx.y);
  for (int64_t tile = blockIdx.y; tile < n_tiles; tile += gridDim.y) {
    __syncthreads();  // the previous tile's LDS reads are done
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int idx = threadIdx.x + p * kThreads;
      if (idx < QUADS) store_planes(vp[0], vp[1], vp[2], (idx / (W / 4)) * LDP + 4 * (idx % (W / 4)), pre[p]);
    }
    __syncthreads();
    if (tile + gridDim.y < n_tiles) fetch(tile + gridDim.y);
    const int64_t row0 = tile * 64;
    auto product = [&](auto full) {
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) {
        floatx4 acc[CT];
#pragma unroll
        for (int j = 0; j < CT; ++j) acc[j] = kZero4;
#pragma unroll
        for (int kc = 0; kc < KC; ++kc) {
          const int at = (16 * rt + c) * LDP + 16 * kc + 4 * q;
          const SplitB b = split_b_planes(*reinterpret_cast<const uint2*>(&vp[0][at]),
                                          *reinterpret_cast<const uint2*>(&vp[1][at]),
                                          *reinterpret_cast<const uint2*>(&vp[2][at]));
#pragma unroll
          for (int j = 0; j < CT; ++j) acc[j] = mfma_split(ma[kc][j], b, acc[j]);
        }
        // Lane (c, q) holds row c's columns 4q.. of both 16-column tiles.  Lanes c and c ^ 8
        // trade halves (c < 8 gives its second tile, c >= 8 its first; one DPP rotate by 8
        // within each 16-lane row), so each of the two stores writes eight whole rows of the
        // wave's 32 columns (128 contiguous bytes a row) instead of 64-byte halves of sixteen.
        const bool lo = c < 8;
        floatx4 sw;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          sw[i] = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(lo ? acc[1][i] : acc[0][i]),
                                                             kDppRowRor8, 0xF, 0xF, false));
#pragma unroll
        for (int h = 0; h < 2; ++h)
          store4<full()>(out, row0 + 16 * rt + 8 * h + (c & 7), col0 + 16 * (c >> 3) + 4 * q, N, C,
                         (h == 0) == lo ? acc[h] : sw, vec_out);
      }
    };
    if (vec_out && row0 + 64 <= N && col0 + 16 * CT <= C)
      product(std::true_type{});
    else
      product(std::false_type{});
  }
}

// Input gradient: tiles of 64 RT rows, each wave 16 RT rows over the whole
// contraction; a 64-column chunk of dmix is staged as fp32 (each wave splits
// its own rows' A operands), the chunk of M as three bf16 planes split once
// per workgroup; running totals every four chunks.
template <int W>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void node_mix_dinput_split(const float* __restrict__ dmix,
                                                                  const float* __restrict__ M, int64_t N, int w,
                                                                  int64_t C, float* __restrict__ dv, int64_t lddv) {
  constexpr int RT = kSplitRT, ROWS = 64 * RT;
  // LDM: a 16-lane 8-byte read covers 32 banks once
  constexpr int KC = 64, LDM = KC + 4, JW = W / 16, KS = KC / 16;
  // dmix rows unpadded, 16-byte unit u of row r at u ^ (r mod 16): a 16-byte read's set of
  // 16 lanes (c < 8 of one lane row, c >= 8 of another) then meets 16 distinct bank quads
  constexpr int LDD = KC;
  constexpr int TOTAL_EVERY = 256 / KC;  // chunks a running sum spans before it joins the total
  constexpr int DQ = ROWS * KC / 4 / kThreads;
  constexpr int MQ = W * KC / 4 / kThreads;
  __shared__ __align__(16) float dt[ROWS * LDD];
  __shared__ __align__(16) uint16_t mp[3][W * LDM];  // M's hi, mid and lo pieces, row k of M at k * LDM
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, c = lane & 15, q = lane >> 4;
  const int64_t row0 = (int64_t)blockIdx.x * ROWS;
  const int64_t n_chunks = (C + KC - 1) / KC;
  constexpr int CQ = KC / 4;  // 16-byte pieces of a chunk row
  float4 pd[DQ], pm[MQ];
  auto fetch = [&](int64_t ch) {
    const int64_t c0 = ch * KC;
#pragma unroll
    for (int p = 0; p < DQ; ++p) {
      const int idx = threadIdx.x + p * kThreads, row = idx / CQ, cq = idx % CQ;
      const int64_t r = row0 + row, col = c0 + 4 * cq;
      pd[p] = (r < N && col < C) ? *reinterpret_cast<const float4*>(dmix + r * C + col)
                                 : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int p = 0; p < MQ; ++p) {
      const int idx = threadIdx.x + p * kThreads, row = idx / CQ, cq = idx % CQ;
      const int64_t col = c0 + 4 * cq;
      pm[p] = (row < w && col < C) ? *reinterpret_cast<const float4*>(M + (int64_t)row * C + col)
                                   : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  };
  floatx4 acc[RT][JW], tot[RT][JW];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int j = 0; j < JW; ++j) acc[rt][j] = tot[rt][j] = kZero4;
  fetch(0);
  for (int64_t ch = 0; ch < n_chunks; ++ch) {
    __syncthreads();
#pragma unroll
    for (int p = 0; p < DQ; ++p) {
      const int idx = threadIdx.x + p * kThreads;
      const int u = (idx % CQ) ^ ((idx / CQ) & 15);
      *reinterpret_cast<float4*>(&dt[(idx / CQ) * LDD + 4 * u]) = pd[p];
    }
#pragma unroll
    for (int p = 0; p < MQ; ++p) {
      const int idx = threadIdx.x + p * kThreads;
      store_planes(mp[0], mp[1], mp[2], (idx / CQ) * LDM + 4 * (idx % CQ), pm[p]);
    }
    __syncthreads();
    if (ch + 1 < n_chunks) fetch(ch + 1);
#pragma unroll
    for (int kc = 0; kc < KS; ++kc) {
      SplitA a[RT];
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        const int u = (4 * kc + q) ^ c;
        const float4 x = *reinterpret_cast<const float4*>(&dt[(16 * RT * wv + 16 * rt + c) * LDD + 4 * u]);
        a[rt] = split_a(x.x, x.y, x.z, x.w);
      }
#pragma unroll
      for (int j = 0; j < JW; ++j) {
        const int at = (16 * j + c) * LDM + 16 * kc + 4 * q;
        const SplitB b = split_b_planes(*reinterpret_cast<const uint2*>(&mp[0][at]),
                                        *reinterpret_cast<const uint2*>(&mp[1][at]),
                                        *reinterpret_cast<const uint2*>(&mp[2][at]));
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) acc[rt][j] = mfma_split(a[rt], b, acc[rt][j]);
      }
    }
    if (ch % TOTAL_EVERY == TOTAL_EVERY - 1 || ch + 1 == n_chunks) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int j = 0; j < JW; ++j) {
          tot[rt][j] += acc[rt][j];
          acc[rt][j] = kZero4;
        }
    }
  }
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int j = 0; j < JW; ++j) {
      const int col = 16 * j + c;
      if (col >= w) continue;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int64_t r = row0 + 16 * RT * wv + 16 * rt + 4 * q + i;
        if (r < N) dv[r * lddv + col] = tot[rt][j][i];
      }
    }
}

// Weight gradient: workgroup (x, y) owns the whole (w x 16 JT)-column tile
// [16 JT x, 16 JT (x + 1)) over rows [y rps, min(N, (y + 1) rps)); its four
// waves take rows 16 wv .. 16 wv + 15 of each 64-row chunk, a wave's 16 rows
// forming one contraction chunk of split products, each wave accumulating the
// whole tile and writing one partial: 4 S partial matrices.
template <int W, typename V = float, typename DM = float>
__global__ __launch_bounds__(kThreads) void node_mix_dweight_split(const V* __restrict__ v, int64_t ldv,
                                                                   const DM* __restrict__ dmix, int64_t N, int w,
                                                                   int64_t C, int64_t rps, float* __restrict__ partial,
                                                                   int vec_v) {
  constexpr int JT = kSplitJT, COLS = 16 * JT;
  // lanes (c, q) read rows 16 wv + 4 q + s: strides with 4 LD = 16 (mod 64) words put a quarter-wave's
  // rows in distinct banks
  constexpr int RC = 64, LDV = W + 4, LDM = COLS + 4, IW = W / 16;
  constexpr int VQ = (RC * W / 4 + kThreads - 1) / kThreads;
  constexpr int CQ = COLS / 4;  // 16-byte pieces of a dmix row
  constexpr int DQ = (RC * CQ + kThreads - 1) / kThreads;
  __shared__ __align__(16) float vt[RC * LDV];
  __shared__ __align__(16) float dt[RC * LDM];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, c = lane & 15, q = lane >> 4;
  const int64_t c0 = (int64_t)blockIdx.x * COLS;
  const int64_t first = (int64_t)blockIdx.y * rps, last = first + rps < N ? first + rps : N;
  float4 pv[VQ], pd[DQ];
  auto fetch = [&](int64_t r0) {
#pragma unroll
    for (int p = 0; p < VQ; ++p) {
      const int idx = threadIdx.x + p * kThreads, row = idx / (W / 4), k = 4 * (idx % (W / 4));
      const int64_t r = r0 + row;
      pv[p] = (idx < RC * W / 4 && r < last) ? load_v4(v + r * ldv + k, k, w, vec_v) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int p = 0; p < DQ; ++p) {
      const int idx = threadIdx.x + p * kThreads, row = idx / CQ, cq = idx % CQ;
      const int64_t r = r0 + row, col = c0 + 4 * cq;
      pd[p] = (idx < RC * CQ && r < last && col < C) ? load_dm4(dmix + r * C + col) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  };
  floatx4 acc[IW][JT];
#pragma unroll
  for (int i = 0; i < IW; ++i)
#pragma unroll
    for (int j = 0; j < JT; ++j) acc[i][j] = kZero4;
  if (first < last) fetch(first);
  for (int64_t r0 = first; r0 < last; r0 += RC) {
    __syncthreads();
#pragma unroll
    for (int p = 0; p < VQ; ++p) {
      const int idx = threadIdx.x + p * kThreads;
      if (idx < RC * W / 4) *reinterpret_cast<float4*>(&vt[(idx / (W / 4)) * LDV + 4 * (idx % (W / 4))]) = pv[p];
    }
#pragma unroll
    for (int p = 0; p < DQ; ++p) {
      const int idx = threadIdx.x + p * kThreads;
      if (idx < RC * CQ) *reinterpret_cast<float4*>(&dt[(idx / CQ) * LDM + 4 * (idx % CQ)]) = pd[p];
    }
    __syncthreads();
    if (r0 + RC < last) fetch(r0 + RC);
    // rows 16 wv + 4 q + s of the chunk are contraction indices 4 q + s
    const int rb = 16 * wv + 4 * q;
    SplitA a[IW];
#pragma unroll
    for (int i = 0; i < IW; ++i)
      a[i] = split_a(vt[rb * LDV + 16 * i + c], vt[(rb + 1) * LDV + 16 * i + c], vt[(rb + 2) * LDV + 16 * i + c],
                     vt[(rb + 3) * LDV + 16 * i + c]);
#pragma unroll
    for (int j = 0; j < JT; ++j) {
      const SplitB b = split_b(dt[rb * LDM + 16 * j + c], dt[(rb + 1) * LDM + 16 * j + c],
                               dt[(rb + 2) * LDM + 16 * j + c], dt[(rb + 3) * LDM + 16 * j + c]);
#pragma unroll
      for (int i = 0; i < IW; ++i) acc[i][j] = mfma_split(a[i], b, acc[i][j]);
    }
  }
  float* out = partial + ((int64_t)blockIdx.y * 4 + wv) * w * C;
#pragma unroll
  for (int i = 0; i < IW; ++i)
#pragma unroll
    for (int j = 0; j < JT; ++j) {
      const int64_t col = c0 + 16 * j + c;
      if (col >= C) continue;
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) {
        const int row = 16 * i + 4 * q + ii;
        if (row < w) out[(int64_t)row * C + col] = acc[i][j][ii];
      }
    }
}

// ---------------------------------------------------------------- 32-deep split products
//
// The same products for vectors of 17 to 128 reals with each operand register
// holding one piece of 32 contraction indices (lane (c, q) the indices 32 kd +
// 8 q + s, s < 8): six instructions per 32 indices, three operand registers
// sets a side (hi, mid, lo) and none of them assembled from halves, so half the
// LDS reads and no register copies next to the 16-deep form.  Bfloat16 operands
// are their own hi piece (P = 1): the products with their mid and lo pieces,
// exact zeros, are left out.
//
// LDS operands are 16-byte units of eight bf16 values of one piece; a row of U
// units keeps unit u at u ^ (row mod U), so that neither the staging writes
// nor a 16-lane set of operand reads meet in a bank.
template <int P>
struct Pieces {
  u32x4 p[P];
};

template <int P>
__device__ __forceinline__ Pieces<P> pieces8(const float (&x)[8]) {
  Pieces<P> r;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (P == 1) {
      r.p[0][i] = pack_bf16(x[2 * i], x[2 * i + 1]);
    } else {
      const SplitPair sp = split_pair(x[2 * i], x[2 * i + 1]);
      r.p[0][i] = sp.hi;
      r.p[1][i] = sp.mid;
      r.p[2][i] = sp.lo;
    }
  }
  return r;
}

// acc[t] += A[t] B over 32 contraction indices for T tiles, the smallest
// products first (pieces of order i + j = 2, 1, 0), the tiles' chains side by side.
template <int T, int PA, int PB>
__device__ __forceinline__ void mfma_pieces(const Pieces<PA> (&a)[T], const Pieces<PB>& b, floatx4 (&acc)[T]) {
#pragma unroll
  for (int order = 2; order >= 0; --order)
#pragma unroll
    for (int i = 0; i <= order; ++i) {
      if (i >= PA || order - i >= PB) continue;
#pragma unroll
      for (int t = 0; t < T; ++t) acc[t] = mfma_bf16(a[t].p[i], b.p[order - i], acc[t]);
    }
}

template <int W>
constexpr int DeepCT = W == 128 ? 2 : 4;  // 16-column tiles a forward wave holds
template <int W>
constexpr int DeepJT = W == 128 ? 2 : 4;  // column tiles a weight-gradient wave owns
template <int U>
__device__ __forceinline__ int deep_unit(int row, int u) {
  return row * U + (u ^ (U >= 8 ? row & (U - 1) : (row >> 2) & (U - 1)));
}

// Eight consecutive reals k .. k + 7 (zero at and past w).
template <typename V>
__device__ __forceinline__ void load8(const V* src, int k, int w, int vec, float (&x)[8]) {
  const float4 a = load_v4(src, k, w, vec), b = load_v4(src + 4, k + 4, w, vec);
  x[0] = a.x, x[1] = a.y, x[2] = a.z, x[3] = a.w;
  x[4] = b.x, x[5] = b.y, x[6] = b.z, x[7] = b.w;
}

// Forward: wave wv of workgroup x owns columns x 64 CT + 16 CT wv + 16 j + c
// (j < CT), M's pieces at them held in registers; each 64-row tile of v is split
// once per workgroup into LDS.
template <int W, typename V = float>
__global__ __launch_bounds__(kThreads, 2) void node_mix_forward_deep(const V* __restrict__ v, int64_t ldv,
                                                                     const float* __restrict__ M, int64_t N, int w,
                                                                     int64_t C, float* __restrict__ out, int vec_v,
                                                                     int vec_out) {
  constexpr int KD = W / 32, CT = DeepCT<W>, U = W / 8, PV = sizeof(V) == 2 ? 1 : 3;
  constexpr int PER = 64 * U / kThreads;  // staged units a thread
  static_assert(PER * kThreads == 64 * U, "whole units a thread");
  __shared__ __align__(16) u32x4 vs[PV][64 * U];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, c = lane & 15, q = lane >> 4;
  const int64_t col0 = (int64_t)blockIdx.x * (64 * CT) + 16 * CT * wv;
  Pieces<3> ma[KD][CT];
#pragma unroll
  for (int kd = 0; kd < KD; ++kd)
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const int64_t col = col0 + 16 * j + c;
      float x[8];
#pragma unroll
      for (int s8 = 0; s8 < 8; ++s8) {
        const int k = 32 * kd + 8 * q + s8;
        x[s8] = (k < w && col < C) ? M[(int64_t)k * C + col] : 0.f;
      }
      ma[kd][j] = pieces8<3>(x);
    }
  const int64_t n_tiles = (N + 63) / 64;
  float pre[PER][8];
  auto fetch = [&](int64_t tile) {
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int idx = threadIdx.x + p * kThreads, row = idx / U, k = 8 * (idx % U);
      const int64_t r = tile * 64 + row;
      if (r < N) {
        load8(v + r * ldv + k, k, w, vec_v, pre[p]);
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) pre[p][i] = 0.f;
      }
    }
  };
  if ((int64_t)blockIdx.y < n_tiles) fetch(blockIdx.y);
  for (int64_t tile = blockIdx.y; tile < n_tiles; tile += gridDim.y) {
    __syncthreads();  // the previous tile's LDS reads are done
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int idx = threadIdx.x + p * kThreads;
      const Pieces<PV> x = pieces8<PV>(pre[p]);
#pragma unroll
      for (int i = 0; i < PV; ++i) vs[i][deep_unit<U>(idx / U, idx % U)] = x.p[i];
    }
    __syncthreads();
    if (tile + gridDim.y < n_tiles) fetch(tile + gridDim.y);
    auto product = [&](auto full) {
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) {
        floatx4 acc[CT];
#pragma unroll
        for (int j = 0; j < CT; ++j) acc[j] = kZero4;
#pragma unroll
        for (int kd = 0; kd < KD; ++kd) {
          Pieces<PV> b;
#pragma unroll
          for (int i = 0; i < PV; ++i) b.p[i] = vs[i][deep_unit<U>(16 * rt + c, 4 * kd + q)];
          mfma_pieces(ma[kd], b, acc);
        }
        if constexpr (W == 32) {
          // lanes c and c ^ 8 trade tile halves by one DPP rotate, so a store writes eight whole
          // 128-byte row runs instead of sixteen 64-byte halves (1.25 -> 1.07 ms; no gain for wider vectors)
          const bool lo = c < 8;
#pragma unroll
          for (int j = 0; j < CT; j += 2) {
            floatx4 sw;
#pragma unroll
            for (int i = 0; i < 4; ++i)
              sw[i] = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(lo ? acc[j + 1][i] : acc[j][i]),
                                                                 kDppRowRor8, 0xF, 0xF, false));
#pragma unroll
            for (int h = 0; h < 2; ++h)
              store4<full()>(out, tile * 64 + 16 * rt + 8 * h + (c & 7), col0 + 16 * (j + (c >> 3)) + 4 * q, N, C,
                             (h == 0) == lo ? acc[j + h] : sw, vec_out);
          }
        } else {
#pragma unroll
          for (int j = 0; j < CT; ++j)
            store4<full()>(out, tile * 64 + 16 * rt + c, col0 + 16 * j + 4 * q, N, C, acc[j], vec_out);
        }
        // a row tile's stores leave before the next one's products (2.93 -> 2.62 ms for 64 reals: interleaved,
        // the held results take 232 registers and leave in bursts)
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    if (vec_out && tile * 64 + 64 <= N && col0 + 16 * CT <= C)
      product(std::true_type{});
    else
      product(std::false_type{});
  }
}

// Input gradient: tiles of 128 rows, each wave 32 rows over the workgroup's
// chunks of the contraction (per_split of them; few rows are split over several
// workgroups, their sums added in order by node_mix_dinput_reduce); its dmix rows come straight from memory into the lanes that
// split them, M's chunk of KC columns is split once per workgroup into LDS
// (two buffers, one barrier a chunk); running totals every 256 columns.
template <int W>
__global__ __launch_bounds__(kThreads, 2) void node_mix_dinput_deep(const float* __restrict__ dmix,
                                                                    const float* __restrict__ M, int64_t N, int w,
                                                                    int64_t C, float* __restrict__ dv, int64_t lddv,
                                                                    int64_t per_split) {
  constexpr int RT = 2, KC = W == 32 ? 64 : 32, KD = KC / 32, JW = W / 16, U = KC / 8;
  constexpr int TOTAL_EVERY = 256 / KC;
  constexpr int MP = (W * U + kThreads - 1) / kThreads;  // units of M's chunk a thread stages
  __shared__ __align__(16) u32x4 ms[2][3][W * U];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, c = lane & 15, q = lane >> 4;
  const int64_t row0 = (int64_t)blockIdx.x * (64 * RT) + 16 * RT * wv;
  const int64_t all = (C + KC - 1) / KC, ch0 = (int64_t)blockIdx.y * per_split;
  const int64_t n_chunks = ch0 + per_split < all ? ch0 + per_split : all;
  dv += (int64_t)blockIdx.y * N * lddv;  // a split's partial sums (one split: the gradient itself)
  float4 pd[RT][KD][2], pm[MP][2];
  auto fetch = [&](int64_t ch) {
    const int64_t c0 = ch * KC;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const int64_t r = row0 + 16 * rt + c;
#pragma unroll
      for (int kd = 0; kd < KD; ++kd)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int64_t col = c0 + 32 * kd + 8 * q + 4 * h;
          pd[rt][kd][h] = (r < N && col < C) ? *reinterpret_cast<const float4*>(dmix + r * C + col)
                                             : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    }
#pragma unroll
    for (int p = 0; p < MP; ++p) {
      const int idx = threadIdx.x + p * kThreads, row = idx / U;  // rows past w (and past W) load zeros
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int64_t col = c0 + 8 * (idx % U) + 4 * h;
        pm[p][h] = (row < w && col < C) ? *reinterpret_cast<const float4*>(M + (int64_t)row * C + col)
                                        : make_float4(0.f, 0.f, 0.f, 0.f);
      }
    }
  };
  auto split8 = [](const float4 (&x)[2]) {
    const float y[8] = {x[0].x, x[0].y, x[0].z, x[0].w, x[1].x, x[1].y, x[1].z, x[1].w};
    return pieces8<3>(y);
  };
  floatx4 acc[JW][RT], tot[JW][RT];
#pragma unroll
  for (int j = 0; j < JW; ++j)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) acc[j][rt] = tot[j][rt] = kZero4;
  if (ch0 < n_chunks) fetch(ch0);
  for (int64_t ch = ch0; ch < n_chunks; ++ch) {
    auto& buf = ms[ch & 1];  // last read two chunks ago, before every wave's last barrier
    Pieces<3> a[KD][RT];
#pragma unroll
    for (int p = 0; p < MP; ++p) {
      const int idx = threadIdx.x + p * kThreads;
      const Pieces<3> x = split8(pm[p]);
      if (idx < W * U) {
#pragma unroll
        for (int i = 0; i < 3; ++i) buf[i][deep_unit<U>(idx / U, idx % U)] = x.p[i];
      }
    }
#pragma unroll
    for (int kd = 0; kd < KD; ++kd)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) a[kd][rt] = split8(pd[rt][kd]);
    if (ch + 1 < n_chunks) fetch(ch + 1);
    __syncthreads();
#pragma unroll
    for (int kd = 0; kd < KD; ++kd)
#pragma unroll
      for (int j = 0; j < JW; ++j) {
        Pieces<3> b;
#pragma unroll
        for (int i = 0; i < 3; ++i) b.p[i] = buf[i][deep_unit<U>(16 * j + c, 4 * kd + q)];
        mfma_pieces(a[kd], b, acc[j]);
      }
    if (ch % TOTAL_EVERY == TOTAL_EVERY - 1 || ch + 1 == n_chunks) {
#pragma unroll
      for (int j = 0; j < JW; ++j)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
          tot[j][rt] += acc[j][rt];
          acc[j][rt] = kZero4;
        }
    }
  }
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int j = 0; j < JW; ++j) {
      const int col = 16 * j + c;
      if (col >= w) continue;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int64_t r = row0 + 16 * rt + 4 * q + i;
        if (r < N) dv[r * lddv + col] = tot[j][rt][i];
      }
    }
}

// dv[r][k] = the sum of the splits' partial sums (rows of w reals), in order.
__global__ __launch_bounds__(kThreads) void node_mix_dinput_reduce(const float* __restrict__ partial, int64_t N, int w,
                                                                   int splits, float* __restrict__ dv, int64_t lddv) {
  const int64_t e = (int64_t)blockIdx.x * kThreads + threadIdx.x, n = N * w;
  if (e >= n) return;
  float s = partial[e];
  for (int y = 1; y < splits; ++y) s += partial[y * n + e];
  dv[e / w * lddv + e % w] = s;
}

// Weight gradient: workgroup (x, y) owns 64 JT columns over rows [y rps,
// min(N, (y + 1) rps)), wave wv the columns x 64 JT + 16 JT wv + JT c + j (so a
// lane's tiles are consecutive columns: one load a row, no LDS), in chunks of
// 32 rows; the chunk of v is split once per workgroup into LDS, transposed
// (a thread splits eight rows of one column: one operand unit), two buffers,
// one barrier a chunk.  One partial matrix a workgroup row.
template <int W, typename V = float, typename DM = float>
__global__ __launch_bounds__(kThreads, 2) void node_mix_dweight_deep(const V* __restrict__ v, int64_t ldv,
                                                                     const DM* __restrict__ dmix, int64_t N, int w,
                                                                     int64_t C, int64_t rps,
                                                                     float* __restrict__ partial, int vec_p) {
  constexpr int JT = DeepJT<W>, IW = W / 16, RC = 32, PV = sizeof(V) == 2 ? 1 : 3, PD = sizeof(DM) == 2 ? 1 : 3;
  constexpr int UNITS = 4 * W, VQ = (UNITS + kThreads - 1) / kThreads;
  __shared__ __align__(16) u32x4 vs[2][PV][UNITS];  // unit (octet o, column k) at o W + k
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, c = lane & 15, q = lane >> 4;
  const int64_t col = (int64_t)blockIdx.x * (64 * JT) + 16 * JT * wv + JT * c;
  const int64_t first = (int64_t)blockIdx.y * rps, last = first + rps < N ? first + rps : N;
  float pv[VQ][8], pd[8][JT];
  auto fetch = [&](int64_t r0) {
#pragma unroll
    for (int p = 0; p < VQ; ++p) {
      const int idx = threadIdx.x + p * kThreads, k = idx % W, o = idx / W;
#pragma unroll
      for (int s8 = 0; s8 < 8; ++s8) {
        const int64_t r = r0 + 8 * o + s8;
        float x = 0.f;
        if (idx < UNITS && r < last && k < w) {
          if constexpr (sizeof(V) == 2)
            x = bf16_at(v + r * ldv + k);
          else
            x = v[r * ldv + k];
        }
        pv[p][s8] = x;
      }
    }
#pragma unroll
    for (int s8 = 0; s8 < 8; ++s8) {
      const int64_t r = r0 + 8 * q + s8;
      const bool in = r < last && col < C;  // C is a multiple of 4, so a lane's columns are in or out together
      const DM* src = dmix + r * C + col;
      if constexpr (JT == 4) {
        const float4 x = in ? load_dm4(src) : make_float4(0.f, 0.f, 0.f, 0.f);
        pd[s8][0] = x.x, pd[s8][1] = x.y, pd[s8][2] = x.z, pd[s8][3] = x.w;
      } else if constexpr (sizeof(DM) == 2) {
        const uint32_t x = in ? *reinterpret_cast<const uint32_t*>(src) : 0u;
        pd[s8][0] = bf16_lo(x), pd[s8][1] = bf16_hi(x);
      } else {
        const float2 x = in ? *reinterpret_cast<const float2*>(src) : make_float2(0.f, 0.f);
        pd[s8][0] = x.x, pd[s8][1] = x.y;
      }
    }
  };
  floatx4 acc[IW][JT];
#pragma unroll
  for (int i = 0; i < IW; ++i)
#pragma unroll
    for (int j = 0; j < JT; ++j) acc[i][j] = kZero4;
  if (first < last) fetch(first);
  int cur = 0;
  for (int64_t r0 = first; r0 < last; r0 += RC, cur ^= 1) {
    auto& buf = vs[cur];  // last read two chunks ago, before every wave's last barrier
#pragma unroll
    for (int p = 0; p < VQ; ++p) {
      const int idx = threadIdx.x + p * kThreads;
      const Pieces<PV> x = pieces8<PV>(pv[p]);
      if (idx < UNITS) {
#pragma unroll
        for (int i = 0; i < PV; ++i) buf[i][idx] = x.p[i];
      }
    }
    Pieces<PD> b[JT];
#pragma unroll
    for (int j = 0; j < JT; ++j) {
      float x[8];
#pragma unroll
      for (int s8 = 0; s8 < 8; ++s8) x[s8] = pd[s8][j];
      b[j] = pieces8<PD>(x);
    }
    if (r0 + RC < last) fetch(r0 + RC);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < IW; ++i) {
      Pieces<PV> a;
#pragma unroll
      for (int p = 0; p < PV; ++p) a.p[p] = buf[p][q * W + 16 * i + c];
#pragma unroll
      for (int order = 2; order >= 0; --order)
#pragma unroll
        for (int p = 0; p <= order; ++p) {
          if (p >= PV || order - p >= PD) continue;
#pragma unroll
          for (int j = 0; j < JT; ++j) acc[i][j] = mfma_bf16(a.p[p], b[j].p[order - p], acc[i][j]);
        }
    }
  }
  if (col >= C) return;
  float* out = partial + (int64_t)blockIdx.y * w * C;
#pragma unroll
  for (int i = 0; i < IW; ++i)
#pragma unroll
    for (int ii = 0; ii < 4; ++ii) {
      const int row = 16 * i + 4 * q + ii;
      if (row >= w) continue;
      float* dst = out + (int64_t)row * C + col;
      if (vec_p && JT == 4) {
        *reinterpret_cast<float4*>(dst) = make_float4(acc[i][0][ii], acc[i][1][ii], acc[i][JT - 2][ii], acc[i][JT - 1][ii]);
      } else {
#pragma unroll
        for (int j = 0; j < JT; ++j) dst[j] = acc[i][j][ii];
      }
    }
}

// dM[e] = sum over y = 0, 1, ..., count - 1 of partial[y stride][e], in that order.
__global__ __launch_bounds__(kThreads) void node_mix_reduce_kernel(const float* __restrict__ partial, int64_t n,
                                                                   int64_t count, int64_t stride,
                                                                   float* __restrict__ dM) {
  const int64_t e = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (e >= n) return;
  float s = 0.f;
  for (int64_t y = 0; y < count; ++y) s += partial[y * stride * n + e];
  dM[e] = s;
}

// Partial sums over slices of kReduceSlice consecutive partial matrices, each
// in order and written over its slice's first matrix (the one partial no other
// thread reads at e), so a second pass adds kReduceSlice times fewer rows.
constexpr int64_t kReduceSlice = 32;

__global__ __launch_bounds__(kThreads) void node_mix_reduce_slices_kernel(float* __restrict__ partial, int64_t n,
                                                                          int64_t parts) {
  const int64_t e = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (e >= n) return;
  const int64_t y0 = (int64_t)blockIdx.y * kReduceSlice;
  const int64_t y1 = y0 + kReduceSlice < parts ? y0 + kReduceSlice : parts;
  float s = 0.f;
  for (int64_t y = y0; y < y1; ++y) s += partial[y * n + e];
  partial[y0 * n + e] = s;
}

// dM = the sum of the `parts` partial matrices of n entries in a fixed order:
// directly for a few, else by slices of kReduceSlice then over the slices.
int launch_reduce(float* partial, int64_t n, int64_t parts, float* dM, hipStream_t stream) {
  const unsigned blocks = (unsigned)((n + kThreads - 1) / kThreads);
  if (parts <= 2 * kReduceSlice) {
    hipLaunchKernelGGL(node_mix_reduce_kernel, dim3(blocks), dim3(kThreads), 0, stream, partial, n, parts, (int64_t)1,
                       dM);
    return check_launch("node_mix_backward_weight (reduce)");
  }
  const int64_t slices = (parts + kReduceSlice - 1) / kReduceSlice;
  hipLaunchKernelGGL(node_mix_reduce_slices_kernel, dim3(blocks, (unsigned)slices), dim3(kThreads), 0, stream, partial,
                     n, parts);
  const int rc = check_launch("node_mix_backward_weight (reduce slices)");
  if (rc != GM_OK) return rc;
  hipLaunchKernelGGL(node_mix_reduce_kernel, dim3(blocks), dim3(kThreads), 0, stream, partial, n, slices,
                     kReduceSlice, dM);
  return check_launch("node_mix_backward_weight (reduce)");
}

int check_shapes(int64_t N, int64_t w, int64_t C) {
  GM_REQUIRE(N >= 0 && C >= 0, "N and C must be non-negative");
  GM_REQUIRE(w >= 1 && w <= 128, "the node vector's width w must be in [1, 128]");
  return GM_OK;
}

int width_class(int64_t w) { return w <= 16 ? 16 : (w <= 32 ? 32 : (w <= 64 ? 64 : 128)); }

// Whether vectors of w reals take the split kernels (`split`) in their 32-deep
// form.  Float vectors take the split kernels unless GM_SPLIT_PRODUCTS=0;
// bfloat16 ones (and float ones with bfloat16 mix gradients) have no others.
bool deep(int64_t w, bool split) { return split && w > 16; }

// Column tile of the weight gradient's workgroups: of the 32-deep kernels; of
// the others 64 columns for vectors up to 64 reals, above 128.
int64_t weight_tile(int64_t w, bool split) {
  if (deep(w, split)) return 64 * (w <= 64 ? DeepJT<64> : DeepJT<128>);
  return w <= 64 ? 64 : 128;
}

// Partial matrices a workgroup row writes: four (one a wave) but for the
// 32-deep kernels and the fp32 kernel of vectors above 64 reals (one).
int64_t weight_partials_per_split(int64_t w, bool split) { return w <= 64 && !deep(w, split) ? 4 : 1; }

// Row groups g of a grid of nx x g workgroups whose rows each workgroup loops
// over in equal shares: about `want` workgroups in whole rounds of the
// `slots` resident ones (g = floor(r slots / nx), r = want / slots rounded,
// at least one), so that no last round runs on a fraction of the chip;
// ceil(want / nx) when the occupancy is unknown or a round holds fewer
// workgroups than there are column tiles.
int64_t round_groups(int64_t nx, int64_t want, int64_t slots) {
  if (nx < 1) nx = 1;
  if (slots < nx) return (want + nx - 1) / nx;
  int64_t r = (want + slots / 2) / slots;
  if (r < 1) r = 1;
  return (r * slots) / nx;
}

// The weight gradient's kernel for vectors of w reals (for bfloat16 vectors
// its float form's occupancy stands in).
const void* dweight_kernel(int64_t w, bool sp) {
  switch (width_class(w)) {
    case 16: return sp ? (const void*)node_mix_dweight_split<16> : (const void*)node_mix_dweight_k_kernel<16>;
    case 32: return sp ? (const void*)node_mix_dweight_deep<32> : (const void*)node_mix_dweight_k_kernel<32>;
    case 64: return sp ? (const void*)node_mix_dweight_deep<64> : (const void*)node_mix_dweight_k_kernel<64>;
    default: return sp ? (const void*)node_mix_dweight_deep<128> : (const void*)node_mix_dweight_kernel<128>;
  }
}

// Rows one accumulator of the 32-deep weight gradient sums at most (about): a
// longer chain costs accuracy (the error of a sequential float sum grows with
// its length), a shorter one partial matrices.  4,096 rows: 2.1e-6 relative
// (2-norm) over 524,288 rows against 3.7e-6 for the 16-deep form's 10,900.
constexpr int64_t kMaxChainRows = 4096;

// The weight gradient's row splits: about 1024 workgroups in whole rounds, whole 64-row chunks per split.
void weight_splits(int64_t N, int64_t w, int64_t C, bool split, int64_t max_splits, int64_t& splits, int64_t& rps) {
  const int64_t tile = weight_tile(w, split);
  const int64_t nx = (C + tile - 1) / tile > 0 ? (C + tile - 1) / tile : 1;
  const int64_t chunks = (N + 63) / 64;
  int64_t want = 1024;
  if (deep(w, split)) want = std::max(want, nx * ((N + kMaxChainRows - 1) / kMaxChainRows));
  int64_t s = round_groups(nx, want, resident_blocks(dweight_kernel(w, split), kThreads));
  if (s > chunks) s = chunks;
  if (s > max_splits) s = max_splits;
  if (s < 1) s = 1;
  rps = ((chunks + s - 1) / s) * 64;
  splits = rps > 0 ? (N + rps - 1) / rps : 1;
  if (splits < 1) splits = 1;
}

const void* dinput_kernel(int64_t w) {
  switch (width_class(w)) {
    case 32: return (const void*)node_mix_dinput_deep<32>;
    case 64: return (const void*)node_mix_dinput_deep<64>;
    default: return (const void*)node_mix_dinput_deep<128>;
  }
}

// Splits of the input gradient's contraction: a workgroup walks its chunks one
// after the other, so a launch takes about (rounds of resident workgroups) x
// (chunks a split + kSplitCost): the splits that make this least.  16 row tiles
// (2,048 rows, w = 64, C = 5,440): 191 us whole, 38 us in 16 splits; from four
// rounds of row tiles up the tail is small and the contraction stays whole.
constexpr int64_t kMaxInputSplits = 16, kSplitCost = 6;

void input_splits(int64_t N, int64_t w, int64_t C, int64_t& splits, int64_t& per_split) {
  const int64_t kc = width_class(w) == 32 ? 64 : 32, chunks = (C + kc - 1) / kc, blocks = (N + 127) / 128;
  const int64_t slots = resident_blocks(dinput_kernel(w), kThreads);
  splits = 1;
  if (slots > 0 && blocks < 4 * slots) {
    int64_t best = 0;
    for (int64_t s = 1; s <= kMaxInputSplits && 4 * s <= chunks; ++s) {
      const int64_t cost = (blocks * s + slots - 1) / slots * ((chunks + s - 1) / s + (s > 1 ? kSplitCost : 0));
      if (best == 0 || cost < best) best = cost, splits = s;
    }
  }
  per_split = chunks > 0 ? (chunks + splits - 1) / splits : 1;
  if (chunks > 0) splits = (chunks + per_split - 1) / per_split;
}

int launch_dinput(const float* dmix, const float* M, int64_t N, int64_t w, int64_t C, int64_t splits,
                  int64_t per_split, float* partial, float* dv, int64_t lddv, hipStream_t s) {
  const dim3 grid((unsigned)((N + 127) / 128), (unsigned)splits), block(kThreads);
  float* to = splits > 1 ? partial : dv;
  const int64_t ld = splits > 1 ? w : lddv;
  switch (width_class(w)) {
    case 32: hipLaunchKernelGGL(node_mix_dinput_deep<32>, grid, block, 0, s, dmix, M, N, (int)w, C, to, ld, per_split); break;
    case 64: hipLaunchKernelGGL(node_mix_dinput_deep<64>, grid, block, 0, s, dmix, M, N, (int)w, C, to, ld, per_split); break;
    default: hipLaunchKernelGGL(node_mix_dinput_deep<128>, grid, block, 0, s, dmix, M, N, (int)w, C, to, ld, per_split); break;
  }
  const int rc = check_launch("node_mix_backward_input");
  if (rc != GM_OK || splits == 1) return rc;
  hipLaunchKernelGGL(node_mix_dinput_reduce, dim3((unsigned)((N * w + kThreads - 1) / kThreads)), block, 0, s, partial,
                     N, (int)w, (int)splits, dv, lddv);
  return check_launch("node_mix_backward_input (reduce)");
}

int launch_dweight(const float* v, int64_t ldv, const float* dmix, int64_t N, int64_t w, int64_t C, int64_t splits,
                   int64_t rps, float* partial, float* dM, hipStream_t stream) {
  const bool sp = split_products();
  const int64_t tile = weight_tile(w, sp), nx = (C + tile - 1) / tile;
  if (N > 0 && nx > 0) {
    const dim3 grid((unsigned)nx, (unsigned)splits), block(kThreads);
    const int vec = aligned(v, 16) && ldv % 4 == 0, vec_p = aligned(partial, 16);
    switch (width_class(w)) {
      case 16:
        if (sp) hipLaunchKernelGGL(node_mix_dweight_split<16>, grid, block, 0, stream, v, ldv, dmix, N, (int)w, C, rps, partial, vec);
        else hipLaunchKernelGGL(node_mix_dweight_k_kernel<16>, grid, block, 0, stream, v, ldv, dmix, N, (int)w, C, rps, partial, vec);
        break;
      case 32:
        if (sp) hipLaunchKernelGGL(node_mix_dweight_deep<32>, grid, block, 0, stream, v, ldv, dmix, N, (int)w, C, rps, partial, vec_p);
        else hipLaunchKernelGGL(node_mix_dweight_k_kernel<32>, grid, block, 0, stream, v, ldv, dmix, N, (int)w, C, rps, partial, vec);
        break;
      case 64:
        if (sp) hipLaunchKernelGGL(node_mix_dweight_deep<64>, grid, block, 0, stream, v, ldv, dmix, N, (int)w, C, rps, partial, vec_p);
        else hipLaunchKernelGGL(node_mix_dweight_k_kernel<64>, grid, block, 0, stream, v, ldv, dmix, N, (int)w, C, rps, partial, vec);
        break;
      default:
        if (sp) hipLaunchKernelGGL(node_mix_dweight_deep<128>, grid, block, 0, stream, v, ldv, dmix, N, (int)w, C, rps, partial, vec_p);
        else hipLaunchKernelGGL(node_mix_dweight_kernel<128>, grid, block, 0, stream, v, ldv, dmix, N, (int)w, C, rps, partial, vec);
        break;
    }
    const int rc = check_launch("node_mix_backward_weight");
    if (rc != GM_OK) return rc;
  }
  const int64_t n = w * C;
  if (n > 0) {
    const int64_t parts = (N > 0 && C > 0) ? splits * weight_partials_per_split(w, sp) : (int64_t)0;
    return launch_reduce(partial, n, parts, dM, stream);
  }
  return GM_OK;
}

constexpr int64_t kScratchFloats = int64_t(1) << 23;
constexpr int kMaxDevices = 64;

// Each device's address of `scratch`, looked up once with that device current,
// and an event per device that orders the calls sharing that device's array:
// each call's stream waits for the previous call's kernels (on whatever stream
// they ran) before it writes the partials, and the call records the event
// after its reduction.  The mutex is held from the wait to the record, so calls
// from several host threads or streams serialise on the GPU instead of racing.
std::mutex scratch_mutex;
float* scratch_address[kMaxDevices] = {};
hipEvent_t scratch_done[kMaxDevices] = {};

int scratch_on_current_device(int* device_out, float** out) {
  int device = -1;
  hipError_t err = hipGetDevice(&device);
  if (err != hipSuccess) return fail(GM_ERR_LAUNCH, std::string("hipGetDevice: ") + hipGetErrorString(err));
  GM_REQUIRE(device >= 0 && device < kMaxDevices, "the current device index is out of the scratch table's range");
  if (scratch_address[device] == nullptr) {
    void* address = nullptr;
    err = hipGetSymbolAddress(&address, HIP_SYMBOL(scratch));
    if (err != hipSuccess || address == nullptr)
      return fail(GM_ERR_LAUNCH, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(err));
    hipEvent_t done = nullptr;
    err = hipEventCreateWithFlags(&done, hipEventDisableTiming);
    if (err != hipSuccess)
      return fail(GM_ERR_LAUNCH, std::string("hipEventCreateWithFlags(scratch): ") + hipGetErrorString(err));
    scratch_done[device] = done;
    scratch_address[device] = static_cast<float*>(address);
  }
  *device_out = device;
  *out = scratch_address[device];
  return GM_OK;
}

}  // namespace
}  // namespace gm

extern "C" int gm_node_mix_forward_f32(const float* v, int64_t ldv, const float* M, int64_t N, int64_t w, int64_t C,
                                       float* out, void* stream) {
  int rc = gm::check_shapes(N, w, C);
  if (rc != GM_OK) return rc;
  if (N == 0 || C == 0) return GM_OK;
  GM_REQUIRE(v && M && out, "v, M and out must be device pointers");
  GM_REQUIRE(ldv >= w, "ldv must be at least w");
  const hipStream_t s = (hipStream_t)stream;
  const int vec_v = gm::aligned(v, 16) && ldv % 4 == 0;
  const int vec_out = gm::aligned(out, 16) && C % 4 == 0;
  const int W = gm::width_class(w);
  const bool sp = gm::split_products();
  const int CT = sp ? (W == 16 ? gm::kSplitCT : (W == 128 ? gm::DeepCT<128> : gm::DeepCT<64>)) : (W == 128 ? 2 : 4);
  const int64_t nx = (C + 64 * CT - 1) / (64 * CT), n_tiles = (N + 63) / 64;
  const void* kernel = nullptr;
  switch (W) {
    case 16: kernel = sp ? (const void*)gm::node_mix_forward_split<16> : (const void*)gm::node_mix_forward_kernel<16, 4>; break;
    case 32: kernel = sp ? (const void*)gm::node_mix_forward_deep<32> : (const void*)gm::node_mix_forward_kernel<32, 4>; break;
    case 64: kernel = sp ? (const void*)gm::node_mix_forward_deep<64> : (const void*)gm::node_mix_forward_kernel<64, 4>; break;
    default: kernel = sp ? (const void*)gm::node_mix_forward_deep<128> : (const void*)gm::node_mix_forward_kernel<128, 2>; break;
  }
  int64_t ny = gm::round_groups(nx, 2048, gm::resident_blocks(kernel, gm::kThreads));
  if (ny > n_tiles) ny = n_tiles;
  if (ny > 65535) ny = 65535;
  const dim3 grid((unsigned)nx, (unsigned)ny), block(gm::kThreads);
  if (sp) {
    switch (W) {
      case 16: hipLaunchKernelGGL((gm::node_mix_forward_split<16>), grid, block, 0, s, v, ldv, M, N, (int)w, C, out, vec_v, vec_out); break;
      case 32: hipLaunchKernelGGL((gm::node_mix_forward_deep<32>), grid, block, 0, s, v, ldv, M, N, (int)w, C, out, vec_v, vec_out); break;
      case 64: hipLaunchKernelGGL((gm::node_mix_forward_deep<64>), grid, block, 0, s, v, ldv, M, N, (int)w, C, out, vec_v, vec_out); break;
      default: hipLaunchKernelGGL((gm::node_mix_forward_deep<128>), grid, block, 0, s, v, ldv, M, N, (int)w, C, out, vec_v, vec_out); break;
    }
    return gm::check_launch("node_mix_forward");
  }
  switch (W) {
    case 16: hipLaunchKernelGGL((gm::node_mix_forward_kernel<16, 4>), grid, block, 0, s, v, ldv, M, N, (int)w, C, out, vec_v, vec_out); break;
    case 32: hipLaunchKernelGGL((gm::node_mix_forward_kernel<32, 4>), grid, block, 0, s, v, ldv, M, N, (int)w, C, out, vec_v, vec_out); break;
    case 64: hipLaunchKernelGGL((gm::node_mix_forward_kernel<64, 4>), grid, block, 0, s, v, ldv, M, N, (int)w, C, out, vec_v, vec_out); break;
    default: hipLaunchKernelGGL((gm::node_mix_forward_kernel<128, 2>), grid, block, 0, s, v, ldv, M, N, (int)w, C, out, vec_v, vec_out); break;
  }
  return gm::check_launch("node_mix_forward");
}

namespace gm {
namespace {

int backward_input(const float* dmix, const float* M, int64_t N, int64_t w, int64_t C, float* partial, float* dv,
                   int64_t lddv, hipStream_t s) {
  const int rc = check_shapes(N, w, C);
  if (rc != GM_OK) return rc;
  if (N == 0) return GM_OK;
  GM_REQUIRE(dv && lddv >= w, "dv must be a device pointer with lddv >= w");
  GM_REQUIRE(C == 0 || (dmix && M), "dmix and M must be device pointers");
  GM_REQUIRE(C % 4 == 0 && aligned(dmix, 16) && aligned(M, 16),
             "dmix and M must be 16-byte aligned with C a multiple of 4");
  if (deep(w, split_products())) {
    int64_t splits = 1, per_split = 0;
    if (partial != nullptr) {
      input_splits(N, w, C, splits, per_split);
    } else {
      per_split = C;  // chunks are of 32 columns or more: every chunk
    }
    return launch_dinput(dmix, M, N, w, C, splits, per_split, partial, dv, lddv, s);
  }
  const dim3 grid((unsigned)((N + 127) / 128)), block(kThreads);
  if (split_products()) {
    hipLaunchKernelGGL(node_mix_dinput_split<16>, grid, block, 0, s, dmix, M, N, (int)w, C, dv, lddv);
    return check_launch("node_mix_backward_input");
  }
  switch (width_class(w)) {
    case 16: hipLaunchKernelGGL(node_mix_dinput_kernel<16>, grid, block, 0, s, dmix, M, N, (int)w, C, dv, lddv); break;
    case 32: hipLaunchKernelGGL(node_mix_dinput_kernel<32>, grid, block, 0, s, dmix, M, N, (int)w, C, dv, lddv); break;
    case 64: hipLaunchKernelGGL(node_mix_dinput_kernel<64>, grid, block, 0, s, dmix, M, N, (int)w, C, dv, lddv); break;
    default: hipLaunchKernelGGL(node_mix_dinput_kernel<128>, grid, block, 0, s, dmix, M, N, (int)w, C, dv, lddv); break;
  }
  return check_launch("node_mix_backward_input");
}

}  // namespace
}  // namespace gm

extern "C" int gm_node_mix_backward_input_f32(const float* dmix, const float* M, int64_t N, int64_t w, int64_t C,
                                              float* dv, int64_t lddv, void* stream) {
  return gm::backward_input(dmix, M, N, w, C, nullptr, dv, lddv, (hipStream_t)stream);
}

extern "C" int64_t gm_node_mix_input_partials(int64_t N, int64_t w, int64_t C) {
  if (N <= 0 || w < 1 || w > 128 || C <= 0 || !gm::deep(w, gm::split_products())) return 0;
  int64_t splits = 1, per_split = 0;
  gm::input_splits(N, w, C, splits, per_split);
  return splits > 1 ? splits * N * w : 0;
}

extern "C" int gm_node_mix_backward_input_split_f32(const float* dmix, const float* M, int64_t N, int64_t w, int64_t C,
                                                    float* partial, float* dv, int64_t lddv, void* stream) {
  return gm::backward_input(dmix, M, N, w, C, partial, dv, lddv, (hipStream_t)stream);
}

extern "C" int64_t gm_node_mix_weight_partials(int64_t N, int64_t w, int64_t C) {
  // one workspace for float and bfloat16 vectors: the larger of what their kernels write
  int64_t most = 0;
  for (const bool split : {gm::split_products(), true}) {
    int64_t splits = 1, rps = 64;
    gm::weight_splits(N, w, C, split, 1 << 20, splits, rps);
    most = std::max(most, splits * gm::weight_partials_per_split(w, split) * w * C);
  }
  return most;
}

extern "C" int gm_node_mix_backward_weight_f32(const float* v, int64_t ldv, const float* dmix, int64_t N, int64_t w,
                                               int64_t C, float* partial, float* dM, void* stream) {
  int rc = gm::check_shapes(N, w, C);
  if (rc != GM_OK) return rc;
  if (w * C == 0) return GM_OK;
  GM_REQUIRE(dM && partial, "partial and dM must be device pointers");
  GM_REQUIRE(N == 0 || (v && dmix && ldv >= w), "v (ldv >= w) and dmix must be device pointers");
  GM_REQUIRE(C % 4 == 0 && (N == 0 || gm::aligned(dmix, 16)), "dmix must be 16-byte aligned with C a multiple of 4");
  int64_t splits = 1, rps = 64;
  gm::weight_splits(N, w, C, gm::split_products(), 1 << 20, splits, rps);
  return gm::launch_dweight(v, ldv, dmix, N, w, C, splits, rps, partial, dM, (hipStream_t)stream);
}

extern "C" int gm_node_mix_backward_weight_noalloc_f32(const float* v, int64_t ldv, const float* dmix, int64_t N,
                                                       int64_t w, int64_t C, float* dM, void* stream) {
  int rc = gm::check_shapes(N, w, C);
  if (rc != GM_OK) return rc;
  if (w * C == 0) return GM_OK;
  GM_REQUIRE(dM, "dM must be a device pointer");
  GM_REQUIRE(N == 0 || (v && dmix && ldv >= w), "v (ldv >= w) and dmix must be device pointers");
  GM_REQUIRE(C % 4 == 0 && (N == 0 || gm::aligned(dmix, 16)), "dmix must be 16-byte aligned with C a multiple of 4");
  const int64_t per_split = gm::weight_partials_per_split(w, gm::split_products()) * w * C;
  const int64_t needed = (w <= 64 || gm::split_products() ? 4 : 1) * w * C;
  GM_REQUIRE(needed <= gm::kScratchFloats,
             "w * C is too large for the no-allocation weight gradient: its partials need " +
                 std::to_string(needed) + " floats a row split, the scratch holds " +
                 std::to_string(gm::kScratchFloats));
  const hipStream_t s = (hipStream_t)stream;
  std::lock_guard<std::mutex> lock(gm::scratch_mutex);
  float* partial = nullptr;
  int device = -1;
  rc = gm::scratch_on_current_device(&device, &partial);
  if (rc != GM_OK) return rc;
  // Under stream capture the ordering is the graph's (an event recorded outside
  // a capture cannot be waited on inside it): replays of the graph and other
  // calls on that GPU must not overlap.
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  hipError_t err = hipStreamIsCapturing(s, &capture);
  if (err != hipSuccess) return gm::fail(GM_ERR_LAUNCH, std::string("hipStreamIsCapturing: ") + hipGetErrorString(err));
  const bool ordered = capture == hipStreamCaptureStatusNone;
  if (ordered) {
    err = hipStreamWaitEvent(s, gm::scratch_done[device], 0);
    if (err != hipSuccess) return gm::fail(GM_ERR_LAUNCH, std::string("hipStreamWaitEvent: ") + hipGetErrorString(err));
  }
  // as many row splits as the scratch holds (every partial is written in full: nothing to clear)
  int64_t splits = 1, rps = 64;
  gm::weight_splits(N, w, C, gm::split_products(), gm::kScratchFloats / per_split, splits, rps);
  rc = gm::launch_dweight(v, ldv, dmix, N, w, C, splits, rps, partial, dM, s);
  if (rc != GM_OK || !ordered) return rc;
  err = hipEventRecord(gm::scratch_done[device], s);
  if (err != hipSuccess) return gm::fail(GM_ERR_LAUNCH, std::string("hipEventRecord: ") + hipGetErrorString(err));
  return GM_OK;
}

// bfloat16 node vectors (the rows of a bfloat16 field): the split kernels widen
// them exactly while staging, so the products and outputs are the float32
// entry points' on the widened values.  Vectors up to 64 reals.
extern "C" int gm_node_mix_forward_bf16(const uint16_t* v, int64_t ldv, const float* M, int64_t N, int64_t w,
                                        int64_t C, float* out, void* stream) {
  int rc = gm::check_shapes(N, w, C);
  if (rc != GM_OK) return rc;
  GM_REQUIRE(w <= 64, "bfloat16 node vectors at most 64 reals wide");
  if (N == 0 || C == 0) return GM_OK;
  GM_REQUIRE(v && M && out, "v, M and out must be device pointers");
  GM_REQUIRE(ldv >= w, "ldv must be at least w");
  const hipStream_t s = (hipStream_t)stream;
  const int vec_v = gm::aligned(v, 8) && ldv % 4 == 0;
  const int vec_out = gm::aligned(out, 16) && C % 4 == 0;
  const int W = gm::width_class(w);
  const int CT = W == 16 ? gm::kSplitCT : gm::DeepCT<64>;
  const int64_t nx = (C + 64 * CT - 1) / (64 * CT), n_tiles = (N + 63) / 64;
  const void* kernel = W == 16 ? (const void*)gm::node_mix_forward_split<16, uint16_t>
                       : W == 32 ? (const void*)gm::node_mix_forward_deep<32, uint16_t>
                                 : (const void*)gm::node_mix_forward_deep<64, uint16_t>;
  int64_t ny = gm::round_groups(nx, 2048, gm::resident_blocks(kernel, gm::kThreads));
  if (ny > n_tiles) ny = n_tiles;
  if (ny > 65535) ny = 65535;
  const dim3 grid((unsigned)nx, (unsigned)ny), block(gm::kThreads);
  switch (W) {
    case 16: hipLaunchKernelGGL((gm::node_mix_forward_split<16, uint16_t>), grid, block, 0, s, v, ldv, M, N, (int)w, C, out, vec_v, vec_out); break;
    case 32: hipLaunchKernelGGL((gm::node_mix_forward_deep<32, uint16_t>), grid, block, 0, s, v, ldv, M, N, (int)w, C, out, vec_v, vec_out); break;
    default: hipLaunchKernelGGL((gm::node_mix_forward_deep<64, uint16_t>), grid, block, 0, s, v, ldv, M, N, (int)w, C, out, vec_v, vec_out); break;
  }
  return gm::check_launch("node_mix_forward (bfloat16 vectors)");
}

namespace gm {
namespace {

// The split weight gradient for node vectors of type V and mix gradients of
// type DM (bfloat16 widened exactly while staged): partials, then the
// fixed-order reduction.
template <typename V, typename DM>
int split_dweight(const V* v, int64_t ldv, const DM* dmix, int64_t N, int64_t w, int64_t C, float* partial, float* dM,
                  hipStream_t s) {
  int64_t splits = 1, rps = 64;
  weight_splits(N, w, C, true, 1 << 20, splits, rps);
  const int64_t tile = weight_tile(w, true), nx = (C + tile - 1) / tile;
  if (N > 0 && nx > 0) {
    const dim3 grid((unsigned)nx, (unsigned)splits), block(kThreads);
    const int vec = aligned(v, sizeof(V) == 2 ? 8 : 16) && ldv % 4 == 0, vec_p = aligned(partial, 16);
    switch (width_class(w)) {
      case 16: hipLaunchKernelGGL((node_mix_dweight_split<16, V, DM>), grid, block, 0, s, v, ldv, dmix, N, (int)w, C, rps, partial, vec); break;
      case 32: hipLaunchKernelGGL((node_mix_dweight_deep<32, V, DM>), grid, block, 0, s, v, ldv, dmix, N, (int)w, C, rps, partial, vec_p); break;
      case 64: hipLaunchKernelGGL((node_mix_dweight_deep<64, V, DM>), grid, block, 0, s, v, ldv, dmix, N, (int)w, C, rps, partial, vec_p); break;
      default:
        if constexpr (sizeof(V) == 4)
          hipLaunchKernelGGL((node_mix_dweight_deep<128, V, DM>), grid, block, 0, s, v, ldv, dmix, N, (int)w, C, rps, partial, vec_p);
        break;
    }
    const int rc = check_launch("node_mix_backward_weight");
    if (rc != GM_OK) return rc;
  }
  const int64_t parts = (N > 0 && C > 0) ? splits * weight_partials_per_split(w, true) : (int64_t)0;
  return launch_reduce(partial, w * C, parts, dM, s);
}

}  // namespace
}  // namespace gm

extern "C" int gm_node_mix_backward_weight_bf16(const uint16_t* v, int64_t ldv, const float* dmix, int64_t N,
                                                int64_t w, int64_t C, float* partial, float* dM, void* stream) {
  int rc = gm::check_shapes(N, w, C);
  if (rc != GM_OK) return rc;
  GM_REQUIRE(w <= 64, "bfloat16 node vectors at most 64 reals wide");
  if (w * C == 0) return GM_OK;
  GM_REQUIRE(dM && partial, "partial and dM must be device pointers");
  GM_REQUIRE(N == 0 || (v && dmix && ldv >= w), "v (ldv >= w) and dmix must be device pointers");
  GM_REQUIRE(C % 4 == 0 && (N == 0 || gm::aligned(dmix, 16)), "dmix must be 16-byte aligned with C a multiple of 4");
  return gm::split_dweight(v, ldv, dmix, N, w, C, partial, dM, (hipStream_t)stream);
}

extern "C" int gm_node_mix_backward_weight_bf16_bf16(const uint16_t* v, int64_t ldv, const uint16_t* dmix, int64_t N,
                                                     int64_t w, int64_t C, float* partial, float* dM, void* stream) {
  int rc = gm::check_shapes(N, w, C);
  if (rc != GM_OK) return rc;
  GM_REQUIRE(w <= 64, "bfloat16 node vectors at most 64 reals wide");
  GM_REQUIRE(gm::split_products(), "bfloat16 mix gradients need the split products (GM_SPLIT_PRODUCTS unset or 1)");
  if (w * C == 0) return GM_OK;
  GM_REQUIRE(dM && partial, "partial and dM must be device pointers");
  GM_REQUIRE(N == 0 || (v && dmix && ldv >= w), "v (ldv >= w) and dmix must be device pointers");
  GM_REQUIRE(C % 4 == 0 && (N == 0 || gm::aligned(dmix, 8)), "dmix must be 8-byte aligned with C a multiple of 4");
  return gm::split_dweight(v, ldv, dmix, N, w, C, partial, dM, (hipStream_t)stream);
}

extern "C" int gm_node_mix_backward_weight_f32_bf16(const float* v, int64_t ldv, const uint16_t* dmix, int64_t N,
                                                    int64_t w, int64_t C, float* partial, float* dM, void* stream) {
  int rc = gm::check_shapes(N, w, C);
  if (rc != GM_OK) return rc;
  GM_REQUIRE(gm::split_products(), "bfloat16 mix gradients need the split products (GM_SPLIT_PRODUCTS unset or 1)");
  if (w * C == 0) return GM_OK;
  GM_REQUIRE(dM && partial, "partial and dM must be device pointers");
  GM_REQUIRE(N == 0 || (v && dmix && ldv >= w), "v (ldv >= w) and dmix must be device pointers");
  GM_REQUIRE(C % 4 == 0 && (N == 0 || gm::aligned(dmix, 8)), "dmix must be 8-byte aligned with C a multiple of 4");
  return gm::split_dweight(v, ldv, dmix, N, w, C, partial, dM, (hipStream_t)stream);
}
