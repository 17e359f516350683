// Calibrated W4 quantization: GPTQ (Frantar et al., "GPTQ: Accurate Post-Training Quantization
// for Generative Pre-trained Transformers", 2022, Algorithm 1, one scale per row and 128-column
// group, columns in their natural order) writing the reference's on-disk format (Wq [N][K/8]
// uint32 low nibble first, S [N][K/128] bf16, w = (q - 8) * s), so that ns_w4_linear and every
// other consumer of the format reads its output unchanged. The reference quantizes by round to
// nearest only (kernels/quant/w4a16.cuh:272-297) and names calibrated methods as its next step
// (README.md:233-235).
//
// Arithmetic, fixed so that a sequential CPU restatement reproduces it bit for bit:
//  * column i of a row is quantized as the round-to-nearest quantizer does (q = clamp(
//    rint_half_even(w / s) + 8, 0, 15)), with the group's scale s = bf16_rne(max|w| / 7) (1 for
//    an all-zero group) taken from the row's group values as they stand when the group starts;
//  * its error e = (w - (q - 8) s) / U[i][i] (the product is exact: |q - 8| <= 8 and s has an
//    8-bit significand) goes onto every later column j of the row as w_j <- fma(-e, U[i][j], w_j),
//    U the upper Cholesky factor of the damped inverse Hessian, computed by the caller;
//  * so every w_j receives its updates from i = 0, 1, ..., j - 1 in that order, one fused
//    multiply-add each, whichever of the two kernels below applies them.
//
// One launch per 128-column group g, holding two kinds of workgroups (rows are independent; a
// group needs the errors E of the group before it):
//  * panel workgroups bring the group's own 128 columns up to date with the errors of group
//    g - 1, quantize them column after column and write codes, scales and the errors of group g;
//  * trailing workgroups apply the errors of group g - 1 to every column after group g. They fill
//    the chip while the panel, a serial chain per row, would leave it idle.
// E lives where it is no longer needed: error i of row n replaces W[n][k0 + i].
//
// Both rank-128 updates run on the fp32 matrix cores. v_mfma_f32_32x32x2_f32 and
// v_mfma_f32_16x16x4_f32 add their products to the accumulator one fused multiply-add after
// another in ascending k (checked bit for bit against the scalar chain, subnormal results
// included), so a sequence of them in ascending i is exactly the order above, at twice the rate
// of the vector unit.
#include <stdint.h>

#include "../../include/nanoserve_w4.h"
#include "w4_common.h"

namespace ns {
namespace {

constexpr int kGq = 128;         // group size: columns per launch
constexpr int kPanelRows = 16;   // rows per panel workgroup, 16 lanes each
constexpr int kPanelBlocks = kGq / 16;
constexpr int kPanelStride = kGq + 4;  // LDS row stride of the panel's 16 x 128 tile
constexpr int kUpTile = 128;     // trailing update: rows and columns per workgroup tile
constexpr int kUpK = 32;         // trailing update: error columns staged per LDS pass
constexpr int kEsStride = kUpK + 1;     // LDS row strides that keep the fragment reads on
constexpr int kUsStride = kUpTile + 32; // distinct banks

// LDS floats before row i = 16 b + s of the panel's triangle of U: rows of block b hold the
// 16-column blocks b .. 7.
constexpr int tri_row(int b) { return 256 * (kPanelBlocks * b - b * (b - 1) / 2); }
constexpr int kTriFloats = tri_row(kPanelBlocks);

struct GptqArgs {
  float* W;
  const float* U;
  uint32_t* Wq;
  uint16_t* S;
  int N, K, k0;
  int panels;  // panel workgroups (the first of the grid)
  int up_rows; // row tiles of the trailing update
};

template <int CTRL>
__device__ __forceinline__ int dpp_i(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, false);
}
template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
  return __builtin_bit_cast(float, dpp_i<CTRL>(__builtin_bit_cast(int, v)));
}

// One column of the serial chain: lane S of each 16-lane row owns column 16 b + S. w[r] is column
// 16 (b + r) + lane; u the same columns of U's row. The owner's w[0] becomes its error.
template <int S>
__device__ __forceinline__ void gptq_column(float (&w)[kPanelBlocks], const float* u_row, int width,
                                            int l16, float sf, int& code) {
  float u[kPanelBlocks];
#pragma unroll
  for (int r = 0; r < kPanelBlocks; ++r) u[r] = u_row[S * width + 16 * r];
  const float c = w[0];
  int q = (int)((uint32_t)f2i_rn(c / sf) + 8u);
  q = q < 0 ? 0 : (q > 15 ? 15 : q);
  const float e = fmaf(-static_cast<float>(q - 8), sf, c) / u[0];
  const float eb = dpp_f<0x150 + S>(e);  // row_newbcast: lane S of the row
#pragma unroll
  for (int r = 1; r < kPanelBlocks; ++r) w[r] = fmaf(-eb, u[r], w[r]);
  const float w0 = fmaf(-eb, u[0], c);
  w[0] = l16 > S ? w0 : (l16 == S ? e : c);
  code = l16 == S ? q : code;
}

// Bound by the latency of the per-column chain (two divisions, the rounding, a lane broadcast and
// one fma). Sixteen lanes per row hold eight columns each, so the other updates of a column are
// eight independent fmas off that chain.
__device__ __forceinline__ void gptq_panel(const GptqArgs& a, float* lds) {
  float* tri = lds;                                   // [kTriFloats] + one row of slack
  float* tile = lds + kTriFloats + kGq;               // [16][kPanelStride]
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, lq = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const long long n0 = (long long)blockIdx.x * kPanelRows;
  const int K = a.K, k0 = a.k0;

  // this wave's 32 columns of U[k0 - 128 ..][k0 ..] (B fragments) and of W (accumulators)
  f32x4_t acc[2];
  float bu[2][kGq / 4];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int col = k0 + 32 * wv + 16 * j + l16;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const long long n = n0 + 4 * lq + r;
      acc[j][r] = n < a.N ? a.W[n * K + col] : 0.f;
    }
    if (k0) {
#pragma unroll
      for (int s = 0; s < kGq / 4; ++s) bu[j][s] = a.U[(size_t)(k0 - kGq + 4 * s + lq) * K + col];
    }
  }
  if (k0) {  // the errors of the group before
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int v = tid + 256 * p, r = v >> 5, c = 4 * (v & 31);
      f32x4_t ev = {0.f, 0.f, 0.f, 0.f};
      if (n0 + r < a.N) ev = *reinterpret_cast<const f32x4_t*>(a.W + (n0 + r) * K + k0 - kGq + c);
      *reinterpret_cast<f32x4_t*>(&tile[r * kPanelStride + c]) = ev;
    }
  }
  // the triangle: 16-column blocks b .. 7 of rows 16 b ..
  for (int v = tid; v < kGq * kGq / 4; v += 256) {
    const int i = v >> 5, c = 4 * (v & 31), b = i >> 4;
    if (c < 16 * b) continue;
    const f32x4_t uv = *reinterpret_cast<const f32x4_t*>(a.U + (size_t)(k0 + i) * K + k0 + c);
    *reinterpret_cast<f32x4_t*>(&tri[tri_row(b) + (i & 15) * 16 * (kPanelBlocks - b) + c - 16 * b]) = uv;
  }
  __syncthreads();
  if (k0) {
#pragma unroll
    for (int s = 0; s < kGq / 4; ++s) {
      const float ea = -tile[l16 * kPanelStride + 4 * s + lq];
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ea, bu[j][s], acc[j], 0, 0, 0);
    }
    __syncthreads();  // every wave has read the errors
  }
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) tile[(4 * lq + r) * kPanelStride + 32 * wv + 16 * j + l16] = acc[j][r];
  __syncthreads();

  const int lr = 4 * wv + lq;  // this lane's row, 16 lanes per row
  const long long row = n0 + lr;
  float w[kPanelBlocks];
#pragma unroll
  for (int r = 0; r < kPanelBlocks; ++r) w[r] = tile[lr * kPanelStride + 16 * r + l16];
  float mx = 0.f;
#pragma unroll
  for (int r = 0; r < kPanelBlocks; ++r) mx = fmaxf(mx, fabsf(w[r]));
  mx = fmaxf(mx, dpp_f<0xB1>(mx));   // quad_perm [1,0,3,2], [2,3,0,1], row_half_mirror, row_mirror
  mx = fmaxf(mx, dpp_f<0x4E>(mx));
  mx = fmaxf(mx, dpp_f<0x141>(mx));
  mx = fmaxf(mx, dpp_f<0x140>(mx));
  const uint32_t sb = f32_to_bf16_rne(mx > 0.f ? mx / 7.f : 1.f);
  const float sf = bf16_bits_to_f32(sb);
  const bool live = row < a.N;
  if (live && l16 == 0) a.S[row * (K / kGq) + k0 / kGq] = static_cast<uint16_t>(sb);

#pragma unroll 1
  for (int b = 0; b < kPanelBlocks; ++b) {
    const int width = 16 * (kPanelBlocks - b);  // reads past it feed registers no column uses
    const float* u_row = tri + tri_row(b) + l16;
    int code = 0;
    gptq_column<0>(w, u_row, width, l16, sf, code);
    gptq_column<1>(w, u_row, width, l16, sf, code);
    gptq_column<2>(w, u_row, width, l16, sf, code);
    gptq_column<3>(w, u_row, width, l16, sf, code);
    gptq_column<4>(w, u_row, width, l16, sf, code);
    gptq_column<5>(w, u_row, width, l16, sf, code);
    gptq_column<6>(w, u_row, width, l16, sf, code);
    gptq_column<7>(w, u_row, width, l16, sf, code);
    gptq_column<8>(w, u_row, width, l16, sf, code);
    gptq_column<9>(w, u_row, width, l16, sf, code);
    gptq_column<10>(w, u_row, width, l16, sf, code);
    gptq_column<11>(w, u_row, width, l16, sf, code);
    gptq_column<12>(w, u_row, width, l16, sf, code);
    gptq_column<13>(w, u_row, width, l16, sf, code);
    gptq_column<14>(w, u_row, width, l16, sf, code);
    gptq_column<15>(w, u_row, width, l16, sf, code);
    int word = code << (4 * (l16 & 7));
    word |= dpp_i<0xB1>(word);
    word |= dpp_i<0x4E>(word);
    word |= dpp_i<0x141>(word);
    if (live) {
      a.W[row * K + k0 + 16 * b + l16] = w[0];
      if ((l16 & 7) == 0)
        a.Wq[row * (K >> 3) + ((k0 + 16 * b + l16) >> 3)] = static_cast<uint32_t>(word);
    }
#pragma unroll
    for (int r = 0; r + 1 < kPanelBlocks; ++r) w[r] = w[r + 1];
    w[kPanelBlocks - 1] = 0.f;
  }
}

// W[n][j] for j >= k0 + 128 with the errors of the group before k0: bound by the fp32 matrix rate.
// 128 x 128 tiles, each wave 64 x 64 as 2 x 2 fragments; errors and U staged through LDS 32 at a
// time, the next 32 already loading into registers.
__device__ __forceinline__ void gptq_trailing(const GptqArgs& a, float* lds) {
  float* es = lds;                        // [128 rows][kEsStride]
  float* us = lds + kUpTile * kEsStride;  // [32][kUsStride]
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, kh = lane >> 5;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int t = blockIdx.x - a.panels;
  const long long n0 = (long long)(t % a.up_rows) * kUpTile;
  const int K = a.K, kp = a.k0 - kGq;
  const int j0 = a.k0 + kGq + (t / a.up_rows) * kUpTile;
  const int wr = 64 * (wv >> 1), wc = 64 * (wv & 1);

  f32x4_t ev[4], uv[4];
  auto load = [&](int i0) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int v = tid + 256 * p;
      const long long n = n0 + (v >> 3);
      ev[p] = n < a.N ? *reinterpret_cast<const f32x4_t*>(a.W + n * K + kp + i0 + 4 * (v & 7))
                      : f32x4_t{0.f, 0.f, 0.f, 0.f};
      uv[p] = *reinterpret_cast<const f32x4_t*>(a.U + (size_t)(kp + i0 + (v >> 5)) * K + j0 + 4 * (v & 31));
    }
  };
  load(0);
  f32x16_t acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const long long n = n0 + wr + 32 * i + 8 * (r >> 2) + 4 * kh + (r & 3);
        acc[i][j][r] = n < a.N ? a.W[n * K + j0 + wc + 32 * j + l32] : 0.f;
      }
#pragma unroll 1
  for (int i0 = 0; i0 < kGq; i0 += kUpK) {
    __syncthreads();
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int v = tid + 256 * p;
#pragma unroll
      for (int e = 0; e < 4; ++e) es[(v >> 3) * kEsStride + 4 * (v & 7) + e] = -ev[p][e];
      *reinterpret_cast<f32x4_t*>(&us[(v >> 5) * kUsStride + 4 * (v & 31)]) = uv[p];
    }
    __syncthreads();
    if (i0 + kUpK < kGq) load(i0 + kUpK);
#pragma unroll
    for (int s = 0; s < kUpK / 2; ++s) {
      float ea[2], ub[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) ea[i] = es[(wr + 32 * i + l32) * kEsStride + 2 * s + kh];
#pragma unroll
      for (int j = 0; j < 2; ++j) ub[j] = us[(2 * s + kh) * kUsStride + wc + 32 * j + l32];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(ea[i], ub[j], acc[i][j], 0, 0, 0);
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const long long n = n0 + wr + 32 * i + 8 * (r >> 2) + 4 * kh + (r & 3);
        if (n < a.N) a.W[n * K + j0 + wc + 32 * j + l32] = acc[i][j][r];
      }
}

__global__ void __launch_bounds__(256, 2) w4_gptq_kernel(GptqArgs a) {
  constexpr int kPanelLds = kTriFloats + kGq + kPanelRows * kPanelStride;
  constexpr int kUpLds = kUpTile * kEsStride + kUpK * kUsStride;
  __shared__ __align__(16) float lds[kPanelLds > kUpLds ? kPanelLds : kUpLds];
  if ((int)blockIdx.x < a.panels)
    gptq_panel(a, lds);
  else
    gptq_trailing(a, lds);
}

bool aligned(const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

}  // namespace
}  // namespace ns

extern "C" {

size_t ns_w4_gptq_workspace(int N) {
  return N > 0 ? static_cast<size_t>(ns::kGq) * static_cast<size_t>(N) * sizeof(float) : 0;
}

int ns_w4_gptq(void* W, const void* U, void* Wq, void* S, void* work, size_t work_bytes, int N,
               int K, int G, void* stream) {
  if (G != ns::kGq || N <= 0 || K <= 0 || K % G) return -2;
  if (!W || !U || !Wq || !S || !work || work_bytes < ns_w4_gptq_workspace(N)) return -2;
  if (!ns::aligned(W, 16) || !ns::aligned(U, 16) || !ns::aligned(Wq, 16) || !ns::aligned(S, 2) ||
      !ns::aligned(work, 16))
    return -2;
  ns::GptqArgs a{static_cast<float*>(W), static_cast<const float*>(U), static_cast<uint32_t*>(Wq),
                 static_cast<uint16_t*>(S), N, K, 0, 0, 0};
  a.panels = (N + ns::kPanelRows - 1) / ns::kPanelRows;
  a.up_rows = (N + ns::kUpTile - 1) / ns::kUpTile;
  for (; a.k0 < K; a.k0 += G) {
    const int after = a.k0 ? (K - a.k0 - G) / ns::kUpTile : 0;  // column tiles past this group
    const long long blocks = a.panels + (long long)a.up_rows * after;
    if (blocks > 0x7fffffff) return -2;
    hipLaunchKernelGGL(ns::w4_gptq_kernel, dim3((unsigned)blocks), dim3(256), 0,
                       static_cast<hipStream_t>(stream), a);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return static_cast<int>(err);
  }
  return 0;
}

}  // extern "C"
