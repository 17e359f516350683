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
//  * trailing workgroups apply the errors of group g - 1 to every column after group g, on the CUs
//    that the panels, a serial chain per row, leave with little to do.
// 4608 x 3584 on MI355X: a launch of panels alone takes 26.7 us, the one with 936 trailing tiles 60.8
// (25.8 us of fp32 matrix work), all 28 launches 1.2 ms without gaps. The trailing work runs close to
// its rate, but the panels' chain adds to it.
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

// The panel's triangle of U in LDS: rows of 16-column blocks b = 4 P .. 4 P + 3 keep NB = 8 - 4 P blocks
// each (block b + r of the row as its r-th; those past the group hold values nobody uses), as
// pairs of blocks interleaved per lane, so that a lane reads two of its columns at once. The
// row's own block (r = 0) starts at its diagonal.
constexpr int tri_base(int p) { return p == 0 ? 0 : tri_base(p - 1) + 64 * 16 * (kPanelBlocks - 4 * (p - 1)); }
constexpr int kTriFloats = tri_base(2);

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
constexpr int kRowBcast0 = 0x150;  // row_newbcast:0, lane 0 of each 16-lane row to all of it
constexpr int kRowNext = 0x12F;    // row_ror:15, lane l takes lane l + 1 (lane 15 lane 0)

// Rows n0 .. of W (or of U) as a buffer: rows past the last read as zero and are not stored.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_rsrc(const float* base, long long row, long long rows,
                                                            int K) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base + row * K), (short)0,
                                           (int)(rows * K * 4), 0x00020000);
}
__device__ __forceinline__ float ldf(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}
__device__ __forceinline__ f32x4_t ldf4(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  return __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}
__device__ __forceinline__ void stf(__amdgpu_buffer_rsrc_t r, float v, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, voff, soff, 0);
}

// 1 / x correctly rounded, or NaN where the arithmetic below could overflow or underflow.
__device__ __forceinline__ float safe_rcp(float x) {
  const float m = fabsf(x);
  return m > 0x1p-60f && m < 0x1p60f ? 1.f / x : __builtin_nanf("");
}

// A row of U and the reciprocal of its diagonal, as the lane needs them.
template <int NB>
struct URow {
  float u[NB], ru;
  __device__ __forceinline__ void load(const float* p, const float* rcp) {
    typedef float f32x2_t __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int r = 0; r < NB; r += 2) {
      const f32x2_t v = *reinterpret_cast<const f32x2_t*>(p + 16 * r);
      u[r] = v[0];
      u[r + 1] = v[1];
    }
    ru = *rcp;
  }
};

// Column s of a 16-column block b, the serial chain. w[r], r > 0, is column 16 (b + r) + lane; w[0] is
// rotated so that lane 0 of the row holds the current column, lanes 1 .. 15 - s those after it and
// the lanes behind them the errors of those done; codes (- 8) rotate with them in vr.
//
// Without EXACT the two divisions are multiplications by reciprocals, arranged so that the results
// are those of IEEE division:
//  * rint(c / sf): c * rs is within 2^-22 |c / sf| of it, so both round to the same integer unless
//    the product lies within 1e-5 of a half (or beyond +-16, where the clamp decides alone);
//  * num / ud: q0 = num ru, one correction by its exact remainder gives e; a second correction
//    applied to a faithful quotient yields the correctly rounded one (Markstein, "Computation of
//    elementary functions on the IBM RISC System/6000 processor", 1990), so e is accepted when it
//    leaves e unchanged.
// `bad` collects where a test fails (a few times in a million) or operands are outside the range in
// which the remainders are exact: the block is then done again with EXACT.
template <int NB, bool EXACT>
__device__ __forceinline__ void gptq_column(float (&w)[kPanelBlocks], const URow<NB>& t, int s, int l16,
                                            float sf, float rs, float& vr, bool& bad) {
  const float c = w[0], ud = t.u[0];
  float v, e;
  if constexpr (EXACT) {
    int q = (int)((uint32_t)f2i_rn(c / sf) + 8u);
    q = q < 0 ? 0 : (q > 15 ? 15 : q);
    v = static_cast<float>(q - 8);
    e = fmaf(-v, sf, c) / ud;
  } else {
    const float tq = c * rs, tr = __builtin_rintf(tq);
    v = __builtin_amdgcn_fmed3f(tr, -8.f, 7.f);
    const float num = fmaf(-v, sf, c);
    const float q0 = num * t.ru;
    e = fmaf(fmaf(-ud, q0, num), t.ru, q0);
    const bool fine = fmaf(fmaf(-ud, e, num), t.ru, e) == e && fabsf(tq) < 0x1p20f &&
                      fabsf(tq - tr) < 0.49999f && (fabsf(num) > 0x1p-60f || num == 0.f);
    bad |= !fine;
  }
  const float eb = dpp_f<kRowBcast0>(e);
#pragma unroll
  for (int r = 1; r < NB; ++r) w[r] = fmaf(-eb, t.u[r], w[r]);
  const float w0 = l16 < 16 - s ? fmaf(-eb, ud, c) : c;
  w[0] = dpp_f<kRowNext>(l16 == 0 ? e : w0);
  vr = dpp_f<kRowNext>(l16 == 0 ? v : vr);
}

// The 16 columns of a block in order; true where `bad` (above) came up for a row of the wave. Rolled,
// as straight code that is not in the instruction cache costs more than it saves (all 16 columns
// unrolled ran twice as long).
template <int NB, bool EXACT>
__device__ __forceinline__ bool gptq_columns(float (&w)[kPanelBlocks], const float* u_row, const float* rcp,
                                             int l16, float sf, float rs, float& vr) {
  URow<NB> ta, tb;
  bool bad = false;
  ta.load(u_row, rcp);
#pragma unroll 1
  for (int s = 0; s < 16; s += 2) {  // the next row of U is read ahead of a column's chain
    tb.load(u_row + 16 * NB, rcp + 1);
    gptq_column<NB, EXACT>(w, ta, s, l16, sf, rs, vr, bad);
    u_row += 2 * 16 * NB;
    rcp += 2;
    ta.load(u_row, rcp);  // (after the last column: whatever follows in LDS, unused)
    gptq_column<NB, EXACT>(w, tb, s + 1, l16, sf, rs, vr, bad);
  }
  return __any(l16 == 0 && bad);
}

// Blocks 4 P .. 4 P + 3, which hold NB = 8 - 4 P column blocks per row: columns in order, then each
// block's codes and errors out and the registers moved up.
template <int P>
__device__ __forceinline__ void gptq_blocks(const GptqArgs& a, float (&w)[kPanelBlocks], const float* tri,
                                            const float* rcp, int l16, float sf, float rs,
                                            __amdgpu_buffer_rsrc_t wres, uint32_t w_off, long long row,
                                            bool live) {
  constexpr int NB = kPanelBlocks - 4 * P;
  const float* u_row = tri + tri_base(P) + 2 * l16;
  rcp += 64 * P;
#pragma unroll 1
  for (int h = 0; h < 4; ++h) {
    float vr = 0.f, saved[NB];
#pragma unroll
    for (int r = 0; r < NB; ++r) saved[r] = w[r];
    if (__builtin_expect(gptq_columns<NB, false>(w, u_row, rcp, l16, sf, rs, vr), 0)) {
#pragma unroll
      for (int r = 0; r < NB; ++r) w[r] = saved[r];
      gptq_columns<NB, true>(w, u_row, rcp, l16, sf, rs, vr);
    }
    u_row += 16 * 16 * NB;
    rcp += 16;
    int word = ((int)vr + 8) << (4 * (l16 & 7));
    word |= dpp_i<0xB1>(word);  // quad_perm [1,0,3,2], [2,3,0,1], row_half_mirror
    word |= dpp_i<0x4E>(word);
    word |= dpp_i<0x141>(word);
    const int col = a.k0 + 64 * P + 16 * h + l16;
    stf(wres, w[0], w_off + 4u * col, 0);
    if (live && (l16 & 7) == 0) a.Wq[row * (a.K >> 3) + (col >> 3)] = static_cast<uint32_t>(word);
#pragma unroll
    for (int r = 0; r + 1 < NB; ++r) w[r] = w[r + 1];
  }
}

// Loads of the triangle for class P, in the order of its LDS layout (one value per thread and step,
// no branches: a b128 load per four columns and conditional stores took 8 us of a 30 us panel).
// idx = tid + 256 k: row i = idx / (16 NB) of the class, r = 2 (d / 32) + d % 2 and lane l = d % 32 / 2
// of d = idx % (16 NB). Columns past the group belong to entries nobody uses.
template <int P>
__device__ __forceinline__ void load_tri(float (&uv)[64 * (kPanelBlocks - 4 * P) / 16], __amdgpu_buffer_rsrc_t ures,
                                         int tid, int k0, uint32_t rb) {
  constexpr int NB = kPanelBlocks - 4 * P, W16 = 16 * NB, RPS = 256 / W16;  // rows per step
  const int d = tid % W16, r = 2 * (d / 32) + (d & 1), l = (d & 31) >> 1, i0 = tid / W16;
  const bool own = r == 0;
  const uint32_t base = i0 * rb + 4u * (own ? i0 + l : 16 * r + l);
#pragma unroll
  for (int k = 0; k < 64 / RPS; ++k) {
    const int i = k * RPS;  // first row of the step, within the class
    uv[k] = ldf(ures, base + (own ? 4u * i : 64u * (i >> 4)), (64u * P + i) * rb + 4u * (k0 + 64 * P));
  }
}
template <int P>
__device__ __forceinline__ void store_tri(const float (&uv)[64 * (kPanelBlocks - 4 * P) / 16], float* tri,
                                          int tid) {
#pragma unroll
  for (int k = 0; k < 64 * (kPanelBlocks - 4 * P) / 16; ++k) tri[tri_base(P) + 256 * k + tid] = uv[k];
}

// Bound by the latency of the per-column chain (a dozen dependent operations, two of them lane
// moves). Sixteen lanes per row hold eight columns each, so the other updates of a column are at
// most eight independent fmas off that chain.
__device__ __forceinline__ void gptq_panel(const GptqArgs& a, float* lds) {
  float* tri = lds;                 // [kTriFloats]
  float* rcp = tri + kTriFloats;    // [128] reciprocals of the diagonal
  float* tile = rcp + kGq;          // [16][kPanelStride]
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, lq = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const long long n0 = (long long)blockIdx.x * kPanelRows;
  const int K = a.K, k0 = a.k0;
  const uint32_t rb = 4u * (uint32_t)K;
  const auto wres = rows_rsrc(a.W, n0, min((long long)kPanelRows, a.N - n0), K);

  // Every load of the prologue is issued before its first use, so that it costs one trip to
  // memory: this wave's 32 columns of W (accumulators) and of U's rows k0 - 128 .. (B fragments),
  // the errors of the group before, and the triangle of U.
  f32x4_t acc[2], ev[2];
  float bu[2][kGq / 4], ua[32], ub[16], ud = 1.f;
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      acc[j][r] = ldf(wres, (4 * lq + r) * rb + 4u * (k0 + 32 * wv + 16 * j + l16), 0);
  if (k0) {
    const auto ures = rows_rsrc(a.U, k0 - kGq, kGq, K);
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int v = tid + 256 * p;
      ev[p] = ldf4(wres, (v >> 5) * rb + 16u * (v & 31), 4u * (k0 - kGq));
    }
#pragma unroll
    for (int s = 0; s < kGq / 4; ++s)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        bu[j][s] = ldf(ures, lq * rb + 4u * (k0 + 32 * wv + 16 * j + l16), 4u * s * rb);
  }
  {
    const auto ures = rows_rsrc(a.U, k0, kGq, K);
    load_tri<0>(ua, ures, tid, k0, rb);
    load_tri<1>(ub, ures, tid, k0, rb);
    ud = ldf(ures, (tid & 127) * (rb + 4u), 4u * k0);
  }
  if (k0) {
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int v = tid + 256 * p;
      *reinterpret_cast<f32x4_t*>(&tile[(v >> 5) * kPanelStride + 4 * (v & 31)]) = ev[p];
    }
    __syncthreads();
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
  store_tri<0>(ua, tri, tid);
  store_tri<1>(ub, tri, tid);
  if (tid < kGq) rcp[tid] = safe_rcp(ud);
  __syncthreads();

  const int lr = 4 * wv + lq;  // this lane's row, 16 lanes per row
  const long long row = n0 + lr;
  const bool live = row < a.N;
  float w[kPanelBlocks];
#pragma unroll
  for (int r = 0; r < kPanelBlocks; ++r) w[r] = tile[lr * kPanelStride + 16 * r + l16];
  float mx = 0.f;
#pragma unroll
  for (int r = 0; r < kPanelBlocks; ++r) mx = fmaxf(mx, fabsf(w[r]));
  mx = fmaxf(mx, dpp_f<0xB1>(mx));  // quad_perm [1,0,3,2], [2,3,0,1], row_half_mirror, row_mirror
  mx = fmaxf(mx, dpp_f<0x4E>(mx));
  mx = fmaxf(mx, dpp_f<0x141>(mx));
  mx = fmaxf(mx, dpp_f<0x140>(mx));
  const uint32_t sb = f32_to_bf16_rne(mx > 0.f ? mx / 7.f : 1.f);
  const float sf = bf16_bits_to_f32(sb), rs = safe_rcp(sf);
  if (live && l16 == 0) a.S[row * (K / kGq) + k0 / kGq] = static_cast<uint16_t>(sb);
  const uint32_t w_off = lr * rb;
  gptq_blocks<0>(a, w, tri, rcp, l16, sf, rs, wres, w_off, row, live);
  gptq_blocks<1>(a, w, tri, rcp, l16, sf, rs, wres, w_off, row, live);
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
  const uint32_t rb = 4u * (uint32_t)K;
  const auto wres = rows_rsrc(a.W, n0, min((long long)kUpTile, a.N - n0), K);
  const auto ures = rows_rsrc(a.U, kp, kGq, K);

  f32x4_t ev[4], uv[4];
  const uint32_t e_off = (tid >> 3) * rb + 16u * (tid & 7), u_off = (tid >> 5) * rb + 16u * (tid & 31);
  auto load = [&](int i0) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      ev[p] = ldf4(wres, e_off, 32u * p * rb + 4u * (kp + i0));
      uv[p] = ldf4(ures, u_off, (i0 + 8u * p) * rb + 4u * j0);
    }
  };
  load(0);
  const uint32_t acc_off = (wr + 4 * kh) * rb + 4u * (j0 + wc + l32);
  f32x16_t acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        acc[i][j][r] = ldf(wres, acc_off + 128u * j, (32 * i + 8 * (r >> 2) + (r & 3)) * rb);
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
    for (int r = 0; r < 16; ++r)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        stf(wres, acc[i][j][r], acc_off + 128u * j, (32 * i + 8 * (r >> 2) + (r & 3)) * rb);
}

__global__ void __launch_bounds__(256, 2) w4_gptq_kernel(GptqArgs a) {
  constexpr int kPanelLds = kTriFloats + kGq + kPanelRows * kPanelStride;  // rows read ahead: in bounds
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
  if (K >= 1 << 22) return -2;  // 128 rows of K floats stay within a 2 GiB buffer
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
