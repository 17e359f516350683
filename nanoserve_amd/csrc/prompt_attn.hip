// The prompt pass's attention step for gfx950: bias + RoPE + KV append in one launch, and causal
// grouped-query attention on bf16 matrix cores (contracts in internal_ops.h). The reference does
// both with PyTorch ops (python/nanoserve/qwen.py:119-133, 147-151).
#include <math.h>
#include <stdint.h>

#include <algorithm>

#include "attn_common.h"
#include "internal_ops.h"
#include "w4_common.h"
#include "w4_kernels.h"

namespace ns {
namespace {

// ------------------------------------------------------------------ bias + RoPE + KV append
// Bound by launch and memory latency (1000 tokens of 36 heads: 9.5 us with the KV append, where
// separate bias, RoPE and cache-copy launches took about 60). Thread (token, head block, chunk c)
// rotates elements 8c .. 8c + 7 with their partners D/2 further on in up to kQkvHeads heads, so the
// eight sincosf of a chunk serve all of them and 2 kQkvHeads 16-byte loads are in flight per thread.
constexpr int kQkvHeads = 6;
__global__ void __launch_bounds__(256)
    prompt_qkv_kernel(uint16_t* __restrict__ qkv, const uint16_t* __restrict__ bias,
                      const float* __restrict__ inv_freq, uint16_t* __restrict__ kc,
                      uint16_t* __restrict__ vc, int T, int Hq, int Hk, int D, int pos0,
                      int max_len) {
  const int chunks = D >> 4, H = Hq + 2 * Hk, nblk = (H + kQkvHeads - 1) / kQkvHeads;
  const long long id = (long long)blockIdx.x * 256 + threadIdx.x;
  const int c = (int)(id % chunks);
  const long long tb = id / chunks;
  const int t = (int)(tb / nblk), h0 = (int)(tb % nblk) * kQkvHeads;
  if (tb / nblk >= T) return;
  uint16_t* row = qkv + (size_t)t * H * D;
  u32x4_t lo[kQkvHeads], hi[kQkvHeads], blo[kQkvHeads], bhi[kQkvHeads];
#pragma unroll
  for (int i = 0; i < kQkvHeads; ++i) {
    const int off = min(h0 + i, H - 1) * D + 8 * c;  // heads past H repeat the last, unstored
    lo[i] = *reinterpret_cast<const u32x4_t*>(row + off);
    hi[i] = *reinterpret_cast<const u32x4_t*>(row + off + D / 2);
    if (bias) {
      blo[i] = *reinterpret_cast<const u32x4_t*>(bias + off);
      bhi[i] = *reinterpret_cast<const u32x4_t*>(bias + off + D / 2);
    }
  }
  float cs[8], sn[8];
  if (h0 < Hq + Hk) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      sincosf(static_cast<float>(pos0 + t) * inv_freq[8 * c + e], &sn[e], &cs[e]);
  }
#pragma unroll
  for (int i = 0; i < kQkvHeads; ++i) {
    const int h = h0 + i;
    if (h >= H) break;
    float a[8], b[8];
    unpack8(lo[i], a);
    unpack8(hi[i], b);
    if (bias) {
      float x[8], y[8];
      unpack8(blo[i], x);
      unpack8(bhi[i], y);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        a[e] = round_bf16(a[e] + x[e]);
        b[e] = round_bf16(b[e] + y[e]);
      }
    }
    if (h < Hq + Hk) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float p = a[e], q = b[e];
        a[e] = p * cs[e] - q * sn[e];
        b[e] = q * cs[e] + p * sn[e];
      }
    }
    uint16_t* dst = row + h * D;
    if (kc && h >= Hq) {
      uint16_t* cache = h < Hq + Hk ? kc : vc;
      const int g = h < Hq + Hk ? h - Hq : h - Hq - Hk;
      dst = cache + ((size_t)g * max_len + pos0 + t) * D;
    }
    *reinterpret_cast<u32x4_t*>(dst + 8 * c) = pack8(a);
    *reinterpret_cast<u32x4_t*>(dst + D / 2 + 8 * c) = pack8(b);
  }
}

// ------------------------------------------------------------------ causal attention
// Bound by the matrix cores and, closely behind, the softmax's VALU work. The rows of a kv
// head's problem are its R = Hq / Hk query heads' tokens, token-major (row = token * R + head), so
// one K / V tile serves all heads of the group and the causal limit of a 128-row tile is tight.
//  * Workgroup: 128 rows (four waves of 32) of one kv head over a range of 64-key blocks; K and V
//    blocks come in by buffer-to-LDS loads, two stages (64 KiB, two workgroups per CU).
//  * Scores are computed transposed, S^T = K Q^T on v_mfma_f32_32x32x16_bf16 (A = K rows from LDS,
//    B = Q held in registers): a lane then owns one query (column l % 32) and 16 of each 32 keys,
//    so the softmax needs one lane swap per reduction, and the score registers are, as they
//    stand, the B operand of O^T = V^T P^T: lane half kh holds keys {4 kh + b, 8 + 4 kh + b} of each
//    16, and ds_read_b64_tr_b16 delivers V^T's fragment for exactly those keys.
//  * Probabilities enter the product as bf16 terms, each the rounding of what the terms before it
//    leave (exact in fp32). Prompts from position 0 take two (16 significant bits, where fused bf16
//    attention holds 8). Chunks after cached positions take three, the whole fp32 probability, as an
//    attention in fp32 holds it: with two, 0.23 % of the outputs are not the rounding of the float64
//    result, with three 0.04 %, for fp32 SDPA 0.07 % (28 / 4 heads, 512 tokens at 3000; 61.1 us
//    against 53.6 with two).
//  * LDS rows are 256 B (16 chunks of 16 B): K chunks are XOR-swizzled by row % 16 (the 16 rows of
//    a fragment read hit distinct banks), V chunks by 4 (row % 4) (the 4-row x 64 B transpose
//    reads spread over all banks).
//  * Few row tiles (short prompts, few kv heads) leave CUs idle: the keys are then split over
//    blockIdx.z and a second kernel merges the fp32 partials.
// MI355X, 28 / 4 heads, with the merge: 1000 tokens from position 0 36.1 us (PyTorch's fused SDPA on
// repeated K / V 67 us and its copies 40); 512 tokens after 3000 cached ones 60.9 us (fp32 SDPA 682
// us and its copies 60).
constexpr int kD = 128;
constexpr int kRows = 128;    // query rows per workgroup
constexpr int kKeys = 64;     // keys per block
constexpr int kTile = kKeys * kD;  // bf16 elements of one K or V block

struct AttnArgs {
  const uint16_t *q, *k, *v;
  uint16_t* out;
  float *opart, *ml;  // [splits][Hk * rows][128] and [splits][Hk * rows][2]
  long long q_stride, kv_stride, kv_head_stride;
  int T, R, Hk, pos0, splits;
};

template <int TERMS>
__global__ void __launch_bounds__(256, 2) prompt_attn_kernel(AttnArgs a) {
  // one array per stage: a read of one stage then provably does not alias the loads in flight
  // into the other, so the compiler puts no wait for those before it
  __shared__ __align__(16) uint16_t ks0[kTile], ks1[kTile], vs0[kTile], vs1[kTile];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = blockIdx.x, split = blockIdx.z;
  const int tile = gridDim.y - 1 - blockIdx.y;  // longest tiles first
  const int rows = a.T * a.R, R = a.R;
  const int r0 = tile * kRows;
  const int jq = lane & 31, kh = lane >> 5;
  const int wrow = r0 + 32 * wv;                       // the wave's first row
  const int row = min(wrow + jq, rows - 1);            // rows past the end repeat the last
  const int tok = row / R, hq = g * R + row % R;
  const int qpos = a.pos0 + tok;
  const int wlo = a.pos0 + min(wrow, rows - 1) / R;             // positions of the wave's rows
  const int whi = a.pos0 + min(wrow + 31, rows - 1) / R;
  const int last = a.pos0 + min(r0 + kRows - 1, rows - 1) / R;  // and the tile's last
  const int nb = last / kKeys + 1;
  const int b0 = (int)((long long)nb * split / a.splits);
  const int b1 = (int)((long long)nb * (split + 1) / a.splits);
  const float c = 0.08838834764831845f * 1.4426950408889634f;  // log2(e) / sqrt(128)

  // B operand of the scores: this lane's query at dims 16 s + 8 kh ..
  u32x4_t qf[8];
  {
    const uint16_t* qp = a.q + (size_t)tok * a.q_stride + (size_t)hq * kD + 8 * kh;
#pragma unroll
    for (int s = 0; s < 8; ++s) qf[s] = *reinterpret_cast<const u32x4_t*>(qp + 16 * s);
  }

  // K / V block loader: rows past the last key read as zero through the buffer range check
  const uint32_t rb = 2u * (uint32_t)a.kv_stride;
  const uint32_t span = (uint32_t)(a.pos0 + a.T - 1) * rb + 2u * kD;
  const auto kres = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(a.k + (size_t)g * a.kv_head_stride), (short)0, (int)span, 0x00020000);
  const auto vres = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(a.v + (size_t)g * a.kv_head_stride), (short)0, (int)span, 0x00020000);
  uint32_t k_off[4], v_off[4];
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const uint32_t lr = 16 * wv + 4 * p + (lane >> 4), ch = lane & 15;
    k_off[p] = lr * rb + 16u * (ch ^ (lr & 15));
    v_off[p] = lr * rb + 16u * (ch ^ ((lr & 3) << 2));
  }
  auto issue = [&](uint16_t* ks, uint16_t* vs, int b) {
    const uint32_t so = (uint32_t)b * kKeys * rb;
#pragma unroll
    for (int p = 0; p < 4; ++p) attn_lds_load16(kres, &ks[512 * (4 * wv + p)], k_off[p], so);
#pragma unroll
    for (int p = 0; p < 4; ++p) attn_lds_load16(vres, &vs[512 * (4 * wv + p)], v_off[p], so);
  };

  f32x16_t o[4];
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[d][r] = 0.f;
  float m = -INFINITY, l = 0.f;

  // transpose-read offsets (elements) of the four 32-dim tiles at key row 4 kh + (lane % 16) / 4
  int vt[4];
  {
    const int rr = (lane & 15) >> 2;
#pragma unroll
    for (int d = 0; d < 4; ++d)
      vt[d] = (4 * kh + rr) * kD + 8 * (((d ^ rr) << 2) + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) +
              4 * (lane & 1);
  }

  auto compute = [&](const uint16_t* kt, const uint16_t* vb, int b) {
    f32x16_t s[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[t][r] = 0.f;
#pragma unroll
      for (int d = 0; d < 8; ++d) {
        const int kr = 32 * t + jq;
        const u32x4_t kf = *reinterpret_cast<const u32x4_t*>(&kt[kr * kD + 8 * ((2 * d + kh) ^ (kr & 15))]);
        s[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, kf),
                                                       __builtin_bit_cast(bf16x8_t, qf[d]), s[t], 0, 0, 0);
      }
    }
    if (b * kKeys + kKeys - 1 > wlo) {  // the block crosses the diagonal of some row
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = b * kKeys + 32 * t + 8 * (r >> 2) + 4 * kh + (r & 3);
          if (key > qpos) s[t][r] = -INFINITY;
        }
    }
    float bm = s[0][0];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) bm = fmaxf(bm, s[t][r]);
    bm = fmaxf(bm, lane_xor32(bm));
    if (__any(bm > m)) {
      const float mn = fmaxf(m, bm);
      const float ms = mn == -INFINITY ? 0.f : mn;
      const float alpha = __builtin_amdgcn_exp2f((m - ms) * c);
      m = mn;
      l *= alpha;
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[d][r] *= alpha;
    }
    const float mc = m == -INFINITY ? 0.f : m * c;
    u32x4_t pt[TERMS][4];  // B operands of the four 16-key steps
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        float p0 = __builtin_amdgcn_exp2f(fmaf(s[t][r], c, -mc));
        float p1 = __builtin_amdgcn_exp2f(fmaf(s[t][r + 1], c, -mc));
        l += p0 + p1;
#pragma unroll
        for (int i = 0; i < TERMS; ++i) {
          const uint32_t term = pack_bf16x2_rne(p0, p1);
          pt[i][2 * t + (r >> 3)][(r & 7) >> 1] = term;
          p0 -= __uint_as_float(term << 16);
          p1 -= __uint_as_float(term & 0xffff0000u);
        }
      }
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const u32x2_t v0 = lds_read_tr16(&vb[vt[d] + 16 * t * kD]);
        const u32x2_t v1 = lds_read_tr16(&vb[vt[d] + (16 * t + 8) * kD]);
        const bf16x8_t vf = __builtin_bit_cast(bf16x8_t, (u32x4_t){v0[0], v0[1], v1[0], v1[1]});
#pragma unroll
        for (int i = 0; i < TERMS; ++i)
          o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, __builtin_bit_cast(bf16x8_t, pt[i][t]), o[d], 0, 0, 0);
      }
  };

  // Block b is ready once every wave's loads of it have landed, and past the barrier nobody reads block
  // b - 1, whose stage takes block b + 1: each wave waits for its loads of b and its reads of b - 1.
  auto ready = [] {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0), lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  if (b0 < b1) issue(ks0, vs0, b0);
  for (int b = b0; b < b1; b += 2) {
    ready();
    if (b + 1 < b1) issue(ks1, vs1, b + 1);
    if (b * kKeys <= whi) compute(ks0, vs0, b);  // else past every row of this wave
    if (b + 1 == b1) break;
    ready();
    if (b + 2 < b1) issue(ks0, vs0, b + 2);
    if ((b + 1) * kKeys <= whi) compute(ks1, vs1, b + 1);
  }

  l += lane_xor32(l);
  if (wrow + jq >= rows) return;
  if (a.splits == 1) {
    const float inv = 1.f / l;
    uint16_t* op = a.out + ((size_t)tok * a.Hk * R + hq) * kD + 4 * kh;
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int r = 0; r < 16; r += 4)
        *reinterpret_cast<u32x2_t*>(op + 32 * d + 2 * r) =
            (u32x2_t){pack_bf16x2_rne(o[d][r] * inv, o[d][r + 1] * inv),
                      pack_bf16x2_rne(o[d][r + 2] * inv, o[d][r + 3] * inv)};
  } else {
    const size_t pr = ((size_t)split * a.Hk + g) * rows + row;
    float* op = a.opart + pr * kD + 4 * kh;
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int r = 0; r < 16; r += 4)
        *reinterpret_cast<f32x4_t*>(op + 32 * d + 2 * r) =
            f32x4_t{o[d][r], o[d][r + 1], o[d][r + 2], o[d][r + 3]};
    if (kh == 0) {
      a.ml[2 * pr] = m * c;
      a.ml[2 * pr + 1] = l;
    }
  }
}

// Merge of the splits' partials: 32 threads per (kv head, row), four values each. A split that
// holds no key of a row has max -inf and sum 0.
__global__ void __launch_bounds__(256) prompt_attn_merge_kernel(AttnArgs a) {
  const int rows = a.T * a.R, all = a.Hk * rows;
  const int id = blockIdx.x * 8 + (threadIdx.x >> 5), d = 4 * (threadIdx.x & 31);
  if (id >= all) return;
  float mx = -INFINITY;
#pragma unroll 8
  for (int s = 0; s < a.splits; ++s) mx = fmaxf(mx, a.ml[2 * ((size_t)s * all + id)]);
  float l = 0.f;
  f32x4_t o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (int s = 0; s < a.splits; ++s) {
    const size_t pr = (size_t)s * all + id;
    const float w = __builtin_amdgcn_exp2f(a.ml[2 * pr] - mx);
    const f32x4_t v = *reinterpret_cast<const f32x4_t*>(a.opart + pr * kD + d);
    l = fmaf(w, a.ml[2 * pr + 1], l);
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = fmaf(w, v[e], o[e]);
  }
  const float inv = 1.f / l;
  const int g = id / rows, row = id % rows;
  uint16_t* op = a.out + ((size_t)(row / a.R) * a.Hk * a.R + g * a.R + row % a.R) * kD + d;
  *reinterpret_cast<u32x2_t*>(op) = (u32x2_t){pack_bf16x2_rne(o[0] * inv, o[1] * inv),
                                              pack_bf16x2_rne(o[2] * inv, o[3] * inv)};
}

// Splits over the keys: enough for one and a half workgroups per CU, each with at least four blocks.
// us (28 / 4 heads) for 1, 1.5, 2 and 3 per CU: 512 tokens at 3000 67.5, 60.9, 68.4, 67.4; 2000 tokens
// at 0 56.4, 56.3, 66.5, 66.0; 200 at 4000 45.8, 39.5, 46.3, 42.1. With two blocks or one at least,
// 20 tokens at 4000 take 26.2 and 30.9 us against 23.1, 200 at 0 14.2 and 16.0 against 10.1.
int attn_splits(int T, int Hq, int Hk, int pos0) {
  int cus = 256;  // the device's CU count (a failed query leaves MI355X's; the launch reports it)
  if (cached_cu_count(&cus) != hipSuccess || cus <= 0) cus = 256;
  const long long tiles = (((long long)T * (Hq / Hk) + kRows - 1) / kRows) * Hk;
  const int blocks = (pos0 + T + kKeys - 1) / kKeys;
  const long long want = (3 * cus / 2 + tiles - 1) / tiles;
  return (int)std::max(1ll, std::min<long long>(want, blocks / 4));
}

bool aligned(const void* p, uintptr_t n) { return (reinterpret_cast<uintptr_t>(p) & (n - 1)) == 0; }

bool attn_sizes_ok(int T, int Hq, int Hk, int pos0) {
  return T > 0 && Hq > 0 && Hk > 0 && Hq % Hk == 0 && pos0 >= 0 &&
         (long long)pos0 + T < (1ll << 30) && (long long)T * Hq < (1ll << 30);
}

unsigned attn_row_tiles(int T, int R) { return (unsigned)((T * R + kRows - 1) / kRows); }

// The kernel's offsets and grid: block offsets past the last key stay below 2^32 and the range of the
// keys' rows below 2^31; row tiles are a grid dimension.
bool attn_fits(int T, int Hq, int Hk, int pos0, long long kv_stride) {
  return attn_sizes_ok(T, Hq, Hk, pos0) && kv_stride >= kD && kv_stride < (1ll << 30) &&
         ((long long)pos0 + T + 2 * kKeys) * kv_stride * 2 < (1ll << 31) &&
         attn_row_tiles(T, Hq / Hk) <= 65535u;
}

}  // namespace
}  // namespace ns

extern "C" {

int ns_prompt_qkv(void* qkv, const void* bias, const void* inv_freq, void* k_cache,
                  void* v_cache, int T, int Hq, int Hk, int D, int pos0, int max_len,
                  void* stream) {
  if (T <= 0 || Hq <= 0 || Hk <= 0 || D <= 0 || D % 16 || D > 512 || pos0 < 0) return -2;
  if (!qkv || !inv_freq || (!k_cache) != (!v_cache)) return -2;
  if (k_cache && (long long)pos0 + T > max_len) return -2;
  if (!ns::aligned(qkv, 16) || !ns::aligned(bias, 16) || !ns::aligned(inv_freq, 4) ||
      !ns::aligned(k_cache, 16) || !ns::aligned(v_cache, 16))
    return -2;
  const long long nblk = (Hq + 2ll * Hk + ns::kQkvHeads - 1) / ns::kQkvHeads;
  const long long threads = T * nblk * (D / 16);
  if (threads >= (1ll << 38)) return -2;
  hipLaunchKernelGGL(ns::prompt_qkv_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), static_cast<uint16_t*>(qkv),
                     static_cast<const uint16_t*>(bias), static_cast<const float*>(inv_freq),
                     static_cast<uint16_t*>(k_cache), static_cast<uint16_t*>(v_cache), T, Hq, Hk, D,
                     pos0, max_len);
  return static_cast<int>(hipGetLastError());
}

int ns_prompt_attention_fits(int T, int Hq, int Hk, int pos0, long long kv_stride) {
  return ns::attn_fits(T, Hq, Hk, pos0, kv_stride);
}

size_t ns_prompt_attention_workspace(int T, int Hq, int Hk, int pos0) {
  if (!ns::attn_sizes_ok(T, Hq, Hk, pos0)) return 0;
  const size_t splits = static_cast<size_t>(ns::attn_splits(T, Hq, Hk, pos0));
  return splits > 1 ? splits * T * Hq * (ns::kD + 2) * sizeof(float) : 0;
}

int ns_prompt_attention(const void* q, long long q_stride, const void* k, const void* v,
                        long long kv_stride, long long kv_head_stride, void* out, void* work,
                        size_t work_bytes, int T, int Hq, int Hk, int pos0, void* stream) {
  if (!ns::attn_fits(T, Hq, Hk, pos0, kv_stride)) return -2;
  if (!q || !k || !v || !out) return -2;
  if (!ns::aligned(q, 16) || !ns::aligned(k, 16) || !ns::aligned(v, 16) || !ns::aligned(out, 16))
    return -2;
  if (q_stride % 8 || kv_stride % 8 || kv_head_stride % 8) return -2;
  if (q_stride < (long long)Hq * ns::kD || kv_head_stride < 0) return -2;
  ns::AttnArgs a{};
  a.splits = ns::attn_splits(T, Hq, Hk, pos0);
  if (a.splits > 1) {
    const size_t rows = static_cast<size_t>(T) * Hq;
    if (!work || !ns::aligned(work, 16) || work_bytes < ns_prompt_attention_workspace(T, Hq, Hk, pos0))
      return -2;
    a.opart = static_cast<float*>(work);
    a.ml = a.opart + a.splits * rows * ns::kD;
  }
  a.q = static_cast<const uint16_t*>(q);
  a.k = static_cast<const uint16_t*>(k);
  a.v = static_cast<const uint16_t*>(v);
  a.out = static_cast<uint16_t*>(out);
  a.q_stride = q_stride;
  a.kv_stride = kv_stride;
  a.kv_head_stride = kv_head_stride;
  a.T = T;
  a.R = Hq / Hk;
  a.Hk = Hk;
  a.pos0 = pos0;
  const int rows = T * a.R;
  const auto st = static_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)Hk, ns::attn_row_tiles(T, a.R), (unsigned)a.splits);
  if (pos0 > 0)
    hipLaunchKernelGGL(ns::prompt_attn_kernel<3>, grid, dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL(ns::prompt_attn_kernel<2>, grid, dim3(256), 0, st, a);
  if (a.splits > 1)
    hipLaunchKernelGGL(ns::prompt_attn_merge_kernel, dim3((unsigned)(((long long)rows * Hk + 7) / 8)),
                       dim3(256), 0, st, a);
  return static_cast<int>(hipGetLastError());
}

}  // extern "C"
