// Decode attention over a long KV cache (gfx950): one query token, grouped-query heads of 128, the
// same operation, workspace layout and merge launch as decode_attn_kernel (decode_ops.hip), for
// caches whose rows are worth streaming.
//
// Bound by HBM. decode_attn_kernel gives each 128 cache rows two workgroups that load everything at
// once and end; over a long cache that is rounds of short-lived workgroups, each reading the K rows
// twice, preparing q and leaving partials for every 128 rows. Here at most one eight-wave workgroup per
// CU streams a contiguous range of rows (whole multiples of 128, so just past a multiple of the launch's
// workgroups fewer of them have rows: 8320 rows of 4 kv heads keep 132 of 256 busy):
//  * Each wave takes every eighth 16-row block of the range through its own two-stage LDS ring
//    (8 KiB of K and V per stage by coalesced buffer-to-LDS loads, 128 KiB per workgroup), waiting
//    only for its own loads: no barrier in the loop, 64 KiB and more in flight per CU.
//  * The arithmetic of a block, and the merge of the eight waves, are decode_attn_kernel's (K as the
//    A operand, heads as columns, probabilities as two bf16 terms), so a range of up to 128 rows
//    gives its bits; more blocks per wave are combined with a running maximum. The value operand
//    (rows 4 (l / 16) .. + 3 of one dimension per lane) is one ds_read_b64_tr_b16 per 16 dimensions.
//  * The workgroups' results are merged by decode_attn_merge_kernel.
// Rows per workgroup come from the position (long_chunk_rows), so that a short conversation in a
// large cache still spreads over workgroups of 128 rows (28 / 4 heads, 32768 rows, position 1000: 24.0
// -> 10.3 us with the merge).
#include <math.h>
#include <stdint.h>

#include "attn_common.h"
#include "w4_kernels.h"

namespace ns {
namespace {

constexpr int kD = 128;
constexpr int kWaves = 8;
constexpr int kRows = 16;             // cache rows per block
constexpr int kBlk = kRows * kD;      // bf16 elements of one K or V block
constexpr int kHeads = 8;             // query heads per kv head at most (of 16 score columns)
constexpr int kQs = kD + 8;           // padded q row

struct LongArgs {
  const uint16_t *q, *bias;
  const float *inv_freq, *rot_tab;
  uint16_t *kc, *vc;
  const int* pos;
  uint16_t* out;
  float *opart, *ml;
  int Hq, Hk, max_len;
  float qscale;
};

// kFused: q is the projection output qkv [(Hq + 2 Hk) * D]; every workgroup applies bias and RoPE to
// its group's q heads, and the one whose range holds row *pos also builds that row's k and v,
// appends them to the cache and puts them into its LDS block (the row in memory may still be old).
template <bool kFused>
__global__ void __launch_bounds__(kWaves * kWave) attn_long_kernel(LongArgs a) {
  // one array per stage, so that reads of a stage do not wait for the loads into the other
  __shared__ __align__(16) uint16_t k0[kWaves][kBlk], k1[kWaves][kBlk], v0[kWaves][kBlk], v1[kWaves][kBlk];
  __shared__ __align__(16) uint16_t qb[kHeads][kQs];
  __shared__ __align__(16) uint16_t knew[kD], vnew[kD];
  __shared__ float rot[2][kD / 2];
  __shared__ float red_m[kWaves][16], red_l[kWaves][16];

  const int split = blockIdx.x, g = blockIdx.y;
  const int R = a.Hq / a.Hk;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int pos = __builtin_amdgcn_readfirstlane(*a.pos);

  // q, bias and angles (independent of the position): thread t < 8 R: head t / 8, chunk pair t % 8;
  // then 8 threads for the k head's chunk pairs and 16 for the v head's chunks
  const int nq = 8 * R, c = tid < nq ? tid % 8 : tid - nq;
  const bool is_q = tid < nq, ld_k = kFused && tid >= nq && tid < nq + 8,
             ld_v = kFused && tid >= nq + 8 && tid < nq + 24;
  u32x4_t a0{}, a1{}, b0{}, b1{};
  float angle = 0.f;
  f32x4_t tc[2], ts[2];
  if (is_q || ld_k || ld_v) {
    const int off = is_q ? (g * R + tid / 8) * kD + 8 * c
                  : ld_k ? (a.Hq + g) * kD + 8 * c : (a.Hq + a.Hk + g) * kD + 8 * (tid - nq - 8);
    a0 = *reinterpret_cast<const u32x4_t*>(a.q + off);
    if (!ld_v) a1 = *reinterpret_cast<const u32x4_t*>(a.q + off + kD / 2);
    if (kFused && a.bias) {
      b0 = *reinterpret_cast<const u32x4_t*>(a.bias + off);
      if (!ld_v) b1 = *reinterpret_cast<const u32x4_t*>(a.bias + off + kD / 2);
    }
  }
  if constexpr (kFused) {
    if (a.rot_tab) {
      const int p = 8 * (c & 7);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        tc[i] = *reinterpret_cast<const f32x4_t*>(a.rot_tab + p + 4 * i);
        ts[i] = *reinterpret_cast<const f32x4_t*>(a.rot_tab + kD / 2 + p + 4 * i);
      }
    } else if (tid < kD / 2) {
      angle = a.inv_freq[tid];
    }
  }

  const int n = min(pos + 1, a.max_len);
  if (n <= 0) {  // no rows: zeros
    if (split == 0)
      for (int i = tid; i < R * kD; i += kWaves * kWave) a.out[(size_t)g * R * kD + i] = 0;
    return;
  }
  const int chunk = long_chunk_rows(n, gridDim.x);
  const int nsplit = (n + chunk - 1) / chunk;
  const int start = split * chunk;
  if (start >= n) return;
  const int end = min(start + chunk, n);
  const int nblk = (end - start + kRows - 1) / kRows;

  // block j of the range: lane l of load p brings row 4 p + l / 16; K chunks (16 B) are XOR-swizzled
  // by row % 16, V chunks by 4 (row % 4); rows past the position read as zero
  const auto kres = __builtin_amdgcn_make_buffer_rsrc(a.kc + (size_t)g * a.max_len * kD, (short)0,
                                                      n * kD * 2, 0x00020000);
  const auto vres = __builtin_amdgcn_make_buffer_rsrc(a.vc + (size_t)g * a.max_len * kD, (short)0,
                                                      n * kD * 2, 0x00020000);
  const uint32_t lr = lane >> 4, ch = lane & 15;
  const uint32_t v_off = lr * 256u + 16u * (ch ^ (lr << 2));
  auto issue = [&](uint16_t* ks, uint16_t* vs, int j) {
    const uint32_t so = (uint32_t)(start + j * kRows) * 256u;
#pragma unroll
    for (int p = 0; p < kRows / 4; ++p) {
      const uint32_t row = 4 * p + lr;
      attn_lds_load16(kres, ks + 512 * p, row * 256u + 16u * (ch ^ (row & 15)), so);
    }
#pragma unroll
    for (int p = 0; p < kRows / 4; ++p) attn_lds_load16(vres, vs + 512 * p, v_off + 1024u * p, so);
  };
  uint16_t *ks0 = k0[wv], *ks1 = k1[wv], *vs0 = v0[wv], *vs1 = v1[wv];
  if (wv < nblk) issue(ks0, vs0, wv);
  if (wv + kWaves < nblk) issue(ks1, vs1, wv + kWaves);

  const bool has_new = kFused && pos < a.max_len && pos >= start && pos < end;
  if constexpr (kFused) {
    if (!a.rot_tab) {
      if (tid < kD / 2) {
        float sn, cs;
        sincosf(static_cast<float>(pos) * angle, &sn, &cs);
        rot[0][tid] = cs;
        rot[1][tid] = sn;
      }
      lds_sync();
    }
    if (is_q || (ld_k && has_new)) {
      float lo[8], hi[8];
      unpack8(a0, lo);
      unpack8(a1, hi);
      if (a.bias) {
        float x[8], y[8];
        unpack8(b0, x);
        unpack8(b1, y);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          lo[e] = round_bf16(lo[e] + x[e]);
          hi[e] = round_bf16(hi[e] + y[e]);
        }
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float cs = a.rot_tab ? tc[e >> 2][e & 3] : rot[0][8 * c + e];
        const float sn = a.rot_tab ? ts[e >> 2][e & 3] : rot[1][8 * c + e];
        const float x1 = lo[e], x2 = hi[e];
        lo[e] = x1 * cs - x2 * sn;
        hi[e] = x2 * cs + x1 * sn;
      }
      a0 = pack8(lo);
      a1 = pack8(hi);
    } else if (ld_v && has_new && a.bias) {
      float x[8], y[8];
      unpack8(a0, x);
      unpack8(b0, y);
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] += y[e];
      a0 = pack8(x);
    }
  }
  if (is_q) {
    *reinterpret_cast<u32x4_t*>(&qb[tid / 8][8 * c]) = a0;
    *reinterpret_cast<u32x4_t*>(&qb[tid / 8][kD / 2 + 8 * c]) = a1;
  } else if (has_new && ld_k) {
    uint16_t* row = a.kc + ((size_t)g * a.max_len + pos) * kD;
    *reinterpret_cast<u32x4_t*>(&knew[8 * c]) = a0;
    *reinterpret_cast<u32x4_t*>(&knew[kD / 2 + 8 * c]) = a1;
    *reinterpret_cast<u32x4_t*>(row + 8 * c) = a0;
    *reinterpret_cast<u32x4_t*>(row + kD / 2 + 8 * c) = a1;
  } else if (has_new && ld_v) {
    const int cv = tid - nq - 8;
    *reinterpret_cast<u32x4_t*>(&vnew[8 * cv]) = a0;
    *reinterpret_cast<u32x4_t*>(a.vc + ((size_t)g * a.max_len + pos) * kD + 8 * cv) = a0;
  }
  lds_sync();

  // B operand of the scores: lane (head l % 16, grp = l / 16), dims 32 s + 8 grp ..; heads past R: 0
  const int r16 = lane & 15, grp = lane >> 4;
  u32x4_t qf[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const u32x4_t v = *reinterpret_cast<const u32x4_t*>(&qb[min(r16, R - 1)][32 * s + 8 * grp]);
    qf[s] = r16 < R ? v : u32x4_t{0u, 0u, 0u, 0u};
  }
  f32x4_t o[8];
#pragma unroll
  for (int d = 0; d < 8; ++d) o[d] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;  // of head r16
  // transpose-read offset (elements) of value dims 0 .. 15 at rows 4 grp ..: this lane's address is
  // row 4 grp + r16 / 4, dims 4 (r16 % 4) ..; dims 16 d .. are chunk 2 d of the (swizzled) row
  const int vr = r16 >> 2, v_row = (4 * grp + vr) * kD + 4 * (lane & 1);
  auto v_chunk = [&](int d) { return 8 * ((2 * d + ((lane & 3) >> 1)) ^ (vr << 2)); };

  auto compute = [&](uint16_t* ks, uint16_t* vs, int j) {
    const int row0 = start + j * kRows;
    if (has_new && pos >= row0 && pos < row0 + kRows) {  // the token's own row (uniform)
      const int r = pos - row0;
      if (lane < 16) {
        *reinterpret_cast<u32x4_t*>(ks + r * kD + 8 * (lane ^ r)) =
            *reinterpret_cast<const u32x4_t*>(&knew[8 * lane]);
        *reinterpret_cast<u32x4_t*>(vs + r * kD + 8 * (lane ^ ((r & 3) << 2))) =
            *reinterpret_cast<const u32x4_t*>(&vnew[8 * lane]);
      }
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
      asm volatile("" ::: "memory");
    }
    f32x4_t sc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const u32x4_t kf = *reinterpret_cast<const u32x4_t*>(ks + r16 * kD + 8 * ((4 * s + grp) ^ r16));
      sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, kf),
                                                   __builtin_bit_cast(bf16x8_t, qf[s]), sc, 0, 0, 0);
    }
    // head r16, rows 4 grp + r (base-2 logits); a row past the range gets probability 0
    float sr[4], bm = -INFINITY;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      sr[r] = row0 + 4 * grp + r < end ? sc[r] * a.qscale : -INFINITY;
      bm = fmaxf(bm, sr[r]);
    }
    bm = fmaxf(bm, lane_xor16(bm));
    bm = fmaxf(bm, lane_xor32(bm));
    const float mn = fmaxf(m, bm);
    if (__any(mn > m)) {
      // o holds heads 4 grp + r of dim r16: their factors come from lanes 4 grp + r
      const float alpha = exp2f(m - (mn == -INFINITY ? 0.f : mn));
      m = mn;
      l *= alpha;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float f = __shfl(alpha, 4 * grp + r, kWave);
#pragma unroll
        for (int d = 0; d < 8; ++d) o[d][r] *= f;
      }
    }
    const float mz = m == -INFINITY ? 0.f : m;
    float ls = 0.f, ph[4], pl[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float p = exp2f(sr[r] - mz);
      ls += p;
      ph[r] = round_bf16(p);
      pl[r] = p - ph[r];
    }
    ls += lane_xor16(ls);
    ls += lane_xor32(ls);
    l += ls;
    const s16x4_t pah = __builtin_bit_cast(
        s16x4_t, make_uint2(pack_bf16x2_rne(ph[0], ph[1]), pack_bf16x2_rne(ph[2], ph[3])));
    const s16x4_t pal = __builtin_bit_cast(
        s16x4_t, make_uint2(pack_bf16x2_rne(pl[0], pl[1]), pack_bf16x2_rne(pl[2], pl[3])));
#pragma unroll
    for (int d = 0; d < 8; ++d) {
      const s16x4_t vb = __builtin_bit_cast(s16x4_t, lds_read_tr16(vs + v_row + v_chunk(d)));
      o[d] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(pah, vb, o[d], 0, 0, 0);
      o[d] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(pal, vb, o[d], 0, 0, 0);
    }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);  // the stage is read before it is loaded again
    asm volatile("" ::: "memory");
  };

  // A block's 8 loads are followed by at most the 8 of the wave's next block (stores before them only
  // make the wait longer), so vmcnt(8) waits for it; the last block waits for everything.
  auto ready = [&](bool last) {
    if (last)
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    else
      __builtin_amdgcn_s_waitcnt(0x0F78);  // vmcnt(8)
    asm volatile("" ::: "memory");
  };
  for (int j = wv; j < nblk; j += 2 * kWaves) {
    ready(j + kWaves >= nblk);
    compute(ks0, vs0, j);
    if (j + 2 * kWaves < nblk) issue(ks0, vs0, j + 2 * kWaves);
    if (j + kWaves >= nblk) break;
    ready(j + 2 * kWaves >= nblk);
    compute(ks1, vs1, j + kWaves);
    if (j + 3 * kWaves < nblk) issue(ks1, vs1, j + 3 * kWaves);
  }

  // ---- merge of the waves through their (then free) V stages: [head][128] fp32 per wave
  float* ored = reinterpret_cast<float*>(vs0);
#pragma unroll
  for (int d = 0; d < 8; ++d)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (4 * grp + r < kHeads) ored[(4 * grp + r) * kD + 16 * d + r16] = o[d][r];
  if (grp == 0) {
    red_m[wv][r16] = m;
    red_l[wv][r16] = l;
  }
  lds_sync();
  const float* oall = reinterpret_cast<const float*>(&v0[0][0]);
  for (int i = tid; i < R * kD; i += kWaves * kWave) {
    const int hh = i / kD, d = i % kD;
    float mt = red_m[0][hh];
#pragma unroll
    for (int k = 1; k < kWaves; ++k) mt = fmaxf(mt, red_m[k][hh]);
    float ov = 0.f, lt = 0.f;
#pragma unroll
    for (int k = 0; k < kWaves; ++k) {
      const float f = exp2f(red_m[k][hh] - mt);  // 0 for a wave without rows
      ov = fmaf(f, oall[k * (kBlk / 2) + i], ov);
      lt = fmaf(f, red_l[k][hh], lt);
    }
    const size_t h = (size_t)g * R + hh;
    if (nsplit == 1) {
      a.out[h * kD + d] = static_cast<uint16_t>(f32_to_bf16_rne(ov / lt));
    } else {
      a.opart[((size_t)split * a.Hq + h) * kD + d] = ov;
      if (d == 0) *reinterpret_cast<float2*>(&a.ml[((size_t)split * a.Hq + h) * 2]) = make_float2(mt, lt);
    }
  }
}

}  // namespace

// At most one workgroup per CU; never more splits than 128-row pieces of the cache (the workspace).
int attn_long_splits(int Hk, int max_len) {
  int cus = 256;
  if (cached_cu_count(&cus) != hipSuccess || cus <= 0) cus = 256;
  const int pieces = (max_len + kAttnDecodeChunk - 1) / kAttnDecodeChunk;
  return max(1, min(pieces, cus / Hk));
}

void launch_attn_long(bool fused, const void* q, const void* bias, const void* inv_freq, void* k_cache,
                      void* v_cache, const int* pos, void* out, float* opart, float* ml, int Hq, int Hk,
                      int max_len, float qscale, const float* rot, hipStream_t st) {
  const LongArgs a{static_cast<const uint16_t*>(q), static_cast<const uint16_t*>(bias),
                   static_cast<const float*>(inv_freq), rot, static_cast<uint16_t*>(k_cache),
                   static_cast<uint16_t*>(v_cache), pos, static_cast<uint16_t*>(out), opart, ml, Hq, Hk,
                   max_len, qscale};
  const dim3 grid(attn_long_splits(Hk, max_len), Hk), block(kWaves * kWave);
  if (fused)
    hipLaunchKernelGGL(attn_long_kernel<true>, grid, block, 0, st, a);
  else
    hipLaunchKernelGGL(attn_long_kernel<false>, grid, block, 0, st, a);
}

}  // namespace ns
