/*
 * internal_ops.h -- entry points of libnanoserve_amd.so that nanoserve_amd/ops.py calls and the
 * public headers do not declare. Conventions of include/nanoserve_decode.h: caller-allocated device
 * memory, bf16 tensors as void*, asynchronous on `stream`, no allocation, capturable; 0 on
 * success, -2 for rejected arguments (checked before any HIP call), else the hipError_t.
 */
#ifndef NANOSERVE_INTERNAL_OPS_H
#define NANOSERVE_INTERNAL_OPS_H

#include <stddef.h>

#ifdef __cplusplus
extern "C" {
#endif

/*
 * Bias + RoPE + KV-cache append of T prompt tokens at positions pos0 .. pos0 + T - 1 (the
 * reference does these with PyTorch ops and ns_rope, python/nanoserve/qwen.py:119-122, 147-151).
 * qkv [T][Hq + 2 Hk][D]: every element gets bf16_rne(qkv + bias) (bias NULL: no add) and the q
 * and k heads are rotated as by ns_rope. q heads are updated in place; with k_cache / v_cache
 * [Hk][max_len][D] the k and v heads go to rows pos0 .. of the caches (qkv keeps their old
 * values), without them (both NULL) they are updated in place.
 * -2 for D % 16 != 0, D > 512, sizes <= 0, pos0 < 0, one cache without the other, rows past
 * max_len, NULL or misaligned pointers (qkv, bias and the caches 16-byte aligned).
 */
int ns_prompt_qkv(void* qkv, const void* bias, const void* inv_freq, void* k_cache,
                  void* v_cache, int T, int Hq, int Hk, int D, int pos0, int max_len,
                  void* stream);

/*
 * 1 if ns_prompt_attention takes these sizes with keys kv_stride elements apart (its size limits: keys
 * whose rows reach 2 GiB and more than 65535 tiles of 128 query rows per kv head are refused), else 0.
 */
int ns_prompt_attention_fits(int T, int Hq, int Hk, int pos0, long long kv_stride);

/*
 * Bytes of workspace ns_prompt_attention uses for these sizes (fp32 partials of the splits over
 * the keys); 0 when the queries alone fill the GPU and nothing is split, or for invalid sizes.
 */
size_t ns_prompt_attention_workspace(int T, int Hq, int Hk, int pos0);

/*
 * Causal grouped-query attention of T prompt tokens at positions pos0 .. pos0 + T - 1 (the
 * reference uses PyTorch SDPA, python/nanoserve/qwen.py:124-133). Query t attends over keys
 * 0 .. pos0 + t. q: token stride q_stride, heads [Hq][128] contiguous; k, v: key j of kv head g
 * at g * kv_head_stride + j * kv_stride (strides in elements), 128 values each; out
 * [T][Hq * 128] bf16. Products of the bf16 operands and all sums in fp32, softmax in fp32; the
 * probabilities enter the second product with all 24 bits of fp32 (three bf16 terms) for pos0 > 0
 * and with 16 (two terms) for pos0 == 0.
 * -2 where ns_prompt_attention_fits is 0, for strides that are not a multiple of 8, NULL or pointers that are not 16-byte aligned, work_bytes too small.
 */
int ns_prompt_attention(const void* q, long long q_stride, const void* k, const void* v,
                        long long kv_stride, long long kv_head_stride, void* out, void* work,
                        size_t work_bytes, int T, int Hq, int Hk, int pos0, void* stream);

/*
 * ns_w4_linear for any M >= 1: above 8 rows the prefill GEMM on M rows as they are (ns_w4_linear takes
 * multiples of 128, and the reference's wrapper pads to them, python/nanoserve/ops.py:88-91). The
 * other conditions and return codes are ns_w4_linear's.
 */
int ns_w4_linear_rows(const void* X, const void* Wq, const void* S, void* Y, int M, int N, int K,
                      int G, void* stream);

/*
 * ns_w4_linear_swiglu for any M >= 1: above 8 rows the GEMM with the SwiGLU epilogue on M rows as
 * they are; M = 2..8 the decode GEMV with SwiGLU in its output where G == 128 and K % 256 == 0
 * up to 20480, and elsewhere ns_w4_linear into `tmp` [M][N] bf16 followed by the activation
 * (g and u rounded to bf16 first in either form). tmp: the workspace function's bytes, 16-byte
 * aligned, or NULL where those are 0. M = 2..8 need Y 16-byte aligned. The other conditions and return
 * codes are ns_w4_linear_swiglu's.
 */
size_t ns_w4_linear_swiglu_rows_workspace(int M, int N, int K, int G);
int ns_w4_linear_swiglu_rows(const void* X, const void* Wq, const void* S, void* Y, void* tmp,
                             size_t tmp_bytes, int M, int N, int K, int G, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* NANOSERVE_INTERNAL_OPS_H */
