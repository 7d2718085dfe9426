/*
 * ecf8_attn.h -- C ABI of the many-query attention kernels in libecf8.so:
 * the causal attention of a prompt over the KV caches, and the operand
 * preparation and attention of the DiT's blocks.
 *
 * None of these replaces a reference interface: the reference runs
 * transformers' and DiffSynth's attention over its decoded weights
 * (dfloat/run/run.py:84-155 hooks the Linears around it).
 *
 * Conventions as in ecf8.h: device pointers, stream as void*, ECF8_*
 * status, asynchronous, no allocation.  bf16 tensors are passed as void*
 * (2-byte elements).  Head dimension 128.  Deterministic.
 */
#ifndef ECF8_ATTN_H
#define ECF8_ATTN_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Elements of each packed buffer (keys, values) for B x Hkv heads of T
 * tokens; the tokens of a head are padded to a multiple of 64. */
int64_t ecf8_packed_kv_elements(int64_t B, int Hkv, int64_t T);

/*
 * Causal attention of a prompt: query t of q bf16 [B, Hq, T, 128] (scores
 * scaled by 1/sqrt(128)) over positions [0, t] of the caches bf16 [B, Hkv,
 * Lmax, 128], Hq a multiple of Hkv.  Scores, softmax and both products in
 * fp32 on bf16 inputs (probabilities keep 24 bits).  out bf16 [B * T, Hq *
 * 128].  k_packed / v_packed: work buffers of ecf8_packed_kv_elements
 * bf16 elements each.  Two launches.
 */
int ecf8_prompt_attention(const void *q, const void *k_cache, const void *v_cache, int64_t B,
                          int Hq, int Hkv, int64_t T, int64_t Lmax, void *k_packed,
                          void *v_packed, void *out, void *stream);

#ifdef __cplusplus
}
#endif

#endif /* ECF8_ATTN_H */
