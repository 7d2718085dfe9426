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

/* One token stream of a DiT block's joint attention: the projection output
 * bf16, row t of batch b at qkv + b * batch_stride + t * row_stride elements
 * (H q heads, H k heads, H v heads of 128), and the head norms' bf16
 * weights [128]. */
typedef struct ecf8_dit_stream {
  const void *qkv;
  const void *q_norm;
  const void *k_norm;
  int64_t tokens;
  int64_t row_stride;
  int64_t batch_stride;
} ecf8_dit_stream;

/*
 * Operands of a DiT block's attention over the T tokens of one or two
 * streams, in that order: q and k heads through RMSNorm (fp32, bf16
 * weights) and the rotary embedding of interleaved pairs (cos_t / sin_t fp32
 * [T, 64]); q times `scale` -> q bf16 [B, H, T, 128]; k and v -> packed
 * buffers of ecf8_packed_kv_elements(B, H, T) bf16 elements each.
 */
int ecf8_dit_qkv(const ecf8_dit_stream *streams, int n_streams, int64_t B, int H, float eps,
                 float scale, const float *cos_t, const float *sin_t, void *q, void *k_packed,
                 void *v_packed, void *stream);

/*
 * Attention of q bf16 [B, H, T, 128] (scaled by log2(e) / sqrt(128): a
 * probability is a power of two of its score) over packed keys and values
 * of the same T tokens: fp32 scores and softmax, bf16 probabilities, fp32
 * sums; row t of batch b goes to out (bf16) +
 * (b * T + t) * out_stride, head h at column 128 h.
 */
int ecf8_packed_attention(const void *q, const void *k_packed, const void *v_packed, int64_t B,
                          int H, int64_t T, void *out, int64_t out_stride, void *stream);

/* out bf16 [B, rows, C] = LayerNorm(x) * (1 + scale) + shift in fp32, x bf16
 * [B, rows, C], shift / scale bf16 [C] of batch b at b * *_batch elements.
 * C a multiple of 8, at most 8192. */
int ecf8_dit_modulate(const void *x, int64_t B, int64_t rows, int64_t C, const void *shift,
                      int64_t shift_batch, const void *scale, int64_t scale_batch, float eps,
                      void *out, void *stream);

/* out bf16 [B, rows, C] = x + gate * y, the product rounded to bf16 before
 * the sum; gate bf16 [C] of batch b at b * gate_batch elements. */
int ecf8_dit_gated_add(const void *x, const void *gate, int64_t gate_batch, const void *y,
                       int64_t B, int64_t rows, int64_t C, void *out, void *stream);

/* out[m, :C] = GELU (tanh form, fp32) of x[m, :C], bf16, with row strides in
 * elements. */
int ecf8_dit_gelu(const void *x, int64_t x_row, int64_t rows, int64_t C, void *out,
                  int64_t out_row, void *stream);

#ifdef __cplusplus
}
#endif

#endif /* ECF8_ATTN_H */
