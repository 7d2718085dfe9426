/*
 * ecf8_head.h -- C ABI of the ends of a decode step in libecf8.so: the bf16
 * linear of a few rows (vocabulary head, modulation Linears), the greedy
 * next token and its embedding.  No reference counterpart: the reference
 * runs transformers' generate around its hooks (scripts/inference_llm.py:
 * 108-142).
 *
 * Conventions as in ecf8.h: device pointers, stream as void*, ECF8_*
 * status, asynchronous, no allocation.  Deterministic.
 */
#ifndef ECF8_HEAD_H
#define ECF8_HEAD_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* out[m, n] (bf16, row stride ldo) = sum_k x[m, k] w[n, k] + bias[n] for 1
 * <= M <= 16 rows: x bf16 (row stride ldx, a multiple of 8), w bf16 [N, K],
 * bias bf16 [N] or NULL, fp32 sums.  K a multiple of 32 up to 4096, N a
 * multiple of 16. */
int ecf8_bf16_linear16(const void *x, int64_t ldx, int64_t M, int64_t K, const void *w, int64_t N,
                       const void *bias, void *out, int64_t ldo, void *stream);

/* Bytes of ecf8_greedy_emit's work buffer. */
#define ECF8_GREEDY_CHUNKS 64
int64_t ecf8_greedy_work_bytes(int64_t B);

/* The index of the largest of each row's V logits (bf16, row stride ld; NaN
 * counts as largest, ties go to the lower index) ->
 * next_token int64 [B] and tokens[b, step[0]] (int64, row stride ld_tokens;
 * skipped past it); then step[0] += 1 and pos[0] += advance (pos may be NULL
 * when advance is 0).  Two launches. */
int ecf8_greedy_emit(const void *logits, int64_t ld, int64_t B, int64_t V, void *work,
                     int64_t work_bytes, int64_t *tokens, int64_t ld_tokens, int64_t *next_token,
                     int64_t *step, int *pos, int advance, void *stream);

/* ecf8_greedy_emit; a step outside the token buffer also sets refused[0]
 * (memory that the device can write, e.g. pinned host memory). */
int ecf8_greedy_emit_checked(const void *logits, int64_t ld, int64_t B, int64_t V, void *work,
                             int64_t work_bytes, int64_t *tokens, int64_t ld_tokens,
                             int64_t *next_token, int64_t *step, int *pos, int advance,
                             int *refused, void *stream);

/* out fp32 [B, H] = rows token[b] of table bf16 [V, H] (zeros for a token
 * outside the table); H a multiple of 8. */
int ecf8_embed_rows(const int64_t *token, int64_t B, const void *table, int64_t V, int64_t H,
                    float *out, void *stream);

/* ecf8_embed_rows; a token outside the table also sets refused[0]. */
int ecf8_embed_rows_checked(const int64_t *token, int64_t B, const void *table, int64_t V,
                            int64_t H, float *out, int *refused, void *stream);

#ifdef __cplusplus
}
#endif

#endif /* ECF8_HEAD_H */
