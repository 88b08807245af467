/*
 * a81w41_dense.h -- parity hooks of liba81w41_dense.so: the mechanisms of the models with dense weights on their own.
 * Device pointers, enqueued on `stream`; element type bf16 != 0: bfloat16, else float.  For tests and measurements.
 */
#ifndef A81W41_DENSE_H
#define A81W41_DENSE_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* C = A W^T: A [M][lda], W [N][ldw] elements, C [M][ldc] floats.  lda, ldw: at least K rounded up to 128 bytes, whole
 * multiples of 128 bytes; the columns of W beyond K are zero, those of A finite. */
int a81w41_dense_gemm(const void *A, int lda, const void *W, int ldw, float *C, int ldc, int M, int N, int K, int bf16, void *stream);
/* The same product with gated units: rows of W come as 16 gates, then their 16 ups, and so on (N a multiple of 32), and C [M][ldc >= N / 2]
 * holds elements g / (1 + exp(-slope g)) (u + shift) of g = min(gate, limit), u = clamp(up, -limit, limit). */
int a81w41_dense_gated(const void *A, int lda, const void *W, int ldw, void *C, int ldc, int M, int N, int K, float limit, float slope,
                       float shift, int bf16, void *stream);
/* Attention in latent space.  q [M heads][ld], cache [max_seq][ld] with rows [latent (rank) | rotated part (rot)] and zeros
 * up to ld (a multiple of 128 bytes); token m sees cache rows 0 .. pos + m.  out [M heads][rank] elements.
 * variant 0: the vector kernel; 1: matrix cores (bfloat16 only), the keys dealt to `splits` (1 .. 64) workgroups, with
 * part [splits M heads][rank rounded up to 4] and stats [splits M heads][2] floats as scratch. */
int a81w41_latent_attention(const void *q, const void *cache, int ld, int rank, int rot, int heads, const int *pos_dev, int max_seq, int M,
                            float scale, void *out, int bf16, int variant, int splits, float *part, float *stats, void *stream);
/* The same for one token over a short context, bfloat16, with the product behind it in the same launch: q [heads][ld] with zeros past
 * rank + rot, uv [heads vdim][ld_uv] (ld_uv a multiple of 8, zeros past rank), gates [heads] floats (before the sigmoid), out [heads vdim]
 * floats.  rank: a multiple of 8, at most 512; rot: 1 .. 64. */
int a81w41_latent_token(const void *q, const void *cache, int ld, int rank, int rot, int heads, int vdim, const int *pos_dev, int max_seq,
                        float scale, const void *uv, int ld_uv, const float *gates, float *out, void *stream);
/* Attention on formed keys and values, bfloat16.  q [M][heads][dim + rot], k [max_seq][heads dim] and k_rot
 * [max_seq][ld_rot] (first rot columns), v_t [heads vdim][ld_v] transposed with ld_v a multiple of 64, at least max_seq;
 * gates [M][heads] floats (before the sigmoid), out [M][heads vdim].  dim, rot, ld_rot: multiples of 8. */
int a81w41_formed_attention(const void *q, const void *k, const void *k_rot, int ld_rot, const void *v_t, int ld_v, const float *gates,
                            int heads, int dim, int rot, int vdim, const int *pos_dev, int max_seq, int M, float scale, void *out,
                            void *stream);
/* Grouped attention.  q [M][heads][key_width], cache rows [max_seq][ld] with [value (value_width) | key (key_width)] for each of
 * kv_heads; query head h reads kv head h / (heads / kv_heads).  Token m sees the rows 0 .. pos + m, with chunk > 0 those from
 * the first position of its own chunk on; sink: a further key of score 0 without a value.  Widths are multiples of 8, the
 * first vdim value columns count; out [M][heads][vdim] elements.  variant, splits, part, stats: as above, with
 * splits M heads rows of scratch, vdim rounded up to 4. */
int a81w41_grouped_attention(const void *q, const void *rows, int ld, int heads, int kv_heads, int key_width, int value_width, int vdim,
                             const int *pos_dev, int max_seq, int M, float scale, int chunk, int sink, void *out, int bf16, int variant,
                             int splits, float *part, float *stats, void *stream);
/* A matrix memory over M tokens at positions *pos_dev .. of a sequence.  in [M][ld_in] floats, columns [q | k | v | output gate |
 * input gate | forget gate] of all heads; q is scaled by dim^-1/2 here.  state: a81w41_matrix_memory_state() floats, zero at
 * position 0; scratch: a81w41_matrix_memory_scratch() floats; all 16-byte aligned.  out [M][heads vdim]: per head divided by its
 * root mean square, times norm, times the sigmoid of the output gate.  variant 0: token by token; 1: in chunks. */
size_t a81w41_matrix_memory_state(int heads, int dim, int vdim);
size_t a81w41_matrix_memory_scratch(int heads, int dim, int vdim, int M);
int a81w41_matrix_memory(const float *in, int ld_in, int M, int heads, int dim, int vdim, float cap, float eps, const float *bias_i,
                         const float *bias_f, const float *norm, float *state, const int *pos_dev, int variant, float *scratch, float *out,
                         void *stream);
/* chosen [M][top]: the largest of logits [M][ld] (first `experts` columns) + bias, largest first; weights [M][top]: the softmax
 * over them. */
int a81w41_router(const float *logits, int ld, const float *bias, int experts, int top, int M, int *chosen, float *weights, void *stream);
/* Test hook, host only: the kernel that a81w41_dense_gemm or _gated takes: tiles of 0: 256 x 256, 1: 128 x 256, 2: 128 x 128, 3: 64 x 128, 64 x 64 with
 * 4: four stages of K, 5: two, 6: 64 x 32; 7: 128 x 128 for strides past 32-bit offsets. */
int a81w41_dense_form_selfcheck(int M, int N, int K, int lda, int ldw, int bf16);
/* Test hook, host only: what a one-token pass reads ahead of a matrix [rows][ld] within `room` bytes (gate_up: of `rows` units, sixteen
 * rows of gate and sixteen of up in turn).  Returns the bytes, *extent: how far into the matrix they reach. */
long long a81w41_dense_ahead_selfcheck(int rows, int ld, int gate_up, long long room, int bf16, long long *extent);

#ifdef __cplusplus
}
#endif
#endif /* A81W41_DENSE_H */
