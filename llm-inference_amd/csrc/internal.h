// Functions shared between the kernel and step translation units (not part of the C ABI).
#pragma once

#include "llm_amd/kernels.h"

// embedding_forward that checks the token against the vocabulary on the device: a token
// outside [0, vocab) sets *err and leaves `out` unchanged.
void embedding_checked(bf16 *out, const bf16 *table, const int *d_token, int hidden, int vocab,
                       int *err, hipStream_t stream);

// Two-stage argmax into *out using caller-owned partials of argmax_partial_count() entries.
void argmax_launch(int *out, const bf16 *x, int n, float *pv, int *pi, hipStream_t stream);
int argmax_partial_count();

// sample_forward for a decode step: the draw goes to *out and, with *err, to the two words at mail
// (host memory the device can write). slot: sample_slot_bytes() bytes, zero before the first call, used
// by one call at a time.
bool sample_step(int *out, const bf16 *x, int n, float inv_temp, float u, void *slot, int *mail,
                 const int *err, hipStream_t stream);
size_t sample_slot_bytes();
// sample_forward draws from a row of n in one launch.
bool sample_takes_one_launch(int n);
// For tests: out[i] = exp_f32 (branches: the form with early returns) of the float with the bits
// first + i, i < n.
extern "C" void llm_exp_bits(float *out, unsigned first, unsigned n, int branches, hipStream_t stream);
// For tests, with no draw in flight: how many of the library's slots for sample_forward are taken (-1
// after an error); then, with set 1 or 0, all are taken or free.
extern "C" int llm_sample_slots(int set);

// inv_freq_j = 1 / fp32(pow(theta, fp32(2j / D))) for j < D/2 (D <= 256), cached per (theta, D).
void rope_inv_freq_table(float theta, int D, float *out);

// qk_norm_rope_attention_one_pass, reporting whether it launched.
bool attention_one_pass_launch(bf16 *out, const bf16 *q, const bf16 *k, const bf16 *v,
                               const bf16 *q_norm_w, const bf16 *k_norm_w, bf16 *key_cache,
                               bf16 *value_cache, void *ws, int *err, const int *d_pos,
                               int n_heads, int n_kv_heads, int head_dim, float eps, float theta,
                               int max_seq, float scale, hipStream_t stream);

// attention_forward, reporting whether it launched; err: the step's device error flag (set to 1 for
// a position outside the cache), or NULL.
bool attention_launch(bf16 *out, const bf16 *q, const bf16 *key_cache, const bf16 *value_cache,
                      float *att, int n_heads, int n_kv_heads, int head_dim, const int *d_pos,
                      int max_seq, float scale, hipStream_t stream, int *err = nullptr);

// qk_norm_rope_attention_forward, reporting whether it launched; with rope_table (the
// rope_table_launch output at *d_pos), the kernel reads the RoPE table instead of computing it;
// err as for attention_launch.
bool qk_norm_rope_attention_launch(bf16 *out, const bf16 *q, const bf16 *k, const bf16 *v,
                                   const bf16 *q_norm_w, const bf16 *k_norm_w, bf16 *key_cache,
                                   bf16 *value_cache, float *att, const int *d_pos, int n_heads,
                                   int n_kv_heads, int head_dim, float eps, float theta,
                                   int max_seq, float scale, hipStream_t stream,
                                   const float *rope_table = nullptr, int *err = nullptr);

// The RoPE table at *d_pos into table[0, head_dim): cos then sin of the head_dim / 2 rotation
// pairs, the values rope_table computes in the kernels (one launch serves every layer).
bool rope_table_launch(float *table, const int *d_pos, int head_dim, float theta,
                       hipStream_t stream);
