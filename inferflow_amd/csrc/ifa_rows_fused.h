// ifa_rows_fused.h -- the second half of a single-token layer as one launch (ifa_rows_fused.hip) and the attention that feeds it
#pragma once
#include "ifa_host.h"
#include "ifa_f32_common.h"
#include "inferflow_amd.h"

// x[n] += ls1[n] (s0 W0[n] . a0 + s1 W1[n] . a1) + ls2[n] (W2[n] . a2 + bias2[n]) for ONE row; k0 / k1 / k2 columns, multiples of 8 (0: that part is missing):
//   a0  attention: a finished row (nsplit 1) or the shares of nsplit workgroups per head ([heads][nsplit][maximum, sum, vdim values], joined here with the sink)
//   a1  o / rms_group(o) * norm_w[c % wlen] * act(gate), act 0 sigmoid, 1 silu
//   a2  gelu_tanh(gate_up[c]) * gate_up[k2 + c]
struct IfaRowOut {
    int N; float *x;
    const ifa32::bf16_t *w0, *w1, *w2; int k0, k1, k2;
    float s0, s1; const ifa32::bf16_t *ls1, *ls2, *bias2;
    const float *a0; int nsplit, vdim; const ifa32::bf16_t *sink;
    const float *o, *gate; const ifa32::bf16_t *norm_w; int group, wlen, gate_act; float eps;
    const float *gate_up;
};
constexpr int IFA_ROW_OUT_SPLITS = 8;
// what ifa_row_out takes: sizes, alignment
bool ifa_row_out_fits(const IfaRowOut &P);
int ifa_row_out(const IfaRowOut &P, ifa_stream stream);

// ifa_argmax_rows_f32, one row in two launches (csrc/ifa_ops_f32.hip; ws of ifa_argmax_parts_bytes); step: a decode step's row, whose token becomes the next step's: tokens[0], ring[pos]
// (modulo its size), position and the sequence's place one further on
struct IfaStepAdvance { int *tokens, *pos; ifa_seq_desc *seqs; int *ring; int ring_size; };
extern "C" size_t ifa_argmax_parts_bytes();
extern "C" int ifa_argmax_parts_f32(const float *logits, size_t n, size_t row_stride, size_t rows, const int *excluded_dev, int *out_dev, void *ws, const IfaStepAdvance *step, ifa_stream stream);

// the mixers of a WINDOW_LINEAR layer for ONE row: ifa_kv_store_f32 (keys normed, values the keys as projected) + ifa_attention_window_f32 + the decayed linear
// attention of ifa_state_scan_f32.  *nsplit workgroups per head share the keys and nobody joins their shares (in ws; at most IFA_ROW_OUT_SPLITS; 1: out holds the row)
struct IfaMixRow {
    const float *q, *k; int heads, kv_heads, dim; float eps, scale, softcap; int window, keep_first, max_keys;
    const ifa32::bf16_t *rel; const int *bucket_of; int n_buckets; const ifa32::bf16_t *sink;
    const ifa_seq_desc *seqs; const int *row_seq; void *const *slot_base; size_t k_off, v_off;
    float *out, *ws; size_t ws_bytes;
    const float *lq, *lk, *lv, *decay; int l_heads, l_dim, l_vdim; size_t l_off; float *lin_out;
};
bool ifa_mix_row_fits(const IfaMixRow &M);
int ifa_mix_row(const IfaMixRow &M, int *nsplit, ifa_stream stream);

// GATED_DELTA layers, ONE row per sequence: ifa_shortconv_silu_f32 + ifa_shortconv_tail_f32 + ifa_delta_gates_f32 in one launch (csrc/ifa_seqmix.hip)
int ifa_delta_row_prep(const float *x, size_t ldx, int channels, int taps, const ifa32::bf16_t *w, const ifa_seq_desc *seqs, const int *row_seq, size_t rows, void *const *slot_base,
                       size_t state_off, int norm_cols, int group_dim, float l2_eps, int scale_cols, float scale, float *y, size_t ldy, const float *b, const float *a, int heads,
                       const ifa32::bf16_t *a_log, const ifa32::bf16_t *dt_bias, float *beta, float *decay, ifa_stream stream);

// grouped products over bfloat16 rows (csrc/ifa_linear_bf16.hip): see ifa_linear_bf16w_grouped.  glu_bf16 not null: the matrices' rows are gate | up (rows / 2 each) and only
// act(gate) up is left, in bfloat16 rows of ldc (whole 64s, zero beyond rows / 2)
int ifa_linear_bf16_grouped(const void *w_bf16, size_t rows, size_t cols, const void *a_bf16, size_t lda, const int *a_rows_dev, const int *tile_map_dev, const int *n_tiles_dev,
                            size_t max_tiles, int tile_rows, const void *row_scale_f32, void *c_f32, size_t ldc, int glu_kind, float glu_limit, void *glu_bf16, ifa_stream stream);
// ifa_linear_bf16_both whose output columns [glu_col0, glu_col0 + 2 glu_cols) are gate | up of a gated feed-forward: glu_bf16[t][c] = act(gate[c]) up[c] in bfloat16 rows of ldg
// (whole 64s, zero beyond glu_cols) in their place; the columns before them as ever, any behind them not at all
extern "C" int ifa_linear_bf16_glu(const void *w_bf16, size_t rows, size_t cols, const void *a_bf16, size_t lda, size_t tokens, const void *bias_bf16, void *c_f32, size_t ldc, int silu_col0,
                        int silu_col1, size_t glu_col0, size_t glu_cols, int glu_kind, float glu_limit, void *glu_bf16, size_t ldg, ifa_stream stream);
// At most eight rows of 32-bit activations.  ifa_linear_bf16w whose columns [glu_col0, glu_col0 + 2 glu_cols) are gate | up: g_f32[t][c] = act(gate[c]) up[c] in their place (false: sizes or
// alignment don't allow it, nothing launched); and a product whose row t is multiplied by sigmoid(row_gate[t * ld_gate])
extern "C" bool ifa_linear_bf16w_glu_rows(const void *w_bf16, size_t rows, size_t cols, const void *a_f32, size_t lda, size_t tokens, const void *bias_bf16, void *c_f32, size_t ldc, int silu_col0,
                               int silu_col1, size_t glu_col0, size_t glu_cols, int glu_kind, float glu_limit, void *g_f32, size_t ldg, ifa_stream stream);
extern "C" int ifa_linear_bf16w_gated_rows(const void *w_bf16, size_t rows, size_t cols, const void *a_f32, size_t lda, size_t tokens, const void *row_gate_f32, size_t ld_gate, int accumulate, void *c_f32,
                                size_t ldc, ifa_stream stream);
// C[t][n] += sum over the parts of alpha mul[n] (W[n] . a[t] + bias[n]): a_bf16's rows hold the parts' operands side by side, each zero-padded to whole 64s (lda: their sum);
// cols: a multiple of 8, 64 and more
constexpr int IFA_SUM_PARTS = 3;
struct IfaSumPart { const void *w; size_t cols; const void *mul, *bias; float alpha; };
extern "C" int ifa_linear_bf16_sum(const IfaSumPart *parts, int n_parts, size_t rows, const void *a_bf16, size_t lda, size_t tokens, void *c_f32, size_t ldc, ifa_stream stream);
// ... with K shared out where that leaves less of the chip idle: the count of planes [tokens][rows] of further summands of C that the second writes (planes null: none, all of them in C)
// and the caller adds, in order, where it next reads C (ifa_layernorm_planes_to_bf16, ifa_add_planes_f32)
constexpr int IFA_SUM_PLANES = 7;
extern "C" int ifa_linear_bf16_sum_plane_count(size_t rows, size_t lda, size_t tokens);
extern "C" int ifa_linear_bf16_sum_planes(const IfaSumPart *parts, int n_parts, size_t rows, const void *a_bf16, size_t lda, size_t tokens, void *c_f32, size_t ldc, float *planes, ifa_stream stream);
extern "C" int ifa_add_planes_f32(float *x_f32, const float *planes, int n_planes, size_t rows, size_t cols, ifa_stream stream);      // rows and planes dense
// ifa_rows_to_bf16 into the first `width` columns (a multiple of 8) of rows of ldy
int ifa_rows_to_bf16_part(const void *x_f32, size_t ldx, size_t rows, size_t cols, void *y_bf16, size_t width, size_t ldy, ifa_stream stream);
// Producers that leave what only products read in bfloat16: rows of ldy, zero from the last column up to `width` (both multiples of 8).  The norms: false where the sizes or the
// alignment don't allow it (nothing launched).
// ifa_layernorm_f32
bool ifa_layernorm_to_bf16(int kind, const void *x_f32, size_t ldx, size_t rows, size_t cols, const void *w_bf16, float eps, void *y_bf16, size_t width, size_t ldy, ifa_stream stream);
// ... of x (dense rows) + planes, which x takes up
extern "C" bool ifa_layernorm_planes_to_bf16(int kind, void *x_f32, const float *planes, int n_planes, size_t rows, size_t cols, const void *w_bf16, float eps, void *y_bf16, size_t width, size_t ldy,
                                  ifa_stream stream);
// ifa_gated_groupnorm_f32 (w as long as a group or as the row)
bool ifa_gated_groupnorm_to_bf16(const void *o_f32, size_t ldo, size_t rows, int channels, int group, const void *w_bf16, int wlen, const void *gate_f32, size_t ldg, int gate_act,
                                 float eps, void *y_bf16, size_t width, size_t ldy, ifa_stream stream);
// What a step brings to an attention's cache: keys and values as projected (k null: the layer reads rows that are there already).  norm: the keys by their root mean square (with norm_w or
// without); rot_dims of them turned by pos * freq; turn_q: the queries (in place) like them, with q_norm_w.  As ifa_kv_store_f32 / ifa_qk_rope_store_f32, which these launches stand for
struct IfaFreshKV { const float *k; size_t ldk; const float *v; size_t ldv; int norm; const ifa32::bf16_t *norm_w; float eps; int rot_dims; const double *freq; int turn_q; const ifa32::bf16_t *q_norm_w; };
// The decayed linear attention of the same rows and slots (ifa_state_chunked_f32 of kind 0, its sizes): in the windowed attention's launches where *side_done says so
struct IfaLinearSide { const float *q, *k, *v; size_t ldq, ldk, ldv; int heads, dk, dv; const float *decay; size_t state_off; void *ws; size_t ws_bytes; float *out; size_t ldo; };
// ifa_kv_store_f32 / ifa_qk_rope_store_f32, then ifa_attention_window_f32 / ifa_attention_kv_f32: *left16 tells whether the output is in out_bf16 (rows of ld16, heads * vdim columns) or, where the step's form writes 32 bits, in out_f32
extern "C" int ifa_attention_window_to_bf16(const void *q_f32, size_t ldq, int heads, int kv_heads, int dim, int norm_q, float eps, float scale, float softcap, int window, int keep_first,
                                 const void *rel_bf16, const int *bucket_of_dev, int n_buckets, const void *sink_bf16, const void *seqs_dev, const int *row_seq_dev, size_t rows,
                                 void *const *slot_base_dev, size_t k_off, size_t v_off, void *out_f32, size_t ldo, void *out_bf16, size_t ld16, bool *left16, const void *seqs_host,
                                 int n_seqs, int tile_min_rows, void *ws_f32, size_t ws_bytes, const IfaFreshKV &fresh, const IfaLinearSide *side, bool *side_done, ifa_stream stream);
extern "C" int ifa_attention_kv_to_bf16(const void *q_f32, size_t ldq, int heads, int kv_heads, int dim, int vdim, float scale, int window, int keep_first, int sink, float sink_score,
                             const void *seqs_dev, const int *row_seq_dev, size_t rows, void *const *slot_base_dev, size_t k_off, size_t v_off, void *out_f32, size_t ldo,
                             void *out_bf16, size_t ld16, bool *left16, const void *seqs_host, int n_seqs, int tile_min_rows, int max_keys, void *ws_f32, size_t ws_bytes,
                             const IfaFreshKV &fresh, ifa_stream stream);
// ifa_moe_experts_gated_f32 of more than eight rows that a norm has left in bfloat16 (rows of `width`), where the first tells that the experts' products read them so
bool ifa_moe_gated_reads_bf16(size_t rows, int width, int ff, int top, int ops32, const void *gate_up_bf16, const void *down_bf16);
int ifa_moe_experts_gated_bf16(const void *h_bf16, size_t rows, int width, int ff, int experts, int top, const void *gate_up_bf16, const void *down_bf16, const int *idx_dev,
                               const void *wgt_f32, void *ws, size_t ws_bytes, void *y_f32, size_t ldy, int accumulate, ifa_stream stream);
// Prompts: choice by the largest logits, experts over bfloat16 rows (ifa_moe_gated_reads_bf16) without the sum of a row's pairs, and beside them the activations of a shared expert (sh_ff > 0):
// sh_act[t] = silu(gate) up [* sigmoid(sh_gate[t * sh_ldg])] in bfloat16 rows of sh_ldo.  pair_pos [rows][top], pair_rows [pairs][width] (in ws): what ifa_norm_add_norm_moe adds up
struct IfaMoePrompt {
    const float *logits; size_t ldl, rows; int width, ff, experts, top; const ifa32::bf16_t *gate_up, *down, *h16; int *idx; float *wgt; void *ws; size_t ws_bytes;
    const float *sh_gate_up; size_t sh_ld; int sh_ff; const float *sh_gate; size_t sh_ldg; ifa32::bf16_t *sh_act; size_t sh_ldo;
};
extern "C" int ifa_moe_prompt(const IfaMoePrompt &P, const int **pair_pos, const float **pair_rows, ifa_stream stream);
// ifa_norm_add_norm_f32 of the row m[t] + m2[t] (rows of ldm; false: sizes or alignment don't allow it, nothing launched)
extern "C" bool ifa_norm_add_two_norm_f32(void *x_f32, size_t ldx, size_t rows, size_t cols, const void *m_f32, const void *m2_f32, size_t ldm, const void *w_after_bf16, const void *w_before_bf16,
                              float w_offset, float eps, void *h_f32, size_t ldh, ifa_stream stream);
// ifa_norm_add_norm_f32 / _to_bf16 (h_f32 or h_bf16) of the row  sum_k pair_rows[pair_pos[t][k]] (+ m[t])
extern "C" int ifa_norm_add_norm_moe(void *x_f32, size_t ldx, size_t rows, size_t cols, const void *m_f32, size_t ldm, const int *pair_pos_dev, const void *pair_rows_f32, int top,
                          const void *w_after_bf16, const void *w_before_bf16, float w_offset, float eps, void *h_f32, void *h_bf16, size_t ldh, ifa_stream stream);
// ifa_moe_route_top_f32 inside the first launch of ifa_moe_experts_gated_f32: at most eight rows, 256 experts.  shared: the shared expert's output product beside the experts' in their launch,
// out[t] = sigmoid(gate[t * ldg]) down . act[t] (ifa_linear_bf16w_gated_rows; rows that ifa_moe_shared_fits allows)
struct IfaMoeShared { const ifa32::bf16_t *down; const float *act; size_t lda; int ff; const float *gate; size_t ldg; float *out; size_t ldo; };
extern "C" bool ifa_moe_shared_fits(const IfaMoeShared &S);
extern "C" bool ifa_moe_shared_pays(size_t rows, size_t width, size_t ff);          // ... and in which the one launch is no slower than two
extern "C" int ifa_moe_experts_gated_top_rows_shared(const void *logits_f32, size_t ldl, const void *h_f32, size_t ldh, size_t rows, int width, int ff, int experts, int top, const void *gate_up_bf16,
                                          const void *down_bf16, int *idx_dev, void *wgt_f32, void *ws, size_t ws_bytes, void *y_f32, size_t ldy, int accumulate, const IfaMoeShared *shared,
                                          ifa_stream stream);
// ifa_glu_ex_f32 whose output only products read: bfloat16 rows, zero up to ldo (a multiple of 8; csrc/ifa_ops_f32.hip)
int ifa_glu_to_bf16(int kind, float limit, const void *gate_up_f32, size_t ld, size_t rows, size_t cols, const void *row_gate_f32, size_t ldg, void *out_bf16, size_t ldo,
                    ifa_stream stream);
