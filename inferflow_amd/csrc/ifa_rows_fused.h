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
int ifa_linear_bf16_glu(const void *w_bf16, size_t rows, size_t cols, const void *a_bf16, size_t lda, size_t tokens, const void *bias_bf16, void *c_f32, size_t ldc, int silu_col0,
                        int silu_col1, size_t glu_col0, size_t glu_cols, int glu_kind, float glu_limit, void *glu_bf16, size_t ldg, ifa_stream stream);
// ifa_glu_ex_f32 whose output only products read: bfloat16 rows, zero up to ldo (a multiple of 8; csrc/ifa_ops_f32.hip)
int ifa_glu_to_bf16(int kind, float limit, const void *gate_up_f32, size_t ld, size_t rows, size_t cols, const void *row_gate_f32, size_t ldg, void *out_bf16, size_t ldo,
                    ifa_stream stream);
