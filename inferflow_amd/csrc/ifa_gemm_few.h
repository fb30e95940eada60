// ifa_gemm_few.h -- the linear layers of 9..192 rows (prompts, large batches) that stream their weights once (ifa_gemm_few.hip)
#pragma once
#include "ifa_gemm_rows_mfma.h"

namespace ifa {

constexpr int FEW_MIN = 9, FEW_MAX = 192;       // rows (few_max_rows: of a model's layers)
constexpr int FEW_PARTS = 8;                    // parts of K at the most

// Rows in FRAGMENT ORDER ([K / 128][tiles of 16 rows][4][64 lanes][8 halves]): lane 16 g + r of piece s holds columns 128 S + 32 g + 8 s .. + 7 of row
// 16 tile + r -- the B operand that goes with a word of the MO layout -- so that a wave's request for a fragment is one KiB.  Rows beyond the last of a tile are
// not read.
inline size_t few_frag_bytes(int rows, size_t cols) { return (size_t)((rows + 15) / 16) * 16 * cols * 2; }

struct FewArgs {
    const uint8_t *W[3];           // MO_WORDS copies; up to three matrices one after the other (rows of 16 each); gated pairs: W[0] with W1
    const uint8_t *W1;
    int rows[3];
    int nsets, K, T;
    const half_t *X;               // FEW_ROWS / FEW_GLU, FEW_SUMS with ldx = 0: in fragment order; FEW_SUMS with ldx > 0: rows
    int ldx;
    const half_t *bias[3];
    const half_t *bias1;
    half_t *Y[3];                  // FEW_ROWS: matrix i's columns of each row, rows of ldy[i]; FEW_GLU: Y[0] in fragment order
    int ldy[3];
    int act_kind;
    float *sums;                   // FEW_SUMS: [parts][T][rows[0]], room for FEW_PARTS parts; few_sum_norm adds them
};
enum FewOut { FEW_ROWS, FEW_GLU, FEW_SUMS };
bool few_ok(size_t rows, size_t cols);                       // a matrix that these launches take
int few_max_rows(size_t dim, size_t ffn);                    // up to how many rows a layer of these sizes goes this way
int few_parts(size_t rows, size_t cols);                     // FEW_SUMS: parts of K of such a matrix
int gemm_few(const FewArgs &P, FewOut out, hipStream_t s);
// x_out[t] = res[t] + half(sum of the parts' rows, in order) (+ bias), parts = 0: x_out not written, res[t]; y (nullable) = its RMS norm in fragment order
int few_sum_norm(const float *sums, int parts, const half_t *bias, const half_t *res, half_t *x_out, int T, int cols, const half_t *norm_w, const half_t *norm_b, float multi_base, float eps,
                 half_t *y, hipStream_t s);

} // namespace ifa
