// ifa_linear_bf16.hip -- linear layers with bfloat16 weights [N][K] and 32-bit activations [T][K]:
//   C[t][n] (+)= alpha * mul[n] * act(sum_k A[t][k] W[n][k] + bias[n])     (mul, bias optional; act = SiLU on a column range, else identity;
//                                                                          C in 32-bit floats)
// The epilogue covers a plain projection (store), a projection with bias, and the residual update of a layer
// (accumulate into the 32-bit residual stream with a per-channel layer scale and a branch scale).
//
//   T <= 8    k_lin_rows: one wave per output row, the weight row streamed once in 16-byte pieces, all T activation rows
//             multiplied against it in fp32 (decode steps: bound by the weight stream); k_lin_rows_group: two outputs a wave
//             (large matrices, gated activations)
//   T  > 8    k_lin_mfma: 64 x 64 output tiles, K in steps of 32 through LDS, four waves of 32 x 32 sub-tiles;
//             OPS32 = false: operands rounded to bfloat16, v_mfma_f32_32x32x16_bf16;
//             OPS32 = true : operands stay 32-bit, v_mfma_f32_32x32x2_f32 (the exact mode of the worker)
//   T  > 8    k_lin_tile (ifa_linear_bf16_both, where the caller has rounded the activations: by their producer or by k_rows_to_bf16): tiles of up to
//             128 x 128 (32 x 32 where there are few), both operands straight to LDS; the same sums in the same order as k_lin_mfma<false>
// Accumulation is fp32 in every path.  No atomics; K is shared out (sums of products) by sizes alone, its parts added in order: a result does not depend on what else runs.
#include <algorithm>
#include <cstring>
#include <type_traits>
#include "ifa_host.h"
#include "ifa_f32_common.h"
#include "ifa_rows_fused.h"

using namespace ifa32;

namespace {

typedef float f32x16v __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8v __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));

struct LinArgs {
    const bf16_t *W; const float *A; float *C;
    const bf16_t *bias, *mul;
    int T, N, K, lda, ldc;
    float alpha; int accumulate, vec;
    int act_c0, act_c1;          // output columns [act_c0, act_c1) pass SiLU after the bias (projections whose consumer wants them activated)
    const bf16_t *norm_w; float norm_eps;      // row kernel, prologue 1: the activations are layer-normed (no bias) on the fly
    // grouped product (k_lin_mfma only): tile blockIdx.y serves rows [row0, row0 + n) of group g (tile_map {g, row0, n}; *n_tiles valid
    // tiles) with the matrix W + g * N * K; activation row of output row r: A[a_rows[r]] (a_rows null: r); row_scale per output row
    const int *tile_map, *n_tiles, *a_rows; const float *row_scale;
    bf16_t *C16;                               // (k_lin_tile with act_kind 2: the output in bfloat16 instead of C)
    int act_kind;                              // every output after the bias passes 1: the exact (erf) GELU, 2: the square of relu
};

// What only some kernels read stands in arguments of their own.  (In one struct, with the gate tested at run time, every product of a few rows took 0.05 to 0.2 us more and one of four rows
// 0.3: 1024 x 1024, 1 / 4 / 8 rows 3.56 / 5.14 / 7.47 us against 3.63 / 5.49 / 7.70.)
// Columns [glu_c0, glu_c0 + 2 glu_f) are gate | up.  k_lin_tile: instead of them G16[t][c] = act(gate[c]) up[c] in bfloat16, glu_w columns (whole 64s, zero beyond glu_f); k_lin_rows_group: G in
// 32 bits
struct LinGluArgs : LinArgs { bf16_t *G16; float *G; int ldg, glu_c0, glu_f, glu_w, glu_kind; float glu_limit; };
// Row t times sigmoid(row_gate[t * ld_gate]) (lin_store)
struct LinGatedArgs : LinArgs { const float *row_gate; int ld_gate; };
// Several products into the same columns (k_lin_tile): A's rows hold their operands side by side, each padded to whole steps; W, K, mul, bias, alpha of each here
struct LinSumArgs : LinArgs { struct Part { const bf16_t *W, *mul, *bias; int K, steps; float alpha; } part[IFA_SUM_PARTS]; float *planes; int ks; };

template <class Args>
__device__ __forceinline__ void lin_store(const Args &P, int t, int n, float acc)
{
    if (P.bias) acc += bf2f(P.bias[n]);
    if (n >= P.act_c0 && n < P.act_c1) acc = silu_exact(acc);
    if (P.act_kind == 1) acc = 0.5f * acc * (1.0f + erff(acc * 0.70710678118654752f));
    if (P.act_kind == 2) { acc = fmaxf(acc, 0.0f); acc *= acc; }
    if (P.row_scale) acc *= P.row_scale[t];
    if constexpr (std::is_same_v<Args, LinGatedArgs>) acc *= sigmoid_f(P.row_gate[(size_t)t * P.ld_gate]);
    if (P.mul) acc *= bf2f(P.mul[n]);
    acc *= P.alpha;
    float *c = P.C + (size_t)t * P.ldc + n;
    *c = P.accumulate ? *c + acc : acc;
}

constexpr int LM_T = 64, LM_N = 64, LM_K = 32;

template <bool OPS32>
__global__ void __launch_bounds__(256) k_lin_mfma(LinArgs P)
{
    // bf16 operands: [64][40] halfs per matrix (row stride 80 bytes: 16-byte aligned fragments);
    // 32-bit operands: [64][33] floats per matrix
    __shared__ __attribute__((aligned(16))) char smem[OPS32 ? 2 * LM_T * 33 * 4 : 2 * LM_T * 40 * 2];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int i = lane & 31, g = lane >> 5;
    const int wm = wave & 1, wn = wave >> 1;
    int t0 = blockIdx.y * LM_T, t_end = P.T;
    const int n0 = blockIdx.x * LM_N;
    const bf16_t *Wg = P.W;
    if (P.tile_map) {
        if ((int)blockIdx.y >= *P.n_tiles) return;
        const int *tm = P.tile_map + 3 * blockIdx.y;
        Wg += (size_t)tm[0] * P.N * P.K; t0 = tm[1]; t_end = tm[1] + tm[2];
    }
    const int lr = tid >> 2, lc = (tid & 3) * 8;      // this thread stages 8 consecutive k of row lr
    const size_t a_row = (t0 + lr < t_end) ? (size_t)(P.a_rows ? P.a_rows[t0 + lr] : t0 + lr) : 0;
    f32x16v acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.0f;

    for (int k0 = 0; k0 < P.K; k0 += LM_K) {
        float a8[8], w8[8];
        {
            const int t = t0 + lr, n = n0 + lr, k = k0 + lc;
            const bool in_a = t < t_end, in_w = n < P.N;
            if (P.vec && k + 8 <= P.K) {
                if (in_a) {
                    const float4 v0 = *reinterpret_cast<const float4 *>(P.A + a_row * P.lda + k);
                    const float4 v1 = *reinterpret_cast<const float4 *>(P.A + a_row * P.lda + k + 4);
                    a8[0] = v0.x; a8[1] = v0.y; a8[2] = v0.z; a8[3] = v0.w; a8[4] = v1.x; a8[5] = v1.y; a8[6] = v1.z; a8[7] = v1.w;
                } else {
#pragma unroll
                    for (int e = 0; e < 8; e++) a8[e] = 0.0f;
                }
                if (in_w) {
                    const u32x4v wv = *reinterpret_cast<const u32x4v *>(Wg + (size_t)n * P.K + k);
#pragma unroll
                    for (int e = 0; e < 4; e++) { w8[2 * e] = __uint_as_float(wv[e] << 16); w8[2 * e + 1] = __uint_as_float(wv[e] & 0xFFFF0000u); }
                } else {
#pragma unroll
                    for (int e = 0; e < 8; e++) w8[e] = 0.0f;
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const bool kin = k + e < P.K;
                    a8[e] = in_a && kin ? P.A[a_row * P.lda + k + e] : 0.0f;
                    w8[e] = in_w && kin ? bf2f(Wg[(size_t)n * P.K + k + e]) : 0.0f;
                }
            }
        }
        __syncthreads();      // the previous step's fragments have been read
        if constexpr (OPS32) {
            float *As = reinterpret_cast<float *>(smem), *Ws = As + LM_T * 33;
#pragma unroll
            for (int e = 0; e < 8; e++) { As[lr * 33 + lc + e] = a8[e]; Ws[lr * 33 + lc + e] = w8[e]; }
        } else {
            bf16_t *As = reinterpret_cast<bf16_t *>(smem), *Ws = As + LM_T * 40;
            u32x4v av, wv;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                av[e] = (uint32_t)f2bf(a8[2 * e]) | ((uint32_t)f2bf(a8[2 * e + 1]) << 16);
                wv[e] = (__float_as_uint(w8[2 * e]) >> 16) | (__float_as_uint(w8[2 * e + 1]) & 0xFFFF0000u);
            }
            *reinterpret_cast<u32x4v *>(As + lr * 40 + lc) = av;
            *reinterpret_cast<u32x4v *>(Ws + lr * 40 + lc) = wv;
        }
        __syncthreads();
        if constexpr (OPS32) {
            const float *As = reinterpret_cast<const float *>(smem), *Ws = As + LM_T * 33;
#pragma unroll
            for (int s = 0; s < LM_K / 2; s++)
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(As[(32 * wm + i) * 33 + 2 * s + g], Ws[(32 * wn + i) * 33 + 2 * s + g], acc, 0, 0, 0);
        } else {
            const bf16_t *As = reinterpret_cast<const bf16_t *>(smem), *Ws = As + LM_T * 40;
#pragma unroll
            for (int s = 0; s < LM_K / 16; s++) {
                const bf16x8v af = __builtin_bit_cast(bf16x8v, *reinterpret_cast<const u32x4v *>(As + (32 * wm + i) * 40 + 16 * s + 8 * g));
                const bf16x8v wf = __builtin_bit_cast(bf16x8v, *reinterpret_cast<const u32x4v *>(Ws + (32 * wn + i) * 40 + 16 * s + 8 * g));
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af, wf, acc, 0, 0, 0);
            }
        }
    }
    const int n = n0 + 32 * wn + i;
    if (n < P.N) {
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int t = t0 + 32 * wm + (r & 3) + 8 * (r >> 2) + 4 * g;
            if (t < t_end) lin_store(P, t, n, acc[r]);
        }
    }
}

// ---- prompts, both operands in bfloat16 already: BM x BN output tiles, WM x WN waves, K in steps of 64 through NB buffers in LDS.  Both operands go from memory to LDS
// directly (global_load_lds_dwordx4: a wave moves 8 rows x 128 bytes per instruction, NB - 1 steps ahead); both images are [rows][64 halfs] with the eight
// 16-byte pieces of row r at slot c ^ ((r >> 1) & 7), so that the fragment reads of 16 consecutive lanes (16 rows, one piece) are free of bank conflicts; the
// loads write LDS linearly, the permutation sits in their SOURCE addresses.  The step's barrier stands before its last group of products: every wave has read
// its last fragments by then, and the first fragments of the next buffer land under that group.
// Workgroups are dealt to the eight XCDs round-robin: the id is remapped so that an XCD works on a compact block of tiles whose operands its L2 shares.
// A's rows are K rounded up to whole steps long, zero beyond K (what W's requests bring in there -- held inside the row -- does not count).
constexpr int LT_BK = 64;
// Up to so many 64 x 64 tiles: 32 x 32 tiles of one wave each, seven steps under way.  us with two buffers of 64 x 64, four of 64 x 64, eight of 32 x 32 -- 16 tiles of 4096 columns
// 30.7, 18.3, 15.4; 64 tiles of 4096 46.0, 19.1, 15.8; 128 of 1024 9.9, 7.1, 6.8; 192 of 1024 10.0, 7.1, 11.3.
constexpr size_t LT_SMALL = 128;
typedef __attribute__((address_space(3))) void lt_lds_t;
typedef const __attribute__((address_space(1))) void lt_glb_t;

// GROUPED: row tiles and matrices from P.tile_map, the rows of A by P.a_rows (null: as they are), each output row times P.row_scale.
// GLU: column tiles from P.glu_c0 on serve BN / 2 outputs of a gated feed-forward: of 32 columns of such a tile 16 are gates and 16 the ups of the same outputs, so that one
// exchange between a wave's rows of 16 lanes brings the two together and the activation is formed here and rounded once (the same values as k_glu_to_bf16's).  The 32-bit gate | up
// rows were written and read again by a launch of their own: 2048 rows of width 2048, 11264 of 19968 columns
// gate | up, 237 + 23 us -> 243 (207 with the tiles as they are); 601 rows of width 1024 31.6 + 7.4 -> 32 (28).
// SUM: the parts of a sum of products one after the other in ONE pass over K: their requests run on without a break, the tile's rows of C are read and written once, and the launches
// but one go.  At a part's last step its columns' scales and biases take it from the step's accumulators into the sum.  (22 products of
// a Gelarax prompt in 8 launches: 2048 rows of width 2048 1268 -> 1202 us (866 with the tiles as they are), 601 of width 1024 312 -> 309 (240), and 14
// launches less.)
// SPLIT (with SUM): the steps shared out over P.ks workgroups a tile (lin_sum_plan).  (As a test at run time it cost the sums that are not shared out 7 %: 2048 rows of width 2048 104 -> 111 us.)
constexpr int LT_GROUPED = 1, LT_GLU = 2, LT_SUM = 4, LT_SPLIT = 8;
template <int MODE>
using LinTileArgs = std::conditional_t<(MODE & LT_SUM) != 0, LinSumArgs, std::conditional_t<(MODE & LT_GLU) != 0, LinGluArgs, LinArgs>>;
template <int BM, int BN, int WM, int WN, int NB, int MODE>
__global__ void __launch_bounds__(64 * WM * WN, BM == 32 ? 1 : 2) k_lin_tile(LinTileArgs<MODE> P, const bf16_t *__restrict__ A16, int lda16, int tiles_m, int tiles_n)
{
    constexpr bool GROUPED = MODE & LT_GROUPED, GLU = MODE & LT_GLU, SUM = MODE & LT_SUM, SPLIT = MODE & LT_SPLIT;
    constexpr int WAVES = WM * WN, TA = BM / (32 * WM), TB = BN / (32 * WN), AI = BM / (8 * WAVES), WI = BN / (8 * WAVES), ROWB = 2 * LT_BK, STEPB = (BM + BN) * ROWB;
    static_assert(AI * 8 * WAVES == BM && WI * 8 * WAVES == BN && TA * 32 * WM == BM && TB * 32 * WN == BN, "whole rows and tiles a wave");
    static_assert((NB - 2) * (AI + WI) < 64, "requests that s_waitcnt can count");
    extern __shared__ __attribute__((aligned(16))) char lt_smem[];          // [NB steps][BM rows of A, BN rows of W]
    char *const smem = lt_smem;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), i = lane & 31, g = lane >> 5, wm = wave % WM, wn = wave / WM;
    int t0, n0, t_end = P.T, kz = 0;
    const bf16_t *Wg = P.W;
    {
        // (grouped: of the tiles that there are, not of the most there can be -- the empty ones, dealt out like the others, left up to five of the XCDs idle: 36 pairs of 64
        // experts of 1024 x 704 66 -> 46 us, 2400 pairs 127 -> 101)
        if constexpr (GROUPED) tiles_m = *P.n_tiles;
        const int nwg = tiles_m * tiles_n;
        int orig = blockIdx.x;
        if constexpr (SPLIT) { kz = orig / nwg; orig -= kz * nwg; }
        const int xcd = orig & 7, q = nwg >> 3, r = nwg & 7;
        if (GROUPED && orig >= nwg) return;
        const int wg = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (orig >> 3);
        constexpr int GM = 1024 / BM;          // bands of 1024 rows of C, the row tiles of a band fastest
        const int band = wg / (GM * tiles_n), within = wg % (GM * tiles_n), band_m = min(GM, tiles_m - band * GM);
        t0 = (band * GM + within % band_m) * BM; n0 = (within / band_m) * BN;
        if constexpr (GROUPED) {
            const int *tm = P.tile_map + 3 * (t0 / BM);
            Wg += (size_t)tm[0] * P.N * P.K; t0 = tm[1]; t_end = tm[1] + tm[2];
        }
    }
    // a tile of gates and ups: o0, its first output
    const int n_end = [&]() { if constexpr (GLU) return P.glu_c0; else return P.N; }(), n_plain = GLU ? (n_end + BN - 1) / BN : 0, o0 = (n0 / BN - n_plain) * (BN / 2);
    const bool glu = GLU && n0 / BN >= n_plain;
    auto swz = [](int r) { return (r >> 1) & 7; };
    // (SPLIT) this workgroup's steps, k0 in front of them; (SUM) counted from k0, the part that the next requested step belongs to, from its first step to the one behind its last; likewise for the
    // next step of products
    int k0 = 0, nsteps = lda16 / LT_BK, q_part = 0, q_from = 0, q_to = 0;
    if constexpr (SUM) q_to = P.part[0].steps;
    if constexpr (SPLIT) {
        const int all = nsteps;
        k0 = kz * all / P.ks; nsteps = (kz + 1) * all / P.ks - k0; q_from = -k0; q_to -= k0;
        while (q_to <= 0) { q_part++; q_from = q_to; q_to += P.part[q_part].steps; }
    }
    const bf16_t *asrc[AI], *wsrc[WI];
    int wlim[WI];          // furthest step offset of the lane's piece inside a row of W
#pragma unroll
    for (int j = 0; j < AI; j++) {
        const int row = (wave * AI + j) * 8 + (lane >> 3), c = (lane & 7) ^ swz(row);
        int at = min(t0 + row, t_end - 1);          // (rows beyond the last: repeated, not stored)
        if (GROUPED && P.a_rows) at = P.a_rows[at];
        asrc[j] = A16 + (size_t)at * lda16 + (SPLIT ? k0 * LT_BK : 0) + c * 8;
    }
#pragma unroll
    for (int j = 0; j < WI; j++) {
        const int row = (wave * WI + j) * 8 + (lane >> 3), c = (lane & 7) ^ swz(row);
        int wr = min(n0 + row, n_end - 1);
        if constexpr (GLU) if (glu) wr = P.glu_c0 + ((row & 16) ? P.glu_f : 0) + min(o0 + 16 * (row >> 5) + (row & 15), P.glu_f - 1);
        const bf16_t *W0 = Wg;
        int K = P.K;
        if constexpr (SUM) { W0 = P.part[q_part].W; K = P.part[q_part].K; }
        wsrc[j] = W0 + (size_t)wr * K + c * 8;
        wlim[j] = K - 8 - c * 8;
    }
    int c_part = q_part, c_to = q_to;
    auto enter = [&](int step) {
        if constexpr (SUM) {
            if (step != q_to) return;
            q_part++; q_from = q_to; q_to += P.part[q_part].steps;
            const int K = P.part[q_part].K;
#pragma unroll
            for (int j = 0; j < WI; j++) {
                const int row = (wave * WI + j) * 8 + (lane >> 3), c = (lane & 7) ^ swz(row);
                wsrc[j] = P.part[q_part].W + (size_t)min(n0 + row, n_end - 1) * K + c * 8;
                wlim[j] = K - 8 - c * 8;
            }
        }
    };
    auto stage_a = [&](int step, char *to, int j) {
        __builtin_amdgcn_global_load_lds((lt_glb_t *)(asrc[j] + step * LT_BK), (lt_lds_t *)(to + (wave * AI + j) * 1024), 16, 0, 0);
    };
    auto stage_w = [&](int step, char *to, int j) {
        __builtin_amdgcn_global_load_lds((lt_glb_t *)(wsrc[j] + min((step - q_from) * LT_BK, wlim[j])), (lt_lds_t *)(to + BM * ROWB + (wave * WI + j) * 1024), 16, 0, 0);
    };
    auto stage = [&](int step, char *to) {
        enter(step);
#pragma unroll
        for (int j = 0; j < AI; j++) stage_a(step, to, j);
#pragma unroll
        for (int j = 0; j < WI; j++) stage_w(step, to, j);
    };
    const int lc = g ^ swz(i), a_off = (wm * (BM / WM) + i) * ROWB, w_off = (BM + wn * (BN / WN) + i) * ROWB;          // (tile rows start at multiples of 32)
    f32x16v acc[TA][TB];
#pragma unroll
    for (int a = 0; a < TA; a++)
#pragma unroll
        for (int b = 0; b < TB; b++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[a][b][r] = 0.0f;
    f32x16v tot[SUM ? TA : 1][SUM ? TB : 1];
    if constexpr (SUM) {
#pragma unroll
        for (int a = 0; a < TA; a++)
#pragma unroll
            for (int b = 0; b < TB; b++) tot[a][b] = acc[a][b];
    }
    // (asked for here: a request behind those of the steps would wait for all of them)
    float p_mul[SUM ? IFA_SUM_PARTS : 1][TB], p_bias[SUM ? IFA_SUM_PARTS : 1][TB];
    if constexpr (SUM) {
#pragma unroll
        for (int k = 0; k < IFA_SUM_PARTS; k++)
#pragma unroll
            for (int b = 0; b < TB; b++) {
                const auto &part = P.part[k];
                const int n = min(n0 + wn * (BN / WN) + 32 * b + i, P.N - 1);
                p_bias[k][b] = part.bias ? bf2f(part.bias[n]) : 0.0f; p_mul[k][b] = part.alpha * (part.mul ? bf2f(part.mul[n]) : 1.0f);
            }
    }
    auto close = [&](int step) {          // (behind the step's products)
        if constexpr (SUM) {
            const bool whole = step + 1 == c_to;          // (else: another workgroup has the rest of the part, and its bias)
            if (!whole && (!SPLIT || step + 1 != nsteps)) return;
#pragma unroll
            for (int b = 0; b < TB; b++) {
                float bv = p_bias[0][b], mv = p_mul[0][b];
#pragma unroll
                for (int k = 1; k < IFA_SUM_PARTS; k++) if (c_part == k) { bv = p_bias[k][b]; mv = p_mul[k][b]; }
#pragma unroll
                for (int a = 0; a < TA; a++)
#pragma unroll
                    for (int r = 0; r < 16; r++) { tot[a][b][r] += (acc[a][b][r] + (!SPLIT || whole ? bv : 0.0f)) * mv; acc[a][b][r] = 0.0f; }
            }
            c_part++;
            if (step + 1 < nsteps) c_to += P.part[c_part].steps;
        }
    };
    bf16x8v af[2][TA], wf[2][TB];
    auto frags = [&](const char *base, int ks, bf16x8v (&fa)[TA], bf16x8v (&fw)[TB]) {
        const int so = ((2 * ks) ^ lc) << 4;
#pragma unroll
        for (int a = 0; a < TA; a++) fa[a] = *reinterpret_cast<const bf16x8v *>(base + a_off + a * 32 * ROWB + so);
#pragma unroll
        for (int b = 0; b < TB; b++) fw[b] = *reinterpret_cast<const bf16x8v *>(base + w_off + b * 32 * ROWB + so);
    };
    auto mma = [&](const bf16x8v (&fa)[TA], const bf16x8v (&fw)[TB]) {
#pragma unroll
        for (int a = 0; a < TA; a++)
#pragma unroll
            for (int b = 0; b < TB; b++) acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[a], fw[b], acc[a][b], 0, 0, 0);
    };
    if constexpr (NB == 2) {
        stage(0, smem);
        __syncthreads();
        frags(smem, 0, af[0], wf[0]);
        for (int step = 0; step + 1 < nsteps; step++) {
            char *cur = smem + (step & 1) * STEPB, *nxt = smem + (~step & 1) * STEPB;
            stage(step + 1, nxt);
#pragma unroll
            for (int ks = 0; ks < 3; ks++) {
                frags(cur, ks + 1, af[(ks + 1) & 1], wf[(ks + 1) & 1]);
                mma(af[ks & 1], wf[ks & 1]);
            }
            __syncthreads();
            frags(nxt, 0, af[0], wf[0]);
            mma(af[1], wf[1]);
            close(step);
        }
        const char *cur = smem + ((nsteps - 1) & 1) * STEPB;
#pragma unroll
        for (int ks = 0; ks < 3; ks++) {
            frags(cur, ks + 1, af[(ks + 1) & 1], wf[(ks + 1) & 1]);
            mma(af[ks & 1], wf[ks & 1]);
        }
        mma(af[1], wf[1]);
        close(nsteps - 1);
    } else if constexpr (BM > 32) {
        // A step's own requests have arrived (those of the NB - 2 steps behind it may be under way), everybody's with the barrier, before which every wave has also read the
        // step before: its buffer takes the step NB - 1 further on.
        auto arrived = [&](auto more) {
            if constexpr (decltype(more)::value) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"((NB - 2) * (AI + WI)) : "memory");
            else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        };
        auto one = [&](int step, int j, auto more, auto last) {
            const char *cur = smem + j * STEPB, *nxt = smem + (j + 1 == NB ? 0 : j + 1) * STEPB;
            if constexpr (decltype(more)::value) stage(step + NB - 1, smem + (j == 0 ? NB - 1 : j - 1) * STEPB);
#pragma unroll
            for (int ks = 0; ks < 3; ks++) {          // (the next fragments under this one's products)
                frags(cur, ks + 1, af[(ks + 1) & 1], wf[(ks + 1) & 1]);
                __builtin_amdgcn_sched_barrier(0);
                mma(af[ks & 1], wf[ks & 1]);
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (!decltype(last)::value) {
                arrived(more);
                frags(nxt, 0, af[0], wf[0]);
                __builtin_amdgcn_sched_barrier(0);
            }
            mma(af[1], wf[1]);
            __builtin_amdgcn_sched_barrier(0);
            close(step);
        };
        // (at least NB steps)
#pragma unroll
        for (int j = 0; j < NB - 1; j++) stage(j, smem + j * STEPB);
        arrived(std::true_type());
        frags(smem, 0, af[0], wf[0]);
        int step = 0, j = 0;
        for (; step + NB - 1 < nsteps; step++) { one(step, j, std::true_type(), std::false_type()); j = j + 1 == NB ? 0 : j + 1; }
        for (; step + 1 < nsteps; step++) { one(step, j, std::false_type(), std::false_type()); j = j + 1 == NB ? 0 : j + 1; }
        one(step, j, std::false_type(), std::true_type());
    } else {
        static_assert(TA == 1 && TB == 1 && AI == 4 && WI == 4, "one wave: one tile of each operand, its requests of a step spread over four products");
        const unsigned lds0 = (unsigned)(uintptr_t)(lt_lds_t *)smem;
        unsigned at[4];
#pragma unroll
        for (int ks = 0; ks < 4; ks++) at[ks] = lds0 + (((2 * ks) ^ lc) << 4);
        // One step: its requests have arrived (those of the NB - 2 steps behind it may be under way) and the step before has been read: its buffer takes the step NB - 1 further on.
        // (The reads and their wait are one block: reads that the compiler sees wait for every request into LDS, once a round of the buffers at the least.)
        auto one = [&](int step, int j, auto more) {
            if constexpr (decltype(more)::value) asm volatile("s_waitcnt vmcnt(%0)" :: "n"((NB - 2) * (AI + WI)) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            char *to = smem + (j == 0 ? NB - 1 : j - 1) * STEPB;
            if constexpr (decltype(more)::value) enter(step + NB - 1);
            const unsigned oa = j * STEPB + a_off, ow = j * STEPB + w_off;
            bf16x8v fa[4], fw[4];
            asm volatile("ds_read_b128 %0, %8\n\tds_read_b128 %4, %12\n\tds_read_b128 %1, %9\n\tds_read_b128 %5, %13\n\tds_read_b128 %2, %10\n\tds_read_b128 %6, %14\n\t"
                         "ds_read_b128 %3, %11\n\tds_read_b128 %7, %15\n\ts_waitcnt lgkmcnt(0)"
                         : "=&v"(fa[0]), "=&v"(fa[1]), "=&v"(fa[2]), "=&v"(fa[3]), "=&v"(fw[0]), "=&v"(fw[1]), "=&v"(fw[2]), "=&v"(fw[3])
                         : "v"(at[0] + oa), "v"(at[1] + oa), "v"(at[2] + oa), "v"(at[3] + oa), "v"(at[0] + ow), "v"(at[1] + ow), "v"(at[2] + ow), "v"(at[3] + ow) : "memory");
#pragma unroll
            for (int ks = 0; ks < 4; ks++) {
                acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[ks], fw[ks], acc[0][0], 0, 0, 0);
                if constexpr (decltype(more)::value) {          // (the only wave: its requests go out under its products, 4096 columns 16.5 -> 15.4 us)
                    __builtin_amdgcn_sched_barrier(0);
                    stage_a(step + NB - 1, to, ks);
                    stage_w(step + NB - 1, to, ks);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            close(step);
        };
        // (at least NB steps)
#pragma unroll
        for (int j = 0; j < NB - 1; j++) stage(j, smem + j * STEPB);
        int step = 0, j = 0;
        for (; step + NB - 1 < nsteps; step++) { one(step, j, std::true_type()); j = j + 1 == NB ? 0 : j + 1; }
        for (; step < nsteps; step++) { one(step, j, std::false_type()); j = j + 1 == NB ? 0 : j + 1; }
    }
    // every (row, column) of the wave's tile: f(C element's place, value behind the bias)
    auto each = [&](auto f) {
#pragma unroll
        for (int b = 0; b < TB; b++) {
            const int n = n0 + wn * (BN / WN) + 32 * b + i;
            if (n >= n_end) continue;
            const float bv = P.bias ? bf2f(P.bias[n]) : 0.0f, mv = P.alpha * (P.mul ? bf2f(P.mul[n]) : 1.0f);
#pragma unroll
            for (int a = 0; a < TA; a++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int t = t0 + wm * (BM / WM) + 32 * a + (r & 3) + 8 * (r >> 2) + 4 * g;
                    if (t < t_end) f((size_t)t * P.ldc + n, n, acc[a][b][r] + bv, mv);
                }
        }
    };
    if constexpr (SUM) {
#pragma unroll
        for (int b = 0; b < TB; b++) {
            const int n = n0 + wn * (BN / WN) + 32 * b + i;
            if (n >= n_end) continue;
#pragma unroll
            for (int a = 0; a < TA; a++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int t = t0 + wm * (BM / WM) + 32 * a + (r & 3) + 8 * (r >> 2) + 4 * g;
                    if (t >= t_end) continue;
                    if (!SPLIT || kz == 0) P.C[(size_t)t * P.ldc + n] += tot[a][b][r];
                    else P.planes[((size_t)(kz - 1) * P.T + t) * P.N + n] = tot[a][b][r];
                }
        }
        return;
    }
    if constexpr (GLU) {
        if (glu) {
            // lanes of a first row of 16 hold gates, those of a second one ups: after the exchange of a second row's r with a first row's r + 8 both hold both, rows r here, r + 8 there
            const int hi = i >> 4;
#pragma unroll
            for (int b = 0; b < TB; b++) {
                const int o = o0 + wn * (BN / (2 * WN)) + 16 * b + (i & 15);
                const float gb = P.bias && o < P.glu_f ? bf2f(P.bias[P.glu_c0 + o]) : 0.0f, ub = P.bias && o < P.glu_f ? bf2f(P.bias[P.glu_c0 + P.glu_f + o]) : 0.0f;
#pragma unroll
                for (int a = 0; a < TA; a++)
#pragma unroll
                    for (int r = 0; r < 8; r++) {
                        const auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[a][b][r]), __float_as_uint(acc[a][b][r + 8]), false, false);
                        const int t = t0 + wm * (BM / WM) + 32 * a + (r & 3) + 8 * (r >> 2) + 16 * hi + 4 * g;
                        const float v = glu_of(P.glu_kind, P.glu_limit, __uint_as_float(x[0]) + gb, __uint_as_float(x[1]) + ub);
                        if (t < t_end && o < P.glu_w) P.G16[(size_t)t * P.ldg + o] = __builtin_bit_cast(bf16_t, (__bf16)(o < P.glu_f ? v : 0.0f));
                    }
            }
            return;
        }
    }
    if constexpr (GROUPED) {          // (the rows' scales take the place of the columns')
#pragma unroll
        for (int a = 0; a < TA; a++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int t = t0 + wm * (BM / WM) + 32 * a + (r & 3) + 8 * (r >> 2) + 4 * g;
                if (t >= t_end) continue;
                const float sc = P.row_scale ? P.row_scale[t] : 1.0f;
#pragma unroll
                for (int b = 0; b < TB; b++) {
                    const int n = n0 + wn * (BN / WN) + 32 * b + i;
                    if (n < P.N) P.C[(size_t)t * P.ldc + n] = acc[a][b][r] * sc;
                }
            }
        return;
    }
    if (P.act_kind == 2) {
        if (P.C16) each([&](size_t at, int, float v, float mv) { v = fmaxf(v, 0.0f); P.C16[at] = __builtin_bit_cast(bf16_t, (__bf16)(v * v * mv)); });
        else each([&](size_t at, int, float v, float mv) { v = fmaxf(v, 0.0f); P.C[at] = v * v * mv; });
    } else if (P.act_kind == 0 && P.act_c0 >= P.act_c1) {
        if (P.accumulate) each([&](size_t at, int, float v, float mv) { P.C[at] += v * mv; });
        else each([&](size_t at, int, float v, float mv) { P.C[at] = v * mv; });
    } else {
        each([&](size_t at, int n, float v, float mv) {
            if (n >= P.act_c0 && n < P.act_c1) v = silu_exact(v);
            if (P.act_kind == 1) v = 0.5f * v * (1.0f + erff(v * 0.70710678118654752f));
            P.C[at] = P.accumulate ? P.C[at] + v * mv : v * mv;
        });
    }
}

// column tiles of a product (gate | up: with G16's padding)
size_t lin_col_tiles(const LinArgs &P, int bn) { return ((size_t)P.N + bn - 1) / bn; }
size_t lin_col_tiles(const LinGluArgs &P, int bn) { return (P.glu_c0 + bn - 1) / bn + ((size_t)P.glu_w + bn / 2 - 1) / (bn / 2); }

template <int BM, int BN, int WM, int WN, int NB, int MODE>
int launch_lin_tile(const LinTileArgs<MODE> &P, const bf16_t *a16, size_t lda16, size_t row_tiles, hipStream_t s)
{
    constexpr int smem = NB * (BM + BN) * 2 * LT_BK;
    const int tm = (int)row_tiles, tn = (int)lin_col_tiles(P, BN);
    const auto fn = k_lin_tile<BM, BN, WM, WN, NB, MODE>;
    if (smem > 64 * 1024) IFA_HIP_CHECK(hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, smem));
    unsigned ks = 1;
    if constexpr ((MODE & LT_SPLIT) != 0) ks = (unsigned)P.ks;
    hipLaunchKernelGGL(fn, dim3((unsigned)tm * (unsigned)tn * ks), dim3(64 * WM * WN), smem, s, P, a16, (int)lda16, tm, tn);
    IFA_LAUNCH_CHECK();
    return IFA_OK;
}

// Tile shapes by what a round of the chip's 256 compute units takes: us a step of 64 columns and beside the steps, measured with weights from memory.  A round that is not full takes less a
// step, the chip's clock and its caches being shared: where a compute unit has one workgroup, from `one` (few of them) to `full`; where it has two, `one` up to 256 workgroups, then from `two`
// to `full`.  (As if every round took what a full one of short rows does, rows of 5632 columns and more ran alone on a compute unit in two rounds: tokens x columns x K 1233 x 4096 x 5632 97 us,
// by twos 85; 4096 x 4096 x 5632 214 and 198; 2048 x 4096 x 8192 156 and 143.  Against the fastest shape of each of 570 sizes from 16 to 4096 tokens, 256 to 11264 columns and 320 to 11008 K
// 1.5 % behind on average and up to 17, now 0.7.)
// us before (128 x 128 and 128 x 64 of 4 waves with two buffers, 64 x 64 with four) / now, tokens x columns x K: 2048 x 2048 x 9728 123 / 90, 1000 x 2048 x 9728 117 / 62,
// 2000 x 1024 x 4864 58 / 32, 2048 x 1024 x 1024 15.4 / 8.7, 730 x 2836 x 1024 16.1 / 12.5, 1024 x 4096 x 2048 29.9 / 22.5, 601 x 1024 x 4864 22.1 / 20.8; in a Gelarax layer 2048 rows' input
// product (19968 columns, gated) 238 / 207, its output product 150 / 108.  (256 x 128 tiles of eight waves, one a compute unit, 225 to 235 there.)
struct LinShape { int per_cu; double one, two, full, beside; };
enum { LT_128x128_PAIR, LT_128x128, LT_128x64, LT_64x64, LT_N_SHAPES };
constexpr LinShape LT_SHAPES[LT_N_SHAPES] = {{2, 0.80, 0.87, 1.13, 4}, {1, 0.42, 0, 0.585, 5}, {1, 0.36, 0, 0.36, 4}, {2, 0.255, 0.44, 0.44, 4}};
double lin_cost(const LinShape &h, size_t tiles, size_t steps)
{
    const size_t cus = 256, slots = cus * h.per_cu, rounds = tiles / slots, rest = tiles % slots;
    const double whole = rounds * (steps * h.full + h.beside);
    if (rest == 0) return whole;
    const double a_step = h.per_cu == 1 ? h.one + (h.full - h.one) * rest / cus : rest <= cus ? h.one : h.two + (h.full - h.two) * (rest - cus) / cus;
    return whole + steps * a_step + h.beside;
}

template <int MODE>
int lin_tile_dispatch(const LinTileArgs<MODE> &P, const bf16_t *a, size_t lda, hipStream_t s)
{
    const size_t T = (size_t)P.T, t128 = (T + 127) / 128, t64 = (T + 63) / 64, n128 = lin_col_tiles(P, 128), n64 = lin_col_tiles(P, 64), steps = lda / LT_BK;
    IFA_REQUIRE(t64 * n64 < (1u << 31), "linear_bf16: too many tiles");
    // 128 x 128 tiles would give some compute units one workgroup and some two, 128 x 64 tiles of four waves, three a compute unit, share out more evenly.  us 128 x 128 / 128 x 64 (as before the
    // shapes below), tokens x columns x K: 411 x 11264 x 256, 512, 1024, 2048 9.4 / 8.7, 13.4 / 12.7, 21.7 / 20.7, 37.5 / 35.4; 601 x 6700 x 1024 19.8 / 18.9, x 2048 33.8 / 31.7;
    // 1233 x 3500 x 704, 1408 15.3 / 14.8, 24.9 / 23.6; beyond 32 steps nothing (1000 x 5632 x 4096 68.2 / 68.4, 1233 x 4600 x 5632 90.9 / 95.6)
    // (few steps, below: where 64 x 64 tiles of two buffers would have no place at once, four a compute unit: gated, 800 x 4816 x 256 8.0 us with those, 10.0 with these; 1000 x 4816 11.2, 10.3)
    if (t128 * n64 > 512 && t128 * n128 < 384 && steps <= 32 && (steps >= 5 || t64 * n64 > 1024)) return launch_lin_tile<128, 64, 2, 2, 2, MODE>(P, a, lda, t128, s);
    if (steps < 5) {
        // Fewer steps than the buffers of the tiles below: two buffers, but 64 x 64 tiles that all have a place at once take four where there are four steps.  us with 64 x 64 of two buffers,
        // 64 x 64 of four, 128 x 64 (four waves, three workgroups a compute unit), 128 x 128 -- four steps, tokens x columns: 16 x 4096 4.4, 3.8, 5.2, 5.6; 1000 x 1024 4.5, 4.2, 5.4, 5.8;
        // 1000 x 2048 5.6, 5.2, 6.3, 6.7; 411 x 5632 6.0, 7.5, 6.8, 6.9; 411 x 11264 9.8, 10.6, 8.7, 9.4; 1233 x 4096 9.9, 10.6, 8.8, 9.3; 601 x 11264 11.2, 13.7, 13.1, 10.0; two steps,
        // 1000 x 4096 6.7, -, 6.9, 7.0; 1000 x 5632 8.1, -, 7.3, 7.7; 1233 x 5632 8.9, -, 10.0, 8.3
        if (t128 * n128 >= 384) return launch_lin_tile<128, 128, 2, 4, 2, MODE>(P, a, lda, t128, s);
        if (steps == 4 && t64 * n64 <= 512) return launch_lin_tile<64, 64, 2, 2, 4, MODE>(P, a, lda, t64, s);
        return launch_lin_tile<64, 64, 2, 2, 2, MODE>(P, a, lda, t64, s);
    }
    if (t64 * n64 <= LT_SMALL && steps >= 8) return launch_lin_tile<32, 32, 1, 1, 8, MODE>(P, a, lda, (T + 31) / 32, s);
    const size_t tiles[LT_N_SHAPES] = {t128 * n128, t128 * n128, t128 * n64, t64 * n64};
    int best = 0;
    for (int k = 1; k < LT_N_SHAPES; k++)
        if (lin_cost(LT_SHAPES[k], tiles[k], steps) < lin_cost(LT_SHAPES[best], tiles[best], steps)) best = k;
    switch (best) {
    case LT_128x128_PAIR: return launch_lin_tile<128, 128, 2, 4, 2, MODE>(P, a, lda, t128, s);
    case LT_128x128: return launch_lin_tile<128, 128, 2, 4, 4, MODE>(P, a, lda, t128, s);
    case LT_128x64: return launch_lin_tile<128, 64, 4, 2, 4, MODE>(P, a, lda, t128, s);
    default: return launch_lin_tile<64, 64, 2, 2, 5, MODE>(P, a, lda, t64, s);
    }
}

template <int MODE>
int lin_grouped_dispatch(const LinTileArgs<MODE> &P, const bf16_t *a, size_t lda, size_t max_tiles, int tile_rows, hipStream_t s)
{
    IFA_REQUIRE(max_tiles * lin_col_tiles(P, 64) < (1u << 31), "linear_bf16_grouped: too many tiles");
    // (8192 pairs of 16 experts, 1408 x 1024 gate | up and 1024 x 704, us: four waves a 128 x 128 tile 54.8 + 46.8, eight 47.9 + 40.4; 2900 pairs: 64 x 64 tiles 34.2 + 18.8, 64 x 128 of
    // eight waves 27.0 + 17.0; whole experts, sort and sums with them, 36 pairs of these 28.7 -> 25.3, 64 pairs 29.5 -> 25.9, 54 pairs of 32 experts 2816 x 2048 and 2048 x 1408 132.6 -> 115.0,
    // 18 pairs of 8 experts 512 x 512 and 512 x 256 19.2 -> 18.4)
    if (tile_rows == 128) return launch_lin_tile<128, 128, 2, 4, 2, MODE>(P, a, lda, max_tiles, s);
    if (lda >= 3 * LT_BK) return launch_lin_tile<64, 128, 2, 4, 3, MODE>(P, a, lda, max_tiles, s);
    return launch_lin_tile<64, 64, 2, 2, 2, MODE>(P, a, lda, max_tiles, s);
}

// rows of 32-bit values to bfloat16, zero up to `width` columns (a multiple of 8) of rows of ldy
__global__ void __launch_bounds__(256) k_rows_to_bf16(const float *__restrict__ x, size_t ldx, int cols, bf16_t *__restrict__ y, int width, int ldy, int vec)
{
    const float *xr = x + (size_t)blockIdx.y * ldx;
    const int c = (blockIdx.x * 256 + threadIdx.x) * 8;
    if (c >= width) return;
    float v[8];
    if (vec && c + 8 <= cols) {
        const float4 a = *reinterpret_cast<const float4 *>(xr + c), b = *reinterpret_cast<const float4 *>(xr + c + 4);
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    } else {
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = c + e < cols ? xr[c + e] : 0.0f;
    }
    bf16x8v h;
#pragma unroll
    for (int e = 0; e < 8; e++) h[e] = (__bf16)v[e];
    *reinterpret_cast<bf16x8v *>(y + (size_t)blockIdx.y * ldy + c) = h;
}

// T <= TT rows; one wave per output row at a time.  PRO: what the activations pass as they are read (steps of a few rows are bound
// by launches and dependent loads, not arithmetic, so the neighbouring element-wise launch is folded in here):
//   1  layer norm without bias: a = (x - mean) / sqrt(var + eps) * w[k]   (every wave forms mean and variance of the T rows itself)
//   2  gated GELU: the row holds gate | up (2 K values), a = gelu_tanh(gate[k]) * up[k]
template <int TT, int PRO, class Args = LinArgs>
__global__ void __launch_bounds__(256) k_lin_rows(Args P)
{
    const int lane = threadIdx.x & 63;
    const int wave = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6), nwaves = gridDim.x * (blockDim.x >> 6);
    float mean[TT], rstd[TT];
    if (PRO == 1) {
#pragma unroll
        for (int t = 0; t < TT; t++) {
            const float *a = P.A + (size_t)min(t, P.T - 1) * P.lda;
            float s = 0.0f;
            for (int k = lane * 4; k < P.K; k += 256) { const float4 v = *reinterpret_cast<const float4 *>(a + k); s += (v.x + v.y) + (v.z + v.w); }
            mean[t] = wave_sum(s) / (float)P.K;
            float q = 0.0f;
            for (int k = lane * 4; k < P.K; k += 256) {
                const float4 v = *reinterpret_cast<const float4 *>(a + k);
                const float d0 = v.x - mean[t], d1 = v.y - mean[t], d2 = v.z - mean[t], d3 = v.w - mean[t];
                q += (d0 * d0 + d1 * d1) + (d2 * d2 + d3 * d3);
            }
            rstd[t] = 1.0f / sqrtf(wave_sum(q) / (float)P.K + P.norm_eps);
        }
    }
    for (int n = wave; n < P.N; n += nwaves) {
        float acc[TT];
#pragma unroll
        for (int t = 0; t < TT; t++) acc[t] = 0.0f;
        const bf16_t *w = P.W + (size_t)n * P.K;
        // (with a prologue its operands and the weight are enough in flight and the activations the longer part; up to four rows the waves are, of a large matrix: 32000 rows of 1024,
        // 2 / 4 rows 14.2 / 20.9 us, pieces first 15.7 / 23.0)
        if (P.vec && (PRO != 0 || TT <= 4)) {
            for (int k = lane * 8; k < P.K; k += 512) {
                const u32x4v wv = *reinterpret_cast<const u32x4v *>(w + k);
                float w8[8], g8[8];
#pragma unroll
                for (int e = 0; e < 4; e++) { w8[2 * e] = __uint_as_float(wv[e] << 16); w8[2 * e + 1] = __uint_as_float(wv[e] & 0xFFFF0000u); }
                if (PRO == 1) {
                    const u32x4v gv = *reinterpret_cast<const u32x4v *>(P.norm_w + k);
#pragma unroll
                    for (int e = 0; e < 4; e++) { g8[2 * e] = __uint_as_float(gv[e] << 16); g8[2 * e + 1] = __uint_as_float(gv[e] & 0xFFFF0000u); }
                }
#pragma unroll
                for (int t = 0; t < TT; t++) {
                    const float *a = P.A + (size_t)min(t, P.T - 1) * P.lda + k;
                    const float4 v0 = *reinterpret_cast<const float4 *>(a), v1 = *reinterpret_cast<const float4 *>(a + 4);
                    float x8[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
                    if (PRO == 1) {
#pragma unroll
                        for (int e = 0; e < 8; e++) x8[e] = (x8[e] - mean[t]) * rstd[t] * g8[e];
                    } else if (PRO == 2) {
                        const float4 u0 = *reinterpret_cast<const float4 *>(a + P.K), u1 = *reinterpret_cast<const float4 *>(a + P.K + 4);
                        const float u8[8] = {u0.x, u0.y, u0.z, u0.w, u1.x, u1.y, u1.z, u1.w};
#pragma unroll
                        for (int e = 0; e < 8; e++) x8[e] = gelu_tanh_f(x8[e]) * u8[e];
                    }
                    float sum = acc[t];
#pragma unroll
                    for (int e = 0; e < 8; e++) sum = fmaf(x8[e], w8[e], sum);
                    acc[t] = sum;
                }
            }
        } else if (P.vec) {
            // the weight's pieces of up to 2048 columns first (they come from memory; the rows come from the caches), past its end a piece again that is not multiplied: a piece
            // asked for behind the products of the one before, and eight rows formed for six, took 9.4 instead of 8.3 us (33 products of six rows a step).  As many pieces
            // as there are.
            auto block = [&](int k0, auto pieces) {
                constexpr int NP = decltype(pieces)::value;
                u32x4v wp[NP];
#pragma unroll
                for (int j = 0; j < NP; j++) wp[j] = *reinterpret_cast<const u32x4v *>(w + min(k0 + 512 * j + lane * 8, P.K - 8));
#pragma unroll
                for (int j = 0; j < NP; j++) {
                    const int k = k0 + 512 * j + lane * 8;
                    if (k0 + 512 * j >= P.K) break;
                    float4 v[TT][2];
#pragma unroll
                    for (int t = 0; t < TT; t++) {
                        const float *a = P.A + (size_t)min(t, P.T - 1) * P.lda + min(k, P.K - 8);
                        v[t][0] = *reinterpret_cast<const float4 *>(a); v[t][1] = *reinterpret_cast<const float4 *>(a + 4);
                    }
                    if (k >= P.K) continue;
                    float w8[8];
#pragma unroll
                    for (int e = 0; e < 4; e++) { w8[2 * e] = __uint_as_float(wp[j][e] << 16); w8[2 * e + 1] = __uint_as_float(wp[j][e] & 0xFFFF0000u); }
#pragma unroll
                    for (int t = 0; t < TT; t++) {
                        const float x8[8] = {v[t][0].x, v[t][0].y, v[t][0].z, v[t][0].w, v[t][1].x, v[t][1].y, v[t][1].z, v[t][1].w};
                        float sum = acc[t];
#pragma unroll
                        for (int e = 0; e < 8; e++) sum = fmaf(x8[e], w8[e], sum);
                        acc[t] = sum;
                    }
                }
            };
            int k0 = 0;
            for (; P.K - k0 > 1024; k0 += 2048) block(k0, std::integral_constant<int, 4>());
            if (P.K - k0 > 512) block(k0, std::integral_constant<int, 2>());
            else if (P.K - k0 > 0) block(k0, std::integral_constant<int, 1>());
        } else {
            for (int k = lane; k < P.K; k += 64) {
                const float wk = bf2f(w[k]);
#pragma unroll
                for (int t = 0; t < TT; t++) acc[t] = fmaf(P.A[(size_t)min(t, P.T - 1) * P.lda + k], wk, acc[t]);
            }
        }
#pragma unroll
        for (int t = 0; t < TT; t++) acc[t] = wave_sum(acc[t]);
#pragma unroll
        for (int t = 0; t < TT; t++)
            if (lane == t && t < P.T) lin_store(P, t, n, acc[t]);
    }
}

// T <= TT rows of many outputs, NR of them a wave at a time: k_lin_rows reads TT rows of activations (32 bytes of each beside 16 of the weight) for one output, and with six rows
// the caches' bandwidth for them bounds large matrices (32000 x 1024, six rows: 38.9 -> 31.0 us, 8192 x 2048
// 21.0 -> 16.7; four outputs 34.9 and 21.0).  GLU: from column glu_c0 on the NR are gates and ups by twos, and the activation leaves instead
// of them (the launch that formed it took 3.7 us).
template <int TT, int NR, class Args>
__global__ void __launch_bounds__(256) k_lin_rows_group(Args P)
{
    constexpr bool GLU = std::is_same_v<Args, LinGluArgs>;
    const int lane = threadIdx.x & 63, wave = blockIdx.x * 4 + (threadIdx.x >> 6), nwaves = gridDim.x * 4;
    int n_end = P.N, more = 0;
    if constexpr (GLU) { n_end = P.glu_c0; more = (P.glu_f + NR / 2 - 1) / (NR / 2); }
    const int plain = (n_end + NR - 1) / NR, groups = plain + more;
    for (int grp = wave; grp < groups; grp += nwaves) {
        const bool glu = GLU && grp >= plain;
        const int n0 = grp * NR, o0 = (grp - plain) * (NR / 2);
        const bf16_t *w[NR];
        int row[NR];
#pragma unroll
        for (int r = 0; r < NR; r++) {
            row[r] = min(n0 + r, n_end - 1);
            if constexpr (GLU) if (glu) row[r] = P.glu_c0 + ((r & 1) ? P.glu_f : 0) + min(o0 + (r >> 1), P.glu_f - 1);
            w[r] = P.W + (size_t)row[r] * P.K;
        }
        float acc[TT][NR];
#pragma unroll
        for (int t = 0; t < TT; t++)
#pragma unroll
            for (int r = 0; r < NR; r++) acc[t][r] = 0.0f;
        // (pieces of the weights first, see k_lin_rows; past the end a piece again that is not multiplied)
        auto block = [&](int k0, auto pieces) {
            constexpr int NP = decltype(pieces)::value;
            u32x4v wp[NP][NR];
#pragma unroll
            for (int j = 0; j < NP; j++)
#pragma unroll
                for (int r = 0; r < NR; r++) wp[j][r] = *reinterpret_cast<const u32x4v *>(w[r] + min(k0 + 512 * j + lane * 8, P.K - 8));
#pragma unroll
            for (int j = 0; j < NP; j++) {
                const int k = k0 + 512 * j + lane * 8;
                if (k0 + 512 * j >= P.K) break;
                float4 v[TT][2];
#pragma unroll
                for (int t = 0; t < TT; t++) {
                    const float *a = P.A + (size_t)min(t, P.T - 1) * P.lda + min(k, P.K - 8);
                    v[t][0] = *reinterpret_cast<const float4 *>(a); v[t][1] = *reinterpret_cast<const float4 *>(a + 4);
                }
                if (k >= P.K) continue;
#pragma unroll
                for (int r = 0; r < NR; r++) {
                    float w8[8];
#pragma unroll
                    for (int e = 0; e < 4; e++) { w8[2 * e] = __uint_as_float(wp[j][r][e] << 16); w8[2 * e + 1] = __uint_as_float(wp[j][r][e] & 0xFFFF0000u); }
#pragma unroll
                    for (int t = 0; t < TT; t++) {
                        const float x8[8] = {v[t][0].x, v[t][0].y, v[t][0].z, v[t][0].w, v[t][1].x, v[t][1].y, v[t][1].z, v[t][1].w};
                        float sum = acc[t][r];
#pragma unroll
                        for (int e = 0; e < 8; e++) sum = fmaf(x8[e], w8[e], sum);
                        acc[t][r] = sum;
                    }
                }
            }
        };
        int k0 = 0;
        if constexpr (NR <= 2) for (; P.K - k0 > 1024; k0 += 2048) block(k0, std::integral_constant<int, 4>());
        for (; P.K - k0 > 512; k0 += 1024) block(k0, std::integral_constant<int, 2>());
        if (P.K - k0 > 0) block(k0, std::integral_constant<int, 1>());
#pragma unroll
        for (int t = 0; t < TT; t++)
#pragma unroll
            for (int r = 0; r < NR; r++) acc[t][r] = wave_sum(acc[t][r]);
#pragma unroll
        for (int t = 0; t < TT; t++) {
            if (lane != t || t >= P.T) continue;
            if constexpr (GLU) if (glu) {
#pragma unroll
                for (int r = 0; r < NR; r += 2) {
                    const float gb = P.bias ? bf2f(P.bias[row[r]]) : 0.0f, ub = P.bias ? bf2f(P.bias[row[r + 1]]) : 0.0f;
                    if (o0 + (r >> 1) < P.glu_f) P.G[(size_t)t * P.ldg + o0 + (r >> 1)] = glu_of(P.glu_kind, P.glu_limit, acc[t][r] + gb, acc[t][r + 1] + ub);
                }
            }
            if (!glu) {
#pragma unroll
                for (int r = 0; r < NR; r++) if (n0 + r < n_end) lin_store(P, t, n0 + r, acc[t][r]);
            }
        }
    }
}

// workgroups: a group of outputs a wave, up to 32 waves a compute unit
template <int NR, class Args>
void launch_lin_rows_group(const Args &P, hipStream_t s)
{
    size_t groups = ((size_t)P.N + NR - 1) / NR;
    if constexpr (std::is_same_v<Args, LinGluArgs>) groups = ((size_t)P.glu_c0 + NR - 1) / NR + ((size_t)P.glu_f + NR / 2 - 1) / (NR / 2);
    const dim3 grid((unsigned)std::min<size_t>((groups + 3) / 4, 8192));
    if (P.T == 1) hipLaunchKernelGGL((k_lin_rows_group<1, NR, Args>), grid, dim3(256), 0, s, P);
    else if (P.T == 2) hipLaunchKernelGGL((k_lin_rows_group<2, NR, Args>), grid, dim3(256), 0, s, P);
    else if (P.T <= 4) hipLaunchKernelGGL((k_lin_rows_group<4, NR, Args>), grid, dim3(256), 0, s, P);
    else if (P.T <= 6) hipLaunchKernelGGL((k_lin_rows_group<6, NR, Args>), grid, dim3(256), 0, s, P);
    else hipLaunchKernelGGL((k_lin_rows_group<8, NR, Args>), grid, dim3(256), 0, s, P);
}

// Whether two outputs a wave are faster: large matrices whose half as many waves still hide the weights' way from memory (the more rows a wave has to sum, the fewer waves that takes), and
// whose rows are long enough for it.  us one by one / by twos, rows of the weight x columns: 8192 x 1024 with 2, 4, 6, 8 rows 7.5 / 7.3, 9.6 / 8.8, 12.5 / 11.3, 15.8 / 15.8; 32000 x 2048
// 34.9 / 28.8, 58 / 39, 70 / 51, 95 / 62; 2816 x 4096 9.6 / 9.9, 14.3 / 12.9, 16.6 / 16.2, 20.1 / 18.9; 2048 x 8192 12.6 / 13.6, 14.9 / 15.3, 22.3 / 18.8, 27.1 / 22.7; 4096 x 2048
// 7.3 / 7.5, 10.2 / 9.2; and beyond the borders 1024 x 8192 10.5 / 10.7, 12.3 / 12.8, 14.6 / 16.2, 17.3 / 21.1; 16384 x 512 7.3 / 7.6, 10.4 / 10.3, 15.6 / 13.8, 18.4 / 20.7; 65536 x 128
// 16.7 / 18.3, 27.8 / 30.2, 48 / 41, 59 / 63.  One row: one by one (only the gated form below takes two, where that saves a launch: 2816 gates of 1024 columns 7.1 / 5.4 with the activation's)
bool lin_rows_by_twos(const LinArgs &P)
{
    if (P.T < 2 || !P.vec || P.K < 1024 || (size_t)P.N * P.K < (size_t)8 << 20) return false;
    return P.N >= (P.T >= 5 ? 2048 : P.T >= 3 ? 2560 : 5120);
}

// products of at most eight rows without a prologue
template <class Args>
void launch_lin_rows(const Args &P, hipStream_t s)
{
    if (lin_rows_by_twos(P)) { launch_lin_rows_group<2>(P, s); return; }
    const dim3 grid((unsigned)std::min<size_t>(((size_t)P.N + 3) / 4, 8192));
    if (P.T == 1) hipLaunchKernelGGL((k_lin_rows<1, 0, Args>), grid, dim3(256), 0, s, P);
    else if (P.T == 2) hipLaunchKernelGGL((k_lin_rows<2, 0, Args>), grid, dim3(256), 0, s, P);
    else if (P.T <= 4) hipLaunchKernelGGL((k_lin_rows<4, 0, Args>), grid, dim3(256), 0, s, P);
    else if (P.T <= 6) hipLaunchKernelGGL((k_lin_rows<6, 0, Args>), grid, dim3(256), 0, s, P);
    else hipLaunchKernelGGL((k_lin_rows<8, 0, Args>), grid, dim3(256), 0, s, P);
}

// ONE row, layer-normed on the way in (k_lin_rows with prologue 1 formed the norm again for every output row of a wave): each wave forms mean and variance
// once and keeps its lanes' normed values in registers, then walks output rows, the next row's weights asked for before this one's are summed.  The first
// row's weights are on their way under the norm, so the norm's own launch (6 us) is saved for about 1 us more here (both 12.4 us, now 7.6, over a token's products of width 1024).
template <int NP>
__global__ void __launch_bounds__(256) k_lin_row_norm(LinArgs P)
{
    const int lane = threadIdx.x & 63, wave = blockIdx.x * 4 + (threadIdx.x >> 6), nwaves = gridDim.x * 4;
    u32x4v w[NP], g[NP];
    float a[NP][8], b = 0.0f;
    auto request = [&](int n, u32x4v (&to)[NP]) {
#pragma unroll
        for (int p = 0; p < NP; p++) to[p] = *reinterpret_cast<const u32x4v *>(P.W + (size_t)n * P.K + min(512 * p + 8 * lane, P.K - 8));
    };
    int n = wave;
    if (n >= P.N) return;
    float s = 0.0f;
#pragma unroll
    for (int p = 0; p < NP; p++) {          // (asked for before the weights: requests come back in order)
        const int k = min(512 * p + 8 * lane, P.K - 8);
        const float4 v0 = *reinterpret_cast<const float4 *>(P.A + k), v1 = *reinterpret_cast<const float4 *>(P.A + k + 4);
        a[p][0] = v0.x; a[p][1] = v0.y; a[p][2] = v0.z; a[p][3] = v0.w; a[p][4] = v1.x; a[p][5] = v1.y; a[p][6] = v1.z; a[p][7] = v1.w;
        g[p] = *reinterpret_cast<const u32x4v *>(P.norm_w + k);
    }
    __builtin_amdgcn_sched_barrier(0);
    request(n, w);
    if (P.bias) b = bf2f(P.bias[n]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int p = 0; p < NP; p++)
        if (512 * p + 8 * lane < P.K) s += ((a[p][0] + a[p][1]) + (a[p][2] + a[p][3])) + ((a[p][4] + a[p][5]) + (a[p][6] + a[p][7]));
    const float mean = wave_sum(s) / (float)P.K;
    float q = 0.0f;
#pragma unroll
    for (int p = 0; p < NP; p++)
        if (512 * p + 8 * lane < P.K) {
#pragma unroll
            for (int e = 0; e < 8; e++) { a[p][e] -= mean; q = fmaf(a[p][e], a[p][e], q); }
        }
    const float rstd = 1.0f / sqrtf(wave_sum(q) / (float)P.K + P.norm_eps);
#pragma unroll
    for (int p = 0; p < NP; p++) {
        const bool in = 512 * p + 8 * lane < P.K;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            a[p][2 * e] = in ? a[p][2 * e] * rstd * __uint_as_float(g[p][e] << 16) : 0.0f;
            a[p][2 * e + 1] = in ? a[p][2 * e + 1] * rstd * __uint_as_float(g[p][e] & 0xFFFF0000u) : 0.0f;
        }
    }
    while (true) {
        const int next = n + nwaves;
        float acc = 0.0f;
        u32x4v w2[NP];
        float b2 = 0.0f;
        if (next < P.N) { request(next, w2); if (P.bias) b2 = bf2f(P.bias[next]); }
#pragma unroll
        for (int p = 0; p < NP; p++)
            if (512 * p + 8 * lane < P.K) {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    acc = fmaf(a[p][2 * e], __uint_as_float(w[p][e] << 16), acc);
                    acc = fmaf(a[p][2 * e + 1], __uint_as_float(w[p][e] & 0xFFFF0000u), acc);
                }
            }
        acc = wave_sum(acc) + b;
        if (lane == 0) {
            if (n >= P.act_c0 && n < P.act_c1) acc = silu_exact(acc);
            P.C[n] = acc;
        }
        if (next >= P.N) break;
        n = next; b = b2;
#pragma unroll
        for (int p = 0; p < NP; p++) w[p] = w2[p];
    }
}

} // namespace

static int linear_launch(const void *w_bf16, size_t rows, size_t cols, const void *a_f32, size_t lda, size_t tokens, const void *bias_bf16,
                         const void *mul_bf16, float alpha, int accumulate, int ops32, void *c_f32, size_t ldc, int silu_col0, int silu_col1, int prologue,
                         const void *norm_w_bf16, float norm_eps, ifa_stream stream, const char *who, int act = 0, const float *row_gate = nullptr, size_t ld_gate = 0)
{
    IFA_REQUIRE(w_bf16 && a_f32 && c_f32, "%s: null pointer", who);
    IFA_REQUIRE(rows > 0 && cols > 0 && tokens > 0 && lda >= cols * (prologue == 2 ? 2 : 1) && ldc >= rows, "%s: bad shape (%zu x %zu, %zu tokens, lda %zu, ldc %zu)", who, rows, cols, tokens, lda, ldc);
    IFA_REQUIRE(rows < (1u << 30) && cols < (1u << 30) && tokens < (1u << 30), "%s: dimension too large", who);
    LinArgs P;
    P.W = (const bf16_t *)w_bf16; P.A = (const float *)a_f32; P.C = (float *)c_f32;
    P.bias = (const bf16_t *)bias_bf16; P.mul = (const bf16_t *)mul_bf16;
    P.T = (int)tokens; P.N = (int)rows; P.K = (int)cols; P.lda = (int)lda; P.ldc = (int)ldc;
    P.alpha = alpha; P.accumulate = accumulate ? 1 : 0; P.act_c0 = silu_col0; P.act_c1 = silu_col1;
    P.norm_w = (const bf16_t *)norm_w_bf16; P.norm_eps = norm_eps;
    P.tile_map = P.n_tiles = P.a_rows = nullptr; P.row_scale = nullptr; P.act_kind = act; P.C16 = nullptr;
    // 16-byte requests need whole 8-element pieces in every row of both operands
    P.vec = (cols % 8 == 0 && lda % 4 == 0 && ((uintptr_t)a_f32 & 15) == 0 && ((uintptr_t)w_bf16 & 15) == 0) ? 1 : 0;
    hipStream_t s = ifa_s(stream);
    if (prologue) {
        IFA_REQUIRE(prologue == 1 || prologue == 2, "%s: prologue %d", who, prologue);
        IFA_REQUIRE(tokens <= 8 && P.vec, "%s: a fused prologue needs at most 8 rows and 16-byte aligned rows of whole 8-element pieces", who);
        IFA_REQUIRE(prologue != 1 || (norm_w_bf16 && ((uintptr_t)norm_w_bf16 & 15) == 0), "%s: the norm's weight is missing or unaligned", who);
    }
    if (tokens == 1 && prologue == 1 && cols <= 8 * 512 && !mul_bf16 && alpha == 1.0f && !accumulate && act == 0) {
        // (up to 16 waves a compute unit: 4096 of them share the output rows)
        const unsigned grid = (unsigned)std::min<size_t>((rows + 3) / 4, 1024);
        if (cols <= 2 * 512) hipLaunchKernelGGL(k_lin_row_norm<2>, dim3(grid), dim3(256), 0, s, P);
        else if (cols <= 4 * 512) hipLaunchKernelGGL(k_lin_row_norm<4>, dim3(grid), dim3(256), 0, s, P);
        else hipLaunchKernelGGL(k_lin_row_norm<8>, dim3(grid), dim3(256), 0, s, P);
    } else if (row_gate) {
        IFA_REQUIRE(tokens <= 8 && !prologue, "%s: %zu rows (at most 8) with a gate", who, tokens);
        LinGatedArgs G;
        static_cast<LinArgs &>(G) = P;
        G.row_gate = row_gate; G.ld_gate = (int)ld_gate;
        launch_lin_rows(G, s);
    } else if (tokens <= 8 && !prologue) {
        launch_lin_rows(P, s);
    } else if (tokens <= 8) {
        const unsigned grid = (unsigned)std::min<size_t>((rows + 3) / 4, 8192);
#define IFA_LR(TT) { if (prologue == 1) hipLaunchKernelGGL((k_lin_rows<TT, 1>), dim3(grid), dim3(256), 0, s, P); else hipLaunchKernelGGL((k_lin_rows<TT, 2>), dim3(grid), dim3(256), 0, s, P); }
        if (tokens == 1) IFA_LR(1) else if (tokens == 2) IFA_LR(2) else if (tokens <= 4) IFA_LR(4) else if (tokens <= 6) IFA_LR(6) else IFA_LR(8)
#undef IFA_LR
    } else {
        const dim3 grid(ifa_cdiv(rows, LM_N), ifa_cdiv(tokens, LM_T));
        if (ops32) hipLaunchKernelGGL(k_lin_mfma<true>, grid, dim3(256), 0, s, P);
        else hipLaunchKernelGGL(k_lin_mfma<false>, grid, dim3(256), 0, s, P);
    }
    IFA_LAUNCH_CHECK();
    return IFA_OK;
}

int ifa_linear_bf16w_gated_rows(const void *w_bf16, size_t rows, size_t cols, const void *a_f32, size_t lda, size_t tokens, const void *row_gate_f32, size_t ld_gate, int accumulate, void *c_f32,
                                size_t ldc, ifa_stream stream)
{
    IFA_REQUIRE(row_gate_f32 && tokens <= 8 && ld_gate < (1u << 30), "linear_bf16w_gated_rows: %zu rows (at most 8), or no gate", tokens);
    return linear_launch(w_bf16, rows, cols, a_f32, lda, tokens, nullptr, nullptr, 1.0f, accumulate, 1, c_f32, ldc, 0, 0, 0, nullptr, 0.0f, stream, "linear_bf16w_gated_rows", 0,
                         (const float *)row_gate_f32, ld_gate);
}

bool ifa_linear_bf16w_glu_rows(const void *w_bf16, size_t rows, size_t cols, const void *a_f32, size_t lda, size_t tokens, const void *bias_bf16, void *c_f32, size_t ldc, int silu_col0,
                               int silu_col1, size_t glu_col0, size_t glu_cols, int glu_kind, float glu_limit, void *g_f32, size_t ldg, ifa_stream stream)
{
    if (!w_bf16 || !a_f32 || !g_f32 || (!c_f32 && glu_col0) || tokens == 0 || tokens > 8 || cols == 0 || cols % 8 || lda < cols || lda % 4 || ((uintptr_t)a_f32 & 15) || ((uintptr_t)w_bf16 & 15)
        || ldc < glu_col0 || glu_cols == 0 || glu_col0 + 2 * glu_cols > rows || ldg < glu_cols || rows >= (1u << 30) || cols >= (1u << 30) || lda >= (1u << 30) || ldc >= (1u << 30)
        || ldg >= (1u << 30) || glu_kind < 0 || glu_kind > 3 || (glu_kind == 3 && !(glu_limit > 0.0f))) return false;
    LinGluArgs P;
    memset(&P, 0, sizeof(P));
    P.W = (const bf16_t *)w_bf16; P.A = (const float *)a_f32; P.C = (float *)c_f32; P.bias = (const bf16_t *)bias_bf16; P.T = (int)tokens; P.N = (int)rows; P.K = (int)cols; P.lda = (int)lda;
    P.ldc = (int)ldc; P.alpha = 1.0f; P.vec = 1; P.act_c0 = silu_col0; P.act_c1 = silu_col1; P.G = (float *)g_f32; P.ldg = (int)ldg; P.glu_c0 = (int)glu_col0; P.glu_f = (int)glu_cols;
    P.glu_kind = glu_kind; P.glu_limit = glu_limit;
    launch_lin_rows_group<2>(P, ifa_s(stream));
    return true;
}

extern "C" int ifa_linear_bf16w(const void *w_bf16, size_t rows, size_t cols, const void *a_f32, size_t lda, size_t tokens,
                                const void *bias_bf16, const void *mul_bf16, float alpha, int accumulate, int ops32,
                                void *c_f32, size_t ldc, int silu_col0, int silu_col1, ifa_stream stream)
{
    return linear_launch(w_bf16, rows, cols, a_f32, lda, tokens, bias_bf16, mul_bf16, alpha, accumulate, ops32, c_f32, ldc, silu_col0, silu_col1, 0, nullptr, 0.0f,
                         stream, "ifa_linear_bf16w");
}

int ifa_rows_to_bf16_part(const void *x_f32, size_t ldx, size_t rows, size_t cols, void *y_bf16, size_t width, size_t ldy, ifa_stream stream)
{
    IFA_REQUIRE(x_f32 && y_bf16, "ifa_rows_to_bf16: null pointer");
    IFA_REQUIRE(rows > 0 && rows < 65536u * 16u && cols > 0 && ldx >= cols && width >= cols && width % 8 == 0 && ldy >= width && ldy % 8 == 0 && ldy < (1u << 30)
                && ((uintptr_t)y_bf16 & 15) == 0, "ifa_rows_to_bf16: bad shape");
    const int vec = ldx % 4 == 0 && ((uintptr_t)x_f32 & 15) == 0;
    for (size_t r0 = 0; r0 < rows; r0 += 65535) {
        const size_t n = std::min<size_t>(65535, rows - r0);
        hipLaunchKernelGGL(k_rows_to_bf16, dim3(ifa_cdiv(width / 8, 256), (unsigned)n), dim3(256), 0, ifa_s(stream), (const float *)x_f32 + r0 * ldx, ldx, (int)cols,
                           (bf16_t *)y_bf16 + r0 * ldy, (int)width, (int)ldy, vec);
    }
    IFA_LAUNCH_CHECK();
    return IFA_OK;
}

extern "C" int ifa_rows_to_bf16(const void *x_f32, size_t ldx, size_t rows, size_t cols, void *y_bf16, size_t ldy, ifa_stream stream)
{
    return ifa_rows_to_bf16_part(x_f32, ldx, rows, cols, y_bf16, ldy, ldy, stream);
}

extern "C" int ifa_linear_bf16_both(const void *w_bf16, size_t rows, size_t cols, const void *a_bf16, size_t lda, size_t tokens, const void *bias_bf16, const void *mul_bf16,
                                    float alpha, int accumulate, int act, void *c_f32, void *c_bf16, size_t ldc, int silu_col0, int silu_col1, ifa_stream stream)
{
    IFA_REQUIRE(w_bf16 && a_bf16 && (c_f32 || c_bf16), "ifa_linear_bf16_both: null pointer");
    IFA_REQUIRE(rows > 0 && cols >= (size_t)LT_BK && cols % 8 == 0 && tokens > 0 && lda % 64 == 0 && lda >= cols && lda - cols < 64 && ldc >= rows && act >= 0 && act <= 2,
                "ifa_linear_bf16_both: bad shape (%zu x %zu, %zu tokens, lda %zu)", rows, cols, tokens, lda);
    IFA_REQUIRE(!c_bf16 || (act == 2 && !accumulate), "ifa_linear_bf16_both: a bfloat16 output goes with the squared relu and no accumulation");
    IFA_REQUIRE(rows < (1u << 30) && cols < (1u << 30) && tokens < (1u << 30) && (((uintptr_t)a_bf16 | (uintptr_t)w_bf16) & 15) == 0, "ifa_linear_bf16_both: dimension too large or unaligned operand");
    LinArgs P;
    memset(&P, 0, sizeof(P));
    P.W = (const bf16_t *)w_bf16; P.C = (float *)c_f32; P.C16 = (bf16_t *)c_bf16; P.bias = (const bf16_t *)bias_bf16; P.mul = (const bf16_t *)mul_bf16;
    P.T = (int)tokens; P.N = (int)rows; P.K = (int)cols; P.ldc = (int)ldc; P.alpha = alpha; P.accumulate = accumulate ? 1 : 0; P.act_c0 = silu_col0; P.act_c1 = silu_col1;
    P.act_kind = act;
    hipStream_t s = ifa_s(stream);
    const bf16_t *a = (const bf16_t *)a_bf16;
    return lin_tile_dispatch<0>(P, a, lda, s);
}

// Few tiles of many steps leave most of the chip idle: the steps are shared out over KS workgroups a tile, the first of which adds into C while the others leave their sums in planes
// [KS - 1][tokens][rows] for the launch that reads C next.  us a Gelarax layer's sum, one workgroup a tile / shared out, width 1024: 37 tokens 28.0 / 12.6 (32 x 32 tiles by eight), 200
// tokens 28 / 16.6 (64 x 64 by eight), 601 29.8 / 22.0 (128 x 64 by two); whole prompts of 9, 37, 128, 411, 601 tokens 643, 817, 1071, 1228, 1267 -> 506, 690, 954, 1146, 1219, width 2048 977, 1139, 1416,
// 1788, 2061 -> 728, 898, 1211, 1740, 1960.  (Of the choices tried at each of those lengths -- four shapes by three, four, six, eight -- the model's is within 3 % of the fastest prompt.)
struct LinSumPlan { int shape, ks; };
static LinSumPlan lin_sum_plan(size_t T, size_t N, size_t steps)
{
    const size_t t128 = (T + 127) / 128, t64 = (T + 63) / 64, t32 = (T + 31) / 32, n128 = (N + 127) / 128, n64 = (N + 63) / 64, n32 = (N + 31) / 32;
    const struct { LinShape h; size_t tiles; int buffers; } shapes[] = {{LT_SHAPES[LT_128x128], t128 * n128, 4}, {LT_SHAPES[LT_128x64], t128 * n64, 4}, {LT_SHAPES[LT_64x64], t64 * n64, 5},
                                                                        {{2, 0.20, 0.32, 0.32, 3.5}, t32 * n32, 8}};
    LinSumPlan best = {-1, 1};
    double cost = 0;
    for (int k = 0; k < 4; k++)
        for (int z = 1; z <= 1 + IFA_SUM_PLANES; z++) {
            if (steps / z < (size_t)shapes[k].buffers || shapes[k].tiles * z >= (1u << 31)) continue;
            // (a plane is written here and read by the next launch, 3 TB/s; not for less than 15 %, what the model is worth)
            const double c = (lin_cost(shapes[k].h, shapes[k].tiles * z, (steps + z - 1) / z) + (z > 1 ? 0.5 : 0.0) + (z - 1) * (0.1 + T * N * 8 / 3.0e6)) / (z > 1 ? 0.85 : 1.0);
            if (best.shape < 0 || c < cost) { best = {k, z}; cost = c; }
        }
    return best;
}

int ifa_linear_bf16_sum_plane_count(size_t rows, size_t lda, size_t tokens) { return rows && tokens && lda ? lin_sum_plan(tokens, rows, lda / LT_BK).ks - 1 : 0; }

int ifa_linear_bf16_sum_planes(const IfaSumPart *parts, int n_parts, size_t rows, const void *a_bf16, size_t lda, size_t tokens, void *c_f32, size_t ldc, float *planes,
                               ifa_stream stream)
{
    IFA_REQUIRE(parts && a_bf16 && c_f32 && n_parts >= 1 && n_parts <= IFA_SUM_PARTS, "linear_bf16_sum: null pointer or %d parts", n_parts);
    IFA_REQUIRE(rows > 0 && tokens > 0 && ldc >= rows && rows < (1u << 30) && tokens < (1u << 30) && lda < (1u << 30) && ((uintptr_t)a_bf16 & 15) == 0, "linear_bf16_sum: bad shape");
    LinSumArgs P;
    memset(&P, 0, sizeof(P));
    P.C = (float *)c_f32; P.T = (int)tokens; P.N = (int)rows; P.ldc = (int)ldc; P.planes = planes; P.ks = 1;
    size_t at = 0;
    for (int k = 0; k < n_parts; k++) {
        const IfaSumPart &p = parts[k];
        IFA_REQUIRE(p.w && ((uintptr_t)p.w & 15) == 0 && p.cols >= (size_t)LT_BK && p.cols % 8 == 0, "linear_bf16_sum: part %d of %zu columns", k, p.cols);
        P.part[k].W = (const bf16_t *)p.w; P.part[k].mul = (const bf16_t *)p.mul; P.part[k].bias = (const bf16_t *)p.bias; P.part[k].K = (int)p.cols;
        P.part[k].steps = (int)((p.cols + LT_BK - 1) / LT_BK); P.part[k].alpha = p.alpha;
        at += (size_t)P.part[k].steps * LT_BK;
    }
    IFA_REQUIRE(at == lda, "linear_bf16_sum: parts of %zu columns in rows of %zu", at, lda);
    const bf16_t *a = (const bf16_t *)a_bf16;
    const LinSumPlan plan = planes ? lin_sum_plan(tokens, rows, lda / LT_BK) : LinSumPlan{0, 1};
    if (plan.ks == 1) return lin_tile_dispatch<LT_SUM>(P, a, lda, ifa_s(stream));
    P.ks = plan.ks;
    const size_t t128 = (tokens + 127) / 128;
    switch (plan.shape) {
    case 0: return launch_lin_tile<128, 128, 2, 4, 4, LT_SUM | LT_SPLIT>(P, a, lda, t128, ifa_s(stream));
    case 1: return launch_lin_tile<128, 64, 4, 2, 4, LT_SUM | LT_SPLIT>(P, a, lda, t128, ifa_s(stream));
    case 2: return launch_lin_tile<64, 64, 2, 2, 5, LT_SUM | LT_SPLIT>(P, a, lda, (tokens + 63) / 64, ifa_s(stream));
    default: return launch_lin_tile<32, 32, 1, 1, 8, LT_SUM | LT_SPLIT>(P, a, lda, (tokens + 31) / 32, ifa_s(stream));
    }
}

int ifa_linear_bf16_sum(const IfaSumPart *parts, int n_parts, size_t rows, const void *a_bf16, size_t lda, size_t tokens, void *c_f32, size_t ldc, ifa_stream stream)
{
    return ifa_linear_bf16_sum_planes(parts, n_parts, rows, a_bf16, lda, tokens, c_f32, ldc, nullptr, stream);
}

int ifa_linear_bf16_glu(const void *w_bf16, size_t rows, size_t cols, const void *a_bf16, size_t lda, size_t tokens, const void *bias_bf16, void *c_f32, size_t ldc, int silu_col0,
                        int silu_col1, size_t glu_col0, size_t glu_cols, int glu_kind, float glu_limit, void *glu_bf16, size_t ldg, ifa_stream stream)
{
    IFA_REQUIRE(w_bf16 && a_bf16 && glu_bf16 && (c_f32 || glu_col0 == 0), "linear_bf16_glu: null pointer");
    IFA_REQUIRE(rows > 0 && cols >= (size_t)LT_BK && cols % 8 == 0 && tokens > 0 && lda % 64 == 0 && lda >= cols && lda - cols < 64 && ldc >= glu_col0 && glu_cols > 0
                && glu_col0 + 2 * glu_cols <= rows && ldg >= ((glu_cols + 63) & ~(size_t)63) && ldg < (1u << 30) && glu_kind >= 0 && glu_kind <= 3 && (glu_kind != 3 || glu_limit > 0.0f),
                "linear_bf16_glu: bad shape (%zu x %zu, %zu tokens, lda %zu, gate | up %zu + 2 x %zu)", rows, cols, tokens, lda, glu_col0, glu_cols);
    IFA_REQUIRE(rows < (1u << 30) && cols < (1u << 30) && tokens < (1u << 30) && (((uintptr_t)a_bf16 | (uintptr_t)w_bf16) & 15) == 0, "linear_bf16_glu: dimension too large or unaligned operand");
    LinGluArgs P;
    memset(&P, 0, sizeof(P));
    P.W = (const bf16_t *)w_bf16; P.C = (float *)c_f32; P.bias = (const bf16_t *)bias_bf16; P.T = (int)tokens; P.N = (int)rows; P.K = (int)cols; P.ldc = (int)ldc; P.alpha = 1.0f;
    P.act_c0 = silu_col0; P.act_c1 = silu_col1; P.G16 = (bf16_t *)glu_bf16; P.ldg = (int)ldg; P.glu_c0 = (int)glu_col0; P.glu_f = (int)glu_cols;
    P.glu_w = (P.glu_f + 63) & ~63; P.glu_kind = glu_kind; P.glu_limit = glu_limit;
    return lin_tile_dispatch<LT_GLU>(P, (const bf16_t *)a_bf16, lda, ifa_s(stream));
}

// ifa_linear_bf16w_grouped over bfloat16 rows (as ifa_linear_bf16_both reads them), tiles of at most tile_rows = 64 or 128 rows of one group
int ifa_linear_bf16_grouped(const void *w_bf16, size_t rows, size_t cols, const void *a_bf16, size_t lda, const int *a_rows_dev, const int *tile_map_dev, const int *n_tiles_dev,
                            size_t max_tiles, int tile_rows, const void *row_scale_f32, void *c_f32, size_t ldc, int glu_kind, float glu_limit, void *glu_bf16, ifa_stream stream)
{
    IFA_REQUIRE(w_bf16 && a_bf16 && (c_f32 || glu_bf16) && tile_map_dev && n_tiles_dev, "linear_bf16_grouped: null pointer");
    IFA_REQUIRE(!glu_bf16 || (rows % 2 == 0 && ldc % 64 == 0 && ldc >= rows / 2 && ldc - rows / 2 < 64 && !row_scale_f32 && glu_kind >= 0 && glu_kind <= 3 && (glu_kind != 3 || glu_limit > 0.0f)),
                "linear_bf16_grouped: bad gate | up (%zu rows, ldc %zu)", rows, ldc);
    IFA_REQUIRE(rows > 0 && cols >= (size_t)LT_BK && cols % 8 == 0 && max_tiles > 0 && lda % 64 == 0 && lda >= cols && lda - cols < 64 && (glu_bf16 || ldc >= rows)
                && (tile_rows == 64 || tile_rows == 128) && rows < (1u << 30) && cols < (1u << 30) && (((uintptr_t)a_bf16 | (uintptr_t)w_bf16) & 15) == 0,
                "linear_bf16_grouped: bad shape (%zu x %zu, lda %zu)", rows, cols, lda);
    LinGluArgs P;
    memset(&P, 0, sizeof(P));
    P.W = (const bf16_t *)w_bf16; P.C = (float *)c_f32; P.N = (int)rows; P.K = (int)cols; P.ldc = (int)ldc; P.alpha = 1.0f;
    P.tile_map = tile_map_dev; P.n_tiles = n_tiles_dev; P.a_rows = a_rows_dev; P.row_scale = (const float *)row_scale_f32;
    const bf16_t *a = (const bf16_t *)a_bf16;
    hipStream_t s = ifa_s(stream);
    if (glu_bf16) {          // (all columns are gate | up)
        P.G16 = (bf16_t *)glu_bf16; P.ldg = P.glu_w = (int)ldc; P.glu_f = (int)(rows / 2); P.glu_kind = glu_kind; P.glu_limit = glu_limit;
        return lin_grouped_dispatch<LT_GROUPED | LT_GLU>(P, a, lda, max_tiles, tile_rows, s);
    }
    return lin_grouped_dispatch<LT_GROUPED>(P, a, lda, max_tiles, tile_rows, s);
}

extern "C" int ifa_linear_bf16w_act(const void *w_bf16, size_t rows, size_t cols, const void *a_f32, size_t lda, size_t tokens, const void *bias_bf16, int act,
                                    int ops32, void *c_f32, size_t ldc, ifa_stream stream)
{
    IFA_REQUIRE(act >= 0 && act <= 2, "ifa_linear_bf16w_act: activation %d", act);
    return linear_launch(w_bf16, rows, cols, a_f32, lda, tokens, bias_bf16, nullptr, 1.0f, 0, ops32, c_f32, ldc, 0, 0, 0, nullptr, 0.0f, stream, "ifa_linear_bf16w_act", act);
}

extern "C" int ifa_linear_bf16w_rows(int prologue, const void *norm_w_bf16, float norm_eps, const void *w_bf16, size_t rows, size_t cols, const void *a_f32,
                                     size_t lda, size_t tokens, const void *bias_bf16, const void *mul_bf16, float alpha, int accumulate, void *c_f32,
                                     size_t ldc, int silu_col0, int silu_col1, ifa_stream stream)
{
    IFA_REQUIRE(tokens <= 8, "ifa_linear_bf16w_rows: %zu rows (at most 8)", tokens);
    return linear_launch(w_bf16, rows, cols, a_f32, lda, tokens, bias_bf16, mul_bf16, alpha, accumulate, 1, c_f32, ldc, silu_col0, silu_col1, prologue,
                         norm_w_bf16, norm_eps, stream, "ifa_linear_bf16w_rows");
}

// Grouped product on the matrix cores: `groups` matrices [rows][cols] back to back in w_bf16; the output rows are sorted by group and
// cut into tiles of at most 64 rows of ONE group: tile_map_dev[3 i] = {group, first row, rows}, *n_tiles_dev tiles (max_tiles bounds the
// grid).  C[r][n] = row_scale[r] * act(sum_k A[a_rows[r]][k] W_group[n][k]); a_rows_dev / row_scale_f32 nullable; act 0 none, 1 erf-GELU.
extern "C" int ifa_linear_bf16w_grouped(const void *w_bf16, size_t rows, size_t cols, int groups, const void *a_f32, size_t lda, const int *a_rows_dev,
                                        const int *tile_map_dev, const int *n_tiles_dev, size_t max_tiles, const void *row_scale_f32, int act, int ops32,
                                        void *c_f32, size_t ldc, ifa_stream stream)
{
    IFA_REQUIRE(w_bf16 && a_f32 && c_f32 && tile_map_dev && n_tiles_dev, "ifa_linear_bf16w_grouped: null pointer");
    IFA_REQUIRE(rows > 0 && cols > 0 && groups > 0 && max_tiles > 0 && max_tiles < 65536 && lda >= cols && ldc >= rows && (act == 0 || act == 1), "ifa_linear_bf16w_grouped: bad shape");
    IFA_REQUIRE(rows < (1u << 30) && cols < (1u << 30), "ifa_linear_bf16w_grouped: dimension too large");
    LinArgs P;
    P.W = (const bf16_t *)w_bf16; P.A = (const float *)a_f32; P.C = (float *)c_f32; P.bias = nullptr; P.mul = nullptr;
    P.T = 0; P.N = (int)rows; P.K = (int)cols; P.lda = (int)lda; P.ldc = (int)ldc; P.alpha = 1.0f; P.accumulate = 0; P.act_c0 = P.act_c1 = 0;
    P.norm_w = nullptr; P.norm_eps = 0.0f;
    P.tile_map = tile_map_dev; P.n_tiles = n_tiles_dev; P.a_rows = a_rows_dev; P.row_scale = (const float *)row_scale_f32; P.act_kind = act; P.C16 = nullptr;
    P.vec = (cols % 8 == 0 && lda % 4 == 0 && ((uintptr_t)a_f32 & 15) == 0 && ((uintptr_t)w_bf16 & 15) == 0 && (rows * cols) % 8 == 0) ? 1 : 0;
    const dim3 grid(ifa_cdiv(rows, LM_N), (unsigned)max_tiles);
    if (ops32) hipLaunchKernelGGL(k_lin_mfma<true>, grid, dim3(256), 0, ifa_s(stream), P);
    else hipLaunchKernelGGL(k_lin_mfma<false>, grid, dim3(256), 0, ifa_s(stream), P);
    IFA_LAUNCH_CHECK();
    return IFA_OK;
}
