// ifa_moe_f32.hip -- mixture of experts on 32-bit activations with bfloat16 expert matrices:
//   router   scores = softmax(logits) over `experts` feed-forward experts followed by `identity` identity experts; the `top` largest
//            (score + correction) are chosen, their weights are the plain scores (not renormalized)
//            (renorm: the chosen scores are divided by their sum and multiplied by a scale)
//            (second kind, k_moe_route_top: the `top` largest logit + bias, weights = softmax over the chosen values only)
//   experts  y[t] (+)= sum_k wgt[t][k] * E_{idx[t][k]}(h[t]),  E_e(h) = W_down[e] act(W_up[e] h),  identity: E(h) = h
//            (gated experts: E_e(h) = W_down[e] (silu(W_gate[e] h) * (W_up[e] h)), gate and up rows of an expert stored back to back)
// Few rows (decode steps): every (row, choice) pair streams its expert's matrices, a wave per output (k_moe_up_rows / k_moe_down_rows).
// Many rows: the pairs are sorted by expert (counts, offsets and tiles of rows of one expert), both products run grouped on the matrix
// cores (gather of the rows in the first, activation in its epilogue, the pair's weight in the second's), and a row's pairs are added in
// the fixed order of its choices.  ifa_moe_prompt (choice by the largest logits, bfloat16 rows, up to 512 experts): sorted by many
// workgroups (k_moe_route_count, k_moe_place_glu), added by the norm behind (k_norm_add_norm_reg, ifa_ops_f32.hip).  Otherwise sorted
// by one (k_moe_sort) and added by k_moe_combine.  No atomics on values: a row's result does not depend on what else is in the step.
#include <algorithm>
#include <cstring>
#include "ifa_host.h"
#include "ifa_f32_common.h"
#include "inferflow_amd.h"
#include "ifa_rows_fused.h"

using namespace ifa32;

namespace {

typedef uint32_t u32x4m __attribute__((ext_vector_type(4)));

// What a choice compares: a score that is no number comes last, with those of -inf, and an entry already taken (NaN from there on) compares with nothing.
// So every pass finds an entry of the row, and no entry twice, whatever the scores are: the experts read their weights by these indices.
__device__ __forceinline__ float choice_of(float v) { return v == v ? v : -INFINITY; }

__device__ __forceinline__ float gelu_erf_f(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }

// one wave per row: softmax over n_all logits, then `top` passes of argmax over score + correction (lowest index on ties)
// (score_kind 1: the scores are the sigmoids of the logits instead of their softmax)
__global__ void __launch_bounds__(64) k_moe_route(const float *__restrict__ logits, size_t ld, int n_all, int top, const bf16_t *__restrict__ corr,
                                                  int *__restrict__ idx, float *__restrict__ wgt, int score_kind, int renorm, float renorm_eps, float wgt_scale)
{
    extern __shared__ float sc[];          // [n_all] scores, [n_all] choice scores
    float *ch = sc + n_all;
    const int t = blockIdx.x, lane = threadIdx.x;
    const float *z = logits + (size_t)t * ld;
    if (score_kind == 1) {
        for (int e = lane; e < n_all; e += 64) { const float s = sigmoid_f(z[e]); sc[e] = s; ch[e] = choice_of(s + (corr ? bf2f(corr[e]) : 0.0f)); }
    } else {
        float mx = -INFINITY;
        for (int e = lane; e < n_all; e += 64) mx = fmaxf(mx, z[e]);
        mx = wave_max(mx);
        float sum = 0.0f;
        for (int e = lane; e < n_all; e += 64) { const float p = expf(z[e] - mx); sc[e] = p; sum += p; }
        sum = wave_sum(sum);
        for (int e = lane; e < n_all; e += 64) { const float s = sc[e] / sum; sc[e] = s; ch[e] = choice_of(s + (corr ? bf2f(corr[e]) : 0.0f)); }
    }
    __syncthreads();
    float sum = 0.0f;          // (lane 0: of the chosen scores)
    for (int k = 0; k < top; k++) {
        float best = -INFINITY; int bi = 0x7FFFFFFF;
        for (int e = lane; e < n_all; e += 64) { const float v = ch[e]; if (v > best || (v == best && e < bi)) { best = v; bi = e; } }
        for (int o = 32; o > 0; o >>= 1) {
            const float ov = __shfl_xor(best, o, 64); const int oi = __shfl_xor(bi, o, 64);
            if (ov > best || (ov == best && oi < bi)) { best = ov; bi = oi; }
        }
        if (lane == 0) { idx[(size_t)t * top + k] = bi; wgt[(size_t)t * top + k] = sc[bi]; ch[bi] = NAN; sum += sc[bi]; }
        __syncthreads();
    }
    if (renorm && lane == 0) { const float den = sum + renorm_eps; for (int k = 0; k < top; k++) wgt[(size_t)t * top + k] = wgt[(size_t)t * top + k] / den * wgt_scale; }
}

// one wave per row: `top` passes of argmax over logit + bias (lowest index on ties), then the softmax over the chosen values
__global__ void __launch_bounds__(64) k_moe_route_top(const float *__restrict__ logits, size_t ld, int n_all, int top, const bf16_t *__restrict__ bias,
                                                      int *__restrict__ idx, float *__restrict__ wgt)
{
    extern __shared__ float ch[];          // [n_all] choice values, [top] weights before the division
    float *pw = ch + n_all;
    const int t = blockIdx.x, lane = threadIdx.x;
    const float *z = logits + (size_t)t * ld;
    for (int e = lane; e < n_all; e += 64) ch[e] = choice_of(z[e] + (bias ? bf2f(bias[e]) : 0.0f));
    __syncthreads();
    float first = 0.0f, sum = 0.0f;
    for (int k = 0; k < top; k++) {
        float best = -INFINITY; int bi = 0x7FFFFFFF;
        for (int e = lane; e < n_all; e += 64) { const float v = ch[e]; if (v > best || (v == best && e < bi)) { best = v; bi = e; } }
        for (int o = 32; o > 0; o >>= 1) {
            const float ov = __shfl_xor(best, o, 64); const int oi = __shfl_xor(bi, o, 64);
            if (ov > best || (ov == best && oi < bi)) { best = ov; bi = oi; }
        }
        if (k == 0) first = best;                      // the largest of all: the softmax's reference
        const float p = expf(best - first);
        sum += p;
        if (lane == 0) { idx[(size_t)t * top + k] = bi; pw[k] = p; ch[bi] = NAN; }
        __syncthreads();
    }
    for (int k = lane; k < top; k += 64) wgt[(size_t)t * top + k] = pw[k] / sum;
}

// Steps of a few rows: the router's product and its choice in one launch.  A workgroup per row: the waves share out the router's outputs
// (a dot of `width` each), then the scores and the `top` passes as in k_moe_route (wave 0; the other waves only keep the barriers).
// (x not null: the row the router reads is formed here first, h[t] = tanh(alpha x[t]) nw + nb, and written for the experts behind)
__global__ void __launch_bounds__(1024) k_moe_route_rows(const float *h, size_t ldh, int W, const bf16_t *__restrict__ router, int n_all, int top,
                                                        const bf16_t *__restrict__ corr, int *__restrict__ idx, float *__restrict__ wgt, int vec, int score_kind,
                                                        const float *__restrict__ x, size_t ldx, const bf16_t *__restrict__ alpha, const bf16_t *__restrict__ nw_,
                                                        const bf16_t *__restrict__ nb_, float *h_out, int renorm, float renorm_eps, float wgt_scale)
{
    extern __shared__ float sc[];          // [n_all] logits, then scores; [n_all] choice scores
    float *ch = sc + n_all;
    const int t = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const float *hr = h + (size_t)t * ldh;
    if (x) {
        const float a = bf2f(alpha[0]);
        for (int c = threadIdx.x; c < W; c += blockDim.x) h_out[(size_t)t * ldh + c] = fmaf(tanhf(a * x[(size_t)t * ldx + c]), bf2f(nw_[c]), bf2f(nb_[c]));
        __syncthreads();          // (the workgroup reads back what it has written itself)
    }
    for (int e = wave; e < n_all; e += nw) {
        const bf16_t *w = router + (size_t)e * W;
        float acc = 0.0f;
        if (vec) {
#pragma unroll 4
            for (int k = lane * 8; k < W; k += 512) {
                const u32x4m wv = *reinterpret_cast<const u32x4m *>(w + k);
                const float4 a0 = *reinterpret_cast<const float4 *>(hr + k), a1 = *reinterpret_cast<const float4 *>(hr + k + 4);
                acc = fmaf(a0.x, __uint_as_float(wv[0] << 16), acc); acc = fmaf(a0.y, __uint_as_float(wv[0] & 0xFFFF0000u), acc);
                acc = fmaf(a0.z, __uint_as_float(wv[1] << 16), acc); acc = fmaf(a0.w, __uint_as_float(wv[1] & 0xFFFF0000u), acc);
                acc = fmaf(a1.x, __uint_as_float(wv[2] << 16), acc); acc = fmaf(a1.y, __uint_as_float(wv[2] & 0xFFFF0000u), acc);
                acc = fmaf(a1.z, __uint_as_float(wv[3] << 16), acc); acc = fmaf(a1.w, __uint_as_float(wv[3] & 0xFFFF0000u), acc);
            }
        } else {
            for (int k = lane; k < W; k += 64) acc = fmaf(hr[k], bf2f(w[k]), acc);
        }
        acc = wave_sum(acc);
        if (lane == 0) sc[e] = acc;
    }
    __syncthreads();
    if (wave == 0 && score_kind == 1) {
        for (int e = lane; e < n_all; e += 64) { const float sv = sigmoid_f(sc[e]); sc[e] = sv; ch[e] = choice_of(sv + (corr ? bf2f(corr[e]) : 0.0f)); }
    } else if (wave == 0) {
        float mx = -INFINITY;
        for (int e = lane; e < n_all; e += 64) mx = fmaxf(mx, sc[e]);
        mx = wave_max(mx);
        float sum = 0.0f;
        for (int e = lane; e < n_all; e += 64) { const float pe = expf(sc[e] - mx); sc[e] = pe; sum += pe; }      // (each lane touches its own entries only)
        sum = wave_sum(sum);
        for (int e = lane; e < n_all; e += 64) { const float sv = sc[e] / sum; sc[e] = sv; ch[e] = choice_of(sv + (corr ? bf2f(corr[e]) : 0.0f)); }
    }
    __syncthreads();
    float chosen = 0.0f;          // (thread 0: the sum of the chosen scores)
    for (int k = 0; k < top; k++) {
        if (wave == 0) {
            float best = -INFINITY; int bi = 0x7FFFFFFF;
            for (int e = lane; e < n_all; e += 64) { const float v = ch[e]; if (v > best || (v == best && e < bi)) { best = v; bi = e; } }
            for (int o = 32; o > 0; o >>= 1) {
                const float ov = __shfl_xor(best, o, 64); const int oi = __shfl_xor(bi, o, 64);
                if (ov > best || (ov == best && oi < bi)) { best = ov; bi = oi; }
            }
            if (lane == 0) { idx[(size_t)t * top + k] = bi; wgt[(size_t)t * top + k] = sc[bi]; ch[bi] = NAN; chosen += sc[bi]; }
        }
        __syncthreads();
    }
    if (renorm && threadIdx.x == 0) { const float den = chosen + renorm_eps; for (int k = 0; k < top; k++) wgt[(size_t)t * top + k] = wgt[(size_t)t * top + k] / den * wgt_scale; }
}

// Steps of a few rows whose choice is made by the first experts' launch itself: every workgroup forms the scores of its row from the router's logits
// and finds the expert of its pair as the one whose RANK (larger choice scores, lower index on ties) is the pair's place; the pair's first
// workgroup leaves expert and weight for the launches behind.  At most 256 router outputs (one per thread).
struct RouteSel {
    const float *logits; size_t ld; int n_all, score_kind, renorm; float renorm_eps, wgt_scale;
    const bf16_t *corr; int *idx; float *wgt;
};

__device__ int route_pair(const RouteSel &R, int t, int k, int top, bool leave)
{
    __shared__ float ch[256], red[17];
    __shared__ int mine;
    const int e = threadIdx.x;
    const bool live = e < R.n_all;
    float s = live ? R.logits[(size_t)t * R.ld + e] : -INFINITY;
    if (R.score_kind == 2) s = s == s ? s : -INFINITY;          // (the logits themselves; one that is no number comes last)
    else if (R.score_kind == 1) s = live ? sigmoid_f(s) : 0.0f;
    else {          // softmax: the maximum over the row, then the sum
        const float wm = wave_max(s);
        if ((e & 63) == 0) red[e >> 6] = wm;
        __syncthreads();
        float mx = -INFINITY;
        for (int w = 0; w < (int)(blockDim.x >> 6); w++) mx = fmaxf(mx, red[w]);
        s = live ? expf(s - mx) : 0.0f;
        s /= block_sum(s, red);
    }
    float c = live ? s + (R.corr ? bf2f(R.corr[e]) : 0.0f) : -INFINITY;
    if (c != c) c = -INFINITY;          // (no number: last, so that the ranks are a permutation and every pair has an expert; its weight stays what it is)
    ch[e] = c;
    __syncthreads();
    int rank = 0;
    if (live) {
#pragma unroll 8
        for (int j = 0; j < R.n_all; j++) { const float v = ch[j]; rank += (v > c || (v == c && j < e)) ? 1 : 0; }
    }
    if (live && rank == k) mine = e;
    if (R.score_kind == 2) {          // weights: softmax over the chosen
        if (leave) {
            const float wm = wave_max(c);
            __syncthreads();
            if ((e & 63) == 0) red[e >> 6] = wm;
            __syncthreads();
            float mx = -INFINITY;
            for (int w = 0; w < (int)(blockDim.x >> 6); w++) mx = fmaxf(mx, red[w]);
            const float pe = live && rank < top ? expf(c - mx) : 0.0f, all = block_sum(pe, red);
            if (live && rank == k) { R.idx[(size_t)t * top + k] = e; R.wgt[(size_t)t * top + k] = pe / all; }
        }
        __syncthreads();
        return mine;
    }
    float sum = 0.0f;
    if (leave && R.renorm) sum = block_sum(live && rank < top ? s : 0.0f, red);
    if (leave && live && rank == k) {
        R.idx[(size_t)t * top + k] = e;
        R.wgt[(size_t)t * top + k] = R.renorm ? s / (sum + R.renorm_eps) * R.wgt_scale : s;
    }
    __syncthreads();
    return mine;
}

// grid (ff chunks, pairs): act[p][n] = gelu(W_up[e][n] . h[t]); a wave per n at a time.  Identity pairs do nothing.
template <bool GATED, bool SEL>
__global__ void __launch_bounds__(256) k_moe_up_rows(const float *__restrict__ h, size_t ldh, int W, int F, int experts, int top, const bf16_t *__restrict__ up,
                                                     const int *__restrict__ idx, float *__restrict__ act, int vec, int glu_kind, float limit, RouteSel R)
{
    const int p = blockIdx.y, e = SEL ? route_pair(R, p / top, p % top, top, blockIdx.x == 0) : idx[p];
    if (e >= experts) return;
    const int lane = threadIdx.x & 63, wave = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6), nwaves = gridDim.x * (blockDim.x >> 6);
    const float *hr = h + (size_t)(p / top) * ldh;
    if (GATED) {      // the expert's matrix holds F gate rows, then F up rows: both dots of an output side by side
        for (int n = wave; n < F; n += nwaves) {
            const bf16_t *wg = up + ((size_t)e * 2 * F + n) * W, *wu = wg + (size_t)F * W;
            float ag = 0.0f, au = 0.0f;
            if (vec) {
#pragma unroll 2
                for (int k = lane * 8; k < W; k += 512) {
                    const u32x4m gv = *reinterpret_cast<const u32x4m *>(wg + k), uv = *reinterpret_cast<const u32x4m *>(wu + k);
                    const float4 a0 = *reinterpret_cast<const float4 *>(hr + k), a1 = *reinterpret_cast<const float4 *>(hr + k + 4);
                    const float a8[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        ag = fmaf(a8[2 * j], __uint_as_float(gv[j] << 16), ag); ag = fmaf(a8[2 * j + 1], __uint_as_float(gv[j] & 0xFFFF0000u), ag);
                        au = fmaf(a8[2 * j], __uint_as_float(uv[j] << 16), au); au = fmaf(a8[2 * j + 1], __uint_as_float(uv[j] & 0xFFFF0000u), au);
                    }
                }
            } else {
                for (int k = lane; k < W; k += 64) { ag = fmaf(hr[k], bf2f(wg[k]), ag); au = fmaf(hr[k], bf2f(wu[k]), au); }
            }
            ag = wave_sum(ag); au = wave_sum(au);
            if (lane == 0) {
                if (glu_kind == 3) { const float g = fminf(ag, limit), u = fminf(fmaxf(au, -limit), limit); act[(size_t)p * F + n] = g * sigmoid_f(1.702f * g) * (u + 1.0f); }
                else act[(size_t)p * F + n] = silu_exact(ag) * au;
            }
        }
        return;
    }
    for (int n = wave; n < F; n += nwaves) {
        const bf16_t *w = up + ((size_t)e * F + n) * W;
        float acc = 0.0f;
        if (vec) {
#pragma unroll 4
            for (int k = lane * 8; k < W; k += 512) {
                const u32x4m wv = *reinterpret_cast<const u32x4m *>(w + k);
                const float4 a0 = *reinterpret_cast<const float4 *>(hr + k), a1 = *reinterpret_cast<const float4 *>(hr + k + 4);
                acc = fmaf(a0.x, __uint_as_float(wv[0] << 16), acc); acc = fmaf(a0.y, __uint_as_float(wv[0] & 0xFFFF0000u), acc);
                acc = fmaf(a0.z, __uint_as_float(wv[1] << 16), acc); acc = fmaf(a0.w, __uint_as_float(wv[1] & 0xFFFF0000u), acc);
                acc = fmaf(a1.x, __uint_as_float(wv[2] << 16), acc); acc = fmaf(a1.y, __uint_as_float(wv[2] & 0xFFFF0000u), acc);
                acc = fmaf(a1.z, __uint_as_float(wv[3] << 16), acc); acc = fmaf(a1.w, __uint_as_float(wv[3] & 0xFFFF0000u), acc);
            }
        } else {
            for (int k = lane; k < W; k += 64) acc = fmaf(hr[k], bf2f(w[k]), acc);
        }
        acc = wave_sum(acc);
        if (lane == 0) act[(size_t)p * F + n] = gelu_erf_f(acc);
    }
}

// grid (width chunks, rows): y[t][c] (+)= sum_k wgt * (identity ? h[t][c] : W_down[e][c] . act[p]); a wave per c at a time.  The chosen
// experts are walked NK at a time with their loads issued side by side (a step is bound by requests in flight: four experts take 130 registers, so that twice as many
// waves are in flight as with eight), their weighted partial sums reduced once (six rows of four experts of 704 columns 21.6 -> 12.4 us).
// SHARED: the first of the rows' workgroups (one more than rows) are the shared expert's output product of all rows (k_lin_rows' sums, times sigmoid of a row's gate) into rows of their own, which
// the norm behind adds: six rows of four experts of 704 and a shared one of 1408 to 1024 columns 13.0 + 9.8 -> 16.5 us.  (With a form for eight rows 17.9; added by the wave that has the row's sum, which reads the shared weights
// once a row: 19.9; the shared expert's workgroups behind the others: 19.7.)  A form for each number of rows (SHARED; 0: without): with eight rows in every step a model of six such layers
// took 446 / 470 / 549 / 565 / 607 / 649 us a step of 1 / 2 / 3 / 4 / 5 / 6 rows, now 432 / 457 / 530 / 555 / 597 / 645 (two launches: 460 / 496 / 555 / 599 / 653 / 680).
template <int SH_ROWS>
__device__ __forceinline__ void shared_down(const IfaMoeShared &S, int W, int wave, int nwaves)
{
    constexpr int SP = 4;          // (pieces of 512 columns asked for ahead)
    const int lane = threadIdx.x & 63;
    for (int c = wave; c < W; c += nwaves) {
        const bf16_t *w = S.down + (size_t)c * S.ff;
        float acc[SH_ROWS];
#pragma unroll
        for (int t = 0; t < SH_ROWS; t++) acc[t] = 0.0f;
        for (int k0 = 0; k0 < S.ff; k0 += 512 * SP) {
            u32x4m wv[SP];
#pragma unroll
            for (int j = 0; j < SP; j++) wv[j] = *reinterpret_cast<const u32x4m *>(w + min(k0 + 512 * j + lane * 8, S.ff - 8));
#pragma unroll
            for (int j = 0; j < SP; j++) {
                if (k0 + 512 * j >= S.ff) break;
                const int k = k0 + 512 * j + lane * 8;
                float4 a[SH_ROWS][2];
#pragma unroll
                for (int t = 0; t < SH_ROWS; t++) {
                    const float *r = S.act + (size_t)t * S.lda + min(k, S.ff - 8);
                    a[t][0] = *reinterpret_cast<const float4 *>(r); a[t][1] = *reinterpret_cast<const float4 *>(r + 4);
                }
                if (k >= S.ff) continue;
#pragma unroll
                for (int t = 0; t < SH_ROWS; t++) {
                    const float v[8] = {a[t][0].x, a[t][0].y, a[t][0].z, a[t][0].w, a[t][1].x, a[t][1].y, a[t][1].z, a[t][1].w};
#pragma unroll
                    for (int e = 0; e < 8; e++) acc[t] = fmaf(v[e], __uint_as_float((e & 1) ? (wv[j][e >> 1] & 0xFFFF0000u) : (wv[j][e >> 1] << 16)), acc[t]);
                }
            }
        }
#pragma unroll
        for (int t = 0; t < SH_ROWS; t++) acc[t] = wave_sum(acc[t]);
#pragma unroll
        for (int t = 0; t < SH_ROWS; t++)
            if (lane == t) S.out[(size_t)t * S.ldo + c] = acc[t] * sigmoid_f(S.gate[(size_t)t * S.ldg]);
    }
}
template <int NK, int SHARED>
__global__ void __launch_bounds__(256) k_moe_down_rows(const float *__restrict__ h, size_t ldh, int W, int F, int experts, int top, const bf16_t *__restrict__ down,
                                                       const int *__restrict__ idx, const float *__restrict__ wgt, const float *__restrict__ act,
                                                       int accumulate, float *__restrict__ y, size_t ldy, int vec, std::conditional_t<(SHARED > 0), IfaMoeShared, int> S)
{
    const int lane = threadIdx.x & 63, wave = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6), nwaves = gridDim.x * (blockDim.x >> 6);
    int t = blockIdx.y;
    if constexpr (SHARED > 0) {
        if (t == 0) { shared_down<SHARED>(S, W, wave, nwaves); return; }
        t--;
    }
    for (int c = wave; c < W; c += nwaves) {
        float out = 0.0f, part = 0.0f;
        for (int k0 = 0; k0 < top; k0 += NK) {
            int e[NK]; float acc[NK];
#pragma unroll
            for (int k = 0; k < NK; k++) { e[k] = k0 + k < top ? idx[t * top + k0 + k] : experts; acc[k] = 0.0f; }
            if (vec) {
                for (int j = lane * 8; j < F; j += 512) {
                    u32x4m wv[NK]; float4 a0[NK], a1[NK];
#pragma unroll
                    for (int k = 0; k < NK; k++)
                        if (e[k] < experts) {
                            wv[k] = *reinterpret_cast<const u32x4m *>(down + ((size_t)e[k] * W + c) * F + j);
                            const float *a = act + (size_t)(t * top + k0 + k) * F + j;
                            a0[k] = *reinterpret_cast<const float4 *>(a); a1[k] = *reinterpret_cast<const float4 *>(a + 4);
                        }
#pragma unroll
                    for (int k = 0; k < NK; k++)
                        if (e[k] < experts) {
                            float s = acc[k];
                            s = fmaf(a0[k].x, __uint_as_float(wv[k][0] << 16), s); s = fmaf(a0[k].y, __uint_as_float(wv[k][0] & 0xFFFF0000u), s);
                            s = fmaf(a0[k].z, __uint_as_float(wv[k][1] << 16), s); s = fmaf(a0[k].w, __uint_as_float(wv[k][1] & 0xFFFF0000u), s);
                            s = fmaf(a1[k].x, __uint_as_float(wv[k][2] << 16), s); s = fmaf(a1[k].y, __uint_as_float(wv[k][2] & 0xFFFF0000u), s);
                            s = fmaf(a1[k].z, __uint_as_float(wv[k][3] << 16), s); s = fmaf(a1[k].w, __uint_as_float(wv[k][3] & 0xFFFF0000u), s);
                            acc[k] = s;
                        }
                }
            } else {
#pragma unroll
                for (int k = 0; k < NK; k++)
                    if (e[k] < experts) {
                        const bf16_t *w = down + ((size_t)e[k] * W + c) * F;
                        const float *a = act + (size_t)(t * top + k0 + k) * F;
                        for (int j = lane; j < F; j += 64) acc[k] = fmaf(a[j], bf2f(w[j]), acc[k]);
                    }
            }
#pragma unroll
            for (int k = 0; k < NK; k++) {      // in the order of the row's choices
                if (k0 + k >= top) break;
                const float wk = wgt[t * top + k0 + k];
                if (e[k] < experts) part = fmaf(wk, acc[k], part);
                else out = fmaf(wk, h[(size_t)t * ldh + c], out);
            }
        }
        out += wave_sum(part);
        if (lane == 0) { float *d = y + (size_t)t * ldy + c; *d = accumulate ? *d + out : out; }
    }
}

// ONE workgroup: pairs (row, choice) sorted by expert.  a_rows[pos] = row of the pair at sorted place pos, pair_pos[p] = place of pair p
// (-1: identity), w_sorted[pos] = its weight, tile_map = tiles of at most tile_rows places of one expert, *n_tiles.  The place of a pair inside
// its expert's range comes from an LDS counter: the order there may differ from run to run, the values computed per pair do not.
__global__ void __launch_bounds__(1024) k_moe_sort(const int *__restrict__ idx, const float *__restrict__ wgt, int n_pairs, int experts, int top,
                                                   int *__restrict__ a_rows, int *__restrict__ pair_pos, float *__restrict__ w_sorted,
                                                   int *__restrict__ tile_map, int *__restrict__ n_tiles, int tile_rows)
{
    extern __shared__ int cnt[];           // [experts] counts, then cursors; [experts + 1] offsets
    int *off = cnt + experts;
    for (int e = threadIdx.x; e < experts; e += blockDim.x) cnt[e] = 0;
    __syncthreads();
    for (int p = threadIdx.x; p < n_pairs; p += blockDim.x) { const int e = idx[p]; if (e < experts) atomicAdd(&cnt[e], 1); }
    __syncthreads();
    if (threadIdx.x == 0) {
        int o = 0, nt = 0;
        for (int e = 0; e < experts; e++) {
            off[e] = o;
            for (int r = 0; r < cnt[e]; r += tile_rows) { tile_map[3 * nt] = e; tile_map[3 * nt + 1] = o + r; tile_map[3 * nt + 2] = min(tile_rows, cnt[e] - r); nt++; }
            o += cnt[e];
            cnt[e] = 0;
        }
        off[experts] = o;
        *n_tiles = nt;
    }
    __syncthreads();
    for (int p = threadIdx.x; p < n_pairs; p += blockDim.x) {
        const int e = idx[p];
        if (e >= experts) { pair_pos[p] = -1; continue; }
        const int pos = off[e] + atomicAdd(&cnt[e], 1);
        a_rows[pos] = p / top; pair_pos[p] = pos; w_sorted[pos] = wgt[p];
    }
}

// The same in two launches of many workgroups, for the choice by the largest logits (k_moe_route_top's, a wave a row): k_moe_route_count leaves, for each block of `rb` rows, how many of its
// pairs chose each expert, k_moe_place_glu adds these counts up and gives the pairs their places, in their order.  One workgroup took 7.8 us for 787 rows of 16 experts, top 4, and 13.6 for 2048:
// the pairs come and go through one compute unit, and its threads' counters wait for each other.  At most 512 experts (LDS) and 256 blocks (a placing workgroup reads all their counts).
constexpr int PLACE_EXPERTS = 512, PLACE_BLOCKS = 256, PLACE_WAVES = 16;
size_t route_count_smem(int experts, int top) { return ((size_t)experts + PLACE_WAVES * (size_t)(experts + top)) * 4; }
__global__ void __launch_bounds__(64 * PLACE_WAVES) k_moe_route_count(const float *__restrict__ logits, size_t ld, int experts, int top, int rows, int rb, int *__restrict__ idx,
                                                                      float *__restrict__ wgt, int *__restrict__ counts)
{
    extern __shared__ int hist[];          // [experts] counts; per wave [experts] choice values, [top] weights before the division
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float *ch = (float *)(hist + experts) + wave * (experts + top), *pw = ch + experts;
    auto in_order = []() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); };          // (a wave's own LDS accesses)
    for (int e = threadIdx.x; e < experts; e += 64 * PLACE_WAVES) hist[e] = 0;
    __syncthreads();
    for (int r = wave; r < rb; r += PLACE_WAVES) {
        const int t = blockIdx.x * rb + r;
        if (t >= rows) break;
        const float *z = logits + (size_t)t * ld;
        for (int e = lane; e < experts; e += 64) ch[e] = choice_of(z[e]);
        in_order();
        float first = 0.0f, sum = 0.0f;
        for (int k = 0; k < top; k++) {
            float best = -INFINITY; int bi = 0x7FFFFFFF;
            for (int e = lane; e < experts; e += 64) { const float v = ch[e]; if (v > best || (v == best && e < bi)) { best = v; bi = e; } }
            for (int o = 32; o > 0; o >>= 1) {
                const float ov = __shfl_xor(best, o, 64); const int oi = __shfl_xor(bi, o, 64);
                if (ov > best || (ov == best && oi < bi)) { best = ov; bi = oi; }
            }
            if (k == 0) first = best;
            const float p = expf(best - first);
            sum += p;
            if (lane == 0) { idx[(size_t)t * top + k] = bi; pw[k] = p; ch[bi] = NAN; atomicAdd(&hist[bi], 1); }
            in_order();
        }
        for (int k = lane; k < top; k += 64) wgt[(size_t)t * top + k] = pw[k] / sum;
        in_order();
    }
    __syncthreads();
    for (int e = threadIdx.x; e < experts; e += 64 * PLACE_WAVES) counts[(size_t)blockIdx.x * experts + e] = hist[e];
}

// what k_moe_sort leaves, and the counts of the blocks
struct MoePlace { const int *idx; const float *wgt; int n_pairs, experts, top; int *a_rows, *pair_pos; float *w_sorted; int *tile_map, *n_tiles; int tile_rows; const int *counts; int blocks, rb; };
size_t place_smem(int experts) { return (size_t)(2 + PLACE_WAVES) * experts * 4; }

// workgroup `wg` places the pairs of PLACE_WAVES blocks, a block a wave; the first one leaves the tiles too
__device__ void moe_place(const MoePlace &S, int wg, int *lds)
{
    const int E = S.experts, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, b0 = wg * PLACE_WAVES, pad = E <= 1 ? 1 : 1 << (32 - __builtin_clz(E - 1));
    int *all = lds, *before = lds + E, *mine = lds + (2 + wave) * E;
    for (int e = tid; e < 2 * E; e += 64 * PLACE_WAVES) lds[e] = 0;
    __syncthreads();
    {
        const int e = tid & (pad - 1);
        int n = 0, f = 0;
        if (e < E)
            for (int b = tid / pad; b < S.blocks; b += 64 * PLACE_WAVES / pad) { const int c = S.counts[(size_t)b * E + e]; n += c; if (b < b0) f += c; }
        if (n) atomicAdd(&all[e], n);
        if (f) atomicAdd(&before[e], f);
    }
    __syncthreads();
    if (wave == 0) {          // where an expert's range begins; its tiles
        int from = 0, tiles = 0;
        for (int e0 = 0; e0 < E; e0 += 64) {
            const int e = e0 + lane, n = e < E ? all[e] : 0, nt = (n + S.tile_rows - 1) / S.tile_rows;
            int upto = n, t_upto = nt;
#pragma unroll
            for (int k = 1; k < 64; k <<= 1) {
                const int x = __shfl_up(upto, k, 64), y = __shfl_up(t_upto, k, 64);
                if (lane >= k) { upto += x; t_upto += y; }
            }
            const int o = from + upto - n;
            if (e < E) before[e] += o;
            if (wg == 0)
                for (int k = 0; k < nt; k++) {
                    int *tm = S.tile_map + 3 * (tiles + t_upto - nt + k);
                    tm[0] = e; tm[1] = o + k * S.tile_rows; tm[2] = min(S.tile_rows, n - k * S.tile_rows);
                }
            from += __builtin_amdgcn_readlane(upto, 63); tiles += __builtin_amdgcn_readlane(t_upto, 63);
        }
        if (wg == 0 && lane == 0) *S.n_tiles = tiles;
    }
    __syncthreads();
    for (int e = tid; e < E; e += 64 * PLACE_WAVES) {          // ... and each wave's part of it
        int c[PLACE_WAVES], at = before[e];
#pragma unroll
        for (int w = 0; w < PLACE_WAVES; w++) c[w] = S.counts[(size_t)min(b0 + w, S.blocks - 1) * E + e];
#pragma unroll
        for (int w = 0; w < PLACE_WAVES; w++) { lds[(2 + w) * E + e] = at; at += c[w]; }
    }
    __syncthreads();
    if (b0 + wave >= S.blocks) return;
    const int p0 = (b0 + wave) * S.rb * S.top, p1 = min(S.n_pairs, p0 + S.rb * S.top), bits = 32 - __builtin_clz(E);          // (E itself stands for no pair)
    for (int q = p0; q < p1; q += 64) {
        const int p = q + lane, e = p < p1 ? S.idx[p] : E;
        const float w = S.wgt[min(p, p1 - 1)];
        uint64_t same = ~(uint64_t)0;          // the lanes of the same expert
        for (int b = 0; b < bits; b++) { const uint64_t set = __builtin_amdgcn_ballot_w64(e >> b & 1); same &= e >> b & 1 ? set : ~set; }
        const int earlier = __builtin_popcountll(same & (((uint64_t)1 << lane) - 1));
        if (p < p1) {
            const int pos = mine[e] + earlier;
            S.a_rows[pos] = p / S.top; S.pair_pos[p] = pos; S.w_sorted[pos] = w;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (p < p1 && earlier == 0) mine[e] += __builtin_popcountll(same);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
}

// ... beside the shared expert's activations (k_glu_to_bf16), which need as little of the choice: the first `placing` workgroups and the others
struct MoeGlu { const float *gate_up; size_t ld; int F; const float *row_gate; size_t ldg; bf16_t *out; int ldo, pieces, vec; size_t total; };
__global__ void __launch_bounds__(64 * PLACE_WAVES) k_moe_place_glu(MoePlace S, int placing, MoeGlu G)
{
    extern __shared__ int place_lds[];
    if ((int)blockIdx.x < placing) { moe_place(S, blockIdx.x, place_lds); return; }
    const size_t id = (size_t)(blockIdx.x - placing) * 1024 + threadIdx.x;
    if (id >= G.total) return;
    if (G.vec) glu_piece<true>(0, 0.0f, G.gate_up, G.ld, G.F, G.row_gate, G.ldg, G.out, G.ldo, G.pieces, id);
    else glu_piece<false>(0, 0.0f, G.gate_up, G.ld, G.F, G.row_gate, G.ldg, G.out, G.ldo, G.pieces, id);
}

// y[t][c] (+)= sum_k (identity ? wgt h[t][c] : yp[pair_pos][c])  (the pair's weight is already inside yp)
__global__ void __launch_bounds__(256) k_moe_combine(const float *__restrict__ h, size_t ldh, int W, int top, const int *__restrict__ pair_pos,
                                                     const float *__restrict__ wgt, const float *__restrict__ yp, int accumulate, float *__restrict__ y, size_t ldy)
{
    const int t = blockIdx.y, c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= W) return;
    float out = 0.0f;
    for (int k = 0; k < top; k++) {
        const int p = t * top + k, pos = pair_pos[p];
        out += pos < 0 ? wgt[p] * h[(size_t)t * ldh + c] : yp[(size_t)pos * W + c];
    }
    float *d = y + (size_t)t * ldy + c;
    *d = accumulate ? *d + out : out;
}

size_t al16(size_t v) { return (v + 15) & ~(size_t)15; }
size_t moe_tiles_max(size_t rows, int top, int experts) { return (rows * (size_t)top + 63) / 64 + (size_t)experts; }

} // namespace

extern "C" {

int ifa_moe_route_scores_f32(int score_kind, const void *logits_f32, size_t ld, size_t rows, int n_all, int top, const void *correction_bf16, int *idx_dev,
                             void *wgt_f32, ifa_stream stream)
{
    return ifa_moe_route_renorm_f32(score_kind, 0, 0.0f, 1.0f, logits_f32, ld, rows, n_all, top, correction_bf16, idx_dev, wgt_f32, stream);
}

int ifa_moe_route_renorm_f32(int score_kind, int renorm, float renorm_eps, float wgt_scale, const void *logits_f32, size_t ld, size_t rows, int n_all, int top,
                             const void *correction_bf16, int *idx_dev, void *wgt_f32, ifa_stream stream)
{
    IFA_REQUIRE(logits_f32 && idx_dev && wgt_f32, "ifa_moe_route_scores_f32: null pointer");
    IFA_REQUIRE(rows > 0 && n_all >= 1 && n_all <= 4096 && top >= 1 && top <= n_all && ld >= (size_t)n_all && (score_kind == 0 || score_kind == 1),
                "ifa_moe_route_scores_f32: bad shape (%d router outputs, %d chosen, scores of kind %d)", n_all, top, score_kind);
    hipLaunchKernelGGL(k_moe_route, dim3((unsigned)rows), dim3(64), (size_t)n_all * 8, ifa_s(stream), (const float *)logits_f32, ld, n_all, top,
                       (const bf16_t *)correction_bf16, idx_dev, (float *)wgt_f32, score_kind, renorm ? 1 : 0, renorm_eps, wgt_scale);
    IFA_LAUNCH_CHECK();
    return IFA_OK;
}

int ifa_moe_route_f32(const void *logits_f32, size_t ld, size_t rows, int n_all, int top, const void *correction_bf16, int *idx_dev, void *wgt_f32,
                      ifa_stream stream)
{
    return ifa_moe_route_scores_f32(0, logits_f32, ld, rows, n_all, top, correction_bf16, idx_dev, wgt_f32, stream);
}

int ifa_moe_route_rows_f32(const void *h_f32, size_t ldh, size_t rows, int width, const void *router_bf16, int n_all, int top, const void *correction_bf16,
                           int *idx_dev, void *wgt_f32, ifa_stream stream)
{
    return ifa_moe_route_rows_scores_f32(0, h_f32, ldh, rows, width, router_bf16, n_all, top, correction_bf16, idx_dev, wgt_f32, stream);
}

int ifa_moe_route_rows_scores_f32(int score_kind, const void *h_f32, size_t ldh, size_t rows, int width, const void *router_bf16, int n_all, int top,
                                  const void *correction_bf16, int *idx_dev, void *wgt_f32, ifa_stream stream)
{
    return ifa_moe_route_rows_renorm_f32(score_kind, 0, 0.0f, 1.0f, h_f32, ldh, rows, width, router_bf16, n_all, top, correction_bf16, idx_dev, wgt_f32, stream);
}

int ifa_moe_route_rows_renorm_f32(int score_kind, int renorm, float renorm_eps, float wgt_scale, const void *h_f32, size_t ldh, size_t rows, int width,
                                  const void *router_bf16, int n_all, int top, const void *correction_bf16, int *idx_dev, void *wgt_f32, ifa_stream stream)
{
    IFA_REQUIRE(h_f32 && router_bf16 && idx_dev && wgt_f32, "ifa_moe_route_rows_f32: null pointer");
    IFA_REQUIRE(rows > 0 && rows <= 64 && width > 0 && n_all >= 1 && n_all <= 4096 && top >= 1 && top <= n_all && ldh >= (size_t)width && (score_kind == 0 || score_kind == 1),
                "ifa_moe_route_rows_f32: bad shape");
    const int vec = (width % 8 == 0 && ldh % 4 == 0 && ((uintptr_t)h_f32 & 15) == 0 && ((uintptr_t)router_bf16 & 15) == 0) ? 1 : 0;
    hipLaunchKernelGGL(k_moe_route_rows, dim3((unsigned)rows), dim3(n_all > 8 ? 1024 : 256), (size_t)n_all * 8, ifa_s(stream), (const float *)h_f32, ldh, width,
                       (const bf16_t *)router_bf16, n_all, top, (const bf16_t *)correction_bf16, idx_dev, (float *)wgt_f32, vec, score_kind, (const float *)nullptr, (size_t)0,
                       (const bf16_t *)nullptr, (const bf16_t *)nullptr, (const bf16_t *)nullptr, (float *)nullptr, renorm ? 1 : 0, renorm_eps, wgt_scale);
    IFA_LAUNCH_CHECK();
    return IFA_OK;
}

int ifa_moe_dyt_route_rows_f32(int score_kind, const void *x_f32, size_t ldx, const void *alpha_bf16, const void *norm_w_bf16, const void *norm_b_bf16, void *h_f32,
                               size_t ldh, size_t rows, int width, const void *router_bf16, int n_all, int top, const void *correction_bf16, int *idx_dev,
                               void *wgt_f32, ifa_stream stream)
{
    IFA_REQUIRE(x_f32 && alpha_bf16 && norm_w_bf16 && norm_b_bf16 && h_f32 && router_bf16 && idx_dev && wgt_f32 && x_f32 != h_f32, "ifa_moe_dyt_route_rows_f32: null pointer");
    IFA_REQUIRE(rows > 0 && rows <= 64 && width > 0 && n_all >= 1 && n_all <= 4096 && top >= 1 && top <= n_all && ldh >= (size_t)width && ldx >= (size_t)width
                && (score_kind == 0 || score_kind == 1), "ifa_moe_dyt_route_rows_f32: bad shape");
    const int vec = (width % 8 == 0 && ldh % 4 == 0 && ((uintptr_t)h_f32 & 15) == 0 && ((uintptr_t)router_bf16 & 15) == 0) ? 1 : 0;
    hipLaunchKernelGGL(k_moe_route_rows, dim3((unsigned)rows), dim3(n_all > 8 ? 1024 : 256), (size_t)n_all * 8, ifa_s(stream), (const float *)h_f32, ldh, width,
                       (const bf16_t *)router_bf16, n_all, top, (const bf16_t *)correction_bf16, idx_dev, (float *)wgt_f32, vec, score_kind, (const float *)x_f32, ldx,
                       (const bf16_t *)alpha_bf16, (const bf16_t *)norm_w_bf16, (const bf16_t *)norm_b_bf16, (float *)h_f32, 0, 0.0f, 1.0f);
    IFA_LAUNCH_CHECK();
    return IFA_OK;
}

int ifa_moe_route_top_f32(const void *logits_f32, size_t ld, size_t rows, int n_all, int top, const void *bias_bf16, int *idx_dev, void *wgt_f32,
                          ifa_stream stream)
{
    IFA_REQUIRE(logits_f32 && idx_dev && wgt_f32, "ifa_moe_route_top_f32: null pointer");
    IFA_REQUIRE(rows > 0 && n_all >= 1 && n_all <= 4096 && top >= 1 && top <= n_all && ld >= (size_t)n_all, "ifa_moe_route_top_f32: bad shape (%d router outputs, %d chosen)", n_all, top);
    hipLaunchKernelGGL(k_moe_route_top, dim3((unsigned)rows), dim3(64), (size_t)(n_all + top) * 4, ifa_s(stream), (const float *)logits_f32, ld, n_all, top,
                       (const bf16_t *)bias_bf16, idx_dev, (float *)wgt_f32);
    IFA_LAUNCH_CHECK();
    return IFA_OK;
}

size_t ifa_moe_workspace_bytes(size_t rows, int top, int width, int ff, int experts)
{
    const size_t pairs = rows * (size_t)top;
    return al16(pairs * ff * 4) + al16(pairs * width * 4) + 3 * al16(pairs * 4) + al16(moe_tiles_max(rows, top, experts) * 12) + 16;
}

// whether gated experts of more than eight rows run over bfloat16 rows (k_lin_tile): sizes and alignment, see moe_experts
static bool moe_in16(size_t rows, int width, int ff, int top, int ops32, const void *up_bf16, const void *down_bf16)
{
    const size_t lda_h = ((size_t)width + 63) & ~(size_t)63, lda_f = ((size_t)ff + 63) & ~(size_t)63;
    return rows > 8 && !ops32 && width % 8 == 0 && width >= 64 && ff % 8 == 0 && ff >= 64 && width + ff >= 512 && lda_f <= 2 * (size_t)ff && lda_h <= 2 * (size_t)width * top
           && (((uintptr_t)up_bf16 | (uintptr_t)down_bf16) & 15) == 0;
}

// the workspace of a step's pairs (ff_ws: 3 ff of gated experts, whose first product leaves gate | up in front of the activations)
struct MoeSpace { float *actb, *yp; int *a_rows, *pair_pos; float *w_sorted; int *tile_map, *n_tiles; };
static MoeSpace moe_space(void *ws, size_t rows, int top, int width, int ff_ws, int experts)
{
    const size_t pairs = rows * (size_t)top;
    char *b = (char *)ws;
    MoeSpace s;
    s.actb = (float *)b; b += al16(pairs * ff_ws * 4);
    s.yp = (float *)b; b += al16(pairs * width * 4);
    s.a_rows = (int *)b; b += al16(pairs * 4);
    s.pair_pos = (int *)b; b += al16(pairs * 4);
    s.w_sorted = (float *)b; b += al16(pairs * 4);
    s.tile_map = (int *)b; b += al16(moe_tiles_max(rows, top, experts) * 12);
    s.n_tiles = (int *)b;
    return s;
}

// row tiles of bfloat16 experts' products, see moe_experts
static int moe_tile_rows16(size_t pairs, int width, int experts)
{
    return pairs >= (size_t)256 * experts && pairs / 128 * (((size_t)width + 127) / 128) >= 256 ? 128 : 64;
}

static int moe_experts(const char *who, int gated, int glu_kind, float limit, const void *h_f32, size_t ldh, size_t rows, int width, int ff, int experts, int identity, int top, int act,
                       const void *up_bf16, const void *down_bf16, const int *idx_dev, const void *wgt_f32, int ops32, void *ws, size_t ws_bytes,
                       void *y_f32, size_t ldy, int accumulate, ifa_stream stream, const RouteSel *sel = nullptr, const void *h_bf16 = nullptr, const IfaMoeShared *shared = nullptr)
{
    IFA_REQUIRE((h_f32 || h_bf16) && idx_dev && wgt_f32 && ws && y_f32 && (experts == 0 || (up_bf16 && down_bf16)), "%s: null pointer", who);
    IFA_REQUIRE(rows > 0 && rows < 65536 && width > 0 && ff > 0 && experts >= 0 && experts <= 4096 && identity >= 0 && top >= 1 && top <= experts + identity && act == 0
                && ldh >= (size_t)width && ldy >= (size_t)width, "%s: bad shape", who);
    // gated experts: the first product leaves gate | up (2 ff values per pair) in front of the activations
    const int ff_ws = gated ? 3 * ff : ff;
    IFA_REQUIRE(ws_bytes >= ifa_moe_workspace_bytes(rows, top, width, ff_ws, experts) && ((uintptr_t)ws & 15) == 0, "%s: workspace of %zu bytes, %zu needed", who, ws_bytes,
                ifa_moe_workspace_bytes(rows, top, width, ff_ws, experts));
    const size_t pairs = rows * (size_t)top;
    const MoeSpace at = moe_space(ws, rows, top, width, ff_ws, experts);
    float *const actb = at.actb, *const gub = actb + pairs * ff;                     // gub: [pairs][2 ff] (gated experts, many rows)
    float *const yp = at.yp, *const w_sorted = at.w_sorted;
    int *const a_rows = at.a_rows, *const pair_pos = at.pair_pos, *const tile_map = at.tile_map, *const n_tiles = at.n_tiles;
    hipStream_t s = ifa_s(stream);
    const float *h = (const float *)h_f32;
    if (rows <= 8 || experts == 0) {
        const int vec_u = (width % 8 == 0 && ldh % 4 == 0 && ((uintptr_t)h_f32 & 15) == 0 && ((uintptr_t)up_bf16 & 15) == 0) ? 1 : 0;
        const int vec_d = (ff % 8 == 0 && ((uintptr_t)down_bf16 & 15) == 0) ? 1 : 0;
        if (experts > 0 && gated && sel)
            hipLaunchKernelGGL((k_moe_up_rows<true, true>), dim3(std::min(512u, ifa_cdiv((size_t)ff, 4)), (unsigned)pairs), dim3(256), 0, s, h, ldh, width, ff, experts, top,
                               (const bf16_t *)up_bf16, idx_dev, actb, vec_u, glu_kind, limit, *sel);
        else if (experts > 0 && gated)
            hipLaunchKernelGGL((k_moe_up_rows<true, false>), dim3(std::min(512u, ifa_cdiv((size_t)ff, 4)), (unsigned)pairs), dim3(256), 0, s, h, ldh, width, ff, experts, top,
                               (const bf16_t *)up_bf16, idx_dev, actb, vec_u, glu_kind, limit, RouteSel());
        else if (experts > 0)
            hipLaunchKernelGGL((k_moe_up_rows<false, false>), dim3(std::min(512u, ifa_cdiv((size_t)ff, 4)), (unsigned)pairs), dim3(256), 0, s, h, ldh, width, ff, experts, top,
                               (const bf16_t *)up_bf16, idx_dev, actb, vec_u, 0, 0.0f, RouteSel());
        const dim3 grid(std::min(1024u, ifa_cdiv((size_t)width, 4)), (unsigned)rows + (shared ? 1u : 0u));
#define IFA_DOWN(NK, SH, S) hipLaunchKernelGGL((k_moe_down_rows<NK, SH>), grid, dim3(256), 0, s, h, ldh, width, ff, experts, top, (const bf16_t *)down_bf16, idx_dev, (const float *)wgt_f32, \
                                               actb, accumulate ? 1 : 0, (float *)y_f32, ldy, vec_d, S)
#define IFA_DOWN_SH(NK) switch (shared ? (int)rows : 0) { \
            case 0: IFA_DOWN(NK, 0, 0); break; case 1: IFA_DOWN(NK, 1, *shared); break; case 2: IFA_DOWN(NK, 2, *shared); break; case 3: IFA_DOWN(NK, 3, *shared); break; \
            case 4: IFA_DOWN(NK, 4, *shared); break; case 5: IFA_DOWN(NK, 5, *shared); break; case 6: IFA_DOWN(NK, 6, *shared); break; case 7: IFA_DOWN(NK, 7, *shared); break; \
            default: IFA_DOWN(NK, 8, *shared); }
        if (top <= 4) IFA_DOWN_SH(4) else IFA_DOWN_SH(8)
#undef IFA_DOWN_SH
#undef IFA_DOWN
        IFA_LAUNCH_CHECK();
        return IFA_OK;
    }
    // gated experts, products over bfloat16 rows where the activations are rounded anyway: h once (in the place of the down products' output, which is not there yet), the experts'
    // activations by the launch that forms them.  From 512 columns on, of both products together: below, the launch that rounds h costs more than the products gain (8 experts,
    // us before / now: 128 x 128 18.7 / 21.6, 256 x 128 20.6 / 21.6, 256 x 256 22.6 / 21.6).  Row tiles of 128 where an expert has several on average and they still fill the
    // chip (4000 pairs of 8 experts: 1408 x 2048 288 -> 197 us; 520 x 136 52, 46 with tiles of 64, 59 with tiles of 128)
    const size_t lda_h = ((size_t)width + 63) & ~(size_t)63, lda_f = ((size_t)ff + 63) & ~(size_t)63;
    const bool in16 = gated && moe_in16(rows, width, ff, top, ops32, up_bf16, down_bf16);
    IFA_REQUIRE(in16 || h_f32, "%s: rows in bfloat16 where the sizes need 32 bits", who);
    const int tile_rows = in16 ? moe_tile_rows16(pairs, width, experts) : 64;
    const size_t max_tiles = (pairs + tile_rows - 1) / tile_rows + (size_t)experts;
    IFA_REQUIRE(max_tiles < 65536, "%s: %zu rows x %d choices exceed one step", who, rows, top);
    hipLaunchKernelGGL(k_moe_sort, dim3(1), dim3(1024), (size_t)(2 * experts + 1) * 4, s, idx_dev, (const float *)wgt_f32, (int)pairs, experts, top, a_rows, pair_pos, w_sorted,
                       tile_map, n_tiles, tile_rows);
    IFA_LAUNCH_CHECK();
    int rc;
    if (in16) {
        bf16_t *h16 = (bf16_t *)yp, *a16 = (bf16_t *)actb;
        if (!h_bf16 && (rc = ifa_rows_to_bf16(h_f32, ldh, rows, (size_t)width, h16, lda_h, stream))) return rc;
        if ((rc = ifa_linear_bf16_grouped(up_bf16, (size_t)2 * ff, (size_t)width, h_bf16 ? h_bf16 : h16, lda_h, a_rows, tile_map, n_tiles, max_tiles, tile_rows, nullptr, nullptr, lda_f, glu_kind, limit, a16, stream))) return rc;
        if ((rc = ifa_linear_bf16_grouped(down_bf16, (size_t)width, (size_t)ff, a16, lda_f, nullptr, tile_map, n_tiles, max_tiles, tile_rows, w_sorted, yp, (size_t)width, 0, 0.0f, nullptr, stream))) return rc;
    } else if (gated) {
        if ((rc = ifa_linear_bf16w_grouped(up_bf16, (size_t)2 * ff, (size_t)width, experts, h_f32, ldh, a_rows, tile_map, n_tiles, max_tiles, nullptr, 0, ops32, gub, (size_t)2 * ff, stream))) return rc;
        if ((rc = ifa_glu_ex_f32(glu_kind, limit, gub, (size_t)2 * ff, pairs, (size_t)ff, nullptr, 0, actb, (size_t)ff, stream))) return rc;
    } else if ((rc = ifa_linear_bf16w_grouped(up_bf16, (size_t)ff, (size_t)width, experts, h_f32, ldh, a_rows, tile_map, n_tiles, max_tiles, nullptr, 1, ops32, actb, (size_t)ff, stream))) return rc;
    if (!in16 && (rc = ifa_linear_bf16w_grouped(down_bf16, (size_t)width, (size_t)ff, experts, actb, (size_t)ff, nullptr, tile_map, n_tiles, max_tiles, w_sorted, 0, ops32, yp, (size_t)width, stream))) return rc;
    hipLaunchKernelGGL(k_moe_combine, dim3(ifa_cdiv((size_t)width, 256), (unsigned)rows), dim3(256), 0, s, h, ldh, width, top, pair_pos, (const float *)wgt_f32, yp,
                       accumulate ? 1 : 0, (float *)y_f32, ldy);
    IFA_LAUNCH_CHECK();
    return IFA_OK;
}

int ifa_moe_experts_f32(const void *h_f32, size_t ldh, size_t rows, int width, int ff, int experts, int identity, int top, int act,
                        const void *up_bf16, const void *down_bf16, const int *idx_dev, const void *wgt_f32, int ops32, void *ws, size_t ws_bytes,
                        void *y_f32, size_t ldy, int accumulate, ifa_stream stream)
{
    return moe_experts("ifa_moe_experts_f32", 0, 0, 0.0f, h_f32, ldh, rows, width, ff, experts, identity, top, act, up_bf16, down_bf16, idx_dev, wgt_f32, ops32, ws, ws_bytes, y_f32,
                       ldy, accumulate, stream);
}

int ifa_moe_experts_gated_f32(const void *h_f32, size_t ldh, size_t rows, int width, int ff, int experts, int top, const void *gate_up_bf16,
                              const void *down_bf16, const int *idx_dev, const void *wgt_f32, int ops32, void *ws, size_t ws_bytes, void *y_f32, size_t ldy,
                              int accumulate, ifa_stream stream)
{
    IFA_REQUIRE(experts > 0, "ifa_moe_experts_gated_f32: no experts");
    return moe_experts("ifa_moe_experts_gated_f32", 1, 0, 0.0f, h_f32, ldh, rows, width, ff, experts, 0, top, 0, gate_up_bf16, down_bf16, idx_dev, wgt_f32, ops32, ws, ws_bytes,
                       y_f32, ldy, accumulate, stream);
}

int ifa_moe_experts_glu_f32(int glu_kind, float limit, const void *h_f32, size_t ldh, size_t rows, int width, int ff, int experts, int top,
                            const void *gate_up_bf16, const void *down_bf16, const int *idx_dev, const void *wgt_f32, int ops32, void *ws, size_t ws_bytes,
                            void *y_f32, size_t ldy, int accumulate, ifa_stream stream)
{
    IFA_REQUIRE(experts > 0 && (glu_kind == 0 || (glu_kind == 3 && limit > 0.0f)), "ifa_moe_experts_glu_f32: no experts, or gate kind %d (0, or 3 with a limit)", glu_kind);
    return moe_experts("ifa_moe_experts_glu_f32", 1, glu_kind, limit, h_f32, ldh, rows, width, ff, experts, 0, top, 0, gate_up_bf16, down_bf16, idx_dev, wgt_f32, ops32, ws,
                       ws_bytes, y_f32, ldy, accumulate, stream);
}

int ifa_moe_experts_routed_rows_f32(int score_kind, int renorm, float renorm_eps, float wgt_scale, const void *logits_f32, size_t ldl, const void *correction_bf16,
                                    int glu_kind, float limit, const void *h_f32, size_t ldh, size_t rows, int width, int ff, int experts, int top,
                                    const void *gate_up_bf16, const void *down_bf16, int *idx_dev, void *wgt_f32, void *ws, size_t ws_bytes, void *y_f32, size_t ldy,
                                    int accumulate, ifa_stream stream)
{
    IFA_REQUIRE(logits_f32 && rows <= 8 && experts > 0 && experts <= 256 && ldl >= (size_t)experts && (score_kind == 0 || score_kind == 1)
                && (glu_kind == 0 || (glu_kind == 3 && limit > 0.0f)), "ifa_moe_experts_routed_rows_f32: bad arguments (%zu rows: at most 8, %d experts: at most 256)", rows, experts);
    RouteSel R;
    R.logits = (const float *)logits_f32; R.ld = ldl; R.n_all = experts; R.score_kind = score_kind; R.renorm = renorm ? 1 : 0; R.renorm_eps = renorm_eps; R.wgt_scale = wgt_scale;
    R.corr = (const bf16_t *)correction_bf16; R.idx = idx_dev; R.wgt = (float *)wgt_f32;
    return moe_experts("ifa_moe_experts_routed_rows_f32", 1, glu_kind, limit, h_f32, ldh, rows, width, ff, experts, 0, top, 0, gate_up_bf16, down_bf16, idx_dev, wgt_f32, 1, ws,
                       ws_bytes, y_f32, ldy, accumulate, stream, &R);
}

} // extern "C"

int ifa_moe_experts_gated_top_rows_shared(const void *logits_f32, size_t ldl, const void *h_f32, size_t ldh, size_t rows, int width, int ff, int experts, int top, const void *gate_up_bf16,
                                   const void *down_bf16, int *idx_dev, void *wgt_f32, void *ws, size_t ws_bytes, void *y_f32, size_t ldy, int accumulate, const IfaMoeShared *shared,
                                   ifa_stream stream)
{
    IFA_REQUIRE(!shared || (shared->down && shared->act && shared->gate && shared->out && shared->ldo >= (size_t)width && ifa_moe_shared_fits(*shared)), "moe_experts_gated_top_rows: shared expert of %d columns", shared ? shared->ff : 0);
    IFA_REQUIRE(logits_f32 && rows <= 8 && experts > 0 && experts <= 256 && ldl >= (size_t)experts, "moe_experts_gated_top_rows: %zu rows (at most 8), %d experts (at most 256)", rows, experts);
    RouteSel R;
    memset(&R, 0, sizeof(R));
    R.logits = (const float *)logits_f32; R.ld = ldl; R.n_all = experts; R.score_kind = 2; R.idx = idx_dev; R.wgt = (float *)wgt_f32;
    return moe_experts("moe_experts_gated_top_rows", 1, 0, 0.0f, h_f32, ldh, rows, width, ff, experts, 0, top, 0, gate_up_bf16, down_bf16, idx_dev, wgt_f32, 1, ws, ws_bytes, y_f32, ldy,
                       accumulate, stream, &R, nullptr, shared);
}

// A wave of the shared expert's workgroups reads all rows' activations for one output: with many weights and three rows and more the launch of its own, which has two outputs a wave there, is the
// faster one.  One launch / two, 2 to 8 rows, two of eight experts: 6144 x 4096 0.96 to 1.00, 4096 x 8192 and 8192 x 4096 0.95 to 1.04 (from four rows on 0.97 to 1.04), 8192 x 8192 0.99 for two
// rows and 1.06 to 1.13 for more; 16.8 M weights and less 0.70 to 0.97.
bool ifa_moe_shared_pays(size_t rows, size_t width, size_t ff) { return rows <= 2 || width * ff <= (size_t)24 << 20; }

bool ifa_moe_shared_fits(const IfaMoeShared &S)
{
    return S.ff >= 8 && S.ff % 8 == 0 && S.lda >= (size_t)S.ff && S.lda % 4 == 0 && (((uintptr_t)S.down | (uintptr_t)S.act) & 15) == 0;
}

bool ifa_moe_gated_reads_bf16(size_t rows, int width, int ff, int top, int ops32, const void *gate_up_bf16, const void *down_bf16)
{
    return width % 64 == 0 && moe_in16(rows, width, ff, top, ops32, gate_up_bf16, down_bf16);
}

int ifa_moe_experts_gated_bf16(const void *h_bf16, size_t rows, int width, int ff, int experts, int top, const void *gate_up_bf16, const void *down_bf16, const int *idx_dev,
                               const void *wgt_f32, void *ws, size_t ws_bytes, void *y_f32, size_t ldy, int accumulate, ifa_stream stream)
{
    IFA_REQUIRE(h_bf16 && ((uintptr_t)h_bf16 & 15) == 0 && experts > 0 && ifa_moe_gated_reads_bf16(rows, width, ff, top, 0, gate_up_bf16, down_bf16), "moe_experts_gated_bf16: bad shape");
    return moe_experts("moe_experts_gated_bf16", 1, 0, 0.0f, nullptr, (size_t)width, rows, width, ff, experts, 0, top, 0, gate_up_bf16, down_bf16, idx_dev, wgt_f32, 0, ws, ws_bytes, y_f32,
                       ldy, accumulate, stream, nullptr, h_bf16);
}

// Choice by the largest logits + the shared expert's activations + ifa_moe_experts_gated_bf16 without the sum of a row's pairs, which the norm behind it forms (ifa_norm_add_norm_moe): rows of
// ifa_moe_gated_reads_bf16, at most 65535, of at most PLACE_EXPERTS experts.  us choice + sort + activations, before / now: 787 rows of 16 experts, top 4, 1408 shared columns
// 4.7 + 7.8 + 5.5 / 5.9 + 5.5, 2048 rows 5.6 + 13.6 + 8.8 / 6.7 + 8.6
int ifa_moe_prompt(const IfaMoePrompt &P, const int **pair_pos, const float **pair_rows, ifa_stream stream)
{
    const size_t pairs = P.rows * (size_t)P.top, lda_f = ((size_t)P.ff + 63) & ~(size_t)63;
    IFA_REQUIRE(P.logits && P.h16 && P.idx && P.wgt && P.ws && P.gate_up && P.down && P.experts >= 1 && P.experts <= PLACE_EXPERTS && P.top >= 1 && P.top <= P.experts && P.rows > 0 && P.rows < 65536
                && P.ldl >= (size_t)P.experts && ((uintptr_t)P.h16 & 15) == 0 && ifa_moe_gated_reads_bf16(P.rows, P.width, P.ff, P.top, 0, P.gate_up, P.down), "moe_prompt: bad arguments");
    IFA_REQUIRE(!P.sh_ff || (P.sh_gate_up && P.sh_act && P.sh_ld >= 2 * (size_t)P.sh_ff && P.sh_ldo % 8 == 0 && P.sh_ldo >= (size_t)P.sh_ff && P.sh_ldo < (1u << 30) && ((uintptr_t)P.sh_act & 15) == 0),
                "moe_prompt: bad shared expert");
    IFA_REQUIRE(P.ws_bytes >= ifa_moe_workspace_bytes(P.rows, P.top, P.width, 3 * P.ff, P.experts) && ((uintptr_t)P.ws & 15) == 0, "moe_prompt: workspace of %zu bytes", P.ws_bytes);
    const int tile_rows = moe_tile_rows16(pairs, P.width, P.experts);
    const size_t max_tiles = (pairs + tile_rows - 1) / tile_rows + (size_t)P.experts;
    IFA_REQUIRE(max_tiles < 65536, "moe_prompt: %zu rows x %d choices exceed one step", P.rows, P.top);
    const MoeSpace at = moe_space(P.ws, P.rows, P.top, P.width, 3 * P.ff, P.experts);
    // (the counts lie where experts of 32-bit rows have their gates and ups: 2 ff >= 128 values a pair, more than 32 a row and 512)
    const int rb = PLACE_WAVES * (int)((P.rows + (size_t)PLACE_WAVES * PLACE_BLOCKS - 1) / ((size_t)PLACE_WAVES * PLACE_BLOCKS)), blocks = (int)((P.rows + rb - 1) / rb);
    int *counts = (int *)(at.actb + pairs * P.ff);
    const MoePlace S = {P.idx, P.wgt, (int)pairs, P.experts, P.top, at.a_rows, at.pair_pos, at.w_sorted, at.tile_map, at.n_tiles, tile_rows, counts, blocks, rb};
    MoeGlu G;
    memset(&G, 0, sizeof(G));
    if (P.sh_ff) {
        G.gate_up = P.sh_gate_up; G.ld = P.sh_ld; G.F = P.sh_ff; G.row_gate = P.sh_gate; G.ldg = P.sh_ldg; G.out = P.sh_act; G.ldo = (int)P.sh_ldo; G.pieces = (int)(P.sh_ldo / 8);
        G.vec = P.sh_ld % 4 == 0 && P.sh_ff % 4 == 0 && ((uintptr_t)P.sh_gate_up & 15) == 0; G.total = P.rows * (size_t)G.pieces;
    }
    int rc;
    const int placing = (blocks + PLACE_WAVES - 1) / PLACE_WAVES;
    const size_t lds = route_count_smem(P.experts, P.top);
    if (lds > 64 * 1024) IFA_HIP_CHECK(hipFuncSetAttribute((const void *)k_moe_route_count, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(k_moe_route_count, dim3((unsigned)blocks), dim3(64 * PLACE_WAVES), lds, ifa_s(stream), P.logits, P.ldl, P.experts, P.top, (int)P.rows, rb, P.idx, P.wgt, counts);
    hipLaunchKernelGGL(k_moe_place_glu, dim3((unsigned)(placing + (G.total + 1023) / 1024)), dim3(64 * PLACE_WAVES), place_smem(P.experts), ifa_s(stream), S, placing, G);
    IFA_LAUNCH_CHECK();
    bf16_t *a16 = (bf16_t *)at.actb;
    if ((rc = ifa_linear_bf16_grouped(P.gate_up, (size_t)2 * P.ff, (size_t)P.width, P.h16, (size_t)P.width, at.a_rows, at.tile_map, at.n_tiles, max_tiles, tile_rows, nullptr, nullptr, lda_f, 0,
                                      0.0f, a16, stream))) return rc;
    if ((rc = ifa_linear_bf16_grouped(P.down, (size_t)P.width, (size_t)P.ff, a16, lda_f, nullptr, at.tile_map, at.n_tiles, max_tiles, tile_rows, at.w_sorted, at.yp, (size_t)P.width, 0, 0.0f,
                                      nullptr, stream))) return rc;
    *pair_pos = at.pair_pos; *pair_rows = at.yp;
    return IFA_OK;
}
