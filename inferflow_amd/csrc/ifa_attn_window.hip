// ifa_attn_window.hip -- softmax attention over a per-sequence key / value cache in 32-bit floats with
//   * a sliding window that keeps the first tokens: query i sees key j iff j <= i and (i - j < window or j < keep_first)
//   * grouped queries (query head h reads key / value head h / (heads / kv_heads))
//   * query and key RMS-normed per head without a weight (the keys when they enter the cache)
//   * score = q.k * scale, optional soft cap (cap * tanh(score / cap)), + a learned bias per (distance bucket, head)
//   * a sink per head: exp(sink) joins the denominator, with no key and no value
// Scores, weights and sums are fp32.  The cache rows are [max_ctx][kv_heads * dim] (K: the normed keys) and [max_ctx][kv_heads * vdim]
// (V) per (slot, layer); a row is addressed by its true position, so kept first tokens keep their distances.
// The same kernels serve attention with rotated queries and keys (ifa_attention_kv_f32): there the norm (with a weight) and the
// rotation are applied by k_qk_rope_store before the keys enter the cache, the values have a size of their own, the sink has a fixed
// score and the window may be unlimited; a layer may read the cache rows that an earlier layer has written.
#include <algorithm>
#include <cstring>
#include <vector>
#include "ifa_host.h"
#include "ifa_f32_common.h"
#include "inferflow_amd.h"
#include "ifa_rows_fused.h"
#include "ifa_chunkscan.h"

using namespace ifa32;

namespace {

// one workgroup per row: K row = k / sqrt(mean_head(k^2) + eps) (norm_k != 0) or k; V row = v as given
__global__ void __launch_bounds__(256) k_kv_store_f32(const float *__restrict__ k, size_t ldk, const float *__restrict__ v, size_t ldv, int kv_heads, int dim,
                                                      int norm_k, float eps, const SeqDesc *__restrict__ seqs, const int *__restrict__ row_seq,
                                                      float *const *__restrict__ slot_base, size_t k_off, size_t v_off)
{
    const int t = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const SeqDesc sd = seqs[row_seq[t]];
    const size_t pos = (size_t)(sd.pos0 + t - sd.row0), kvd = (size_t)kv_heads * dim;
    float *kc = slot_base[sd.slot] + k_off + pos * kvd, *vc = slot_base[sd.slot] + v_off + pos * kvd;
    for (int g = wave; g < kv_heads; g += nw) {
        const float *kr = k + (size_t)t * ldk + (size_t)g * dim, *vr = v + (size_t)t * ldv + (size_t)g * dim;
        float r = 1.0f;
        if (norm_k) {
            float s = 0.0f;
            for (int c = lane; c < dim; c += 64) s = fmaf(kr[c], kr[c], s);
            r = 1.0f / sqrtf(wave_sum(s) / (float)dim + eps);
        }
        for (int c = lane; c < dim; c += 64) { vc[(size_t)g * dim + c] = vr[c]; kc[(size_t)g * dim + c] = kr[c] * r; }
    }
}

typedef float f32x4w __attribute__((ext_vector_type(4)));
// device memory, said so: loads through a pointer that came out of memory would be FLAT, and those hold up the waits for LDS
typedef const __attribute__((address_space(1))) float gfloat;
typedef const __attribute__((address_space(1))) f32x4w gf32x4;

struct WinAttnArgs {
    const float *q; size_t ldq;
    int heads, kv_heads, dim, vdim;
    int norm_q; float eps, scale, softcap;
    int window, keep_first;
    const bf16_t *rel; const int *bucket_of; int n_buckets;      // rel [n_buckets][heads]; bucket_of [distance]
    const bf16_t *sink;                                          // [heads] or null
    int sink_fixed; float sink_score;                            // sink_fixed != 0 (and sink null): every head's sink has this score
    const SeqDesc *seqs; const int *row_seq; float *const *slot_base; size_t k_off, v_off;
    float *out; size_t ldo;
    bf16_t *out16; size_t ld16;      // (k_attn_tile, k_attn_tile_combine) not null: the output in bfloat16 instead, for the product behind
    float *ws; int nsplit;           // nsplit > 1: the keys of a (row, head) are shared out to nsplit workgroups; partial results in ws [rows][heads][nsplit][dim + 2]
};

__device__ __forceinline__ bool has_sink(const WinAttnArgs &P) { return P.sink != nullptr || P.sink_fixed != 0; }
__device__ __forceinline__ float sink_of(const WinAttnArgs &P, int h) { return P.sink ? bf2f(P.sink[h]) : (P.sink_fixed ? P.sink_score : -INFINITY); }

constexpr int WA_DPL_MAX = 16;    // dim <= 64 * DPL: a lane holds DPL value columns (1, 2, 4, 10 or 16: up to 1024, the row of a latent-attention cache)

// grid (rows, heads, splits), four waves: the visible keys (kept first tokens, then the window) are walked in chunks of 16, four
// lanes per key for the score, one value column per lane for the weighted sum; chunks go round-robin to the waves, each
// with its own running maximum / sum / accumulator, merged through LDS at the end together with the sink.
// FRESH (steps of one row): the row's own key and value are not in the cache yet.  They are read as projected (F.k, F.v; norm_k: the key by its root mean
// square) and the first workgroup of their head leaves them there.
struct FreshRow { const float *k, *v; int norm_k; };

template <int WA_DPL, bool FRESH>
__device__ __forceinline__ void attn_row(const WinAttnArgs &P, const FreshRow &F, const int t, const int h, const int split, float *sm)
{
    float *qn = sm;                                   // [dim]
    float *wm = sm + P.dim, *wl = wm + 4;             // per wave: maximum, sum
    float *wacc = wl + 4;                             // [4][vdim]
    __shared__ float red[17];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int dim = P.dim, vdim = P.vdim, g = h / (P.heads / P.kv_heads);
    // FRESH: the query first, then the first keys and values, whose places do not depend on it: they are on their way under its norm, and a chunk's values under the scores of its keys
    // (the mixers' launch of a token 8.9 -> 8.15 us; with many rows the registers for it cost more: six rows 12.1 -> 13.9)
    const float *qr = P.q + (size_t)t * P.ldq + (size_t)h * dim;
    float qv[4];
#pragma unroll
    for (int e = 0; e < 4; e++) qv[e] = e == 0 || 256 * e < dim ? qr[min(tid + 256 * e, dim - 1)] : 0.0f;
    const SeqDesc sd = P.seqs[P.row_seq[t]];
    const int i = sd.pos0 + t - sd.row0;
    gfloat *own_k = nullptr, *own_v = nullptr;
    if constexpr (FRESH) { own_k = (gfloat *)F.k + (size_t)g * dim; own_v = (gfloat *)F.v + (size_t)g * vdim; }
    const int lo = max(0, i - P.window + 1), nkeep = min(P.keep_first, lo), nk = nkeep + (i - lo + 1);
    const size_t kvd = (size_t)P.kv_heads * dim, vvd = (size_t)P.kv_heads * vdim;
    gfloat *kc = (gfloat *)(P.slot_base[sd.slot] + P.k_off + (size_t)g * dim), *vc = (gfloat *)(P.slot_base[sd.slot] + P.v_off + (size_t)g * vdim);
    // 16 keys per wave and step, four lanes per key (each a quarter of the dot product in interleaved 16-byte pieces, finished by a quad sum)
    const int nchunks = (nk + 15) / 16, sub = lane & 3;
    const int nsplit = max(1, P.nsplit);
    // (heads of whole 16s up to 128: the key's pieces are held; value rows VB at a time, asked for side by side -- keys past the last: the row's own, not counted)
    constexpr int VB = WA_DPL <= 2 ? 16 : WA_DPL <= 4 ? 8 : 2;
    const bool held = FRESH && (dim & 15) == 0 && dim <= 128;
    f32x4w kq[8];
    float v[VB][WA_DPL];
    auto place = [&](int ch) { const int vi = ch * 16 + (lane >> 2); return vi < nk ? (vi < nkeep ? vi : lo + (vi - nkeep)) : i; };
    auto key_row = [&](int j) { return FRESH && j == i ? own_k : kc + (size_t)j * kvd; };
    auto ask_k = [&](int j) {
        if (!held) return;
        gfloat *kr = key_row(j);
#pragma unroll
        for (int u = 0; u < 8; u++) kq[u] = *(gf32x4 *)(kr + min(4 * sub + 16 * u, dim - 4));
    };
    auto ask_v = [&](int j, int j0) {
#pragma unroll
        for (int jj = 0; jj < VB; jj++) {
            const int kj = __shfl(j, 4 * (j0 + jj), 64);
            gfloat *vr = FRESH && kj == i ? own_v : vc + (size_t)kj * vvd;
#pragma unroll
            for (int e = 0; e < WA_DPL; e++) v[jj][e] = vr[min(lane + 64 * e, vdim - 1)];
        }
    };
    int ch = split * 4 + wave, j = place(ch);
    if (FRESH && ch < nchunks) { ask_k(j); __builtin_amdgcn_sched_barrier(0); ask_v(j, 0); }
    if constexpr (FRESH) __builtin_amdgcn_sched_barrier(0);
    {
        float s = 0.0f;
#pragma unroll
        for (int e = 0; e < 4; e++) if (tid + 256 * e < dim) s = fmaf(qv[e], qv[e], s);
        const float r = P.norm_q ? 1.0f / sqrtf(block_sum(s, red) / (float)dim + P.eps) : 1.0f;
#pragma unroll
        for (int e = 0; e < 4; e++) if (tid + 256 * e < dim) qn[tid + 256 * e] = qv[e] * r;
    }
    __syncthreads();
    float own_r = 1.0f;
    if constexpr (FRESH) {
        if (F.norm_k) {
            float s = 0.0f;
            for (int c = tid; c < dim; c += blockDim.x) s = fmaf(own_k[c], own_k[c], s);
            own_r = 1.0f / sqrtf(block_sum(s, red) / (float)dim + P.eps);
        }
        if (split == 0 && h % (P.heads / P.kv_heads) == 0) {
            float *kd = P.slot_base[sd.slot] + P.k_off + ((size_t)i * P.kv_heads + g) * dim, *vd = P.slot_base[sd.slot] + P.v_off + ((size_t)i * P.kv_heads + g) * vdim;
            for (int c = tid; c < dim; c += blockDim.x) kd[c] = own_k[c] * own_r;
            for (int c = tid; c < vdim; c += blockDim.x) vd[c] = own_v[c];
        }
    }
    float m = -INFINITY, l = 0.0f, acc[WA_DPL];
#pragma unroll
    for (int e = 0; e < WA_DPL; e++) acc[e] = 0.0f;
    while (ch < nchunks) {
        const int next = ch + 4 * nsplit;
        const bool valid = ch * 16 + (lane >> 2) < nk;
        float s = 0.0f;
        if (held) {
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const int c = 4 * sub + 16 * u;
                if (c < dim) { s = fmaf(qn[c], kq[u].x, s); s = fmaf(qn[c + 1], kq[u].y, s); s = fmaf(qn[c + 2], kq[u].z, s); s = fmaf(qn[c + 3], kq[u].w, s); }
            }
        } else {
            gfloat *kr = key_row(j);
            if ((dim & 3) == 0) {
#pragma unroll 8
                for (int c = 4 * sub; c < dim; c += 16) {
                    const f32x4w kv = *(gf32x4 *)(kr + c);
                    s = fmaf(qn[c], kv.x, s); s = fmaf(qn[c + 1], kv.y, s); s = fmaf(qn[c + 2], kv.z, s); s = fmaf(qn[c + 3], kv.w, s);
                }
            } else {
                for (int c = sub; c < dim; c += 4) s = fmaf(qn[c], kr[c], s);
            }
        }
        const int jn = place(next);
        if (FRESH && next < nchunks) ask_k(jn);
        s = quad_sum(s) * P.scale;
        if (FRESH && j == i) s *= own_r;
        if (P.softcap > 0.0f) s = P.softcap * tanhf(s / P.softcap);
        if (P.rel) s += bf2f(P.rel[(size_t)P.bucket_of[i - j] * P.heads + h]);
        if (!valid) s = -INFINITY;
        const float m_new = fmaxf(m, wave_max(s));          // finite: the chunk holds at least one visible key
        const float p = valid ? expf(s - m_new) : 0.0f;
        const float corr = m == -INFINITY ? 0.0f : expf(m - m_new);
        l = l * corr + wave_sum(sub == 0 ? p : 0.0f);
#pragma unroll
        for (int e = 0; e < WA_DPL; e++) acc[e] *= corr;
        m = m_new;
        for (int j0 = 0; j0 < 16; j0 += VB) {
            if (!FRESH || j0 > 0) ask_v(j, j0);
#pragma unroll
            for (int jj = 0; jj < VB; jj++) {
                const float pj = __shfl(p, 4 * (j0 + jj), 64);
#pragma unroll
                for (int e = 0; e < WA_DPL; e++) acc[e] = ch * 16 + j0 + jj < nk ? fmaf(pj, v[jj][e], acc[e]) : acc[e];
            }
        }
        if (FRESH && next < nchunks) ask_v(jn, 0);
        ch = next; j = jn;
    }
    if (lane == 0) { wm[wave] = m; wl[wave] = l; }
#pragma unroll
    for (int e = 0; e < WA_DPL; e++) { const int d = lane + 64 * e; if (d < vdim) wacc[wave * vdim + d] = acc[e]; }
    __syncthreads();
    if (nsplit > 1) {      // this workgroup's share: maximum, sum and weighted values relative to that maximum; the sink joins in the combine
        float M = -INFINITY;
        for (int w = 0; w < 4; w++) M = fmaxf(M, wm[w]);
        float L = 0.0f, f[4];
        for (int w = 0; w < 4; w++) { f[w] = wm[w] == -INFINITY ? 0.0f : expf(wm[w] - M); L += wl[w] * f[w]; }
        float *dst = P.ws + (((size_t)t * P.heads + h) * nsplit + split) * (vdim + 2);
        if (tid == 0) { dst[0] = M; dst[1] = L; }
        for (int d = tid; d < vdim; d += blockDim.x) {
            float o = 0.0f;
            for (int w = 0; w < 4; w++) o = fmaf(wacc[w * vdim + d], f[w], o);
            dst[2 + d] = o;
        }
        return;
    }
    const float snk = sink_of(P, h);
    float M = snk;
    for (int w = 0; w < 4; w++) M = fmaxf(M, wm[w]);
    float L = has_sink(P) ? expf(snk - M) : 0.0f;
    float f[4];
    for (int w = 0; w < 4; w++) { f[w] = wm[w] == -INFINITY ? 0.0f : expf(wm[w] - M); L += wl[w] * f[w]; }
    for (int d = tid; d < vdim; d += blockDim.x) {
        float o = 0.0f;
        for (int w = 0; w < 4; w++) o = fmaf(wacc[w * vdim + d], f[w], o);
        P.out[(size_t)t * P.ldo + (size_t)h * vdim + d] = o / L;
    }
}

template <int WA_DPL>
__global__ void __launch_bounds__(256) k_attn_window(WinAttnArgs P)
{
    extern __shared__ float sm[];
    attn_row<WA_DPL, false>(P, FreshRow(), blockIdx.x, blockIdx.y, blockIdx.z, sm);
}

// One token of decayed linear attention, S <- d S + k v^T, o = S^T q, for 64 columns of a head: four waves of dk / 4 rows each
struct StateRow { const float *q, *k, *v, *decay; int heads, dk, dv; size_t state_off; float *out; };
template <int DK4>
__device__ __forceinline__ void state_row(const StateRow &R, const SeqDesc &sd, float *state_base, const int h, const int c0, float *sm)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = min(c0 + lane, R.dv - 1), k0 = wave * DK4;
    float *S = state_base + R.state_off + ((size_t)h * R.dk + k0) * R.dv + c;
    const float *q = R.q + (size_t)h * R.dk + k0, *k = R.k + (size_t)h * R.dk + k0;
    const float d = R.decay[h], v = R.v[(size_t)h * R.dv + c];
    float x[DK4], o = 0.0f;
#pragma unroll
    for (int e = 0; e < DK4; e++) x[e] = ((gfloat *)S)[(size_t)e * R.dv];          // (whatever is there before a sequence's first token does not count)
#pragma unroll
    for (int e = 0; e < DK4; e++) {
        x[e] = fmaf(sd.pos0 > 0 ? x[e] : 0.0f, d, k[e] * v);
        o = fmaf(q[e], x[e], o);
    }
    if (c0 + lane < R.dv) {
#pragma unroll
        for (int e = 0; e < DK4; e++) S[(size_t)e * R.dv] = x[e];
    }
    sm[wave * 64 + lane] = o;
    __syncthreads();
    if (wave == 0 && c0 + lane < R.dv) R.out[(size_t)h * R.dv + c] = (sm[lane] + sm[64 + lane]) + (sm[128 + lane] + sm[192 + lane]);
}

// The mixers of a WINDOW_LINEAR layer for a step of one row in one launch: workgroups [0, heads * nsplit) the attention with the row's own key and value, the rest
// the decayed linear attention (9 us; three launches of 4, 7.5 and 4 otherwise)
template <int WA_DPL, int DK4>
__global__ void __launch_bounds__(256) k_mix_row(WinAttnArgs P, FreshRow F, StateRow R)
{
    extern __shared__ float sm[];
    const int nsplit = max(1, P.nsplit), na = P.heads * nsplit, id = blockIdx.x;
    if (id < na) { attn_row<WA_DPL, true>(P, F, 0, id % P.heads, id / P.heads, sm); return; }
    const int per = (R.dv + 63) / 64;
    const SeqDesc sd = P.seqs[0];
    state_row<DK4>(R, sd, P.slot_base[sd.slot], (id - na) / per, (id - na) % per * 64, sm);
}

// grid (rows, heads), one or two waves (a group of 64 columns each): the shares of a (row, head) and its sink into the output row.  Lane sp holds share sp's maximum and
// sum, so the scale factors come from two wave reductions; the weighted values are then read for all shares at once.
constexpr int WA_MAX_SPLITS = 32;

__global__ void __launch_bounds__(128) k_attn_window_combine(WinAttnArgs P)
{
    const int t = blockIdx.x, h = blockIdx.y, dim = P.vdim, nsplit = P.nsplit, lane = threadIdx.x & 63;      // (dim: columns of a value row)
    const float *src = P.ws + ((size_t)t * P.heads + h) * nsplit * (dim + 2);
    const float snk = sink_of(P, h);
    const float m_sp = lane < nsplit ? src[(size_t)lane * (dim + 2)] : -INFINITY, l_sp = lane < nsplit ? src[(size_t)lane * (dim + 2) + 1] : 0.0f;
    const float M = fmaxf(snk, wave_max(m_sp));
    const float f_sp = m_sp == -INFINITY ? 0.0f : expf(m_sp - M);
    const float L = wave_sum(l_sp * f_sp) + (has_sink(P) ? expf(snk - M) : 0.0f);
    // (every lane walks every group of 64 columns, also where it has no column of its own: the scale factors come from other lanes)
    for (int d0 = threadIdx.x & 64; d0 < dim; d0 += blockDim.x) {
        const int d = d0 + lane;
        float v[WA_MAX_SPLITS];
#pragma unroll
        for (int sp = 0; sp < WA_MAX_SPLITS; sp++) v[sp] = src[(size_t)min(sp, nsplit - 1) * (dim + 2) + 2 + min(d, dim - 1)];      // (no branch: all at once)
        float o = 0.0f;
#pragma unroll
        for (int sp = 0; sp < WA_MAX_SPLITS; sp++) o = sp < nsplit ? fmaf(v[sp], __shfl(f_sp, sp, 64), o) : o;
        if (d < dim) P.out[(size_t)t * P.ldo + (size_t)h * dim + d] = o / L;
    }
}

typedef float f32x16w __attribute__((ext_vector_type(16)));
constexpr int WT_K = 32;          // keys of a block

// ---- prompts without a workspace: 128 queries of one sequence per workgroup, the visible keys walked in blocks of 32 that are staged ONCE per workgroup
// in LDS; each wave owns 32 queries, one per lane of each half: S^T = K Q^T and O^T += V^T P^T on the fp32 matrix cores
// (v_mfma_f32_32x32x2_f32: scores and weights stay 32-bit).  In the transposed products a lane's accumulators hold 16 keys of ITS
// query, so the online softmax (running maximum, weights, rescaling of O^T) is lane-local but for one exchange between the halves,
// and the weights are the second product's B operand as they lie in the accumulators: no trip through LDS.
constexpr int WT_Q = 128;

// Key rows of dim <= 32 NTK and value rows of vdim <= 32 NTV floats; the columns beyond are zero in LDS.
template <int NTK, int NTV>
__global__ void __launch_bounds__(256) k_attn_window_tile(WinAttnArgs P, int n_seqs, int vec)
{
    constexpr int DK = 32 * NTK, DKP = DK + 1, DV = 32 * NTV, DVP = DV + 1;
    extern __shared__ float sm[];
    float *Qs = sm;                          // [128][DKP]
    float *Ks = Qs + WT_Q * DKP;             // [32][DKP]
    float *Vs = Ks + WT_K * DKP;             // [32][DVP]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i = lane & 31, g = lane >> 5;
    const int h = blockIdx.x, kvh = h / (P.heads / P.kv_heads), dk = P.dim, dv = P.vdim;
    // which sequence and which of its 128-row tiles.  The grid runs over (head, tile) with the head as the fast index and the tiles from
    // the last one down: the tiles with the most key blocks start first, and the query heads of a group, which read the same key and
    // value rows, run side by side.
    int tile = (int)(gridDim.y - 1 - blockIdx.y), sq = 0;
    for (; sq < n_seqs; sq++) {
        const int nt = (P.seqs[sq].n + WT_Q - 1) / WT_Q;
        if (tile < nt) break;
        tile -= nt;
    }
    if (sq >= n_seqs) return;
    const SeqDesc sd = P.seqs[sq];
    const int r0 = sd.row0 + tile * WT_Q, nq = min(WT_Q, sd.n - tile * WT_Q), p0 = sd.pos0 + tile * WT_Q;
    const size_t kvd = (size_t)P.kv_heads * dk, vvd = (size_t)P.kv_heads * dv;
    const float *kc = P.slot_base[sd.slot] + P.k_off + (size_t)kvh * dk, *vc = P.slot_base[sd.slot] + P.v_off + (size_t)kvh * dv;
    // Q rows of this wave, normed, into LDS
    for (int rr = 0; rr < 32; rr++) {
        const int q = 32 * wave + rr;
        float v[NTK > 2 ? 2 : 1];
        float ssum = 0.0f;
#pragma unroll
        for (int e = 0; e < (NTK > 2 ? 2 : 1); e++) {
            const int c = lane + 64 * e;
            v[e] = (q < nq && c < dk) ? P.q[(size_t)(r0 + q) * P.ldq + (size_t)h * dk + c] : 0.0f;
            ssum = fmaf(v[e], v[e], ssum);
        }
        const float rinv = P.norm_q ? 1.0f / sqrtf(wave_sum(ssum) / (float)dk + P.eps) : 1.0f;
#pragma unroll
        for (int e = 0; e < (NTK > 2 ? 2 : 1); e++) { const int c = lane + 64 * e; if (c < DK) Qs[q * DKP + c] = v[e] * rinv; }
    }
    const int nq_w = min(32, max(0, nq - 32 * wave));             // queries of this wave
    const int qlo = p0 + 32 * wave, qhi = qlo + nq_w - 1;          // their positions
    const int lo_min = max(0, p0 - P.window + 1), nkeep = min(P.keep_first, lo_min), p_last = p0 + nq - 1;
    const int nb_keep = (nkeep + WT_K - 1) / WT_K, nb_win = (p_last - lo_min + 1 + WT_K - 1) / WT_K;
    f32x16w o[NTV];
    float m = -INFINITY, l = 0.0f;          // of the lane's query (lane & 31)
#pragma unroll
    for (int nt = 0; nt < NTV; nt++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[nt][r] = 0.0f;
    // 16-byte path: a thread stages NTK pieces of the key block and NTV of the value block; the pieces of block b + 1 are asked for
    // before block b is worked on and wait in registers meanwhile, so that the loads run behind the matrix-core work
    float4 kreg[NTK], vreg[NTV];
    auto fetch = [&](int b) {
        const bool kept = b < nb_keep;
        const int kb0 = kept ? b * WT_K : lo_min + (b - nb_keep) * WT_K;
        const int kc_n = kept ? min(WT_K, nkeep - kb0) : min(WT_K, p_last - kb0 + 1);
#pragma unroll
        for (int u = 0; u < NTK; u++) {
            const int e = tid + 256 * u, row = e / (DK / 4), c4 = (e % (DK / 4)) * 4;
            kreg[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (row < kc_n && c4 < dk) kreg[u] = *reinterpret_cast<const float4 *>(kc + (size_t)(kb0 + row) * kvd + c4);
        }
#pragma unroll
        for (int u = 0; u < NTV; u++) {
            const int e = tid + 256 * u, row = e / (DV / 4), c4 = (e % (DV / 4)) * 4;
            vreg[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (row < kc_n && c4 < dv) vreg[u] = *reinterpret_cast<const float4 *>(vc + (size_t)(kb0 + row) * vvd + c4);
        }
    };
    const int nb_all = nb_keep + nb_win;
    if (vec && nb_all > 0) fetch(0);
    for (int b = 0; b < nb_all; b++) {
        const bool kept = b < nb_keep;
        const int kb0 = kept ? b * WT_K : lo_min + (b - nb_keep) * WT_K;
        const int kc_n = kept ? min(WT_K, nkeep - kb0) : min(WT_K, p_last - kb0 + 1);
        __syncthreads();                 // the previous block's K / V reads are done (and Q is staged)
        if (vec) {
#pragma unroll
            for (int u = 0; u < NTK; u++) {
                const int e = tid + 256 * u, row = e / (DK / 4), c4 = (e % (DK / 4)) * 4;
                float *kd = Ks + row * DKP + c4;
                kd[0] = kreg[u].x; kd[1] = kreg[u].y; kd[2] = kreg[u].z; kd[3] = kreg[u].w;
            }
#pragma unroll
            for (int u = 0; u < NTV; u++) {
                const int e = tid + 256 * u, row = e / (DV / 4), c4 = (e % (DV / 4)) * 4;
                float *vd = Vs + row * DVP + c4;
                vd[0] = vreg[u].x; vd[1] = vreg[u].y; vd[2] = vreg[u].z; vd[3] = vreg[u].w;
            }
            if (b + 1 < nb_all) fetch(b + 1);
        } else {
            for (int e = tid; e < WT_K * DK; e += 256) {
                const int row = e / DK, c = e % DK;
                Ks[row * DKP + c] = (row < kc_n && c < dk) ? kc[(size_t)(kb0 + row) * kvd + c] : 0.0f;
            }
            for (int e = tid; e < WT_K * DV; e += 256) {
                const int row = e / DV, c = e % DV;
                Vs[row * DVP + c] = (row < kc_n && c < dv) ? vc[(size_t)(kb0 + row) * vvd + c] : 0.0f;
            }
        }
        __syncthreads();
        const bool active = nq_w > 0 && kb0 <= qhi && (kept || kb0 + kc_n - 1 >= qlo - P.window + 1 || kb0 < P.keep_first);
        if (active) {
            // S^T = K Q^T: the lane's 16 accumulators are 16 KEYS of ITS query (lane & 31), so the running maximum, the weights and the
            // rescaling stay inside the lane but for one exchange between the two halves of the wave
            f32x16w acc;
#pragma unroll
            for (int r = 0; r < 16; r++) acc[r] = 0.0f;
            const float *qa = Qs + (32 * wave + i) * DKP + g, *ka = Ks + i * DKP + g;
#pragma unroll 8
            for (int s2 = 0; s2 < DK / 2; s2++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(ka[2 * s2], qa[2 * s2], acc, 0, 0, 0);
            const int iq = qlo + i;
            const bool qin = i < nq_w;
            float mloc = -INFINITY;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int kk = (r & 3) + 8 * (r >> 2) + 4 * g, j = kb0 + kk;
                const bool vis = qin && kk < kc_n && j <= iq && (iq - j < P.window || j < P.keep_first);
                float sc = acc[r] * P.scale;
                if (P.softcap > 0.0f) sc = P.softcap * tanhf(sc / P.softcap);
                if (P.rel && vis) sc += bf2f(P.rel[(size_t)P.bucket_of[iq - j] * P.heads + h]);
                sc = vis ? sc : -INFINITY;
                acc[r] = sc;
                mloc = fmaxf(mloc, sc);
            }
            mloc = fmaxf(mloc, __shfl_xor(mloc, 32, 64));
            const float m_new = fmaxf(m, mloc);
            const float corr = m == -INFINITY ? 1.0f : expf(m - m_new);      // (m_new == -inf only while nothing was visible: sums are 0)
            float psum = 0.0f;
#pragma unroll
            for (int r = 0; r < 16; r++) { acc[r] = acc[r] == -INFINITY ? 0.0f : expf(acc[r] - m_new); psum += acc[r]; }
            l = l * corr + psum;             // (the keys of this half of the wave; the halves are added at the end)
            m = m_new;
            // O^T += V^T P^T: the weights are the B operand as they lie in the accumulators (step s2 takes keys (s2 & 3) + 8 (s2 >> 2) + 4 g)
#pragma unroll
            for (int nt = 0; nt < NTV; nt++) {
#pragma unroll
                for (int r = 0; r < 16; r++) o[nt][r] *= corr;
                const float *va = Vs + 4 * g * DVP + 32 * nt + i;
#pragma unroll
                for (int s2 = 0; s2 < 16; s2++)
                    o[nt] = __builtin_amdgcn_mfma_f32_32x32x2f32(va[((s2 & 3) + 8 * (s2 >> 2)) * DVP], acc[s2], o[nt], 0, 0, 0);
            }
        }
    }
    // the lane holds value columns 32 nt + (r & 3) + 8 (r >> 2) + 4 g of its query
    const float snk = sink_of(P, h);
    const float ls = l + __shfl_xor(l, 32, 64);
    if (i < nq_w) {
        const float M = fmaxf(m, snk);
        const float f = expf(m - M);
        const float L = ls * f + (has_sink(P) ? expf(snk - M) : 0.0f);
        const float sc = f / L;
        float *dst = P.out + (size_t)(r0 + 32 * wave + i) * P.ldo + (size_t)h * dv;
#pragma unroll
        for (int nt = 0; nt < NTV; nt++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int c = 32 * nt + (r & 3) + 8 * (r >> 2) + 4 * g;
                if (c < dv) dst[c] = o[nt][r] * sc;
            }
    }
}

// ---- prompts with a workspace, on the bfloat16 matrix cores.  A workgroup of eight waves holds 32 queries of up to four query heads that share a key / value head
// (hpw heads; the waves take further queries beyond them) and walks a share of their visible keys in blocks of 32.  The products are transposed as above.
// Arithmetic: every 32-bit operand is the sum of three bfloat16 values (24 bits: nothing is lost but the last rounding), and a product takes
// the six of the nine partial products that reach 2^-24 of the largest: 6 x 32 matrix-core cycles per 16 columns where the fp32 instructions
// take 512.  Error against 64 bits: no larger than the fp32 instructions' (test_tiled_attention_with_a_workspace_against_64_bits_and_the_fp32_tiles).
// In blocks with an infinity or NaN among the keys or values (k_attn_parts marks them) the queries' and weights' parts are formed so that no lower part of 0 meets an infinity.  (An
// infinity in a query is not looked for: its scores are infinities of both signs, their weights NaN.)
// The fp32 tiles above took 487 us for 2048 causal tokens of 8 heads of 128 (16 tiles x 8 heads on half of the compute units, the last tile alone walking 64 blocks)
// and 420 us for 16 heads with a window of 1024, soft cap and bias; this form 83 and 146 us, of it 6 us for the operands and 14 us for joining the
// shares.  Bound by matrix cores and vector instructions in turn (3072 and ~2500 cycles per wave and block; the waves of a SIMD do not drift apart enough to
// overlap them).  Hence the operands are split and laid out once per layer by k_attn_parts, not by every tile that reads them (staged and split per
// workgroup: 126 us), and the key blocks of long tiles go to several workgroups (chunks of cb blocks, joined by k_attn_tile_combine).
typedef __bf16 bf16x8w __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4w __attribute__((ext_vector_type(4)));
constexpr int WT_WAVES = 8, WT_MAX_CHUNKS = 32, WT_SLOTS = 256;

typedef const __attribute__((address_space(1))) void wa_glb_t;
typedef __attribute__((address_space(3))) void wa_lds_t;

struct Parts { bf16x8w p[3]; };

// CHECKED false: of values that do not round to infinity
template <bool CHECKED = true>
__device__ __forceinline__ Parts parts_of(const float *v)
{
    Parts r;
    float big = 0.0f, d[8];
    if constexpr (CHECKED) {
#pragma unroll
        for (int e = 0; e < 8; e++) big = fmaxf(big, __builtin_fabsf(v[e]));
    }
#pragma unroll
    for (int e = 0; e < 8; e++) { r.p[0][e] = (__bf16)v[e]; d[e] = v[e] - (float)r.p[0][e]; }
    if (CHECKED && __builtin_amdgcn_ballot_w64(big > 3.38e38f)) {          // (the first part of what would round to infinity is cut off instead; infinities stay in it)
#pragma unroll
        for (int e = 0; e < 8; e++)
            if (__builtin_fabsf(v[e]) > 3.38e38f) {
                const float cut = __uint_as_float(__float_as_uint(v[e]) & 0xFFFF0000u);
                r.p[0][e] = (__bf16)cut; d[e] = __builtin_fabsf(v[e]) == INFINITY ? 0.0f : v[e] - cut;
            }
    }
#pragma unroll
    for (int e = 0; e < 8; e++) { r.p[1][e] = (__bf16)d[e]; r.p[2][e] = (__bf16)(d[e] - (float)r.p[1][e]); }
    return r;
}

// For products with an infinity: the same values (zero apart) in three parts of one sign, none of them zero, so that each partial product is an infinity of the sum's sign.
// Cut off instead of rounded; where nothing is left the smallest normal number, which adds nothing to a finite product.
__device__ __forceinline__ Parts one_sign(const Parts &t)
{
    Parts r;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const float x = (float)t.p[0][e] + ((float)t.p[1][e] + (float)t.p[2][e]), least = x == 0.0f ? 0.0f : __builtin_copysignf(1.17549435e-38f, x);
        const float a = __uint_as_float(__float_as_uint(x) & 0xFFFF0000u), d = x - a, b = __uint_as_float(__float_as_uint(d) & 0xFFFF0000u), c = d - b;
        r.p[0][e] = (__bf16)a; r.p[1][e] = (__bf16)(b == 0.0f ? least : b); r.p[2][e] = (__bf16)(c == 0.0f ? least : c);
    }
    return r;
}
// (back again)
__device__ __forceinline__ Parts rounded(const Parts &t)
{
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = (float)t.p[0][e] + ((float)t.p[1][e] + (float)t.p[2][e]);
    return parts_of(v);
}

__device__ __forceinline__ bool not_finite(const float *v)
{
    float z = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; e++) z = fmaf(v[e], 0.0f, z);
    return z != 0.0f;          // (0, or NaN from any of them)
}

// the five partial products below the leading one, smallest first
__device__ __forceinline__ f32x16w mfma_rest(const Parts &a, const Parts &b, f32x16w c)
{
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.p[2], b.p[0], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.p[0], b.p[2], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.p[1], b.p[1], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.p[1], b.p[0], c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.p[0], b.p[1], c, 0, 0, 0);
}

// exp(x) for x <= 0 to within a rounding or two: the rounding of x log2(e) is carried along (the exponential of a plain fp32 product would be off
// by |x| 2^-24); NaN stays NaN
__device__ __forceinline__ float exp_neg(float x)
{
    x = x < -1.0e4f ? -1.0e4f : x;
    const float hi = x * 1.44269502f, lo = fmaf(x, 1.92596299e-8f, fmaf(x, 1.44269502f, -hi));
    const float e = __builtin_amdgcn_exp2f(hi);
    return fmaf(e, lo * 0.693147182f, e);
}

// tanh(y) to within two roundings, without a branch: the continued fraction y / (1 + y^2 / (3 + y^2 / (5 + y^2 / (7 + y^2 / 9)))) as a quotient where |y| < 0.6
// (its remainder is below 1e-9 there), (1 - e) / (1 + e) with e = exp(-2 |y|) elsewhere
__device__ __forceinline__ float tanh_sel(float y)
{
    const float a = __builtin_fabsf(y), z = y * y, e = exp_neg(-2.0f * a);
    const bool small = a < 0.6f;
    const float n = small ? a * fmaf(z, z + 105.0f, 945.0f) : 1.0f - e, d = small ? fmaf(z, fmaf(z, 15.0f, 420.0f), 945.0f) : 1.0f + e;
    const float r = __builtin_amdgcn_rcpf(d), t = n * r;
    return __builtin_copysignf(fmaf(fmaf(-t, d, n), r, t), y);
}

// The key blocks of a sequence are counted in absolute positions (block = position / 32).  What k_attn_parts lays out for a step: the blocks of the
// kept first tokens, then those from the first one that the step's first query sees to the last.
struct SeqBlocks { int kept, first, count; };
__host__ __device__ __forceinline__ SeqBlocks seq_blocks(int pos0, int n, int window, int keep_first)
{
    const int lo = pos0 - window + 1 > 0 ? pos0 - window + 1 : 0, end = pos0 + n, keep = keep_first < end ? keep_first : end;
    SeqBlocks s;
    s.kept = (keep + WT_K - 1) / WT_K;
    s.first = s.kept > lo / WT_K ? s.kept : lo / WT_K;
    const int more = (end - 1) / WT_K - s.first + 1;
    s.count = s.kept + (more > 0 ? more : 0);
    return s;
}
// the blocks that nq queries from position p0 on see: 0 .. kept - 1, then `first` and on, nb in all
struct TileBlocks { int kept, first, nb; };
__host__ __device__ __forceinline__ TileBlocks tile_blocks(int p0, int nq, int window, int keep_first)
{
    const int lo = p0 - window + 1 > 0 ? p0 - window + 1 : 0, keep = keep_first < lo ? keep_first : lo;
    TileBlocks t;
    t.kept = (keep + WT_K - 1) / WT_K;
    t.first = t.kept > lo / WT_K ? t.kept : lo / WT_K;
    const int more = (p0 + nq - 1) / WT_K - t.first + 1;
    t.nb = t.kept + (more > 0 ? more : 0);
    return t;
}

// marks, shares: where the blocks' marks and the chunks' partial results begin in the workspace (floats), behind the operands
// few: a step's sequences, where there are up to FEW, and the chunks of those behind, the tiles and the operand blocks of those in front of each: tables in memory, each behind the other, were a
// microsecond a trip in front of everything else.  Four: every further one is 28 bytes of arguments and a choice in front of each place, in three launches a layer.  With eight, steps of five to
// eight sequences are 0.2 to 1 % of a whole prompt faster (Sopulorn of width 1024, 5 x 400 tokens 1326 -> 1317 us, 8 x 200 1208 -> 1198) and steps of one to four, the most frequent ones, 0.3 to
// 1.3 % slower (1 x 16 770 -> 780, 1 x 601 1112 -> 1118, 3 x 411 1152 -> 1160); with sixteen everything is 1 to 2 % slower (Gelarax 1 x 601 1052 -> 1067, Sopulorn 16 x 100 1095 -> 1115)
constexpr int FEW = 4;
struct FewSeq { SeqDesc sd; int chunk0, tile0, block0; };
struct TileArgs { int n_seqs, hpw, cb, tiles; size_t marks, shares; int n_few; FewSeq few[FEW]; };
// the sequence that holds an item, the first items of the sequences given by `at`
template <class At>
__device__ __forceinline__ FewSeq few_of(const TileArgs &A, int id, At at)
{
    FewSeq f = A.few[0];
#pragma unroll
    for (int s = 1; s < FEW; s++) if (s < A.n_few && id >= at(A.few[s])) f = A.few[s];
    return f;
}

// The windowed attention's launches may bring the decayed linear attention's of the same layer with them (IfaLinearSide): chunk sums beside the keys' operands, the states from chunk to chunk
// beside the tiles, the chunks' outputs beside the shares.  Alone, each of them left most of the chip idle: 601 rows of width 1024 (8 heads, 2 of keys) 4.8 + 6.1 + 15.0, 27.6 + 4.9 and
// 9.0 + 11.2 us, together 15.9, 24.8 and 12.8; 2048 rows of width 2048 (16 heads, 4) 6.2 + 8.4 + 30.2, 114.9 + 9.9 and 11.6 + 23.8, together 38.2, 111.3 and 32.5 (tiles whose queries are asked
// for at once, see k_attn_tile, in the second figures only)
// At most SIDE_SEQS sequences: a chunk's workgroup finds its sequence by going through them, and has more others beside it to hide that in launches of its own; and the states beside the tiles up
// to SIDE_PASS workgroups, each of which takes a tile's place on its compute unit (100 KB of LDS), in a launch of their own beyond.  A model's prompts, us, with the launches of its own / shared /
// shared but for the states, n sequences of up to l tokens: width 1024, 128 such workgroups a sequence: 16 x 300 1884 / 1808 / 1813, 24 x 200 2263 / 2218 / 2202, 32 x 130 2185 / 2176 / 2129,
// 32 x 400 4418 / 4461 / 4385, 64 x 130 3632 / 3898 / 3641, 64 x 200 4707 / 4991 / 4752, 128 x 150 7578 / 8711 / 7958; width 2048, 256 a sequence: 1 x 2048 4372 / 4265 / 4328, 16 x 200
// 3144 / 3170 / 3127, 32 x 200 6075 / 6245 / 6059
constexpr int SIDE_SEQS = 32, SIDE_PASS = 2048;
struct SideArgs { ifachunk::ChunkArgs c; int chunks, zc, first, pass, per; };          // zc: pieces of 64 value columns; workgroups of the first and third launch, of the second (per: a head's)

// The item (of n) that a number running over all items' counts falls into, or -1; id becomes the number inside it.  A wave looks at 64 items at a time (walked by one thread,
// a step of 1024 sequences behind 100 keys each took 10.6 ms, now 0.37; 512 behind 200 2.0 ms, now 0.26).  count: called by all lanes, -1 for none.
template <class Count>
__device__ __forceinline__ int item_of(int n, int &id, Count count)
{
    const int lane = threadIdx.x & 63;
    for (int s0 = 0; s0 < n; s0 += 64) {
        const int c = count(s0 + lane < n ? s0 + lane : -1);
        int upto = c;
#pragma unroll
        for (int k = 1; k < 64; k <<= 1) { const int x = __shfl_up(upto, k, 64); if (lane >= k) upto += x; }
        const uint64_t past = __builtin_amdgcn_ballot_w64(upto > id);
        if (past) {
            const int at = __builtin_ctzll(past);
            id -= __builtin_amdgcn_readlane(upto, at) - __builtin_amdgcn_readlane(c, at);
            return s0 + at;
        }
        id -= __builtin_amdgcn_readlane(upto, 63);
    }
    return -1;
}
__device__ __forceinline__ int wave_sum_i(int v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// The id-th chunk of the step, the chunks numbered tile by tile from the last sequence's last tile on: its sequence, its tile there (of qw queries) and over the step, its number
// in the tile, the operand blocks of the sequences before.  A grid of tiles x chunks would do without this, but its empty places leave some XCD with more chunks
// than compute units, and the launch takes twice as long (100 against 50 us at 2048 tokens).
struct ChunkPlace { SeqDesc sd; int tile, tile_g, chunk, block0; };
__device__ __forceinline__ bool chunk_of(const WinAttnArgs &P, const TileArgs &A, int qw, int id, ChunkPlace &at)
{
    const int lane = threadIdx.x & 63;
    auto chunks = [&](int pos0, int n, int tile) { return (tile_blocks(pos0 + tile * qw, min(qw, n - tile * qw), P.window, P.keep_first).nb + A.cb - 1) / A.cb; };
    auto place = [&](const SeqDesc &sd) {          // (id: inside the sequence)
        const int nt = (sd.n + qw - 1) / qw, back = item_of(nt, id, [&](int x) { return x >= 0 ? chunks(sd.pos0, sd.n, nt - 1 - x) : 0; });
        at.sd = sd; at.chunk = id; at.tile = nt - 1 - back;
        return back >= 0;
    };
    if (A.n_few) {
        FewSeq f = A.few[0];          // (numbered from the last one on: its chunk0 is 0)
#pragma unroll
        for (int s = FEW - 1; s >= 0; s--) if (s < A.n_few && id >= A.few[s].chunk0) f = A.few[s];
        id -= f.chunk0;
        if (!place(f.sd)) return false;
        at.block0 = f.block0; at.tile_g = f.tile0 + at.tile;
        return true;
    }
    int sq = 0;
    {
        const int back = item_of(A.n_seqs, id, [&](int x) {
            int pos0 = 0, n = 0, c = 0;
            if (x >= 0) { const SeqDesc &sd = P.seqs[A.n_seqs - 1 - x]; pos0 = sd.pos0; n = sd.n; }
            const int nt = (n + qw - 1) / qw;
            if (nt <= 4) for (int t = 0; t < nt; t++) c += chunks(pos0, n, t);
            for (uint64_t many = __builtin_amdgcn_ballot_w64(nt > 4); many; many &= many - 1) {          // (sequences of many tiles: the wave counts them together)
                const int l = __builtin_ctzll(many), p = __builtin_amdgcn_readlane(pos0, l), m = __builtin_amdgcn_readlane(n, l), mt = __builtin_amdgcn_readlane(nt, l);
                int part = 0;
                for (int t = lane; t < mt; t += 64) part += chunks(p, m, t);
                part = wave_sum_i(part);
                if (lane == l) c = part;
            }
            return c;
        });
        if (back < 0) return false;
        sq = A.n_seqs - 1 - back;
    }
    if (!place(P.seqs[sq])) return false;
    int blocks = 0, tiles = 0;
    for (int s = lane; s < sq; s += 64) {
        const SeqDesc &b = P.seqs[s];
        blocks += seq_blocks(b.pos0, b.n, P.window, P.keep_first).count;
        tiles += (b.n + qw - 1) / qw;
    }
    if (sq > 0) { blocks = wave_sum_i(blocks); tiles = wave_sum_i(tiles); }
    at.block0 = __builtin_amdgcn_readfirstlane(blocks);
    at.tile_g = __builtin_amdgcn_readfirstlane(tiles) + at.tile;
    return true;
}

// Operands of one block of 32 keys as the matrix instructions take them, [part][16 columns][lane][8]: keys (lane = 32 g + key, columns 16 ks + 8 g ..), then
// values transposed (lane = 32 g + column, keys in the order in which the scores' accumulators hold them).  Columns beyond the rows' ends are zero.
template <int NTK, int NTV> constexpr int kBlockPieces = 3 * 64 * (2 * NTK + 2 * NTV);

// One head of a row: its root mean square norm (with a weight), then the turn of its first rot_dims dimensions in pairs (see k_qk_rope_store); cs: [rot_dims / 2] cos, [rot_dims / 2] sin of
// its position.  A wave; every lane reads both members of its pairs before anything is written, so that dst may be src (dim <= 64 CPL)
template <int CPL>
__device__ __forceinline__ void turn_head(const float *src, float *dst, int dim, bool norm, const bf16_t *nw_, float eps, int rot_dims, int pairing, const float *cs, int lane)
{
    const int half = rot_dims / 2;
    float r = 1.0f;
    if (norm) {
        float s = 0.0f;
        for (int c = lane; c < dim; c += 64) s = fmaf(src[c], src[c], s);
        r = 1.0f / sqrtf(wave_sum(s) / (float)dim + eps);
    }
    float val[CPL], oth[CPL];
#pragma unroll
    for (int e = 0; e < CPL; e++) {
        const int c = lane + 64 * e;
        val[e] = oth[e] = 0.0f;
        if (c < dim) {
            val[e] = src[c] * r * (nw_ ? bf2f(nw_[c]) : 1.0f);
            if (c < rot_dims) { const int pc = pairing ? c ^ 1 : (c < half ? c + half : c - half); oth[e] = src[pc] * r * (nw_ ? bf2f(nw_[pc]) : 1.0f); }
        }
    }
#pragma unroll
    for (int e = 0; e < CPL; e++) {
        const int c = lane + 64 * e;
        if (c >= dim) continue;
        float out = val[e];
        if (c < rot_dims) {
            const bool first = pairing ? (c & 1) == 0 : c < half;          // first or second member of its pair
            const int fi = pairing ? c >> 1 : (c < half ? c : c - half);
            out = first ? val[e] * cs[fi] - oth[e] * cs[half + fi] : val[e] * cs[fi] + oth[e] * cs[half + fi];
        }
        dst[c] = out;
    }
}

__device__ __forceinline__ void angle_of(int pos, const double *__restrict__ freq, int i, int half, float *cs)
{
    const double a = (double)pos * freq[i];
    double sn, cn; sincos(a, &sn, &cn);          // (one argument reduction for both)
    cs[i] = (float)cn; cs[half + i] = (float)sn;
}

// turn_head of a head of at most 64 E that a wave holds, E values a lane (lane and lane + 64); w: the norm's weights (1: none), cs: the cosines and sines of the lane's pairs
template <int E> struct Turn { int half, from[E]; bool first[E]; float w[E]; };
template <int E>
__device__ __forceinline__ Turn<E> turn_of(int dim, int rot_dims, const bf16_t *nw_, int lane)
{
    Turn<E> u;
    u.half = rot_dims / 2;
#pragma unroll
    for (int e = 0; e < E; e++) { const int c = lane + 64 * e; u.w[e] = nw_ ? bf2f(nw_[min(c, dim - 1)]) : 1.0f; u.first[e] = c < u.half; u.from[e] = c < u.half ? c + u.half : c - u.half; }
    return u;
}
// the factor of a held head's root mean square norm
template <int E>
__device__ __forceinline__ float norm_held(const float (&v)[E], int dim, float eps, int lane)
{
    float s = 0.0f;
#pragma unroll
    for (int e = 0; e < E; e++) if (lane + 64 * e < dim) s = fmaf(v[e], v[e], s);
    return 1.0f / sqrtf(wave_sum(s) / (float)dim + eps);
}
template <int E>
__device__ __forceinline__ void turn_held(float (&v)[E], const Turn<E> &u, int dim, bool norm, float eps, int rot_dims, const float (&cv)[E], const float (&sv)[E], int lane)
{
    float r = 1.0f, val[E];
    if (norm) r = norm_held<E>(v, dim, eps, lane);
#pragma unroll
    for (int e = 0; e < E; e++) val[e] = v[e] * r * u.w[e];
#pragma unroll
    for (int e = 0; e < E; e++) {
        float oth = __shfl(val[0], u.from[e] & 63, 64);
        if constexpr (E == 2) { const float b = __shfl(val[1], u.from[e] & 63, 64); oth = u.from[e] < 64 ? oth : b; }
        v[e] = lane + 64 * e >= rot_dims ? val[e] : (u.first[e] ? val[e] * cv[e] - oth * sv[e] : val[e] * cv[e] + oth * sv[e]);
    }
}
template <int E>
__device__ __forceinline__ void turn_angles(const float *cs, const Turn<E> &u, int rot_dims, int lane, float (&cv)[E], float (&sv)[E])
{
#pragma unroll
    for (int e = 0; e < E; e++) {
        const int c = lane + 64 * e, fi = u.first[e] ? c : c - u.half;
        const bool in = c < rot_dims;
        cv[e] = in ? cs[fi] : 1.0f; sv[e] = in ? cs[u.half + fi] : 0.0f;
    }
}

// a row's heads in place, eight at a time (those of part `part` of `parts`), all their values asked for beside the row's place: a wave (cs: its own)
constexpr int HB = 8;
template <int E, class Pos>
__device__ __forceinline__ void turn_row(float *q, int heads, int part, int parts, int dim, const bf16_t *nw_, float eps, int rot_dims, const double *freq, float *cs, int lane, Pos position)
{
    const Turn<E> u = turn_of<E>(dim, rot_dims, nw_, lane);
    float cv[E], sv[E];
    for (int h0 = HB * part; h0 < heads; h0 += HB * parts) {
        float v[HB][E];
#pragma unroll
        for (int h = 0; h < HB; h++)
#pragma unroll
            for (int e = 0; e < E; e++) v[h][e] = q[(size_t)min(h0 + h, heads - 1) * dim + min(lane + 64 * e, dim - 1)];
        if (h0 == HB * part) {
            const int pos = position();
            for (int i = lane; i < u.half; i += 64) angle_of(pos, freq, i, u.half, cs);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");          // (the wave's own)
            turn_angles<E>(cs, u, rot_dims, lane, cv, sv);
        }
#pragma unroll
        for (int h = 0; h < HB; h++) {
            turn_held<E>(v[h], u, dim, nw_ != nullptr, eps, rot_dims, cv, sv, lane);
#pragma unroll
            for (int e = 0; e < E; e++) if (h0 + h < heads && lane + 64 * e < dim) q[(size_t)(h0 + h) * dim + lane + 64 * e] = v[h][e];
        }
    }
}

// What a step brings to the cache (k null: nothing, or it is there already): keys as projected, normed and turned as k_kv_store_f32 and k_qk_rope_store do, and values; q_rows: the step's
// queries are normed and turned in place by waves behind the blocks' workgroups, q_parts of them a row.
struct FreshKV { const float *k; size_t ldk; const float *v; size_t ldv; int norm; const bf16_t *norm_w; float eps; int rot_dims; const double *freq; int q_rows, q_parts, q_wgs; const bf16_t *q_norm_w; float *q; };          // (q_rows 0: the queries are not turned)

// the sequence of the step's block `at`, which becomes the number inside it; false: there is none
__device__ __forceinline__ bool block_seq(const WinAttnArgs &P, const TileArgs &A, int &at, SeqDesc &sd)
{
    if (A.n_few) { const FewSeq f = few_of(A, at, [](const FewSeq &x) { return x.block0; }); sd = f.sd; at -= f.block0; return true; }
    const int sq = item_of(A.n_seqs, at, [&](int x) { if (x < 0) return 0; const SeqDesc &b = P.seqs[x]; return seq_blocks(b.pos0, b.n, P.window, P.keep_first).count; });
    if (sq < 0) return false;
    sd = P.seqs[sq];
    return true;
}

// grid (kv heads, blocks of the step): the cache rows of a block into its operands, where everything is in the cache already -- once per layer and step, not once per tile that reads the block.
// Bound by its launch and one trip to memory (reads 4, writes 6 bytes per value).  Rows past the sequence's last: that row again (their scores are masked).
template <int NTK, int NTV>
__global__ void __launch_bounds__(256) k_attn_parts_kept(WinAttnArgs P, TileArgs A)
{
    constexpr int DK = 32 * NTK, DV = 32 * NTV, KS = 2 * NTK;
    const int tid = threadIdx.x, kvh = blockIdx.x, dk = P.dim, dv = P.vdim;
    int at = blockIdx.y;
    SeqDesc sd;
    if (!block_seq(P, A, at, sd)) return;
    const SeqBlocks sb = seq_blocks(sd.pos0, sd.n, P.window, P.keep_first);
    const int kb0 = (at < sb.kept ? at : sb.first + at - sb.kept) * WT_K, last = sd.pos0 + sd.n - 1;
    const size_t kvd = (size_t)P.kv_heads * dk, vvd = (size_t)P.kv_heads * dv;
    gfloat *kc = (gfloat *)(P.slot_base[sd.slot] + P.k_off + (size_t)kvh * dk), *vc = (gfloat *)(P.slot_base[sd.slot] + P.v_off + (size_t)kvh * dv);
    bf16x8w *dst = (bf16x8w *)P.ws + ((size_t)blockIdx.y * P.kv_heads + kvh) * kBlockPieces<NTK, NTV>;
    const bool vec = dk % 4 == 0 && P.k_off % 4 == 0;      // (arena bases are 256-byte aligned)
    bool odd = false;          // an infinity or NaN among the thread's values
    for (int e = tid; e < WT_K * (DK / 8); e += 256) {
        const int key = e / (DK / 8), c8 = e % (DK / 8), c = 8 * c8;
        gfloat *row = kc + (size_t)min(kb0 + key, last) * kvd;
        float v[8];
        if (vec) {
            const f32x4w lo = *(gf32x4 *)(row + min(c, dk - 4)), hi = *(gf32x4 *)(row + min(c + 4, dk - 4));
#pragma unroll
            for (int x = 0; x < 4; x++) { v[x] = c < dk ? lo[x] : 0.0f; v[4 + x] = c + 4 < dk ? hi[x] : 0.0f; }
        } else {
#pragma unroll
            for (int x = 0; x < 8; x++) { const float f = row[min(c + x, dk - 1)]; v[x] = c + x < dk ? f : 0.0f; }
        }
        odd |= not_finite(v);
        const Parts t = parts_of(v);
#pragma unroll
        for (int pl = 0; pl < 3; pl++) dst[(pl * KS + (c8 >> 1)) * 64 + 32 * (c8 & 1) + key] = t.p[pl];
    }
    dst += 3 * KS * 64;
    for (int e = tid; e < 4 * DV; e += 256) {
        const int d = e % DV, sg = e / DV, k0 = 16 * (sg >> 1) + 4 * (sg & 1);
        float v[8];
#pragma unroll
        for (int x = 0; x < 8; x++) { const float f = vc[(size_t)min(kb0 + k0 + 8 * (x >> 2) + (x & 3), last) * vvd + min(d, dv - 1)]; v[x] = d < dv ? f : 0.0f; }
        odd |= not_finite(v);
        const Parts t = parts_of(v);
#pragma unroll
        for (int pl = 0; pl < 3; pl++) dst[((pl * NTV + (d >> 5)) * 2 + (sg >> 1)) * 64 + 32 * (sg & 1) + (d & 31)] = t.p[pl];
    }
    const int any = __syncthreads_or(odd);
    if (tid < 4) ((uint32_t *)(P.ws + A.marks))[4 * ((size_t)blockIdx.y * P.kv_heads + kvh) + tid] = any ? 1u : 0u;
}

// Workgroups that a block's keys and its values of so many 32s are shared out to: the chain of a step of a few rows (a head's angles in double, its norm, its turn) is as long as the keys a wave has.
// us with the attention, keys of 64 columns in one and in two: 16 heads (4 of keys) turned, 16 rows 18.7 / 15.5, 200 28.4 / 25.4, 2048 87.0 / 86.4; normed alone 18.4 / 16.3, 29.7 / 27.7, 57.4 / 55.4
// (two launches 17.0, 29.0, 59).
__host__ __device__ constexpr int key_shares(int NT) { return NT > 1 ? 2 : 1; }
__host__ __device__ constexpr int value_shares(int NT) { return NT > 2 ? 2 : 1; }

// ... with rows that the step brings: a workgroup per (head of keys, block of the step, share of its keys or values) lays a block's rows out as operands and stores those of the step into the cache on
// their way: a position is in one of the step's blocks, and only there.  Fresh keys go through LDS, all asked for at once.  In front of them, for they take longest, the step's queries, normed and turned
// in place: a wave per row and up to all of its heads, fewer where there are few rows.  Rows past the sequence's last: that row as it came (their scores are masked).
// TURN: something is turned, or normed with a weight.  Without it (keys that are normed at most) the angles' and the turns' code is not there: steps of a few rows walk through the kernel's code once.
// us, the launch that stored the rows + the one that read them back -> this one: 2 heads of keys of 128, 19 rows 3.3 + 5.4 -> 6.6, 100 rows 4.0 + 6.3 -> 6.5; with 8 heads of queries, 64 of 128 columns
// turned, 639 rows 8.7 + 6.4 -> 9.6, 2048 12.4 + 6.9 -> 12.9.  See fresh_pays for where the two launches stay.
template <int NTK, int NTV, bool TURN, bool SIDE>
__global__ void __launch_bounds__(256) k_attn_parts(WinAttnArgs P, TileArgs A, FreshKV F, std::conditional_t<SIDE, SideArgs, int> side)
{
    constexpr int DK = 32 * NTK, DV = 32 * NTV, KS = 2 * NTK, KROW = DK + 4, E = (DK + 63) / 64;
    constexpr int KH = key_shares(NTK), VH = value_shares(NTV), KN = WT_K / KH, KI = (KN * (DK / 8) + 255) / 256, VN = 4 * DV / VH, VI = (VN + 255) / 256;
    int id = blockIdx.x;
    if constexpr (SIDE) {
        if (id < side.first) { ifachunk::linear_chunk(side.c, id % side.chunks, id / side.chunks % side.c.heads, id / side.chunks / side.c.heads); return; }
        id -= side.first;
    }
    extern __shared__ __attribute__((aligned(16))) float part_lds[];          // [KN][KROW], [KN][rot_dims] (queries: [4][rot_dims])
    float *rows = part_lds, *cs = part_lds + KN * KROW;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, dk = P.dim, dv = P.vdim, half = F.rot_dims / 2;
    if constexpr (TURN) {
        if (id < F.q_wgs) {          // queries
            const int w = 4 * id + wave, t = w / F.q_parts;
            if (t < F.q_rows) turn_row<E>(F.q + (size_t)t * P.ldq, P.heads, w % F.q_parts, F.q_parts, dk, F.q_norm_w, F.eps, F.rot_dims, F.freq, cs + wave * F.rot_dims, lane, [&]() {
                    const SeqDesc sd = A.n_few ? few_of(A, t, [](const FewSeq &x) { return x.sd.row0; }).sd : P.seqs[P.row_seq[t]];
                    return sd.pos0 + t - sd.row0;
                });
            return;
        }
        id -= F.q_wgs;
    }
    const int share = id % (KH + VH), kvh = id / (KH + VH) % P.kv_heads, place = id / (KH + VH) / P.kv_heads;
    const bool keys = share < KH;
    int at = place;
    SeqDesc sd;
    if (!block_seq(P, A, at, sd)) return;
    const SeqBlocks sb = seq_blocks(sd.pos0, sd.n, P.window, P.keep_first);
    const int kb0 = (at < sb.kept ? at : sb.first + at - sb.kept) * WT_K, k0b = keys ? KN * share : 0, last = sd.pos0 + sd.n - 1, fresh0 = F.k ? sd.pos0 : 0x7FFFFFFF;          // positions from fresh0 on are the step's
    typedef __attribute__((address_space(1))) float gfloat_w;
    bf16x8w *dst = (bf16x8w *)P.ws + ((size_t)place * P.kv_heads + kvh) * kBlockPieces<NTK, NTV>;
    bool odd = false;          // an infinity or NaN among the thread's values
    if (keys && kb0 + WT_K <= fresh0) {          // cached rows alone: pieces of eight columns as they are read
        gfloat *kc = (gfloat *)(P.slot_base[sd.slot] + P.k_off + (size_t)kvh * dk);
        const bool vec = dk % 4 == 0 && P.k_off % 4 == 0;          // (arena bases are 256-byte aligned)
        f32x4w raw[KI][2];
#pragma unroll
        for (int u = 0; u < KI; u++) {
            const int e = min(tid + 256 * u, KN * (DK / 8) - 1), key = k0b + e / (DK / 8), c = 8 * (e % (DK / 8));
            gfloat *row = kc + (size_t)min(kb0 + key, last) * P.kv_heads * dk;
            if (vec) { raw[u][0] = *(gf32x4 *)(row + min(c, dk - 4)); raw[u][1] = *(gf32x4 *)(row + min(c + 4, dk - 4)); }
            else {
#pragma unroll
                for (int x = 0; x < 8; x++) raw[u][x >> 2][x & 3] = row[min(c + x, dk - 1)];
            }
        }
#pragma unroll
        for (int u = 0; u < KI; u++) {
            const int e = tid + 256 * u, key = k0b + e / (DK / 8), c8 = e % (DK / 8);
            if (e >= KN * (DK / 8)) break;
            float f[8];
#pragma unroll
            for (int x = 0; x < 8; x++) f[x] = 8 * c8 + x < dk ? raw[u][x >> 2][x & 3] : 0.0f;
            odd |= not_finite(f);
            const Parts t = parts_of(f);
#pragma unroll
            for (int pl = 0; pl < 3; pl++) dst[(pl * KS + (c8 >> 1)) * 64 + 32 * (c8 & 1) + key] = t.p[pl];
        }
    } else if (keys) {
        const size_t kvd = (size_t)P.kv_heads * dk;
        gfloat_w *kc = (gfloat_w *)(P.slot_base[sd.slot] + P.k_off + (size_t)kvh * dk);
        constexpr int KW = KN / 4;          // keys a wave, E values of each a lane
        float v[KW][E];
#pragma unroll
        for (int x = 0; x < KW; x++) {
            const int j = min(kb0 + k0b + KW * wave + x, last);
            gfloat *row = (gfloat *)F.k + (size_t)(sd.row0 + j - sd.pos0) * F.ldk + (size_t)kvh * dk;
            if (kb0 < fresh0 && j < fresh0) row = (gfloat *)kc + (size_t)j * kvd;          // (blocks of the step alone do not wait for the slot's place)
#pragma unroll
            for (int e = 0; e < E; e++) v[x][e] = row[min(lane + 64 * e, dk - 1)];
        }
        Turn<E> u;
        if constexpr (TURN) {
            u = turn_of<E>(dk, F.rot_dims, F.norm_w, lane);
            for (int e = lane; e < KW * half; e += 64) {
                const int key = KW * wave + e / half, j = kb0 + k0b + key;
                if (j >= fresh0 && j <= last) angle_of(j, F.freq, e % half, half, cs + key * F.rot_dims);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");          // (the wave's own)
        }
#pragma unroll
        for (int x = 0; x < KW; x++) {
            const int key = KW * wave + x, j = kb0 + k0b + key;
            if (j >= fresh0 && j <= last) {          // (beyond the last: that row as it came, masked)
                if constexpr (TURN) {
                    float cv[E], sv[E];
                    turn_angles<E>(cs + key * F.rot_dims, u, F.rot_dims, lane, cv, sv);
                    turn_held<E>(v[x], u, dk, F.norm != 0, F.eps, F.rot_dims, cv, sv, lane);
                } else if (F.norm) {
                    const float r = norm_held<E>(v[x], dk, F.eps, lane);
#pragma unroll
                    for (int e = 0; e < E; e++) v[x][e] *= r;
                }
            }
#pragma unroll
            for (int e = 0; e < E; e++) {
                const int c = lane + 64 * e;
                if (c < DK) rows[key * KROW + c] = c < dk ? v[x][e] : 0.0f;
                if (c < dk && j >= fresh0 && j <= last) kc[(size_t)j * kvd + c] = v[x][e];
            }
        }
        __syncthreads();
        for (int e = tid; e < KN * (DK / 8); e += 256) {
            const int key = e / (DK / 8), c8 = e % (DK / 8);
            const float *row = rows + key * KROW + 8 * c8;
            float f[8];
            const f32x4w lo = *(const f32x4w *)row, hi = *(const f32x4w *)(row + 4);
#pragma unroll
            for (int x = 0; x < 4; x++) { f[x] = lo[x]; f[4 + x] = hi[x]; }
            odd |= not_finite(f);
            const Parts t = parts_of(f);
#pragma unroll
            for (int pl = 0; pl < 3; pl++) dst[(pl * KS + (c8 >> 1)) * 64 + 32 * (c8 & 1) + k0b + key] = t.p[pl];
        }
    } else {
        const size_t vvd = (size_t)P.kv_heads * dv;
        gfloat_w *vc = (gfloat_w *)(P.slot_base[sd.slot] + P.v_off + (size_t)kvh * dv);
        float v[VI][8];
#pragma unroll
        for (int u = 0; u < VI; u++) {
            const int e = (share - KH) * VN + min(tid + 256 * u, VN - 1), d = e % DV, sg = e / DV, k0 = 16 * (sg >> 1) + 4 * (sg & 1);
#pragma unroll
            for (int x = 0; x < 8; x++) {
                const int j = min(kb0 + k0 + 8 * (x >> 2) + (x & 3), last);
                gfloat *row = (gfloat *)F.v + (size_t)(sd.row0 + j - sd.pos0) * F.ldv + (size_t)kvh * dv;
                if (kb0 < fresh0 && j < fresh0) row = (gfloat *)vc + (size_t)j * vvd;
                v[u][x] = row[min(d, dv - 1)];
            }
        }
        dst += 3 * KS * 64;
#pragma unroll
        for (int u = 0; u < VI; u++) {
            const int e = (share - KH) * VN + tid + 256 * u, d = e % DV, sg = e / DV, k0 = 16 * (sg >> 1) + 4 * (sg & 1);
            if (tid + 256 * u >= VN) break;
#pragma unroll
            for (int x = 0; x < 8; x++) {
                const int j = kb0 + k0 + 8 * (x >> 2) + (x & 3);
                if (j >= fresh0 && j <= last && d < dv) vc[(size_t)j * vvd + d] = v[u][x];
                if (d >= dv) v[u][x] = 0.0f;
            }
            odd |= not_finite(v[u]);
            const Parts t = parts_of(v[u]);
#pragma unroll
            for (int pl = 0; pl < 3; pl++) dst[((pl * NTV + (d >> 5)) * 2 + (sg >> 1)) * 64 + 32 * (sg & 1) + (d & 31)] = t.p[pl];
        }
    }
    const int any = __syncthreads_or(odd);
    if (tid == 0) ((uint32_t *)(P.ws + A.marks))[4 * ((size_t)place * P.kv_heads + kvh) + share] = any ? 1u : 0u;
}

// Key rows of dim <= 32 NTK and value rows of vdim <= 32 NTV floats.  VEC: rows of whole, aligned 16-byte pieces in q and the output.
template <int NTK, int NTV, bool VEC>
__global__ void __launch_bounds__(64 * WT_WAVES, 2) k_attn_tile(WinAttnArgs P, TileArgs A, int hx, int groups, SideArgs side)
{
    constexpr int KS = 2 * NTK, PIECES = kBlockPieces<NTK, NTV>;
    const int bx = blockIdx.x % hx, by = blockIdx.x / hx;
    if (by >= groups) {
        const int id = blockIdx.x - hx * groups, e = id % side.per * (64 * WT_WAVES) + threadIdx.x;
        if (e < side.c.dk * side.c.dv) ifachunk::linear_pass(side.c, e, id / side.per % side.c.heads, id / side.per / side.c.heads);
        return;
    }
    extern __shared__ bf16x8w ops[];                          // two blocks' operands, then a bias table per wave
    float *bias = (float *)(ops + 2 * PIECES) + 64 * (threadIdx.x >> 6);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), i = lane & 31, g = lane >> 5;
    const int h = bx * A.hpw + wave % A.hpw, qsub = wave / A.hpw, kvh = bx * A.hpw / (P.heads / P.kv_heads), dk = P.dim, dv = P.vdim;
    const int qw = 32 * (WT_WAVES / A.hpw);
    ChunkPlace at;
    if (!chunk_of(P, A, qw, by, at)) return;
    const SeqDesc sd = at.sd;
    const int tile = at.tile, tile_g = at.tile_g, chunk = at.chunk, block0 = at.block0;
    const int r0 = sd.row0 + tile * qw, nq = min(qw, sd.n - tile * qw), p0 = sd.pos0 + tile * qw;
    const SeqBlocks sb = seq_blocks(sd.pos0, sd.n, P.window, P.keep_first);
    const TileBlocks tb = tile_blocks(p0, nq, P.window, P.keep_first);
    const int nch = (tb.nb + A.cb - 1) / A.cb, b0 = chunk * A.cb, b1 = min(tb.nb, b0 + A.cb);
    const int nq_w = min(32, max(0, nq - 32 * qsub)), qlo = p0 + 32 * qsub, qhi = qlo + nq_w - 1;          // queries of this wave, their positions
    const bool qin = i < nq_w;
    const float inv_cap = P.softcap > 0.0f ? 1.0f / P.softcap : 0.0f;
    // a block's operands go from memory to LDS directly, asked for behind the scores of the block before (whose operand reads would wait for them):
    // they land under its softmax
    auto fetch = [&](int b) {
        const int block = b < tb.kept ? b : tb.first + b - tb.kept, at = block < sb.kept ? block : sb.kept + block - sb.first;
        const bf16x8w *src = (const bf16x8w *)P.ws + ((size_t)(block0 + at) * P.kv_heads + kvh) * PIECES;
        bf16x8w *dst = ops + (b & 1) * PIECES;
#pragma unroll
        for (int u = 0; u < PIECES / 64; u += WT_WAVES)
            if (u + wave < PIECES / 64)
                __builtin_amdgcn_global_load_lds((wa_glb_t *)(src + (u + wave) * 64 + lane), (wa_lds_t *)(dst + (u + wave) * 64), 16, 0, 0);
    };
    // which of the chunk's blocks (64 at a time) have a mark
    typedef uint32_t u32x4w __attribute__((ext_vector_type(4)));          // (its shares, see k_attn_parts)
    auto mark_of = [&](int b) -> u32x4w {
        const int x = min(b + lane, b1 - 1), block = x < tb.kept ? x : tb.first + x - tb.kept, at = block < sb.kept ? block : sb.kept + block - sb.first;
        return ((const __attribute__((address_space(1))) u32x4w *)(P.ws + A.marks))[(size_t)(block0 + at) * P.kv_heads + kvh];
    };
    auto marked = [&](int b, u32x4w m) -> uint64_t {
        uint32_t any = m[0] | m[1];
        if constexpr (key_shares(NTK) + value_shares(NTV) > 2) any |= m[2];
        if constexpr (key_shares(NTK) + value_shares(NTV) > 3) any |= m[3];
        return __builtin_amdgcn_ballot_w64(any != 0 && b + lane < b1);
    };
    u32x4w first;
    // All of the lane's query at once (queries past the tile's last: that one again, not stored), in front of the first block's operands, behind whose requests it would wait for them: asked
    // for by fours behind these, and every eight values looked at for ones that would round to infinity, a launch took 28.3 us for 601 rows of 8 heads,
    // now 25.3 (2048 rows of 16 heads 122.8, 118.9; of 8 heads, whose tiles take ten blocks each, 60.1, 60.3).
    float qv[KS][8];
    {
        gfloat *qr = (gfloat *)P.q + (size_t)(r0 + min(32 * qsub + i, nq - 1)) * P.ldq + (size_t)h * dk;
        f32x4w raw[KS][2];
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const int c = 16 * ks + 8 * g;
#pragma unroll
            for (int e = 0; e < 2; e++)
                if constexpr (VEC) raw[ks][e] = *(gf32x4 *)(qr + min(c + 4 * e, dk - 4));
                else {
#pragma unroll
                    for (int x = 0; x < 4; x++) raw[ks][e][x] = qr[min(c + 4 * e + x, dk - 1)];
                }
        }
        __builtin_amdgcn_sched_barrier(0);
        first = mark_of(b0);
        __builtin_amdgcn_sched_barrier(0);
        fetch(b0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
#pragma unroll
            for (int x = 0; x < 8; x++) qv[ks][x] = 16 * ks + 8 * g + x < dk ? raw[ks][x >> 2][x & 3] : 0.0f;
    }
    uint64_t odd = marked(b0, first);
    // the lane's query, normed, in three parts
    Parts q[KS];
    {
        float r = 1.0f;
        if (P.norm_q) {
            float sum = 0.0f;
#pragma unroll
            for (int ks = 0; ks < KS; ks++)
#pragma unroll
                for (int x = 0; x < 8; x++) sum = fmaf(qv[ks][x], qv[ks][x], sum);
            r = 1.0f / sqrtf((sum + __shfl_xor(sum, 32, 64)) / (float)dk + P.eps);
        }
        float big = 0.0f;
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
#pragma unroll
            for (int x = 0; x < 8; x++) { qv[ks][x] *= r; big = fmaxf(big, __builtin_fabsf(qv[ks][x])); }
        if (__builtin_amdgcn_ballot_w64(big > 3.38e38f)) {
#pragma unroll
            for (int ks = 0; ks < KS; ks++) q[ks] = parts_of(qv[ks]);
        } else {
#pragma unroll
            for (int ks = 0; ks < KS; ks++) q[ks] = parts_of<false>(qv[ks]);
        }
    }
    f32x16w o[NTV];
    float m = -INFINITY, l = 0.0f;          // of the lane's query
#pragma unroll
    for (int nt = 0; nt < NTV; nt++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[nt][r] = 0.0f;
    for (int b = b0; b < b1; b++) {
        if (((b - b0) & 63) == 0 && b > b0) odd = marked(b, mark_of(b));
        const bool infinite = odd >> ((b - b0) & 63) & 1;
        const int kb0 = (b < tb.kept ? b : tb.first + b - tb.kept) * WT_K;
        const bool active = nq_w > 0 && kb0 <= qhi && (kb0 + WT_K - 1 >= qlo - P.window + 1 || kb0 < P.keep_first);
        // this wave's share of the block has landed, and behind the barrier every wave's, and no wave reads the other buffer any more
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (!active) { if (b + 1 < b1) fetch(b + 1); continue; }
        const bf16x8w *Kp = ops + (b & 1) * PIECES, *Vp = Kp + 3 * KS * 64;
        f32x16w acc;
#pragma unroll
        for (int r = 0; r < 16; r++) acc[r] = 0.0f;
        if (infinite) {
#pragma unroll
            for (int ks = 0; ks < KS; ks++) q[ks] = one_sign(q[ks]);
        }
        {
            Parts k[2];
            auto read_k = [&](int ks) {
#pragma unroll
                for (int pl = 0; pl < 3; pl++) k[ks & 1].p[pl] = Kp[(pl * KS + ks) * 64 + lane];
            };
            read_k(0);
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {          // (the next operands are on their way behind the products of these; no further ahead: registers)
                if (ks + 1 < KS) read_k(ks + 1);
                acc = mfma_rest(k[ks & 1], q[ks], acc);
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k[ks & 1].p[0], q[ks].p[0], acc, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (infinite) {
#pragma unroll
            for (int ks = 0; ks < KS; ks++) q[ks] = rounded(q[ks]);
        }
#pragma unroll
        for (int r = 0; r < 16; r++) acc[r] *= P.scale;
        if (P.softcap > 0.0f) {
            __builtin_amdgcn_sched_barrier(0);          // (or the branch is turned into computing it always)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[r] = P.softcap * tanh_sel(acc[r] * inv_cap);
        }
        if (P.rel) {           // the bias by distance, one distance a lane: entry 31 + i - kk of the block
            const int dist = qlo - kb0 - 31 + lane;
            bias[lane] = dist >= 0 && dist <= qhi - kb0 && (dist < P.window || kb0 < P.keep_first) ? bf2f(P.rel[(size_t)P.bucket_of[dist] * P.heads + h]) : 0.0f;
#pragma unroll
            for (int r = 0; r < 16; r++) acc[r] += bias[31 + i - ((r & 3) + 8 * (r >> 2) + 4 * g)];
        }
        __builtin_amdgcn_sched_barrier(0);
        if (b + 1 < b1) fetch(b + 1);
        __builtin_amdgcn_sched_barrier(0);
        // (blocks that every query of the wave sees whole need no masks)
        if (!(nq_w == 32 && kb0 + WT_K - 1 <= qlo && (qhi - kb0 < P.window || kb0 + WT_K <= P.keep_first))) {
            const int iq = qlo + i;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int j = kb0 + (r & 3) + 8 * (r >> 2) + 4 * g;
                if (!(qin && j <= iq && (iq - j < P.window || j < P.keep_first))) acc[r] = -INFINITY;
            }
        }
        float mloc = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; r++) mloc = fmaxf(mloc, acc[r]);
        mloc = fmaxf(mloc, __shfl_xor(mloc, 32, 64));
        const float m_new = fmaxf(m, mloc), m_use = m_new == -INFINITY ? 0.0f : m_new;      // (-inf only while nothing was visible: sums are 0)
        const float corr = m == -INFINITY ? 1.0f : exp_neg(m - m_new);
        float psum = 0.0f, w[2][8];
#pragma unroll
        for (int r = 0; r < 16; r++) { const float p = exp_neg(acc[r] - m_use); w[r >> 3][r & 7] = p; psum += p; }
        l = l * corr + psum;             // (the keys of this half of the wave; the halves are added at the end)
        m = m_new;
        Parts w0 = parts_of<false>(w[0]), w1 = parts_of<false>(w[1]);          // (at most 1)
        if (infinite) { w0 = one_sign(w0); w1 = one_sign(w1); }
        __builtin_amdgcn_sched_barrier(0);
        Parts v[2];
        auto read_v = [&](int u) {
#pragma unroll
            for (int pl = 0; pl < 3; pl++) v[u & 1].p[pl] = Vp[(pl * NTV * 2 + u) * 64 + lane];
        };
        read_v(0);
#pragma unroll
        for (int u = 0; u < 2 * NTV; u++) {
            if (u + 1 < 2 * NTV) read_v(u + 1);
            f32x16w &on = o[u >> 1];
            if (!(u & 1)) {
#pragma unroll
                for (int r = 0; r < 16; r++) on[r] *= corr;
            }
            on = mfma_rest(v[u & 1], u & 1 ? w1 : w0, on);
            on = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v[u & 1].p[0], (u & 1 ? w1 : w0).p[0], on, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // the lane holds value columns 32 nt + (r & 3) + 8 (r >> 2) + 4 g of its query
    const float ls = l + __shfl_xor(l, 32, 64);
    if (nch > 1) {                       // this chunk's share: [maximum][sum][columns] x 32 queries
        float *dst = P.ws + A.shares + ((((size_t)tile_g * hx + bx) * P.nsplit + chunk) * WT_WAVES + wave) * 32 * (dv + 2) + i;
        if (g == 0) { dst[0] = m; dst[32] = ls; }
#pragma unroll
        for (int nt = 0; nt < NTV; nt++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int c = 32 * nt + (r & 3) + 8 * (r >> 2) + 4 * g;
                if (c < dv) dst[(size_t)(2 + c) * 32] = o[nt][r];
            }
        return;
    }
    if (!qin) return;
    const float snk = sink_of(P, h);
    const float M = fmaxf(m, snk);
    const float f = expf(m - M);
    const float sc = f / (ls * f + (has_sink(P) ? expf(snk - M) : 0.0f));
    if (P.out16) {
        bf16_t *d16 = P.out16 + (size_t)(r0 + 32 * qsub + i) * P.ld16 + (size_t)h * dv;
#pragma unroll
        for (int nt = 0; nt < NTV; nt++)
#pragma unroll
            for (int r = 0; r < 16; r += 4) {
                const int c = 32 * nt + 8 * (r >> 2) + 4 * g;
                bf16x4w v;
#pragma unroll
                for (int x = 0; x < 4; x++) v[x] = (__bf16)(o[nt][r + x] * sc);
                if constexpr (VEC) { if (c < dv) *reinterpret_cast<bf16x4w *>(d16 + c) = v; }
                else {
#pragma unroll
                    for (int x = 0; x < 4; x++) if (c + x < dv) { const __bf16 one = v[x]; d16[c + x] = __builtin_bit_cast(bf16_t, one); }          // (the builtin of a vector element takes the first one)
                }
            }
        return;
    }
    float *dst = P.out + (size_t)(r0 + 32 * qsub + i) * P.ldo + (size_t)h * dv;
#pragma unroll
    for (int nt = 0; nt < NTV; nt++)
#pragma unroll
        for (int r = 0; r < 16; r += 4) {
            const int c = 32 * nt + 8 * (r >> 2) + 4 * g;
            if constexpr (VEC) { if (c < dv) *reinterpret_cast<float4 *>(dst + c) = make_float4(o[nt][r] * sc, o[nt][r + 1] * sc, o[nt][r + 2] * sc, o[nt][r + 3] * sc); }
            else {
#pragma unroll
                for (int x = 0; x < 4; x++) if (c + x < dv) dst[c + x] = o[nt][r + x] * sc;
            }
        }
}

// the chunks' shares of 32 queries of a head and its sink into the output rows: 256 threads for head group bx (of hx), tile tile_g and z (waves of k_attn_tile x 4), 32 value columns a workgroup.
// A chain of requests (the sequence, the maxima, the shares), not their bytes: the shares of four chunks are asked for beside the maxima, which all threads fetch, and four workgroups do what one
// did for all 128 columns, two chunks at a time.  us: Sopulorn 2048 tokens 13.7 -> 11.0, three prompts of 730 in all 10.4 -> 6.9; Gelarax 2048 of width 2048 13.7 -> 12.1, 601 of width 1024
// 11.3 -> 9.0.  (The shares of all 32 possible chunks asked for at once: 208 registers, twice as long.)
constexpr int WC_COLS = 32;
__device__ __forceinline__ void tile_combine(const WinAttnArgs &P, const TileArgs &A, bool few, int hx, int bx, int tile_g, int z)
{
    __shared__ float ms[WT_MAX_CHUNKS][32], ls[WT_MAX_CHUNKS][32], rows[32][WC_COLS + 1];
    const int tid = threadIdx.x, wave = z % WT_WAVES, c0 = z / WT_WAVES * WC_COLS, h = bx * A.hpw + wave % A.hpw, qsub = wave / A.hpw, dv = P.vdim;
    const int qw = 32 * (WT_WAVES / A.hpw), ncol = min(WC_COLS, dv - c0);
    int tile = tile_g;
    SeqDesc sd;
    if (few) { const FewSeq f = few_of(A, tile_g, [](const FewSeq &x) { return x.tile0; }); sd = f.sd; tile -= f.tile0; }
    else {
        const int sq = item_of(A.n_seqs, tile, [&](int x) { return x >= 0 ? (P.seqs[x].n + qw - 1) / qw : 0; });
        if (sq < 0) return;
        sd = P.seqs[sq];
    }
    const int nq = min(qw, sd.n - tile * qw), nq_w = min(32, nq - 32 * qsub);
    const int nch = (tile_blocks(sd.pos0 + tile * qw, nq, P.window, P.keep_first).nb + A.cb - 1) / A.cb;
    if (nch <= 1 || nq_w <= 0) return;
    const int share = WT_WAVES * 32 * (dv + 2), q = tid & 31, nowhere = nch * share * 4;
    // (requests behind the last chunk return zeros, without traffic)
    const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc(P.ws + A.shares + (((size_t)tile_g * hx + bx) * P.nsplit * WT_WAVES + wave) * 32 * (dv + 2), 0,
                                                                         nowhere, 0x00020000);
    auto at = [&](int c, int piece) { return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(src, c < nch ? (c * share + piece * 32 + q) * 4 : nowhere, 0, 0)); };
    // four chunks of shares beside the maxima and sums (thread: query q, chunks j, j + 8 ..), then four at a time
    constexpr int AHEAD = 4;
    float s[AHEAD][WC_COLS / 8];
    auto ask = [&](int from) {
#pragma unroll
        for (int c = 0; c < AHEAD; c++)
#pragma unroll
            for (int k = 0; k < WC_COLS / 8; k++) s[c][k] = at(from + c, 2 + min(c0 + (tid >> 5) + 8 * k, dv - 1));
    };
    for (int c = tid >> 5; c < nch; c += 8) { ms[c][q] = at(c, 0); ls[c][q] = at(c, 1); }
    ask(0);
    const float snk = sink_of(P, h);
    __syncthreads();
    float M = snk, L = 0.0f;
    for (int c = 0; c < nch; c++) M = fmaxf(M, ms[c][q]);
    __syncthreads();
    for (int c = tid >> 5; c < nch; c += 8) { const float m = ms[c][q]; ms[c][q] = m == -INFINITY ? 0.0f : expf(m - M); }
    __syncthreads();
    for (int c = 0; c < nch; c++) L += ls[c][q] * ms[c][q];
    if (has_sink(P)) L += expf(snk - M);
    float o[WC_COLS / 8];
#pragma unroll
    for (int k = 0; k < WC_COLS / 8; k++) o[k] = 0.0f;
    for (int from = 0; from < nch; from += AHEAD) {
        if (from > 0) ask(from);
#pragma unroll
        for (int c = 0; c < AHEAD; c++)
            if (from + c < nch) {
                const float f = ms[from + c][q] / L;
#pragma unroll
                for (int k = 0; k < WC_COLS / 8; k++) o[k] = fmaf(s[c][k], f, o[k]);
            }
    }
#pragma unroll
    for (int k = 0; k < WC_COLS / 8; k++) rows[q][(tid >> 5) + 8 * k] = o[k];
    __syncthreads();
    const int row0 = sd.row0 + tile * qw + 32 * qsub, col = tid % WC_COLS;
    if (col >= ncol) return;
    for (int r = tid / WC_COLS; r < nq_w; r += 256 / WC_COLS) {
        if (P.out16) P.out16[(size_t)(row0 + r) * P.ld16 + (size_t)h * dv + c0 + col] = __builtin_bit_cast(bf16_t, (__bf16)rows[r][col]);
        else P.out[(size_t)(row0 + r) * P.ldo + (size_t)h * dv + c0 + col] = rows[r][col];
    }
}

// (FEW_SEQS: a kernel for either side, the choice in front of a place costs 0.5 us: 16 sequences behind 300 keys 7.0 -> 6.5 us, 12 of 30 rows 7.6 -> 7.0, one of 2000 10.4 -> 10.1)
template <bool FEW_SEQS>
__global__ void __launch_bounds__(256) k_attn_tile_combine(WinAttnArgs P, TileArgs A) { tile_combine(P, A, FEW_SEQS, gridDim.x, blockIdx.x, blockIdx.y, blockIdx.z); }

// ... behind the chunks' outputs of the linear attention beside it
template <int DK, bool VEC>
__global__ void __launch_bounds__(256, ifachunk::chunk_out_waves(0, DK)) k_attn_join_out(WinAttnArgs P, TileArgs A, SideArgs side, int hx)
{
    int id = blockIdx.x;
    if (id < side.first) { ifachunk::chunk_out<0, DK, VEC>(side.c, id % side.chunks, id / side.chunks % side.c.heads, id / side.chunks / side.c.heads); return; }
    id -= side.first;
    tile_combine(P, A, A.n_few != 0, hx, id % hx, id / hx % A.tiles, id / hx / A.tiles);
}

// How a step's tiles are shared out: hpw query heads and qw queries per workgroup, cb key blocks per chunk, up to `chunks` chunks per tile, so that the
// chunks just fill the compute units once (one workgroup each: registers and LDS); below two blocks a chunk the partial results cost more than
// the wait they save.  op_bytes: workspace of the blocks' operands and marks (from mark_at on), bytes: with the chunks' shares (none with one chunk).
struct TilePlan { int hpw, qw, cb, chunks; size_t tiles, groups, blocks, mark_at, op_bytes, bytes; };
TilePlan tile_plan(const ifa_seq_desc *sh, int n_seqs, int heads, int kv_heads, int dim, int vdim, int window, int keep_first, size_t ws_bytes)
{
    TilePlan t;
    const int group = heads / kv_heads, NTK = (dim + 31) / 32, NTV = (vdim + 31) / 32;
    t.hpw = group % 4 == 0 ? 4 : group % 2 == 0 ? 2 : 1;
    t.qw = 32 * (WT_WAVES / t.hpw);
    t.blocks = 0;
    std::vector<int> nbs;
    size_t total = 0, most = 1;
    for (int q = 0; q < n_seqs; q++) {
        t.blocks += (size_t)seq_blocks(sh[q].pos0, sh[q].n, window, keep_first).count;
        for (int at = 0; at < sh[q].n; at += t.qw) {
            nbs.push_back(tile_blocks(sh[q].pos0 + at, std::min(t.qw, sh[q].n - at), window, keep_first).nb);
            total += (size_t)nbs.back(); most = std::max(most, (size_t)nbs.back());
        }
    }
    t.tiles = nbs.size();
    t.mark_at = t.blocks * (size_t)kv_heads * 3 * 64 * 16 * (size_t)(2 * NTK + 2 * NTV);
    t.op_bytes = t.mark_at + t.blocks * (size_t)kv_heads * 16;
    const size_t hx = (size_t)(heads / t.hpw), share = (size_t)WT_WAVES * 32 * ((size_t)vdim + 2) * 4;
    size_t cb = std::max<size_t>({2, total * hx / WT_SLOTS, (most + WT_MAX_CHUNKS - 1) / WT_MAX_CHUNKS});
    auto chunks = [&]() { return (most + cb - 1) / cb; };
    auto groups = [&]() { size_t n = 0; for (int nb : nbs) n += ((size_t)nb + cb - 1) / cb; return n; };
    if (chunks() > 1 && groups() * hx > WT_SLOTS) {          // the smallest that fits, or one chunk a tile (fewer groups the larger it is: found by halves)
        size_t lo = cb, hi = most;
        while (hi - lo > 1) { cb = lo + (hi - lo) / 2; (groups() * hx > WT_SLOTS ? lo : hi) = cb; }
        cb = hi;
    }
    while (chunks() > 1 && t.op_bytes + t.tiles * hx * chunks() * share > ws_bytes) cb = std::max(cb + 1, (most + chunks() - 2) / (chunks() - 1));
    t.cb = (int)cb; t.chunks = (int)chunks(); t.groups = groups();
    t.bytes = t.op_bytes + (t.chunks > 1 ? t.tiles * hx * (size_t)t.chunks * share : 0);
    return t;
}

// Whether a step's rows are stored, and its queries turned, by the launch that lays the operands out (one) or by a launch in front of it (two).  One saves a launch and the rows' way back, and shares a
// row's heads out where rows are few; two has smaller kernels, of which twice as many workgroups are on the chip: where there are more than fit at once (fresh blocks: a workgroup counts whole, a
// cached one for an eighth) they win, unless the queries are so many that their own launch takes long.  us one / two: 8 heads, 8 of keys, of 128: 16 rows 19.5 / 24.4, 200 33 / 38, 2048 93 / 94,
// 64 prompts of 20 54.6 / 49.8, 32 of 100 77 / 70; 2 heads of keys, a token each of 16 users behind 300 37.7 / 43.2, of 64 behind 500 81.0 / 79.0; 64 heads, 8 of keys: 16 rows 20.7 / 41.4, 32 of 100
// 193 / 243; 32 heads, as many of keys, of 64: 30 rows behind 4000 81 / 98.
constexpr int TURN_WAVES = 1024;          // waves that turn queries, as many as stand on the chip at once: a row's heads are shared out to get there
bool fresh_pays(const ifa_seq_desc *sh, int n_seqs, size_t rows, size_t blocks, int wgs, bool own, int turned_heads)
{
    size_t fresh = 0;
    if (own) for (int q = 0; q < n_seqs; q++) fresh += (size_t)((sh[q].pos0 + sh[q].n - 1) / WT_K - sh[q].pos0 / WT_K + 1);
    return fresh * wgs + (blocks - fresh) * wgs / 8 <= 1024 + rows * turned_heads / 24;
}

// (the rows of a step's sequences follow each other)
void few_seqs(TileArgs &A, const ifa_seq_desc *sh, int n_seqs, const TilePlan &t, int window, int keep_first)
{
    A.n_few = 0;
    memset(A.few, 0, sizeof(A.few));
    if (n_seqs > FEW) return;
    int tiles = 0, blocks = 0, row = sh[0].row0;
    for (int q = 0; q < n_seqs; q++) {
        if (sh[q].row0 != row || sh[q].n <= 0) return;
        A.few[q].sd = {sh[q].row0, sh[q].n, sh[q].pos0, sh[q].slot};
        A.few[q].tile0 = tiles; A.few[q].block0 = blocks;
        tiles += (sh[q].n + t.qw - 1) / t.qw; blocks += seq_blocks(sh[q].pos0, sh[q].n, window, keep_first).count; row += sh[q].n;
    }
    int chunks = 0;
    for (int q = n_seqs - 1; q >= 0; q--) {
        A.few[q].chunk0 = chunks;
        for (int at = 0; at < sh[q].n; at += t.qw) chunks += (tile_blocks(sh[q].pos0 + at, std::min(t.qw, sh[q].n - at), window, keep_first).nb + t.cb - 1) / t.cb;
    }
    A.n_few = n_seqs;
}

// ---- rotated queries and keys.  One workgroup per row, a wave per head at a time: RMS norm over the head's dim values with a weight
// (norm_w bf16 [dim], null: none), then the first rot_dims dimensions turn in pairs (i, i + rot_dims / 2) -- pairing 1: (2i, 2i + 1) -- by the angle pos * freq[i]
// (formed in double: at position 1000 one fp32 ulp of the angle is already 1e-4); the rest pass unchanged.  Query heads are rewritten in
// place; key heads go into the K rows of the cache, the value heads (as projected) into its V rows.  k null: the row brings no keys
// and values of its own (the layer reads another layer's cache rows).
// VX: the values are treated too (v_norm: each value head divided by its root mean square; v_freq: the head then turns by the row's position over
// all vdim dimensions, pair (m, m + vdim / 2) by pos * v_freq[m]) instead of entering the V rows as projected.
template <int RS_CPL, bool VX>
__global__ void __launch_bounds__(256) k_qk_rope_store(float *__restrict__ q, size_t ldq, int heads, const float *__restrict__ k, size_t ldk,
                                                       const float *__restrict__ v, size_t ldv, int kv_heads, int dim, int vdim,
                                                       const bf16_t *__restrict__ q_norm_w, const bf16_t *__restrict__ k_norm_w, float eps, int rot_dims,
                                                       const double *__restrict__ freq, const SeqDesc *__restrict__ seqs, const int *__restrict__ row_seq,
                                                       float *const *__restrict__ slot_base, size_t k_off, size_t v_off, int v_norm,
                                                       const double *__restrict__ v_freq, int pairing, int v_heads)
{
    extern __shared__ float cs[];          // [rot_dims / 2] cos, [rot_dims / 2] sin; VX: [vdim / 2] cos, [vdim / 2] sin behind them
    const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = blockDim.x >> 6;
    const SeqDesc sd = seqs[row_seq[t]];
    const int pos = sd.pos0 + t - sd.row0, half = rot_dims / 2;
    // VX: two workgroups per row, blockIdx.y 0 for the queries and keys, 1 for the values (each forms only the angles it needs)
    const bool do_qk = !VX || blockIdx.y == 0, do_v = VX && blockIdx.y == 1;
    if (do_qk)
    for (int i = tid; i < half; i += blockDim.x) angle_of(pos, freq, i, half, cs);
    float *vcs = cs + 2 * half;
    const int vhalf = vdim / 2;
    if (do_v && k && v_freq) {
        for (int i = tid; i < vhalf; i += blockDim.x) {
            const double a = (double)pos * v_freq[i];
            double sn, cn; sincos(a, &sn, &cn);
            vcs[i] = (float)cn; vcs[vhalf + i] = (float)sn;
        }
    }
    __syncthreads();
    const int n_items = do_qk ? heads + (k ? kv_heads : 0) : 0;
    // (steps of a few rows: a row's heads are shared out over gridDim.z workgroups)
    const int w0 = blockIdx.z * nw + wave, wn = nw * gridDim.z;
    for (int it = w0; it < n_items; it += wn) {
        const bool is_q = it < heads;
        const int hd = is_q ? it : it - heads;
        const float *src = is_q ? q + (size_t)t * ldq + (size_t)hd * dim : k + (size_t)t * ldk + (size_t)hd * dim;
        float *dst = is_q ? q + (size_t)t * ldq + (size_t)hd * dim : slot_base[sd.slot] + k_off + ((size_t)pos * kv_heads + hd) * dim;
        const bf16_t *nw_ = is_q ? q_norm_w : k_norm_w;
        turn_head<RS_CPL>(src, dst, dim, nw_ != nullptr, nw_, eps, rot_dims, pairing, cs, lane);
    }
    if (VX) {
        if (!k || !do_v) return;
        // a wave per value head: weightless RMS norm, then the turn by the position (a lane reads both members of a pair from the input row)
        for (int hd = w0; hd < kv_heads; hd += wn) {
            const float *src = v + (size_t)t * ldv + (size_t)hd * vdim;
            float *dst = slot_base[sd.slot] + v_off + ((size_t)pos * kv_heads + hd) * vdim;
            float r = 1.0f;
            if (v_norm) {
                float s = 0.0f;
                for (int c = lane; c < vdim; c += 64) s = fmaf(src[c], src[c], s);
                r = 1.0f / sqrtf(wave_sum(s) / (float)vdim + eps);
            }
            for (int c = lane; c < vdim; c += 64) {
                float out = src[c] * r;
                if (v_freq && c < 2 * vhalf) {
                    const int fi = c < vhalf ? c : c - vhalf;
                    const float oth = src[c < vhalf ? c + vhalf : c - vhalf] * r;
                    out = c < vhalf ? out * vcs[fi] - oth * vcs[vhalf + fi] : out * vcs[fi] + oth * vcs[vhalf + fi];
                }
                dst[c] = out;
            }
        }
        return;
    }
    if (k) {
        float *vd = slot_base[sd.slot] + v_off + (size_t)pos * v_heads * vdim;
        const float *vs = v + (size_t)t * ldv;
        for (int c = blockIdx.z * blockDim.x + tid; c < v_heads * vdim; c += blockDim.x * gridDim.z) vd[c] = vs[c];
    }
}

// heads of a row turned in place by sign * position over their first rot_dims dimensions, pairs (m, m + rot_dims / 2); a workgroup per row
__global__ void __launch_bounds__(256) k_rotate_heads(float *__restrict__ x, size_t ldx, int heads, int dim, int rot_dims, const double *__restrict__ freq, float sign,
                                                      const SeqDesc *__restrict__ seqs, const int *__restrict__ row_seq)
{
    extern __shared__ float cs[];          // [rot_dims / 2] cos, [rot_dims / 2] sin
    const int t = blockIdx.x, tid = threadIdx.x, half = rot_dims / 2;
    const SeqDesc sd = seqs[row_seq[t]];
    const int pos = sd.pos0 + t - sd.row0;
    for (int i = tid; i < half; i += blockDim.x) {
        const double a = (double)sign * (double)pos * freq[i];
        double sn, cn; sincos(a, &sn, &cn);          // (one argument reduction for both)
        cs[i] = (float)cn; cs[half + i] = (float)sn;
    }
    __syncthreads();
    float *xr = x + (size_t)t * ldx;
    for (int e = tid; e < heads * half; e += blockDim.x) {      // a thread owns a pair: both members read before either is written
        const int hd = e / half, i = e % half;
        float *p = xr + (size_t)hd * dim;
        const float u = p[i], w = p[i + half];
        p[i] = u * cs[i] - w * cs[half + i];
        p[i + half] = w * cs[i] + u * cs[half + i];
    }
}

} // namespace

extern "C" {

int ifa_kv_store_f32(const void *k_f32, size_t ldk, const void *v_f32, size_t ldv, int kv_heads, int dim, int norm_k, float eps, const void *seqs_dev,
                     const int *row_seq_dev, size_t rows, void *const *slot_base_dev, size_t k_off, size_t v_off, ifa_stream stream)
{
    IFA_REQUIRE(k_f32 && v_f32 && seqs_dev && row_seq_dev && slot_base_dev, "ifa_kv_store_f32: null pointer");
    IFA_REQUIRE(kv_heads > 0 && dim > 0 && rows > 0 && ldk >= (size_t)kv_heads * dim && ldv >= (size_t)kv_heads * dim, "ifa_kv_store_f32: bad shape");
    hipLaunchKernelGGL(k_kv_store_f32, dim3((unsigned)rows), dim3(256), 0, ifa_s(stream), (const float *)k_f32, ldk, (const float *)v_f32, ldv, kv_heads, dim,
                       norm_k, eps, (const SeqDesc *)seqs_dev, row_seq_dev, (float *const *)slot_base_dev, k_off, v_off);
    IFA_LAUNCH_CHECK();
    return IFA_OK;
}

static int attention_launch(const char *who, const void *q_f32, size_t ldq, int heads, int kv_heads, int dim, int vdim, int norm_q, float eps, float scale, float softcap,
                            int window, int keep_first, const void *rel_bf16, const int *bucket_of_dev, int n_buckets, const void *sink_bf16, int sink_fixed,
                            float sink_score, const void *seqs_dev, const int *row_seq_dev, size_t rows, void *const *slot_base_dev, size_t k_off, size_t v_off,
                            void *out_f32, size_t ldo, const void *seqs_host, int n_seqs, int tile_min_rows, int max_keys, void *ws_f32, size_t ws_bytes,
                            ifa_stream stream, void *out_bf16 = nullptr, size_t ld16 = 0, bool *left16 = nullptr, const IfaFreshKV *fresh = nullptr, const IfaLinearSide *side = nullptr,
                            bool *side_done = nullptr)
{
    if (left16) *left16 = false;
    if (side_done) *side_done = false;
    IFA_REQUIRE(!out_bf16 || (left16 && ld16 >= (size_t)heads * vdim), "%s: bad bfloat16 output", who);
    IFA_REQUIRE(q_f32 && seqs_dev && row_seq_dev && slot_base_dev && out_f32, "%s: null pointer", who);
    IFA_REQUIRE(heads > 0 && kv_heads > 0 && heads % kv_heads == 0 && dim > 0 && vdim > 0 && rows > 0 && window >= 1 && keep_first >= 0, "%s: bad shape", who);
    IFA_REQUIRE(dim <= 64 * WA_DPL_MAX && vdim <= 64 * WA_DPL_MAX, "%s: head size %d / %d above %d", who, dim, vdim, 64 * WA_DPL_MAX);
    IFA_REQUIRE(ldq >= (size_t)heads * dim && ldo >= (size_t)heads * vdim, "%s: row strides %zu / %zu too small", who, ldq, ldo);
    IFA_REQUIRE(!rel_bf16 || (bucket_of_dev && n_buckets > 0), "%s: a bias table needs its bucket map", who);
    WinAttnArgs P;
    P.q = (const float *)q_f32; P.ldq = ldq; P.heads = heads; P.kv_heads = kv_heads; P.dim = dim; P.vdim = vdim; P.norm_q = norm_q; P.eps = eps; P.scale = scale;
    P.softcap = softcap; P.window = window; P.keep_first = keep_first; P.rel = (const bf16_t *)rel_bf16; P.bucket_of = bucket_of_dev; P.n_buckets = n_buckets;
    P.sink = (const bf16_t *)sink_bf16; P.sink_fixed = sink_fixed; P.sink_score = sink_score;
    P.seqs = (const SeqDesc *)seqs_dev; P.row_seq = row_seq_dev; P.slot_base = (float *const *)slot_base_dev;
    P.k_off = k_off; P.v_off = v_off; P.out = (float *)out_f32; P.ldo = ldo; P.out16 = nullptr; P.ld16 = 0; P.ws = nullptr; P.nsplit = 1;
    auto store_fresh = [&]() -> int {
        return fresh->turn_q ? ifa_qk_rope_store_f32((void *)q_f32, ldq, heads, fresh->k, fresh->ldk, fresh->v, fresh->ldv, kv_heads, dim, vdim, fresh->q_norm_w, fresh->norm_w, fresh->eps,
                                                     fresh->rot_dims, fresh->freq, seqs_dev, row_seq_dev, rows, slot_base_dev, k_off, v_off, stream)
                             : ifa_kv_store_f32(fresh->k, fresh->ldk, fresh->v, fresh->ldv, kv_heads, dim, fresh->norm, fresh->eps, seqs_dev, row_seq_dev, rows, slot_base_dev, k_off, v_off, stream);
    };
    // prompts: the tiled matrix-core kernels (heads of up to 128 dimensions, zero-padded to whole 32s); single tokens and other sizes: a workgroup per row.
    // With a workspace the bfloat16 form, from the smallest tiled step on (8 heads of 128: 16 rows 15.5 against 17.8 us, 256 rows 33 against 71, 64 rows behind 3000 keys 49 against 719).
    // Not for one row: its grids follow from the HOST's positions, and a step of one row is captured once and replayed while the position on the device goes on.
    if (rows > 1 && rows >= (size_t)tile_min_rows && n_seqs > 0 && dim <= 128 && vdim <= 128 && ws_f32 && (uintptr_t)ws_f32 % 16 == 0) {
        const TilePlan t = tile_plan((const ifa_seq_desc *)seqs_host, n_seqs, heads, kv_heads, dim, vdim, window, keep_first, ws_bytes);
        if (t.bytes <= ws_bytes && t.tiles < 65536 && t.groups < 65536 && t.blocks < 65536) {          // (a grid's limits; beyond them the tiles below, as without a workspace)
            const int NTK = (dim + 31) / 32, NTV = (vdim + 31) / 32;
            TileArgs A;
            A.n_seqs = n_seqs; A.hpw = t.hpw; A.cb = t.cb; A.tiles = (int)t.tiles; A.marks = t.mark_at / 4; A.shares = t.op_bytes / 4;
            few_seqs(A, (const ifa_seq_desc *)seqs_host, n_seqs, t, window, keep_first);
            P.ws = (float *)ws_f32; P.nsplit = t.chunks;
            if (out_bf16) { P.out16 = (bf16_t *)out_bf16; P.ld16 = ld16; *left16 = true; }
            const bool vec = dim % 4 == 0 && vdim % 4 == 0 && ldq % 4 == 0 && ldo % 4 == 0 && (uintptr_t)q_f32 % 16 == 0 && (uintptr_t)out_f32 % 16 == 0
                             && (!out_bf16 || (ld16 % 4 == 0 && (uintptr_t)out_bf16 % 8 == 0));
            const int hx = heads / t.hpw;
            if (n_seqs > SIDE_SEQS) side = nullptr;          // (*side_done stays false)
            if (fresh && !side && !fresh_pays((const ifa_seq_desc *)seqs_host, n_seqs, rows, t.blocks, kv_heads * (key_shares(NTK) + value_shares(NTV)), fresh->k != nullptr,
                                              fresh->turn_q ? heads : 0)) {
                if (const int rc = store_fresh()) return rc;
                fresh = nullptr;
            }
            FreshKV F;
            memset(&F, 0, sizeof(F));
            if (fresh) {
                F.k = fresh->k; F.ldk = fresh->ldk; F.v = fresh->v; F.ldv = fresh->ldv; F.norm = fresh->norm; F.norm_w = fresh->norm_w; F.eps = fresh->eps; F.rot_dims = fresh->rot_dims;
                F.freq = fresh->freq; F.q_rows = fresh->turn_q ? (int)rows : 0; F.q_norm_w = fresh->q_norm_w; F.q = (float *)q_f32;
            }
            F.q_parts = (int)std::max<size_t>(1, std::min<size_t>(TURN_WAVES / rows, ((size_t)heads + HB - 1) / HB));
            F.q_wgs = (int)(((size_t)F.q_rows * F.q_parts + 3) / 4);
            SideArgs S;
            memset(&S, 0, sizeof(S));
            if (side) {
                size_t chunks = 0;
                const int rc = ifa_chunk_args(&S.c, &chunks, 0, side->q, side->ldq, side->k, side->ldk, side->v, side->ldv, side->heads, side->heads, side->dk, side->dv, side->decay, nullptr,
                                              nullptr, seqs_dev, seqs_host, n_seqs, slot_base_dev, side->state_off, side->ws, side->ws_bytes, side->out, side->ldo);
                if (rc) return rc;
                S.chunks = (int)chunks; S.zc = (side->dv + 63) / 64; S.first = S.chunks * side->heads * S.zc; S.per = (side->dk * side->dv + 64 * WT_WAVES - 1) / (64 * WT_WAVES);
                const size_t pass = (size_t)S.per * side->heads * n_seqs;
                S.pass = pass <= SIDE_PASS ? (int)pass : 0;
            }
            const bool turn = F.rot_dims > 0 || F.q_rows > 0 || F.norm_w, kept = !F.k && !F.q_rows && !side;
            IFA_REQUIRE(!side || !turn, "%s: the linear attention goes beside keys that are not turned", who);
            const unsigned part_wgs = (unsigned)(S.first + (size_t)(key_shares(NTK) + value_shares(NTV)) * kv_heads * t.blocks + F.q_wgs), tile_wgs = (unsigned)(hx * t.groups + S.pass);
#define IFA_WT(K, V) { const size_t smem_p = ((size_t)(WT_K / key_shares(K)) * (32 * K + 4) + (size_t)std::max(WT_K / key_shares(K), 4) * F.rot_dims) * 4; \
                       const size_t smem_t = (size_t)2 * kBlockPieces<K, V> * 16 + WT_WAVES * 64 * 4; \
                       const void *fn = vec ? (const void *)k_attn_tile<K, V, true> : (const void *)k_attn_tile<K, V, false>; \
                       IFA_HIP_CHECK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem_t)); \
                       if (kept) hipLaunchKernelGGL((k_attn_parts_kept<K, V>), dim3((unsigned)kv_heads, (unsigned)t.blocks), dim3(256), 0, ifa_s(stream), P, A); \
                       else if (side) hipLaunchKernelGGL((k_attn_parts<K, V, false, true>), dim3(part_wgs), dim3(256), smem_p, ifa_s(stream), P, A, F, S); \
                       else if (turn) hipLaunchKernelGGL((k_attn_parts<K, V, true, false>), dim3(part_wgs), dim3(256), smem_p, ifa_s(stream), P, A, F, 0); \
                       else hipLaunchKernelGGL((k_attn_parts<K, V, false, false>), dim3(part_wgs), dim3(256), smem_p, ifa_s(stream), P, A, F, 0); \
                       if (side && !S.pass) ifa_linear_pass(S.c, stream); \
                       if (vec) hipLaunchKernelGGL((k_attn_tile<K, V, true>), dim3(tile_wgs), dim3(64 * WT_WAVES), smem_t, ifa_s(stream), P, A, hx, (int)t.groups, S); \
                       else hipLaunchKernelGGL((k_attn_tile<K, V, false>), dim3(tile_wgs), dim3(64 * WT_WAVES), smem_t, ifa_s(stream), P, A, hx, (int)t.groups, S); }
#define IFA_WTV(K) { if (NTV == 1) IFA_WT(K, 1) else if (NTV == 2) IFA_WT(K, 2) else if (NTV == 3) IFA_WT(K, 3) else IFA_WT(K, 4) }
            if (NTK == 1) IFA_WTV(1) else if (NTK == 2) IFA_WTV(2) else if (NTK == 3) IFA_WTV(3) else IFA_WTV(4)
#undef IFA_WTV
#undef IFA_WT
            const unsigned joins = t.chunks > 1 ? (unsigned)(WT_WAVES * ((vdim + WC_COLS - 1) / WC_COLS)) : 0u;
            if (side) {
                const dim3 grid((unsigned)S.first + (unsigned)(hx * t.tiles) * joins);
                const bool v16 = side->ldv % 4 == 0 && ((uintptr_t)side->v & 15) == 0;
#define IFA_JO(D) { if (v16) hipLaunchKernelGGL((k_attn_join_out<D, true>), grid, dim3(256), 0, ifa_s(stream), P, A, S, hx); \
                    else hipLaunchKernelGGL((k_attn_join_out<D, false>), grid, dim3(256), 0, ifa_s(stream), P, A, S, hx); }
                if (side->dk == 64) IFA_JO(64) else IFA_JO(128)
#undef IFA_JO
                *side_done = true;
            } else if (joins && A.n_few) hipLaunchKernelGGL(k_attn_tile_combine<true>, dim3((unsigned)hx, (unsigned)t.tiles, joins), dim3(256), 0, ifa_s(stream), P, A);
            else if (joins) hipLaunchKernelGGL(k_attn_tile_combine<false>, dim3((unsigned)hx, (unsigned)t.tiles, joins), dim3(256), 0, ifa_s(stream), P, A);
            IFA_LAUNCH_CHECK();
            return IFA_OK;
        }
    }
    if (fresh) { if (const int rc = store_fresh()) return rc; }
    // prompts without a workspace (or with one that the operands do not fit, or of more key blocks than a grid has)
    if (rows >= (size_t)tile_min_rows && n_seqs > 0 && dim <= 128 && vdim <= 128) {
        const ifa_seq_desc *sh = (const ifa_seq_desc *)seqs_host;
        size_t tiles = 0;
        for (int q = 0; q < n_seqs; q++) tiles += ((size_t)sh[q].n + WT_Q - 1) / WT_Q;
        const int NTK = (dim + 31) / 32, NTV = (vdim + 31) / 32;
        const size_t smem_t = ((size_t)(WT_Q + WT_K) * (32 * NTK + 1) + (size_t)WT_K * (32 * NTV + 1)) * 4;
        const int vec = (dim % 4 == 0 && vdim % 4 == 0 && k_off % 4 == 0 && v_off % 4 == 0) ? 1 : 0;      // (arena bases are 256-byte aligned)
        IFA_REQUIRE(tiles < 65536, "%s: %zu query tiles in one step", who, tiles);
        const dim3 grid((unsigned)heads, (unsigned)tiles);
#define IFA_WT(K, V) { IFA_HIP_CHECK(hipFuncSetAttribute((const void *)k_attn_window_tile<K, V>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem_t)); \
                       hipLaunchKernelGGL((k_attn_window_tile<K, V>), grid, dim3(256), smem_t, ifa_s(stream), P, n_seqs, vec); }
#define IFA_WTV(K) { if (NTV == 1) IFA_WT(K, 1) else if (NTV == 2) IFA_WT(K, 2) else if (NTV == 3) IFA_WT(K, 3) else IFA_WT(K, 4) }
        if (NTK == 1) IFA_WTV(1) else if (NTK == 2) IFA_WTV(2) else if (NTK == 3) IFA_WTV(3) else IFA_WTV(4)
#undef IFA_WTV
#undef IFA_WT
        IFA_LAUNCH_CHECK();
        return IFA_OK;
    }
    const size_t smem = ((size_t)dim + 8 + 4 * (size_t)vdim) * 4;
    // few rows: a (row, head)'s keys are shared out to several workgroups (one workgroup pulls its keys through ONE compute unit)
    int nsplit = 1;
    if (ws_f32 && rows * (size_t)heads <= 512) {
        size_t keys = (size_t)window + (size_t)keep_first;
        if (max_keys > 0) keys = std::min(keys, (size_t)max_keys);
        nsplit = (int)std::min<size_t>(WA_MAX_SPLITS, (keys + 63) / 64);
        while (nsplit > 1 && rows * (size_t)heads * nsplit * ((size_t)vdim + 2) * 4 > ws_bytes) nsplit--;
    }
    P.ws = (float *)ws_f32; P.nsplit = nsplit;
    const dim3 grid_rows((unsigned)rows, (unsigned)heads, (unsigned)nsplit);
    if (vdim <= 64) hipLaunchKernelGGL(k_attn_window<1>, grid_rows, dim3(256), smem, ifa_s(stream), P);
    else if (vdim <= 128) hipLaunchKernelGGL(k_attn_window<2>, grid_rows, dim3(256), smem, ifa_s(stream), P);
    else if (vdim <= 256) hipLaunchKernelGGL(k_attn_window<4>, grid_rows, dim3(256), smem, ifa_s(stream), P);
    else if (vdim <= 640) hipLaunchKernelGGL(k_attn_window<10>, grid_rows, dim3(256), smem, ifa_s(stream), P);
    else hipLaunchKernelGGL(k_attn_window<WA_DPL_MAX>, grid_rows, dim3(256), smem, ifa_s(stream), P);
    if (nsplit > 1) hipLaunchKernelGGL(k_attn_window_combine, dim3((unsigned)rows, (unsigned)heads), dim3(vdim <= 64 ? 64 : 128), 0, ifa_s(stream), P);
    IFA_LAUNCH_CHECK();
    return IFA_OK;
}

size_t ifa_attention_tile_workspace_bytes(const void *seqs_host, int n_seqs, int heads, int kv_heads, int dim, int vdim, int window, int keep_first)
{
    if (!seqs_host || n_seqs <= 0 || heads <= 0 || kv_heads <= 0 || heads % kv_heads || dim <= 0 || vdim <= 0 || dim > 128 || vdim > 128) return 0;
    return tile_plan((const ifa_seq_desc *)seqs_host, n_seqs, heads, kv_heads, dim, vdim, window > 0 ? window : (1 << 30), keep_first, (size_t)-1).bytes;
}

int ifa_attention_window_f32(const void *q_f32, size_t ldq, int heads, int kv_heads, int dim, int norm_q, float eps, float scale, float softcap,
                             int window, int keep_first, const void *rel_bf16, const int *bucket_of_dev, int n_buckets, const void *sink_bf16,
                             const void *seqs_dev, const int *row_seq_dev, size_t rows, void *const *slot_base_dev, size_t k_off, size_t v_off,
                             void *out_f32, size_t ldo, const void *seqs_host, int n_seqs, int tile_min_rows, void *ws_f32, size_t ws_bytes, ifa_stream stream)
{
    // (the tiled kernel of this entry keeps to whole 32s: other head sizes take a workgroup per row, as before)
    const int tile_ok = dim % 32 == 0 && k_off % 4 == 0 && v_off % 4 == 0;
    return attention_launch("ifa_attention_window_f32", q_f32, ldq, heads, kv_heads, dim, dim, norm_q, eps, scale, softcap, window, keep_first, rel_bf16, bucket_of_dev,
                            n_buckets, sink_bf16, 0, 0.0f, seqs_dev, row_seq_dev, rows, slot_base_dev, k_off, v_off, out_f32, ldo, seqs_host, tile_ok ? n_seqs : 0,
                            tile_min_rows, 0, ws_f32, ws_bytes, stream);
}

int ifa_attention_kv_f32(const void *q_f32, size_t ldq, int heads, int kv_heads, int dim, int vdim, float scale, int window, int keep_first, int sink,
                         float sink_score, const void *seqs_dev, const int *row_seq_dev, size_t rows, void *const *slot_base_dev, size_t k_off, size_t v_off,
                         void *out_f32, size_t ldo, const void *seqs_host, int n_seqs, int tile_min_rows, int max_keys, void *ws_f32, size_t ws_bytes,
                         ifa_stream stream)
{
    const int win = window > 0 ? window : (1 << 30);
    return attention_launch("ifa_attention_kv_f32", q_f32, ldq, heads, kv_heads, dim, vdim, 0, 0.0f, scale, 0.0f, win, keep_first, nullptr, nullptr, 0, nullptr,
                            sink ? 1 : 0, sink_score, seqs_dev, row_seq_dev, rows, slot_base_dev, k_off, v_off, out_f32, ldo, seqs_host, n_seqs, tile_min_rows,
                            max_keys, ws_f32, ws_bytes, stream);
}

// workgroups that share a row's heads: one head per wave for steps of a few rows
static unsigned rope_parts(size_t rows, int heads, int k_heads) { return rows <= 8 ? (unsigned)std::min(16, (heads + k_heads + 3) / 4) : 1u; }

int ifa_qk_rope_store_pairs_f32(int pairing, void *q_f32, size_t ldq, int heads, const void *k_f32, size_t ldk, const void *v_f32, size_t ldv, int k_heads, int v_heads,
                                int dim, int vdim, const void *q_norm_w_bf16, const void *k_norm_w_bf16, float eps, int rot_dims, const double *freq_f64_dev,
                                const void *seqs_dev, const int *row_seq_dev, size_t rows, void *const *slot_base_dev, size_t k_off, size_t v_off, ifa_stream stream)
{
    IFA_REQUIRE(q_f32 && seqs_dev && row_seq_dev && slot_base_dev && (!k_f32 || v_f32), "ifa_qk_rope_store_f32: null pointer");
    IFA_REQUIRE(heads > 0 && k_heads > 0 && v_heads > 0 && dim > 0 && dim <= 1024 && vdim > 0 && rows > 0 && rot_dims >= 0 && rot_dims <= dim && rot_dims % 2 == 0
                && (rot_dims == 0 || freq_f64_dev) && (pairing == 0 || pairing == 1), "ifa_qk_rope_store_f32: bad shape (head size %d, %d rotated)", dim, rot_dims);
    IFA_REQUIRE(ldq >= (size_t)heads * dim && (!k_f32 || (ldk >= (size_t)k_heads * dim && ldv >= (size_t)v_heads * vdim)), "ifa_qk_rope_store_f32: row strides too small");
#define IFA_RS(N) hipLaunchKernelGGL((k_qk_rope_store<N, false>), dim3((unsigned)rows, 1u, rope_parts(rows, heads, k_f32 ? k_heads : 0)), dim3(256), (size_t)std::max(rot_dims, 2) * 4, ifa_s(stream), (float *)q_f32, ldq, heads, \
                                     (const float *)k_f32, ldk, (const float *)v_f32, ldv, k_heads, dim, vdim, (const bf16_t *)q_norm_w_bf16, (const bf16_t *)k_norm_w_bf16, eps, \
                                     rot_dims, freq_f64_dev, (const SeqDesc *)seqs_dev, row_seq_dev, (float *const *)slot_base_dev, k_off, v_off, 0, (const double *)nullptr, \
                                     pairing, v_heads)
    if (dim <= 128) IFA_RS(2); else if (dim <= 256) IFA_RS(4); else IFA_RS(16);
#undef IFA_RS
    IFA_LAUNCH_CHECK();
    return IFA_OK;
}

int ifa_qk_rope_store_f32(void *q_f32, size_t ldq, int heads, const void *k_f32, size_t ldk, const void *v_f32, size_t ldv, int kv_heads, int dim, int vdim,
                          const void *q_norm_w_bf16, const void *k_norm_w_bf16, float eps, int rot_dims, const double *freq_f64_dev, const void *seqs_dev,
                          const int *row_seq_dev, size_t rows, void *const *slot_base_dev, size_t k_off, size_t v_off, ifa_stream stream)
{
    return ifa_qk_rope_store_pairs_f32(0, q_f32, ldq, heads, k_f32, ldk, v_f32, ldv, kv_heads, kv_heads, dim, vdim, q_norm_w_bf16, k_norm_w_bf16, eps, rot_dims, freq_f64_dev,
                                       seqs_dev, row_seq_dev, rows, slot_base_dev, k_off, v_off, stream);
}

int ifa_qkv_rope_store_f32(void *q_f32, size_t ldq, int heads, const void *k_f32, size_t ldk, const void *v_f32, size_t ldv, int kv_heads, int dim, int vdim,
                           const void *q_norm_w_bf16, const void *k_norm_w_bf16, float eps, int rot_dims, const double *freq_f64_dev, int v_norm,
                           const double *v_freq_f64_dev, const void *seqs_dev, const int *row_seq_dev, size_t rows, void *const *slot_base_dev, size_t k_off,
                           size_t v_off, ifa_stream stream)
{
    IFA_REQUIRE(q_f32 && seqs_dev && row_seq_dev && slot_base_dev && (!k_f32 || v_f32), "ifa_qkv_rope_store_f32: null pointer");
    IFA_REQUIRE(heads > 0 && kv_heads > 0 && dim > 0 && dim <= 1024 && vdim > 0 && vdim <= 4096 && rows > 0 && rot_dims >= 0 && rot_dims <= dim && rot_dims % 2 == 0
                && (rot_dims == 0 || freq_f64_dev) && (!v_freq_f64_dev || vdim % 2 == 0), "ifa_qkv_rope_store_f32: bad shape (head sizes %d / %d, %d rotated)", dim, vdim, rot_dims);
    IFA_REQUIRE(ldq >= (size_t)heads * dim && (!k_f32 || (ldk >= (size_t)kv_heads * dim && ldv >= (size_t)kv_heads * vdim)), "ifa_qkv_rope_store_f32: row strides too small");
    const size_t smem = ((size_t)std::max(rot_dims, 2) + (size_t)vdim + 2) * 4;
#define IFA_RS(N) hipLaunchKernelGGL((k_qk_rope_store<N, true>), dim3((unsigned)rows, k_f32 ? 2u : 1u, rope_parts(rows, heads, k_f32 ? kv_heads : 0)), dim3(256), smem, ifa_s(stream), (float *)q_f32, ldq, heads, \
                                     (const float *)k_f32, ldk, (const float *)v_f32, ldv, kv_heads, dim, vdim, (const bf16_t *)q_norm_w_bf16, (const bf16_t *)k_norm_w_bf16, eps, \
                                     rot_dims, freq_f64_dev, (const SeqDesc *)seqs_dev, row_seq_dev, (float *const *)slot_base_dev, k_off, v_off, v_norm ? 1 : 0, v_freq_f64_dev, 0, kv_heads)
    if (dim <= 128) IFA_RS(2); else if (dim <= 256) IFA_RS(4); else IFA_RS(16);
#undef IFA_RS
    IFA_LAUNCH_CHECK();
    return IFA_OK;
}

int ifa_rotate_heads_f32(void *x_f32, size_t ldx, int heads, int dim, int rot_dims, const double *freq_f64_dev, float sign, const void *seqs_dev,
                         const int *row_seq_dev, size_t rows, ifa_stream stream)
{
    IFA_REQUIRE(x_f32 && seqs_dev && row_seq_dev && (rot_dims == 0 || freq_f64_dev), "ifa_rotate_heads_f32: null pointer");
    IFA_REQUIRE(heads > 0 && dim > 0 && rows > 0 && rot_dims >= 0 && rot_dims <= dim && rot_dims % 2 == 0 && rot_dims <= 8192 && ldx >= (size_t)heads * dim,
                "ifa_rotate_heads_f32: bad shape (head size %d, %d rotated)", dim, rot_dims);
    if (rot_dims == 0) return IFA_OK;
    hipLaunchKernelGGL(k_rotate_heads, dim3((unsigned)rows), dim3(256), (size_t)rot_dims * 4, ifa_s(stream), (float *)x_f32, ldx, heads, dim, rot_dims, freq_f64_dev, sign,
                       (const SeqDesc *)seqs_dev, row_seq_dev);
    IFA_LAUNCH_CHECK();
    return IFA_OK;
}

int ifa_attention_kv_sinks_f32(const void *q_f32, size_t ldq, int heads, int kv_heads, int dim, int vdim, float scale, int window, int keep_first,
                               const void *sink_bf16, const void *seqs_dev, const int *row_seq_dev, size_t rows, void *const *slot_base_dev, size_t k_off,
                               size_t v_off, void *out_f32, size_t ldo, const void *seqs_host, int n_seqs, int tile_min_rows, int max_keys, void *ws_f32,
                               size_t ws_bytes, ifa_stream stream)
{
    const int win = window > 0 ? window : (1 << 30);
    return attention_launch("ifa_attention_kv_sinks_f32", q_f32, ldq, heads, kv_heads, dim, vdim, 0, 0.0f, scale, 0.0f, win, keep_first, nullptr, nullptr, 0, sink_bf16,
                            0, 0.0f, seqs_dev, row_seq_dev, rows, slot_base_dev, k_off, v_off, out_f32, ldo, seqs_host, n_seqs, tile_min_rows, max_keys, ws_f32, ws_bytes,
                            stream);
}

} // extern "C"

int ifa_attention_window_to_bf16(const void *q_f32, size_t ldq, int heads, int kv_heads, int dim, int norm_q, float eps, float scale, float softcap, int window, int keep_first,
                                 const void *rel_bf16, const int *bucket_of_dev, int n_buckets, const void *sink_bf16, const void *seqs_dev, const int *row_seq_dev, size_t rows,
                                 void *const *slot_base_dev, size_t k_off, size_t v_off, void *out_f32, size_t ldo, void *out_bf16, size_t ld16, bool *left16, const void *seqs_host,
                                 int n_seqs, int tile_min_rows, void *ws_f32, size_t ws_bytes, const IfaFreshKV &fresh, const IfaLinearSide *side, bool *side_done, ifa_stream stream)
{
    IFA_REQUIRE(fresh.k && fresh.v && !fresh.turn_q && !fresh.norm_w && fresh.rot_dims == 0 && fresh.ldk >= (size_t)kv_heads * dim && fresh.ldv >= (size_t)kv_heads * dim && (!side || side_done),
                "attention_window_to_bf16: bad keys");
    const int tile_ok = dim % 32 == 0 && k_off % 4 == 0 && v_off % 4 == 0;          // (as ifa_attention_window_f32)
    return attention_launch("attention_window_to_bf16", q_f32, ldq, heads, kv_heads, dim, dim, norm_q, eps, scale, softcap, window, keep_first, rel_bf16, bucket_of_dev, n_buckets,
                            sink_bf16, 0, 0.0f, seqs_dev, row_seq_dev, rows, slot_base_dev, k_off, v_off, out_f32, ldo, seqs_host, tile_ok ? n_seqs : 0, tile_min_rows, 0, ws_f32,
                            ws_bytes, stream, out_bf16, ld16, left16, &fresh, side, side_done);
}

int ifa_attention_kv_to_bf16(const void *q_f32, size_t ldq, int heads, int kv_heads, int dim, int vdim, float scale, int window, int keep_first, int sink, float sink_score,
                             const void *seqs_dev, const int *row_seq_dev, size_t rows, void *const *slot_base_dev, size_t k_off, size_t v_off, void *out_f32, size_t ldo,
                             void *out_bf16, size_t ld16, bool *left16, const void *seqs_host, int n_seqs, int tile_min_rows, int max_keys, void *ws_f32, size_t ws_bytes,
                             const IfaFreshKV &fresh, ifa_stream stream)
{
    IFA_REQUIRE(fresh.turn_q && (!fresh.k || (fresh.v && fresh.ldk >= (size_t)kv_heads * dim && fresh.ldv >= (size_t)kv_heads * vdim)) && fresh.norm == (fresh.norm_w != nullptr)
                && fresh.rot_dims >= 0 && fresh.rot_dims <= dim && fresh.rot_dims % 2 == 0 && (fresh.rot_dims == 0 || fresh.freq), "attention_kv_to_bf16: bad keys");
    return attention_launch("attention_kv_to_bf16", q_f32, ldq, heads, kv_heads, dim, vdim, 0, 0.0f, scale, 0.0f, window > 0 ? window : (1 << 30), keep_first, nullptr, nullptr, 0,
                            nullptr, sink ? 1 : 0, sink_score, seqs_dev, row_seq_dev, rows, slot_base_dev, k_off, v_off, out_f32, ldo, seqs_host, n_seqs, tile_min_rows, max_keys,
                            ws_f32, ws_bytes, stream, out_bf16, ld16, left16, &fresh);
}

int ifa_mix_row(const IfaMixRow &M, int *nsplit, ifa_stream stream)
{
    IFA_REQUIRE(M.q && M.k && M.lq && M.lk && M.lv && M.decay && M.seqs && M.row_seq && M.slot_base && M.out && M.lin_out && nsplit, "mix_row: null pointer");
    IFA_REQUIRE(ifa_mix_row_fits(M), "mix_row: %d / %d heads of %d, %d heads of %d x %d", M.heads, M.kv_heads, M.dim, M.l_heads, M.l_dim, M.l_vdim);
    WinAttnArgs P;
    memset(&P, 0, sizeof(P));
    P.q = M.q; P.heads = M.heads; P.kv_heads = M.kv_heads; P.dim = P.vdim = M.dim; P.norm_q = 1; P.eps = M.eps; P.scale = M.scale; P.softcap = M.softcap;
    P.window = M.window; P.keep_first = M.keep_first; P.rel = M.rel; P.bucket_of = M.bucket_of; P.n_buckets = M.n_buckets; P.sink = M.sink;
    P.seqs = (const SeqDesc *)M.seqs; P.row_seq = M.row_seq; P.slot_base = (float *const *)M.slot_base; P.k_off = M.k_off; P.v_off = M.v_off;
    P.out = M.out; P.out16 = nullptr; P.ldo = P.ldq = (size_t)M.heads * M.dim;
    const size_t keys = std::min((size_t)M.window + (size_t)M.keep_first, (size_t)M.max_keys);
    int ns = (int)std::min<size_t>(IFA_ROW_OUT_SPLITS, (keys + 63) / 64);
    while (ns > 1 && (size_t)M.heads * ns * ((size_t)M.dim + 2) * 4 > M.ws_bytes) ns--;
    P.ws = M.ws; P.nsplit = *nsplit = std::max(ns, 1);
    const FreshRow F{M.k, M.k, 1};
    const StateRow R{M.lq, M.lk, M.lv, M.decay, M.l_heads, M.l_dim, M.l_vdim, M.l_off, M.lin_out};
    const size_t smem = std::max((size_t)M.dim + 8 + 4 * (size_t)M.dim, (size_t)256) * 4;
    const dim3 grid((unsigned)(M.heads * P.nsplit + M.l_heads * ((M.l_vdim + 63) / 64)));
#define IFA_MR(D) { if (M.l_dim == 64) hipLaunchKernelGGL((k_mix_row<D, 16>), grid, dim3(256), smem, ifa_s(stream), P, F, R); \
                    else hipLaunchKernelGGL((k_mix_row<D, 32>), grid, dim3(256), smem, ifa_s(stream), P, F, R); }
    if (M.dim <= 64) IFA_MR(1) else IFA_MR(2)
#undef IFA_MR
    IFA_LAUNCH_CHECK();
    return IFA_OK;
}

bool ifa_mix_row_fits(const IfaMixRow &M)
{
    // (more keys than the shares' workgroups take in eight rounds of 64: more workgroups and a launch that joins them do better)
    return M.dim <= 128 && M.dim % 4 == 0 && M.k_off % 4 == 0 && M.v_off % 4 == 0 && (uintptr_t)M.k % 16 == 0 && (M.l_dim == 64 || M.l_dim == 128) && M.l_vdim > 0
           && std::min((size_t)M.window + (size_t)M.keep_first, (size_t)M.max_keys) <= 64 * 8 * IFA_ROW_OUT_SPLITS;
}
