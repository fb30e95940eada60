// ifa_attn.hip -- attention over a KV cache (op-level, any q_tokens).
//
// Replaces the reference sequence GetKRows(+dequant) / TransposeYZ / RepeatKV /
// Gemm_Alg2 / ALiBi / SoftMax / GetVRows / Transpose / RepeatKV / Gemm_Alg2 /
// TransposeYZ+Assign (src/transformer/inference_worker.cc:1116-1312, :1639-1724)
// with one kernel per (head, query token): GQA by indexing, Q8 rows read in
// place, scores kept in LDS.  Rounding points are the reference's:
//   S = half(alpha * sum_d q.k)        (Gemm_Alg2_Kernel, src/kernels/gemm.h:83-178)
//   P = half(half(exp(scale*S - max)) * (1/sum))   (Tensor_SoftMax_Alg2_Kernel)
//   O = half(sum_j P_j * V_j)          (Gemm_Alg2_Kernel)
// q.k and P.V are accumulated in fp32 in index order (products of halfs are
// exact in fp32), so S and O match the restated reference bit-for-bit given the
// same P; P differs by the device expf and the softmax summation order.
#include <map>
#include <mutex>
#include "ifa_host.h"
#include "ifa_device.h"
#include "ifa_math.h"

namespace ifa {

// element d of kv-row j: F16 cache or Q8_B32T2 rows (dequantised to half as q*scale)
template <bool Q8>
__device__ __forceinline__ float kv_elem(const uint8_t *cache, size_t row_bytes, int j, int e)
{
    if constexpr (Q8) {
        const uint8_t *blk = cache + (size_t)j * row_bytes + (size_t)(e >> 5) * 34;
        const float scale = hbits2f(*reinterpret_cast<const uint16_t *>(blk));
        const int q = (int)(int8_t)blk[2 + (e & 31)];
        return h2f(f2h((float)q * scale));
    } else {
        return h2f(reinterpret_cast<const half_t *>(cache + (size_t)j * row_bytes)[e]);
    }
}

// rows != nullptr: dynamic batching -- row t is ONE new token of its own query: K/V cache and context length come from
// rows[t] (the query's KV cache set), smem is sized for the longest context of the batch
struct AttnRow { const uint8_t *kc, *vc; int n_ctx, pad; };

template <bool Q8>
__global__ void __launch_bounds__(256) k_attention(const half_t *__restrict__ q, const uint8_t *__restrict__ kc,
                                                   const uint8_t *__restrict__ vc, int n_ctx, int q_tokens,
                                                   int prefix_len, int heads, int kv_heads, int head_dim,
                                                   float kq_scale, int alibi, int alibi_base, int alibi_total,
                                                   half_t *__restrict__ out, const AttnRow *__restrict__ rows = nullptr)
{
    extern __shared__ __attribute__((aligned(16))) char smem[];
    half_t *S = reinterpret_cast<half_t *>(smem);                       // [n_ctx]
    float *red = reinterpret_cast<float *>(smem + (((size_t)n_ctx * 2 + 15) & ~(size_t)15));  // [8]  (n_ctx: batch maximum)
    const int h = blockIdx.x, t = blockIdx.y;
    if (rows) { kc = rows[t].kc; vc = rows[t].vc; n_ctx = rows[t].n_ctx; prefix_len = n_ctx - 1 - t; }
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int kvh = h / (heads / kv_heads);
    const int kv_dim = kv_heads * head_dim;
    const size_t row_bytes = Q8 ? (size_t)(kv_dim / 32) * 34 : (size_t)kv_dim * 2;
    const half_t *qv = q + ((size_t)t * heads + h) * head_dim;
    const float alpha = 1.0f / sqrtf((float)head_dim) / kq_scale;
    const int n_valid = min(n_ctx, prefix_len + t + 1);   // causal: xi <= prefix_len + t
    const float mk = alibi ? alibi_slope(h + alibi_base, alibi_total) : 0.0f;

    // ---- scores
    float lmax = -INFINITY;
    for (int j = tid; j < n_ctx; j += 256) {
        float c = 0.0f;
        for (int d = 0; d < head_dim; d++) c = __builtin_fmaf(h2f(qv[d]), kv_elem<Q8>(kc, row_bytes, j, kvh * head_dim + d), c);
        half_t s = f2h(alpha * c);
        if (alibi) { float a = (float)j * mk; s = f2h(a + h2f(s)); }
        S[j] = s;
        if (j < n_valid) lmax = fmaxf(lmax, kq_scale * h2f(s));
    }
    lmax = wave_max(lmax);
    if (lane == 0) red[wave] = lmax;
    __syncthreads();
    const float mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    __syncthreads();
    // ---- exp + sum
    float lsum = 0.0f;
    for (int j = tid; j < n_ctx; j += 256) {
        float e = 0.0f;
        if (j < n_valid) e = expf(kq_scale * h2f(S[j]) - mx);
        lsum += e;
        S[j] = f2h(e);
    }
    lsum = wave_sum(lsum);
    if (lane == 0) red[4 + wave] = lsum;
    __syncthreads();
    const float inv = 1.0f / (((red[4] + red[5]) + red[6]) + red[7]);
    for (int j = tid; j < n_ctx; j += 256) S[j] = f2h(h2f(S[j]) * inv);
    __syncthreads();
    // ---- O = P.V, one thread per output dim, j ascending (reference order)
    for (int d = tid; d < head_dim; d += 256) {
        float c = 0.0f;
        for (int j = 0; j < n_valid; j++)
            c = __builtin_fmaf(h2f(S[j]), kv_elem<Q8>(vc, row_bytes, j, kvh * head_dim + d), c);
        out[(size_t)t * heads * head_dim + (size_t)h * head_dim + d] = f2h(c);
    }
}


// ---------------------------------------------------------------- prefill (q_tokens >= 4): MFMA tiles
// One workgroup per (32-query tile, head); same three stages and the same rounding points as k_attention
// (S and P are half tensors between the stages, like the reference's Gemm_Alg2 -> SoftMax -> Gemm_Alg2), but
//   S tile  = Q[32 x HD] . K^T          v_mfma_f32_32x32x16_f16, keys of a 32-block = B columns, straight from the cache
//   P       = row softmax of the [32 x n_keys] half tile kept in LDS (a wave per 8 rows)
//   O tile  = P . V                     V blocks transposed through LDS ([dim][key]) so a lane's 8 keys are contiguous
// fp32 accumulation in MFMA order instead of index order (products of halfs are exact either way).
typedef _Float16 half8v __attribute__((ext_vector_type(8)));
typedef float f32x16v __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));

// 8 consecutive elements e0..e0+7 (e0 % 8 == 0) of kv-row j as halfs
template <bool Q8>
__device__ __forceinline__ half8v kv_load8(const uint8_t *cache, size_t row_bytes, int j, int e0)
{
    if constexpr (Q8) {
        const uint8_t *blk = cache + (size_t)j * row_bytes + (size_t)(e0 >> 5) * 34;
        const uint16_t *p16 = reinterpret_cast<const uint16_t *>(blk);
        const float scale = hbits2f(p16[0]);
        half8v r;
#pragma unroll
        for (int w = 0; w < 4; w++) {
            const uint32_t two = p16[1 + ((e0 & 31) >> 1) + w];
            r[2 * w] = f2h((float)(int)(int8_t)(two & 0xFF) * scale);
            r[2 * w + 1] = f2h((float)(int)(int8_t)(two >> 8) * scale);
        }
        return r;
    } else {
        return __builtin_bit_cast(half8v, *reinterpret_cast<const u32x4v *>(cache + (size_t)j * row_bytes + (size_t)e0 * 2));
    }
}

constexpr int PF_QT = 32;            // queries per workgroup
constexpr int PF_VROW = 40;          // halfs per row of the transposed V block (32 keys + pad: conflict-free b128 reads)

__host__ __device__ inline int pf_nkp(int n_keys) { return (n_keys + 31) / 32 * 32 + 8; }

__device__ unsigned long long g_attn_trace[8];     // wall_clock64 stamps of the longest tile of head 0 (tools/probes)

// SG: the [32 x n_keys] score tile lives in a global workspace (sg_ws: [heads][tiles][32][sg_nkp] halfs) instead of the LDS
// -- contexts past ~2300 keys, where the tile no longer fits the 160 KiB; same stages, same rounding points, the tile is
// written once and walked three times through L2 (a fraction of the K / V traffic of the same tile)
template <int HD, bool Q8, bool SG = false>
__global__ void __launch_bounds__(256) k_attention_mfma(const half_t *__restrict__ q, const uint8_t *__restrict__ kc,
                                                        const uint8_t *__restrict__ vc, int n_ctx, int q_tokens,
                                                        int prefix_len, int heads, int kv_heads, float kq_scale,
                                                        int alibi, int alibi_base, int alibi_total, half_t *__restrict__ out,
                                                        half_t *__restrict__ sg_ws = nullptr, int sg_nkp = 0)
{
    extern __shared__ __attribute__((aligned(16))) char smem[];
    constexpr int KS = HD / 16;          // MFMA k-steps over the head dimension
    constexpr int NT = HD / 32;          // 32-wide output tiles
    // workgroups go to the 8 XCDs round-robin in launch order: give every XCD a fixed eighth of the heads, so a head's
    // K/V rows (re-read by each of its query tiles) stay in ONE 4 MB L2, and start the longest (last) tiles first
    int tile = blockIdx.x, h = blockIdx.y;
    if (heads % 8 == 0) {
        const int w = blockIdx.y * gridDim.x + blockIdx.x, xcd = w & 7, r = w >> 3;
        h = (r / (int)gridDim.x) * 8 + xcd;
        tile = (int)gridDim.x - 1 - r % (int)gridDim.x;
    }
    const int t0 = tile * PF_QT;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int i = lane & 31, g = lane >> 5;
    const int kvh = h / (heads / kv_heads);
    const int kv_dim = kv_heads * HD;
    const size_t row_bytes = Q8 ? (size_t)(kv_dim / 32) * 34 : (size_t)kv_dim * 2;
    const int hoff = kvh * HD;
    const int t_last = min(t0 + PF_QT, q_tokens) - 1;
    const int n_keys = min(n_ctx, prefix_len + t_last + 1);      // causal bound of the whole tile
    const int nkb = (n_keys + 31) / 32;
    const int NKP = SG ? sg_nkp : pf_nkp(n_keys);
    half_t *S = SG ? sg_ws + ((size_t)h * gridDim.x + tile) * PF_QT * (size_t)sg_nkp : reinterpret_cast<half_t *>(smem);     // [32][NKP]
    half_t *Vt = SG ? reinterpret_cast<half_t *>(smem) : S + (size_t)PF_QT * NKP;   // [HD][PF_VROW]
    const float alpha = 1.0f / sqrtf((float)HD) / kq_scale;
    const float mk = alibi ? alibi_slope(h + alibi_base, alibi_total) : 0.0f;

    const bool tracer = h == 0 && tile == (int)gridDim.x - 1 && tid == 0;
    if (tracer) g_attn_trace[0] = wall_clock64();
    // ---- S = half(alpha * Q.K^T) (+ALiBi), key blocks strided over the waves
    {
        half8v qa[KS];
        const int tq = min(t0 + i, q_tokens - 1);
#pragma unroll
        for (int s2 = 0; s2 < KS; s2++)
            qa[s2] = __builtin_bit_cast(half8v, *reinterpret_cast<const u32x4v *>(q + ((size_t)tq * heads + h) * HD + 16 * s2 + 8 * g));
        // two register sets of K fragments: the next block of this wave is in flight while one is multiplied
        half8v ka[KS], kb2[KS];
        auto kload = [&](half8v (&kf)[KS], int kb) {
            const int j = min(32 * kb + i, n_ctx - 1);
#pragma unroll
            for (int s2 = 0; s2 < KS; s2++) kf[s2] = kv_load8<Q8>(kc, row_bytes, j, hoff + 16 * s2 + 8 * g);
        };
        auto kscore = [&](const half8v (&kf)[KS], int kb) {
            f32x16v acc;
#pragma unroll
            for (int r = 0; r < 16; r++) acc[r] = 0.0f;
#pragma unroll
            for (int s2 = 0; s2 < KS; s2++) acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(qa[s2], kf[s2], acc, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int row = (r & 3) + 8 * (r >> 2) + 4 * g;
                half_t sv = f2h(alpha * acc[r]);
                if (alibi) { float a = (float)(32 * kb + i) * mk; sv = f2h(a + h2f(sv)); }
                S[(size_t)row * NKP + 32 * kb + i] = sv;
            }
        };
        if (wave < nkb) kload(ka, wave);
        if (wave + 4 < nkb) kload(kb2, wave + 4);
        for (int kb = wave; kb < nkb; kb += 8) {
            kscore(ka, kb);
            if (kb + 8 < nkb) kload(ka, kb + 8);
            if (kb + 4 < nkb) {
                kscore(kb2, kb + 4);
                if (kb + 12 < nkb) kload(kb2, kb + 12);
            }
        }
    }
    __syncthreads();
    if (tracer) g_attn_trace[1] = wall_clock64();
    // (V rows: the first two key blocks go out in front of the softmax)
    constexpr int CH = HD / 8;               // 16-byte chunks per V row
    constexpr int KPI = 256 / CH;            // keys staged per pass of the workgroup
    constexpr int NIT = (32 + KPI - 1) / KPI;
    half8v va[NIT], vb[NIT];                 // V rows of the next two key blocks, requested two blocks ahead
    // lane bits: key parity | key pair (8) | chunk low (4); waves: chunk high, then further key groups.  Lane pairs swap
    // halves of their rows so that every lane stores (even key, odd key) dwords of 4 dims: half the LDS stores of a
    // 2-byte transpose, spread over 32 banks instead of 8
    const int vpar = tid & 1, vpair = (tid >> 1) & 7;
    const int vch = ((tid >> 4) & 3) + 4 * ((tid >> 6) % (CH / 4));
    const int vkey0 = 16 * ((tid >> 6) / (CH / 4)) + 2 * vpair;             // even key of the lane pair within a pass
    auto vload = [&](half8v (&v)[NIT], int kt) {
#pragma unroll
        for (int it = 0; it < NIT; it++) {
            const int key = min(vkey0 + vpar + it * KPI, 31);
            const int j = min(32 * kt + key, n_ctx - 1);
            v[it] = kv_load8<Q8>(vc, row_bytes, j, hoff + 8 * vch);
        }
    };
    if (nkb > 0) vload(va, 0);
    if (nkb > 1) vload(vb, 1);
    // ---- P = softmax rows (Tensor_SoftMax_Alg2_Kernel rounding: half(e), then half(half(e) * 1/sum))
    // 16-byte LDS accesses, 8 scores per lane and step (a 2-byte walk is one LDS round trip per element); the phase is
    // VALU-bound (32 x n_keys exponentials per workgroup), so whole chunks skip the per-element causal mask
    // Up to 512 keys a row is one piece a lane: four rows at a time in registers, their reductions side by side (row after row each waited for the ones before: 37 queries
    // 13.3 -> 10.0 us a layer, with the first V rows requested up here)
    if (4 * nkb <= 64) {
        const int nch = 4 * nkb;
#pragma unroll
        for (int r4 = 0; r4 < 8; r4 += 4) {
            half8v v[4];
            float lmax[4], lsum[4];
            int nv[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int row = 8 * wave + r4 + u, t = t0 + row;
                nv[u] = t < q_tokens ? min(n_ctx, prefix_len + t + 1) : 0;
                v[u] = *reinterpret_cast<const half8v *>(S + (size_t)row * NKP + 8 * min(lane, nch - 1));
                if (lane >= nch) nv[u] = 0;
                lmax[u] = -INFINITY;
#pragma unroll
                for (int e = 0; e < 8; e++) if (8 * lane + e < nv[u]) lmax[u] = fmaxf(lmax[u], kq_scale * h2f(v[u][e]));
            }
#pragma unroll
            for (int u = 0; u < 4; u++) lmax[u] = wave_max(lmax[u]);
#pragma unroll
            for (int u = 0; u < 4; u++) {
                lsum[u] = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const float ev = 8 * lane + e < nv[u] ? __expf(kq_scale * h2f(v[u][e]) - lmax[u]) : 0.0f;
                    lsum[u] += ev;
                    v[u][e] = f2h(ev);
                }
            }
#pragma unroll
            for (int u = 0; u < 4; u++) lsum[u] = wave_sum(lsum[u]);
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const float inv = lsum[u] > 0.0f ? 1.0f / lsum[u] : 0.0f;
                if (8 * lane < nv[u]) {
#pragma unroll
                    for (int e = 0; e < 8; e++) v[u][e] = f2h(h2f(v[u][e]) * inv);
                }
                if (lane < nch) *reinterpret_cast<half8v *>(S + (size_t)(8 * wave + r4 + u) * NKP + 8 * lane) = v[u];
            }
        }
    } else
    for (int rr = 0; rr < 8; rr++) {
        const int row = 8 * wave + rr;
        const int t = t0 + row;
        half_t *Sr = S + (size_t)row * NKP;
        const int n_valid = t < q_tokens ? min(n_ctx, prefix_len + t + 1) : 0;
        const int nch = 4 * nkb;
        float lmax = -INFINITY;
        for (int c = lane; c < nch; c += 64) {
            const half8v v = *reinterpret_cast<const half8v *>(Sr + 8 * c);
#pragma unroll
            for (int e = 0; e < 8; e++)
                if (8 * c + e < n_valid) lmax = fmaxf(lmax, kq_scale * h2f(v[e]));
        }
        lmax = wave_max(lmax);
        float lsum = 0.0f;
        for (int c = lane; c < nch; c += 64) {
            const half8v v = *reinterpret_cast<const half8v *>(Sr + 8 * c);
            half8v o;
            if (8 * c + 8 <= n_valid) {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const float ev = __expf(kq_scale * h2f(v[e]) - lmax);
                    lsum += ev;
                    o[e] = f2h(ev);
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    float ev = 0.0f;
                    if (8 * c + e < n_valid) ev = __expf(kq_scale * h2f(v[e]) - lmax);
                    lsum += ev;
                    o[e] = f2h(ev);
                }
            }
            *reinterpret_cast<half8v *>(Sr + 8 * c) = o;
        }
        lsum = wave_sum(lsum);
        const float inv = lsum > 0.0f ? 1.0f / lsum : 0.0f;      // rows past q_tokens: all zero
        const int nch_valid = min(nch, (n_valid + 7) / 8);        // beyond: already zero
        for (int c = lane; c < nch_valid; c += 64) {
            const half8v v = *reinterpret_cast<const half8v *>(Sr + 8 * c);
            half8v o;
#pragma unroll
            for (int e = 0; e < 8; e++) o[e] = f2h(h2f(v[e]) * inv);
            *reinterpret_cast<half8v *>(Sr + 8 * c) = o;
        }
    }
    if (tracer) g_attn_trace[2] = wall_clock64();
    // ---- O = P.V
    f32x16v oacc;
#pragma unroll
    for (int r = 0; r < 16; r++) oacc[r] = 0.0f;
    auto vstage = [&](const half8v (&v)[NIT]) {
#pragma unroll
        for (int it = 0; it < NIT; it++) {
            const u32x4v w = __builtin_bit_cast(u32x4v, v[it]);
            const uint32_t m0 = vpar ? w[2] : w[0], m1 = vpar ? w[3] : w[1];            // the 4 dims this lane stores
            const uint32_t r0 = __shfl_xor(vpar ? w[0] : w[2], 1), r1 = __shfl_xor(vpar ? w[1] : w[3], 1);
            const uint32_t e0 = vpar ? r0 : m0, e1 = vpar ? r1 : m1;                      // even key's values
            const uint32_t o0 = vpar ? m0 : r0, o1 = vpar ? m1 : r1;                      // odd key's values
            const int key = vkey0 + it * KPI;
            if (key < 32) {
                uint32_t *dst = reinterpret_cast<uint32_t *>(Vt + (size_t)(8 * vch + 4 * vpar) * PF_VROW + key);
                dst[0 * PF_VROW / 2] = (e0 & 0xFFFFu) | (o0 << 16);
                dst[1 * PF_VROW / 2] = (e0 >> 16) | (o0 & 0xFFFF0000u);
                dst[2 * PF_VROW / 2] = (e1 & 0xFFFFu) | (o1 << 16);
                dst[3 * PF_VROW / 2] = (e1 >> 16) | (o1 & 0xFFFF0000u);
            }
        }
    };
    auto pv = [&](int kt) {
        if (wave < NT) {
#pragma unroll
            for (int s2 = 0; s2 < 2; s2++) {
                const half8v pf = *reinterpret_cast<const half8v *>(S + (size_t)i * NKP + 32 * kt + 16 * s2 + 8 * g);
                const half8v vf = *reinterpret_cast<const half8v *>(Vt + (size_t)(32 * wave + i) * PF_VROW + 16 * s2 + 8 * g);
                oacc = __builtin_amdgcn_mfma_f32_32x32x16_f16(pf, vf, oacc, 0, 0, 0);
            }
        }
    };
    for (int kt = 0; kt < nkb; kt += 2) {
        __syncthreads();                     // previous block consumed (and, first time, P complete)
        vstage(va);
        if (kt + 2 < nkb) vload(va, kt + 2);
        __syncthreads();
        pv(kt);
        if (kt + 1 < nkb) {
            __syncthreads();
            vstage(vb);
            if (kt + 3 < nkb) vload(vb, kt + 3);
            __syncthreads();
            pv(kt + 1);
        }
    }
    if (tracer) g_attn_trace[3] = wall_clock64();
    if (wave < NT) {
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int t = t0 + (r & 3) + 8 * (r >> 2) + 4 * g;
            if (t < q_tokens) out[((size_t)t * heads + h) * HD + 32 * wave + i] = f2h(oacc[r]);
        }
    }
}

// ---------------------------------------------------------------- short prompts from position 0 (4 .. 63 tokens, F16 cache, heads of 128 turned whole)
// What k_rope_qk_store and k_attention_mfma do for such a step in one launch, a workgroup per (32-query tile, head): its queries, keys and values are in the step's own q / k / v rows, asked for
// at once; the tile's own keys, turned, and values go into the cache on their way.  The cosines and sines come from a table of the step (tab [token][64] pairs, formed where the embedding rows
// are gathered): the angles of every key again in every head's workgroup would be 8 us.  The same expressions in the same order, the same bits.
// Bound by its launch and one chain (rows, LDS, scores, softmax, LDS, products): 37 tokens of 32 heads 4.8 + 10.9 -> 4.8 us a layer (a whole prompt of 37 2503 -> 2198).
constexpr int FR_MAX = 64, FR_ROW = 128 + 8, FR_S = FR_MAX + 8;          // keys; halfs per row of queries / keys and of scores
template <int ORDER>
__global__ void __launch_bounds__(256) k_attention_fresh(const half_t *__restrict__ q, const half_t *__restrict__ k, const half_t *__restrict__ v, const float *__restrict__ tab, int T, int heads,
                                                         int kv_heads, float kq_scale, half_t *__restrict__ kcache, half_t *__restrict__ vcache, size_t cache_row, half_t *__restrict__ out)
{
    constexpr int HD = 128, KS = HD / 16;
    __shared__ __attribute__((aligned(16))) half_t Qs[32 * FR_ROW], Ks[FR_MAX * FR_ROW], S[32 * FR_S], Vt[2][HD * PF_VROW];
    const int tile = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i = lane & 31, g = lane >> 5, group = heads / kv_heads, kvh = h / group;
    const int t0 = 32 * tile, nkb = tile + 1;
    const bool stores = h % group == 0;          // (one head of those that share the keys)
    const size_t q_row = (size_t)heads * HD, kv_row = (size_t)kv_heads * HD;
    // a row's head in pieces of eight pairs: halfs a0 .. a0 + 7 and b0 .. b0 + 7
    const int row = tid >> 3, c0 = 8 * (tid & 7), a0 = ORDER == 2 ? c0 : 2 * c0, b0 = ORDER == 2 ? c0 + HD / 2 : 2 * c0 + 8;
    const int tq = min(t0 + row, T - 1);
    auto pair_at = [&](const half_t *p, half8v (&x)[2]) { x[0] = *reinterpret_cast<const half8v *>(p + a0); x[1] = *reinterpret_cast<const half8v *>(p + b0); };
    auto angles_at = [&](int t, float4 (&cs)[4]) {
#pragma unroll
        for (int e = 0; e < 4; e++) cs[e] = *reinterpret_cast<const float4 *>(tab + ((size_t)t * (HD / 2) + c0) * 2 + 4 * e);
    };
    half8v qv[2], kv[2][2], va[2][2];
    float4 cs[2][4];
    pair_at(q + (size_t)tq * q_row + (size_t)h * HD, qv);
    const int vpar = tid & 1, vpair = (tid >> 1) & 7, vch = ((tid >> 4) & 3) + 4 * wave, vkey0 = 2 * vpair;          // (as in k_attention_mfma)
#pragma unroll
    for (int kb = 0; kb < 2; kb++)
        if (kb < nkb) {
            const int t = min(32 * kb + row, T - 1);
            pair_at(k + (size_t)t * kv_row + (size_t)kvh * HD, kv[kb]);
            angles_at(t, cs[kb]);
#pragma unroll
            for (int it = 0; it < 2; it++) va[kb][it] = *reinterpret_cast<const half8v *>(v + (size_t)min(32 * kb + vkey0 + vpar + 16 * it, T - 1) * kv_row + (size_t)kvh * HD + 8 * vch);
        }
    auto turned = [&](const half8v (&x)[2], const float4 (&a)[4], half8v (&y)[2]) {          // rope_rotate's expressions (ifa_math.h)
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float x0 = ORDER == 2 ? h2f(x[0][e]) : h2f(e < 4 ? x[0][2 * e & 7] : x[1][(2 * e - 8) & 7]);
            const float x1 = ORDER == 2 ? h2f(x[1][e]) : h2f(e < 4 ? x[0][(2 * e + 1) & 7] : x[1][(2 * e - 7) & 7]);
            const float c = e & 1 ? a[e >> 1].z : a[e >> 1].x, sn = e & 1 ? a[e >> 1].w : a[e >> 1].y;
            const float p0 = x0 * c, p1 = x1 * sn, p2 = x0 * sn, p3 = x1 * c;
            const half_t r0 = f2h(p0 - p1), r1 = f2h(p2 + p3);
            if (ORDER == 2) { y[0][e] = r0; y[1][e] = r1; }
            else if (e < 4) { y[0][(2 * e) & 7] = r0; y[0][(2 * e + 1) & 7] = r1; }
            else { y[1][(2 * e - 8) & 7] = r0; y[1][(2 * e - 7) & 7] = r1; }
        }
    };
#pragma unroll
    for (int kb = 0; kb < 2; kb++)
        if (kb < nkb) {
            half8v y[2];
            turned(kv[kb], cs[kb], y);
            half_t *dst = Ks + (size_t)(32 * kb + row) * FR_ROW;
            *reinterpret_cast<half8v *>(dst + a0) = y[0]; *reinterpret_cast<half8v *>(dst + b0) = y[1];
            if (kb == tile) {
                half8v z[2];
                turned(qv, cs[kb], z);
                half_t *qd = Qs + (size_t)row * FR_ROW;
                *reinterpret_cast<half8v *>(qd + a0) = z[0]; *reinterpret_cast<half8v *>(qd + b0) = z[1];
                if (stores && t0 + row < T) {
                    half_t *kd = kcache + (size_t)(t0 + row) * cache_row + (size_t)kvh * HD;
                    *reinterpret_cast<half8v *>(kd + a0) = y[0]; *reinterpret_cast<half8v *>(kd + b0) = y[1];
                }
            }
            // values: [dim][key], two keys a dword (as in k_attention_mfma)
#pragma unroll
            for (int it = 0; it < 2; it++) {
                const int key = 32 * kb + vkey0 + vpar + 16 * it;
                if (kb == tile && stores && key < T) *reinterpret_cast<half8v *>(vcache + (size_t)key * cache_row + (size_t)kvh * HD + 8 * vch) = va[kb][it];
                const u32x4v w = __builtin_bit_cast(u32x4v, va[kb][it]);
                const uint32_t m0 = vpar ? w[2] : w[0], m1 = vpar ? w[3] : w[1];
                const uint32_t r0 = __shfl_xor(vpar ? w[0] : w[2], 1), r1 = __shfl_xor(vpar ? w[1] : w[3], 1);
                const uint32_t e0 = vpar ? r0 : m0, e1 = vpar ? r1 : m1, o0 = vpar ? m0 : r0, o1 = vpar ? m1 : r1;
                uint32_t *d = reinterpret_cast<uint32_t *>(Vt[kb] + (size_t)(8 * vch + 4 * vpar) * PF_VROW + vkey0 + 16 * it);
                d[0 * PF_VROW / 2] = (e0 & 0xFFFFu) | (o0 << 16);
                d[1 * PF_VROW / 2] = (e0 >> 16) | (o0 & 0xFFFF0000u);
                d[2 * PF_VROW / 2] = (e1 & 0xFFFFu) | (o1 << 16);
                d[3 * PF_VROW / 2] = (e1 >> 16) | (o1 & 0xFFFF0000u);
            }
        }
    __syncthreads();
    if (wave < nkb) {
        const float alpha = 1.0f / sqrtf((float)HD) / kq_scale;
        f32x16v acc;
#pragma unroll
        for (int r = 0; r < 16; r++) acc[r] = 0.0f;
#pragma unroll
        for (int s2 = 0; s2 < KS; s2++)
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const half8v *>(Qs + (size_t)i * FR_ROW + 16 * s2 + 8 * g),
                                                         *reinterpret_cast<const half8v *>(Ks + (size_t)(32 * wave + i) * FR_ROW + 16 * s2 + 8 * g), acc, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 16; r++) S[(size_t)((r & 3) + 8 * (r >> 2) + 4 * g) * FR_S + 32 * wave + i] = f2h(alpha * acc[r]);
    }
    __syncthreads();
    {   // softmax, a row eight lanes (wave_max and wave_sum over these)
        const int r = 8 * wave + (lane >> 3), c = lane & 7, nch = 4 * nkb, nv = t0 + r < T && c < nch ? t0 + r + 1 : 0;
        half8v p = *reinterpret_cast<const half8v *>(S + (size_t)r * FR_S + 8 * min(c, nch - 1));
        float most = -INFINITY, sum = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; e++) if (8 * c + e < nv) most = fmaxf(most, kq_scale * h2f(p[e]));
        most = fmaxf(most, dpp_xor1(most)); most = fmaxf(most, dpp_xor2(most)); most = fmaxf(most, dpp_half_mirror(most));
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float ev = 8 * c + e < nv ? __expf(kq_scale * h2f(p[e]) - most) : 0.0f;
            sum += ev;
            p[e] = f2h(ev);
        }
        sum += dpp_xor1(sum); sum += dpp_xor2(sum); sum += dpp_half_mirror(sum);
        const float inv = sum > 0.0f ? 1.0f / sum : 0.0f;
        if (8 * c < nv) {
#pragma unroll
            for (int e = 0; e < 8; e++) p[e] = f2h(h2f(p[e]) * inv);
        }
        if (c < nch) *reinterpret_cast<half8v *>(S + (size_t)r * FR_S + 8 * c) = p;
    }
    __syncthreads();
    f32x16v o;
#pragma unroll
    for (int r = 0; r < 16; r++) o[r] = 0.0f;
    for (int kb = 0; kb < nkb; kb++)
#pragma unroll
        for (int s2 = 0; s2 < 2; s2++)
            o = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const half8v *>(S + (size_t)i * FR_S + 32 * kb + 16 * s2 + 8 * g),
                                                       *reinterpret_cast<const half8v *>(Vt[kb] + (size_t)(32 * wave + i) * PF_VROW + 16 * s2 + 8 * g), o, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int t = t0 + (r & 3) + 8 * (r >> 2) + 4 * g;
        if (t < T) out[((size_t)t * heads + h) * HD + 32 * wave + i] = f2h(o[r]);
    }
}

// ---------------------------------------------------------------- long prompts (q_tokens >= 128): two passes over the keys
// One workgroup per (128-query tile, head), a wave per 32 queries.  The three-stage kernel above keeps a [32 x n_keys]
// score tile (LDS, past ~2300 keys a global workspace) and re-reads a head's K / V once per 32 queries: at 4096 tokens it
// moves more score-tile and K / V bytes through L2 than the matrix cores can hide (1.2 ms per layer).  Here nothing of size
// n_keys is stored: pass 1 streams the K blocks and keeps each query's running max / sum, pass 2 streams K and V, REcomputes
// the scores, rounds them exactly like the staged kernel (S half, e = half(exp), P = half(e * 1/sum)) and multiplies by V
// from registers.  K / V blocks of 32 keys are staged through LDS once per 128 queries.
//   S^T = K . Q^T: keys are the MFMA rows, so a lane holds 16 keys of ONE query (its column): max / sum / P need no
//                  cross-lane traffic except one exchange between the lane halves at the end of pass 1;
//   O^T = V^T . P^T: P^T is then already the B operand (lane = query column, 8 keys per k-step); a lane's registers hold keys
//                  4g + {0-3, 8-11, 16-19, 24-27}, so the V block is transposed into LDS with its key columns in THAT order
//                  (f2_col) -- the sum over keys does not care.
constexpr int F2_QT = 128;
constexpr int F2_VROW = 40;          // halfs per row of the transposed V block (32 key columns + pad)
__host__ __device__ constexpr int f2_col(int k) { return (k & 16) | (((k >> 2) & 1) << 3) | (k & 3) | (((k >> 3) & 1) << 2); }
template <int HD> __device__ __forceinline__ int f2_swz(int row) { return HD == 128 ? (row & 15) : ((row >> 1) & 7); }

template <int HD, bool Q8>
__global__ void __launch_bounds__(256, 2) k_attention_2pass(const half_t *__restrict__ q, const uint8_t *__restrict__ kc,
                                                         const uint8_t *__restrict__ vc, int n_ctx, int q_tokens,
                                                         int prefix_len, int heads, int kv_heads, float kq_scale,
                                                         int alibi, int alibi_base, int alibi_total, half_t *__restrict__ out)
{
    static_assert(HD == 128 || HD == 64, "two-pass attention: head_dim 64 / 128");
    constexpr int KS = HD / 16, NT = HD / 32, CHK = HD / 8;
    constexpr int NKC = 32 * CHK / 256;              // 16-byte chunks of the K block per thread
    // two buffers each: block kb + 1 is staged while block kb is multiplied (one barrier per block)
    __shared__ __attribute__((aligned(16))) char Ks2[2][32 * HD * 2];             // [key][HD halfs], 16-byte chunks swizzled
    __shared__ __attribute__((aligned(16))) half_t Vt2[2][HD * F2_VROW];         // [dim][key column]
    int tile = blockIdx.x, h = blockIdx.y;
    if (heads % 8 == 0) {            // an XCD keeps a fixed eighth of the heads (their K / V in ONE L2); longest tiles first
        const int w = blockIdx.y * gridDim.x + blockIdx.x, xcd = w & 7, r = w >> 3;
        h = (r / (int)gridDim.x) * 8 + xcd;
        tile = (int)gridDim.x - 1 - r % (int)gridDim.x;
    }
    const int t0 = tile * F2_QT;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i = lane & 31, g = lane >> 5;
    const int kvh = h / (heads / kv_heads);
    const int kv_dim = kv_heads * HD;
    const size_t row_bytes = Q8 ? (size_t)(kv_dim / 32) * 34 : (size_t)kv_dim * 2;
    const int hoff = kvh * HD;
    const int n_keys = min(n_ctx, prefix_len + min(t0 + F2_QT, q_tokens));        // causal bound of the whole tile
    const int nkb = (n_keys + 31) / 32;
    const int tw = t0 + 32 * wave, tq = tw + i;
    const int n_valid = tq < q_tokens ? min(n_ctx, prefix_len + tq + 1) : 0;      // keys this lane's query may see
    const int wave_keys = tw < q_tokens ? min(n_ctx, prefix_len + min(tw + 32, q_tokens)) : 0;
    const int wave_nkb = (wave_keys + 31) / 32;                                   // blocks past it are fully masked for this wave
    const float alpha = 1.0f / sqrtf((float)HD) / kq_scale;
    const float mk = alibi ? alibi_slope(h + alibi_base, alibi_total) : 0.0f;

    half8v qf[KS];
    {
        const int tqc = min(tq, q_tokens - 1);
#pragma unroll
        for (int s2 = 0; s2 < KS; s2++)
            qf[s2] = __builtin_bit_cast(half8v, *reinterpret_cast<const u32x4v *>(q + ((size_t)tqc * heads + h) * HD + 16 * s2 + 8 * g));
    }
    // ---- staging: K block rows as they are (swizzled chunks), V block transposed with permuted key columns
    half8v kreg[NKC];
    auto kload = [&](int kb) {
#pragma unroll
        for (int it = 0; it < NKC; it++) {
            const int idx = tid + it * 256, row = idx / CHK, c = idx % CHK;
            kreg[it] = kv_load8<Q8>(kc, row_bytes, min(32 * kb + row, n_ctx - 1), hoff + 8 * c);
        }
    };
    auto kstage = [&](int buf) {
#pragma unroll
        for (int it = 0; it < NKC; it++) {
            const int idx = tid + it * 256, row = idx / CHK, c = idx % CHK;
            *reinterpret_cast<half8v *>(Ks2[buf] + (size_t)row * (HD * 2) + (size_t)((c ^ f2_swz<HD>(row)) << 4)) = kreg[it];
        }
    };
    constexpr int KPI = 256 / CHK;           // keys staged per pass of the workgroup
    constexpr int NIT = (32 + KPI - 1) / KPI;
    half8v vreg[NIT];
    const int vpar = tid & 1, vpair = (tid >> 1) & 7;
    const int vch = ((tid >> 4) & 3) + 4 * ((tid >> 6) % (CHK / 4));
    const int vkey0 = 16 * ((tid >> 6) / (CHK / 4)) + 2 * vpair;                  // even key of the lane pair within a pass
    auto vload = [&](int kb) {
#pragma unroll
        for (int it = 0; it < NIT; it++) {
            const int key = min(vkey0 + vpar + it * KPI, 31);
            vreg[it] = kv_load8<Q8>(vc, row_bytes, min(32 * kb + key, n_ctx - 1), hoff + 8 * vch);
        }
    };
    auto swap1 = [](uint32_t v) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, false); };   // lane ^ 1 (quad_perm [1, 0, 3, 2])
    auto vstage = [&](int buf) {             // lane pairs trade halves of their rows: (even key, odd key) dwords of 4 dims
        half_t *Vt = Vt2[buf];
#pragma unroll
        for (int it = 0; it < NIT; it++) {
            const u32x4v w = __builtin_bit_cast(u32x4v, vreg[it]);
            const uint32_t m0 = vpar ? w[2] : w[0], m1 = vpar ? w[3] : w[1];
            const uint32_t r0 = swap1(vpar ? w[0] : w[2]), r1 = swap1(vpar ? w[1] : w[3]);
            const uint32_t e0 = vpar ? r0 : m0, e1 = vpar ? r1 : m1;              // even key's values
            const uint32_t o0 = vpar ? m0 : r0, o1 = vpar ? m1 : r1;              // odd key's values
            const int key = vkey0 + it * KPI;
            if (key < 32) {
                uint32_t *dst = reinterpret_cast<uint32_t *>(Vt + (size_t)(8 * vch + 4 * vpar) * F2_VROW + f2_col(key));
                dst[0 * F2_VROW / 2] = (e0 & 0xFFFFu) | (o0 << 16);
                dst[1 * F2_VROW / 2] = (e0 >> 16) | (o0 & 0xFFFF0000u);
                dst[2 * F2_VROW / 2] = (e1 & 0xFFFFu) | (o1 << 16);
                dst[3 * F2_VROW / 2] = (e1 >> 16) | (o1 & 0xFFFF0000u);
            }
        }
    };
    // scores of key block kb for this wave's 32 queries: x[r] = kq_scale * half(alpha * q.k (+ ALiBi)), key = 32 kb + row(r)
    // scores of key block kb for this wave's 32 queries:  x[r] = half(alpha * q.k (+ ALiBi)) as float,  key = 32 kb + row(r);
    // masked keys: -inf.  exp(kq_scale * x - max) is then exp2(fma(log2(e) * kq_scale, x, c)) with c = -log2(e) * kq_scale * max.
    // (the kernel is VALU-bound -- ~10 instructions per score and pass against 16 MFMAs per 512 scores -- so the mask is
    // applied only in blocks that reach past the wave's first query, and the exponent is one fma + v_exp_f32)
    const float l2e_kq = 1.44269504088896341f * kq_scale;
    const int full_keys = tw < q_tokens ? min(n_ctx, prefix_len + tw + 1) : 0;   // every query of the wave sees keys below this
    auto scores = [&](int kb, float (&x)[16]) {
        const char *Ks = Ks2[kb & 1];
        f32x16v acc;
#pragma unroll
        for (int r = 0; r < 16; r++) acc[r] = 0.0f;
#pragma unroll
        for (int s2 = 0; s2 < KS; s2++) {
            const half8v kf = *reinterpret_cast<const half8v *>(Ks + (size_t)i * (HD * 2) + (size_t)(((2 * s2 + g) ^ f2_swz<HD>(i)) << 4));
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[s2], acc, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 16; r++) {
            half_t sv = f2h(alpha * acc[r]);
            if (alibi) sv = f2h((float)(32 * kb + (r & 3) + 8 * (r >> 2) + 4 * g) * mk + h2f(sv));
            x[r] = h2f(sv);
        }
        if (32 * kb + 32 > full_keys) {                   // (wave-uniform: only the blocks on the causal edge)
#pragma unroll
            for (int r = 0; r < 16; r++)
                if (32 * kb + (r & 3) + 8 * (r >> 2) + 4 * g >= n_valid) x[r] = -INFINITY;
        }
    };
    auto exp2_fast = [](float v) { return __builtin_amdgcn_exp2f(v); };

    // ---- pass 1: running max / sum of every query over its keys
    float m = -INFINITY, sum = 0.0f;
    kload(0);
    kstage(0);
    kload(min(1, nkb - 1));
    __syncthreads();
    for (int kb = 0; kb < nkb; kb++) {
        kstage((kb + 1) & 1);                // (block kb + 1, or a harmless repeat of the last one)
        kload(min(kb + 2, nkb - 1));
        if (kb < wave_nkb) {
            float x[16];
            scores(kb, x);
            float bm = x[0];
#pragma unroll
            for (int r = 1; r < 16; r++) bm = fmaxf(bm, x[r]);
            if (bm > m) { sum *= exp2_fast(l2e_kq * (m - bm)); m = bm; }             // (m = -inf: sum is 0 and stays 0)
            if (m > -INFINITY) {
                const float c = -l2e_kq * m;
#pragma unroll
                for (int r = 0; r < 16; r++) sum += exp2_fast(__builtin_fmaf(l2e_kq, x[r], c));   // masked: 2^-inf = 0
            }
        }
        __syncthreads();
    }
    float M, inv;
    {
        const float m2 = __shfl_xor(m, 32), s2v = __shfl_xor(sum, 32);
        M = fmaxf(m, m2);
        const float tot = (m > -INFINITY ? sum * exp2_fast(l2e_kq * (m - M)) : 0.0f) + (m2 > -INFINITY ? s2v * exp2_fast(l2e_kq * (m2 - M)) : 0.0f);
        inv = tot > 0.0f ? 1.0f / tot : 0.0f;
    }
    // ---- pass 2: P = half(half(exp(x - M)) / sum) from recomputed scores, O^T += V^T . P^T
    f32x16v oacc[NT];
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int r = 0; r < 16; r++) oacc[nt][r] = 0.0f;
    kload(0);
    vload(0);
    kstage(0);
    vstage(0);
    kload(min(1, nkb - 1));
    vload(min(1, nkb - 1));
    __syncthreads();
    for (int kb = 0; kb < nkb; kb++) {
        kstage((kb + 1) & 1);
        vstage((kb + 1) & 1);
        kload(min(kb + 2, nkb - 1));
        vload(min(kb + 2, nkb - 1));
        if (kb < wave_nkb) {
            const half_t *Vt = Vt2[kb & 1];
            float x[16];
            scores(kb, x);
            half8v pb[2];
            const float c = M > -INFINITY ? -l2e_kq * M : 0.0f;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const half_t e = f2h(exp2_fast(__builtin_fmaf(l2e_kq, x[r], c)));       // masked keys: 2^-inf = 0
                pb[r >> 3][r & 7] = f2h(h2f(e) * inv);
            }
#pragma unroll
            for (int s2 = 0; s2 < 2; s2++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++) {
                    const half8v vf = *reinterpret_cast<const half8v *>(Vt + (size_t)(32 * nt + i) * F2_VROW + 16 * s2 + 8 * g);
                    oacc[nt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, pb[s2], oacc[nt], 0, 0, 0);
                }
        }
        __syncthreads();
    }
    if (tq < q_tokens) {
        half_t *orow = out + ((size_t)tq * heads + h) * HD;
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                typedef _Float16 half4v __attribute__((ext_vector_type(4)));
                half4v o4;
#pragma unroll
                for (int e = 0; e < 4; e++) o4[e] = f2h(oacc[nt][4 * j + e]);
                *reinterpret_cast<half4v *>(orow + 32 * nt + 8 * j + 4 * g) = o4;
            }
    }
}

template <int HD, bool Q8, bool ALIBI>
__global__ void __launch_bounds__(256, 2) k_attention_2pass_ks(const half_t *__restrict__ q, const uint8_t *__restrict__ kc,
                                                         const uint8_t *__restrict__ vc, int n_ctx, int q_tokens,
                                                         int prefix_len, int heads, int kv_heads, float kq_scale,
                                                         int alibi_base, int alibi_total, half_t *__restrict__ out)
{
    static_assert(HD == 128 || HD == 64, "two-pass attention: head_dim 64 / 128");
    constexpr int KS = HD / 16, NT = HD / 32, CHK = HD / 8;
    constexpr int NKC = 32 * CHK / 256;              // 16-byte chunks of the K block per thread
    // 64 queries per workgroup: waves 0 / 1 take the even key blocks for queries 0-31 / 32-63, waves 2 / 3 the odd ones; a
    // stage is TWO key blocks (one barrier per 64 keys), the halves' running max / sum and output tiles meet through LDS
    constexpr int KBYTES = 32 * HD * 2, VHALFS = HD * F2_VROW;
    extern __shared__ __attribute__((aligned(16))) char smem[];                   // [2 stages][2 parities] K blocks, then V blocks
    auto KsP = [&](int buf, int p) { return smem + (size_t)(buf * 2 + p) * KBYTES; };
    auto VtP = [&](int buf, int p) { return reinterpret_cast<half_t *>(smem + (size_t)4 * KBYTES) + (size_t)(buf * 2 + p) * VHALFS; };
    int tile = blockIdx.x, h = blockIdx.y;
    if (heads % 8 == 0) {            // an XCD keeps a fixed eighth of the heads (their K / V in ONE L2); longest tiles first
        const int w = blockIdx.y * gridDim.x + blockIdx.x, xcd = w & 7, r = w >> 3;
        h = (r / (int)gridDim.x) * 8 + xcd;
        tile = (int)gridDim.x - 1 - r % (int)gridDim.x;
    }
    const int t0 = tile * 64;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int qw = wave & 1, kp = wave >> 1;          // query half, key-block parity
    const int i = lane & 31, g = lane >> 5;
    const int kvh = h / (heads / kv_heads);
    const int kv_dim = kv_heads * HD;
    const size_t row_bytes = Q8 ? (size_t)(kv_dim / 32) * 34 : (size_t)kv_dim * 2;
    const int hoff = kvh * HD;
    const int n_keys = min(n_ctx, prefix_len + min(t0 + 64, q_tokens));           // causal bound of the whole tile
    const int nkb = (n_keys + 31) / 32, nit = (nkb + 1) / 2;
    const int tw = t0 + 32 * qw, tq = tw + i;
    const int n_valid = tq < q_tokens ? min(n_ctx, prefix_len + tq + 1) : 0;      // keys this lane's query may see
    const int wave_keys = tw < q_tokens ? min(n_ctx, prefix_len + min(tw + 32, q_tokens)) : 0;
    const int wave_nkb = (wave_keys + 31) / 32;                                   // blocks past it are fully masked for this wave
    const float alpha = 1.0f / sqrtf((float)HD) / kq_scale;
    const float mk = ALIBI ? alibi_slope(h + alibi_base, alibi_total) : 0.0f;

    half8v qf[KS];
    {
        const int tqc = min(tq, q_tokens - 1);
#pragma unroll
        for (int s2 = 0; s2 < KS; s2++)
            qf[s2] = __builtin_bit_cast(half8v, *reinterpret_cast<const u32x4v *>(q + ((size_t)tqc * heads + h) * HD + 16 * s2 + 8 * g));
    }
    // ---- staging: K block rows as they are (swizzled chunks), V block transposed with permuted key columns
    half8v kreg[2][NKC];
    // A pair of whole blocks inside the context: the pair's place is a scalar, a lane's place in it does not change (F16 cache; row by row every request cost a multiplication of 16 cycles)
    auto whole = [&](int itn) { return !Q8 && 64 * itn + 64 <= n_ctx && 2 * itn + 1 < nkb; };
    auto load_at = [&](const uint8_t *base, int row, int c) {
        return __builtin_bit_cast(half8v, *reinterpret_cast<const u32x4v *>(base + ((uint32_t)row * (uint32_t)row_bytes + (uint32_t)(2 * (hoff + 8 * c)))));
    };
    auto kload = [&](int itn) {
        if (whole(itn)) {
            const uint8_t *base = kc + (size_t)(64 * itn) * row_bytes;
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int it = 0; it < NKC; it++) { const int idx = tid + it * 256; kreg[p][it] = load_at(base, 32 * p + idx / CHK, idx % CHK); }
            return;
        }
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const int kb = min(2 * itn + p, nkb - 1);
#pragma unroll
            for (int it = 0; it < NKC; it++) {
                const int idx = tid + it * 256, row = idx / CHK, c = idx % CHK;
                kreg[p][it] = kv_load8<Q8>(kc, row_bytes, min(32 * kb + row, n_ctx - 1), hoff + 8 * c);
            }
        }
    };
    auto kstage = [&](int buf) {
#pragma unroll
        for (int p = 0; p < 2; p++)
#pragma unroll
            for (int it = 0; it < NKC; it++) {
                const int idx = tid + it * 256, row = idx / CHK, c = idx % CHK;
                *reinterpret_cast<half8v *>(KsP(buf, p) + (size_t)row * (HD * 2) + (size_t)((c ^ f2_swz<HD>(row)) << 4)) = kreg[p][it];
            }
    };
    constexpr int KPI = 256 / CHK;           // keys staged per pass of the workgroup
    constexpr int NIT = (32 + KPI - 1) / KPI;
    half8v vreg[2][NIT];
    const int vpar = tid & 1, vpair = (tid >> 1) & 7;
    const int vch = ((tid >> 4) & 3) + 4 * ((tid >> 6) % (CHK / 4));
    const int vkey0 = 16 * ((tid >> 6) / (CHK / 4)) + 2 * vpair;                  // even key of the lane pair within a pass
    auto vload = [&](int itn) {
        if (whole(itn)) {
            const uint8_t *base = vc + (size_t)(64 * itn) * row_bytes;
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int it = 0; it < NIT; it++) vreg[p][it] = load_at(base, 32 * p + min(vkey0 + vpar + it * KPI, 31), vch);
            return;
        }
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const int kb = min(2 * itn + p, nkb - 1);
#pragma unroll
            for (int it = 0; it < NIT; it++) {
                const int key = min(vkey0 + vpar + it * KPI, 31);
                vreg[p][it] = kv_load8<Q8>(vc, row_bytes, min(32 * kb + key, n_ctx - 1), hoff + 8 * vch);
            }
        }
    };
    auto swap1 = [](uint32_t v) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, false); };   // lane ^ 1 (quad_perm [1, 0, 3, 2])
    auto vstage = [&](int buf) {             // lane pairs trade halves of their rows: (even key, odd key) dwords of 4 dims
#pragma unroll
      for (int p = 0; p < 2; p++) {
        half_t *Vt = VtP(buf, p);
#pragma unroll
        for (int it = 0; it < NIT; it++) {
            const u32x4v w = __builtin_bit_cast(u32x4v, vreg[p][it]);
            const uint32_t m0 = vpar ? w[2] : w[0], m1 = vpar ? w[3] : w[1];
            const uint32_t r0 = swap1(vpar ? w[0] : w[2]), r1 = swap1(vpar ? w[1] : w[3]);
            const uint32_t e0 = vpar ? r0 : m0, e1 = vpar ? r1 : m1;              // even key's values
            const uint32_t o0 = vpar ? m0 : r0, o1 = vpar ? m1 : r1;              // odd key's values
            const int key = vkey0 + it * KPI;
            if (key < 32) {
                uint32_t *dst = reinterpret_cast<uint32_t *>(Vt + (size_t)(8 * vch + 4 * vpar) * F2_VROW + f2_col(key));
                dst[0 * F2_VROW / 2] = (e0 & 0xFFFFu) | (o0 << 16);
                dst[1 * F2_VROW / 2] = (e0 >> 16) | (o0 & 0xFFFF0000u);
                dst[2 * F2_VROW / 2] = (e1 & 0xFFFFu) | (o1 << 16);
                dst[3 * F2_VROW / 2] = (e1 >> 16) | (o1 & 0xFFFF0000u);
            }
        }
      }
    };
    // scores of key block kb for this wave's 32 queries: x[r] = kq_scale * half(alpha * q.k (+ ALiBi)), key = 32 kb + row(r)
    // scores of key block kb for this wave's 32 queries:  x[r] = half(alpha * q.k (+ ALiBi)) as float,  key = 32 kb + row(r);
    // masked keys: -inf.  exp(kq_scale * x - max) is then exp2(fma(log2(e) * kq_scale, x, c)) with c = -log2(e) * kq_scale * max.
    // (ALiBi is a template parameter: its test inside the unrolled loop was sixteen branches a block.  Scores and probabilities stay pairs of halves, converted and compared two at a time:
    // 32 heads of 128, 2048 tokens 147 -> 125 -> 120 us, 512 tokens 26 -> 22, 512 behind 1500 82 -> 65)
    // (the kernel is VALU-bound -- ~10 instructions per score and pass against 16 MFMAs per 512 scores -- so the mask is
    // applied only in blocks that reach past the wave's first query, and the exponent is one fma + v_exp_f32)
    const float l2e_kq = 1.44269504088896341f * kq_scale;
    const int full_keys = tw < q_tokens ? min(n_ctx, prefix_len + tw + 1) : 0;   // every query of the wave sees keys below this
    typedef _Float16 f16x2v __attribute__((ext_vector_type(2)));
    typedef float f32x2v __attribute__((ext_vector_type(2)));
    auto pair = [](float a, float b) { return __builtin_convertvector((f32x2v{a, b}), f16x2v); };      // (both rounded to nearest in one instruction)
    auto scores = [&](int kb, int buf, f16x2v (&x)[8]) {
        const char *Ks = KsP(buf, kp);
        f32x16v acc;
#pragma unroll
        for (int r = 0; r < 16; r++) acc[r] = 0.0f;
#pragma unroll
        for (int s2 = 0; s2 < KS; s2++) {
            const half8v kf = *reinterpret_cast<const half8v *>(Ks + (size_t)i * (HD * 2) + (size_t)(((2 * s2 + g) ^ f2_swz<HD>(i)) << 4));
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[s2], acc, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 8; r++) {
            x[r] = pair(alpha * acc[2 * r], alpha * acc[2 * r + 1]);
            if constexpr (ALIBI) {
                const int key = 32 * kb + ((2 * r) & 3) + 8 * (r >> 1) + 4 * g;
                x[r] = pair((float)key * mk + (float)x[r][0], (float)(key + 1) * mk + (float)x[r][1]);
            }
        }
        if (32 * kb + 32 > full_keys) {                   // (wave-uniform: only the blocks on the causal edge)
#pragma unroll
            for (int r = 0; r < 16; r++)
                if (32 * kb + (r & 3) + 8 * (r >> 2) + 4 * g >= n_valid) x[r >> 1][r & 1] = (_Float16)-INFINITY;
        }
    };
    auto exp2_fast = [](float v) { return __builtin_amdgcn_exp2f(v); };

    // ---- pass 1: running max / sum of every query over its keys
    float m = -INFINITY, sum = 0.0f;
    kload(0);
    kstage(0);
    kload(min(1, nit - 1));
    __syncthreads();
    for (int itn = 0; itn < nit; itn++) {
        const int kb = 2 * itn + kp;
        kstage((itn + 1) & 1);               // (the next pair of blocks, or a harmless repeat of the last one)
        kload(min(itn + 2, nit - 1));
        if (kb < wave_nkb && kb < nkb) {
            f16x2v x[8];
            scores(kb, itn & 1, x);
            f16x2v b2 = x[0];
#pragma unroll
            for (int r = 1; r < 8; r++) b2 = __builtin_elementwise_max(b2, x[r]);
            const float bm = fmaxf((float)b2[0], (float)b2[1]);
            if (bm > m) { sum *= exp2_fast(l2e_kq * (m - bm)); m = bm; }             // (m = -inf: sum is 0 and stays 0)
            if (m > -INFINITY) {
                const float c = -l2e_kq * m;
#pragma unroll
                for (int r = 0; r < 16; r++) sum += exp2_fast(__builtin_fmaf(l2e_kq, (float)x[r >> 1][r & 1], c));   // masked: 2^-inf = 0
            }
        }
        __syncthreads();
    }
    float M, inv;
    {
        const float m2 = __shfl_xor(m, 32), s2v = __shfl_xor(sum, 32);
        float Mw = fmaxf(m, m2);
        float totw = (m > -INFINITY ? sum * exp2_fast(l2e_kq * (m - Mw)) : 0.0f) + (m2 > -INFINITY ? s2v * exp2_fast(l2e_kq * (m2 - Mw)) : 0.0f);
        // the two key parities of a query meet through LDS (the staging area is idle between the passes)
        float *ms = reinterpret_cast<float *>(smem);             // [query half][32][2]
        if (kp == 1 && g == 0) { ms[(qw * 32 + i) * 2] = Mw; ms[(qw * 32 + i) * 2 + 1] = totw; }
        __syncthreads();
        M = Mw; inv = 0.0f;
        if (kp == 0) {
            const float m1 = ms[(qw * 32 + i) * 2], t1 = ms[(qw * 32 + i) * 2 + 1];
            M = fmaxf(Mw, m1);
            const float tot = (Mw > -INFINITY ? totw * exp2_fast(l2e_kq * (Mw - M)) : 0.0f) + (m1 > -INFINITY ? t1 * exp2_fast(l2e_kq * (m1 - M)) : 0.0f);
            inv = tot > 0.0f ? 1.0f / tot : 0.0f;
        }
        __syncthreads();
        if (kp == 0 && g == 0) { ms[(qw * 32 + i) * 2] = M; ms[(qw * 32 + i) * 2 + 1] = inv; }
        __syncthreads();
        if (kp == 1) { M = ms[(qw * 32 + i) * 2]; inv = ms[(qw * 32 + i) * 2 + 1]; }
        __syncthreads();
    }
    // ---- pass 2: P = half(half(exp(x - M)) / sum) from recomputed scores, O^T += V^T . P^T
    f32x16v oacc[NT];
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int r = 0; r < 16; r++) oacc[nt][r] = 0.0f;
    kload(0);
    vload(0);
    kstage(0);
    vstage(0);
    kload(min(1, nit - 1));
    vload(min(1, nit - 1));
    __syncthreads();
    for (int itn = 0; itn < nit; itn++) {
        const int kb = 2 * itn + kp;
        kstage((itn + 1) & 1);
        vstage((itn + 1) & 1);
        kload(min(itn + 2, nit - 1));
        vload(min(itn + 2, nit - 1));
        if (kb < wave_nkb && kb < nkb) {
            const half_t *Vt = VtP(itn & 1, kp);
            f16x2v x[8];
            scores(kb, itn & 1, x);
            half8v pb[2];
            const float c = M > -INFINITY ? -l2e_kq * M : 0.0f;
#pragma unroll
            for (int r = 0; r < 8; r++) {
                const f16x2v e = pair(exp2_fast(__builtin_fmaf(l2e_kq, (float)x[r][0], c)), exp2_fast(__builtin_fmaf(l2e_kq, (float)x[r][1], c)));       // masked keys: 2^-inf = 0
                const f16x2v w = pair((float)e[0] * inv, (float)e[1] * inv);
                pb[r >> 2][2 * (r & 3)] = w[0]; pb[r >> 2][2 * (r & 3) + 1] = w[1];
            }
#pragma unroll
            for (int s2 = 0; s2 < 2; s2++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++) {
                    const half8v vf = *reinterpret_cast<const half8v *>(Vt + (size_t)(32 * nt + i) * F2_VROW + 16 * s2 + 8 * g);
                    oacc[nt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, pb[s2], oacc[nt], 0, 0, 0);
                }
        }
        __syncthreads();
    }
    {   // the odd-parity half hands its output tiles over (staging area: idle after the last barrier)
        float *os = reinterpret_cast<float *>(smem);             // [query half][NT][16][64]
        if (kp == 1) {
#pragma unroll
            for (int nt = 0; nt < NT; nt++)
#pragma unroll
                for (int r = 0; r < 16; r++) os[((qw * NT + nt) * 16 + r) * 64 + lane] = oacc[nt][r];
        }
        __syncthreads();
        if (kp == 0) {
#pragma unroll
            for (int nt = 0; nt < NT; nt++)
#pragma unroll
                for (int r = 0; r < 16; r++) oacc[nt][r] += os[((qw * NT + nt) * 16 + r) * 64 + lane];
        }
    }
    if (kp == 0 && tq < q_tokens) {
        half_t *orow = out + ((size_t)tq * heads + h) * HD;
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                typedef _Float16 half4v __attribute__((ext_vector_type(4)));
                half4v o4;
#pragma unroll
                for (int e = 0; e < 4; e++) o4[e] = f2h(oacc[nt][4 * j + e]);
                *reinterpret_cast<half4v *>(orow + 32 * nt + 8 * j + 4 * g) = o4;
            }
    }
}

} // namespace ifa

using namespace ifa;

template <int HD>
static int launch_attention_mfma(const void *q, const void *kcache, const void *vcache, int kv_dtype, int n_ctx, int q_tokens,
                                 int prefix_len, int heads, int kv_heads, float kq_scale, int alibi, int alibi_base,
                                 int alibi_total, void *out, size_t smem, hipStream_t s, half_t *sg_ws = nullptr, int sg_nkp = 0)
{
    dim3 grid((unsigned)((q_tokens + PF_QT - 1) / PF_QT), (unsigned)heads);
#define IFA_PFA(Q8V, SGV) { auto kern = k_attention_mfma<HD, Q8V, SGV>; \
        if (smem > 48 * 1024) IFA_HIP_CHECK(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem)); \
        kern<<<grid, dim3(256), smem, s>>>((const half_t *)q, (const uint8_t *)kcache, (const uint8_t *)vcache, n_ctx, q_tokens, \
                                           prefix_len, heads, kv_heads, kq_scale, alibi, alibi_base, alibi_total, (half_t *)out, sg_ws, sg_nkp); }
    if (kv_dtype == Q8_B32T2) { if (sg_ws) IFA_PFA(true, true) else IFA_PFA(true, false) }
    else { if (sg_ws) IFA_PFA(false, true) else IFA_PFA(false, false) }
#undef IFA_PFA
    IFA_LAUNCH_CHECK();
    return IFA_OK;
}

// workspace of the global-score-tile variant, one per (device, stream), grown on demand (growth synchronises the stream)
namespace {
struct SgWs { void *p = nullptr; size_t bytes = 0; };
std::mutex g_sg_mutex;
std::map<std::pair<int, hipStream_t>, SgWs> g_sg_ws;
}
namespace ifa {
void attn_release_stream(int dev, hipStream_t s)          // called by ifa_gemm_release_stream (ifa_gemm.hip)
{
    std::lock_guard<std::mutex> lock(g_sg_mutex);
    auto it = g_sg_ws.find({dev, s});
    if (it == g_sg_ws.end()) return;
    if (it->second.p) (void)hipFree(it->second.p);
    g_sg_ws.erase(it);
}
}
static int sg_workspace(hipStream_t s, size_t bytes, half_t **out)
{
    int dev = 0;
    IFA_HIP_CHECK(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(g_sg_mutex);
    SgWs &w = g_sg_ws[{dev, s}];
    if (bytes > w.bytes) {
        if (w.p) { IFA_HIP_CHECK(hipStreamSynchronize(s)); IFA_HIP_CHECK(hipFree(w.p)); w.p = nullptr; w.bytes = 0; }
        IFA_HIP_CHECK(hipMalloc(&w.p, bytes));
        w.bytes = bytes;
    }
    *out = (half_t *)w.p;
    return IFA_OK;
}

static int g_attn_2pass_min = 64;        // chunks of at least this many queries take the two-pass kernels (ifa_attention_two_pass_min)
static int g_attn_2pass_min_keys = 1 << 30;      // contexts of at least this many keys: the 128-query variant instead of the 64-query one (never by default;
                                                 // 128 / 256 / 512 / 1024 / 2048 / 4096 tokens: 64-query 11.9 / 16.9 / 27.4 / 60.2 / 165 / 492 us, staged kernel 15.6 / 18.9 / 32.7 / 77 / 334 / 1202,
                                                 // 128-query variant - / - / - / 75 / 175 / 519 -- Llama-2-7B heads, profiles/r02_attention_two_pass.log)

// prompts that k_attention_fresh takes: those that k_attention_mfma would, with two blocks of keys at the most (fewer than four rows: a workgroup a row; 64 and more: the two-pass kernel)
extern "C" bool attention_fresh_fits(int tokens, int head_dim, int rope_order, float partial_rotary_factor)
{
    return tokens >= 4 && tokens < g_attn_2pass_min && tokens <= FR_MAX && head_dim == 128 && (rope_order == 1 || rope_order == 2) && (partial_rotary_factor <= 0 || partial_rotary_factor == 1.0f);
}

extern "C" int ifa_attention_two_pass_min(int min_tokens)
{
    const int prev = g_attn_2pass_min;
    if (min_tokens >= 0) g_attn_2pass_min = min_tokens > 0 ? min_tokens : (1 << 30);
    return prev;
}

extern "C" int ifa_attention_two_pass_min_keys(int min_keys)
{
    const int prev = g_attn_2pass_min_keys;
    if (min_keys >= 0) g_attn_2pass_min_keys = min_keys;
    return prev;
}

extern "C" int ifa_debug_attn_trace(unsigned long long *out8)
{
    IFA_HIP_CHECK(hipMemcpyFromSymbol(out8, HIP_SYMBOL(ifa::g_attn_trace), 64));
    return IFA_OK;
}

// engine-internal: ifa_rope_qk_store and ifa_attention of a prompt from position 0 in one launch (k_attention_fresh); tab: (cos, sin) of [token][head_dim / 2]; IFA_ERR_STATE where the two take
// other kernels or the shape isn't covered (nothing launched)
extern "C" int ifa_attention_fresh(const void *q, const void *k, const void *v, const float *tab, int tokens, int heads, int kv_heads, int head_dim, float kq_scale, int rope_order,
                                   float partial_rotary_factor, void *kcache, void *vcache, size_t cache_row_elems, void *out, ifa_stream stream)
{
    IFA_REQUIRE(q && k && v && tab && kcache && vcache && out, "ifa_attention_fresh: null pointer");
    IFA_REQUIRE(heads > 0 && kv_heads > 0 && heads % kv_heads == 0 && kq_scale > 0, "ifa_attention_fresh: heads %d kv_heads %d", heads, kv_heads);
    if (!attention_fresh_fits(tokens, head_dim, rope_order, partial_rotary_factor) || cache_row_elems % 8
        || (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)tab | (uintptr_t)kcache | (uintptr_t)vcache) & 15)) return IFA_ERR_STATE;
    const dim3 grid((unsigned)((tokens + 31) / 32), (unsigned)heads);
#define IFA_FRESH(O) k_attention_fresh<O><<<grid, dim3(256), 0, ifa_s(stream)>>>((const half_t *)q, (const half_t *)k, (const half_t *)v, tab, tokens, heads, kv_heads, kq_scale, (half_t *)kcache, \
                                                                                 (half_t *)vcache, cache_row_elems, (half_t *)out)
    if (rope_order == 2) IFA_FRESH(2); else IFA_FRESH(1);
#undef IFA_FRESH
    IFA_LAUNCH_CHECK();
    return IFA_OK;
}

// engine-internal: n query rows, each one token on its own KV cache (rows_dev[t]); max_ctx = longest context
extern "C" int ifa_attention_rows(const void *q, const void *rows_dev, int kv_dtype, int n_rows, int max_ctx, int heads, int kv_heads,
                                  int head_dim, float kq_scale, int alibi, int alibi_base_head, int alibi_total_heads, void *out,
                                  ifa_stream stream)
{
    IFA_REQUIRE(q && rows_dev && out && n_rows > 0 && max_ctx > 0, "ifa_attention_rows: bad arguments");
    const size_t smem = (((size_t)max_ctx * 2 + 15) & ~(size_t)15) + 64;
    dim3 grid((unsigned)heads, (unsigned)n_rows);
    const int total_heads = alibi_total_heads > 0 ? alibi_total_heads : heads;
    if (kv_dtype == Q8_B32T2) {
        if (smem > 48 * 1024) IFA_HIP_CHECK(hipFuncSetAttribute((const void *)k_attention<true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
        k_attention<true><<<grid, dim3(256), smem, ifa_s(stream)>>>((const half_t *)q, nullptr, nullptr, max_ctx, n_rows, 0, heads, kv_heads, head_dim, kq_scale,
                                                                    alibi, alibi_base_head, total_heads, (half_t *)out, (const AttnRow *)rows_dev);
    } else {
        if (smem > 48 * 1024) IFA_HIP_CHECK(hipFuncSetAttribute((const void *)k_attention<false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
        k_attention<false><<<grid, dim3(256), smem, ifa_s(stream)>>>((const half_t *)q, nullptr, nullptr, max_ctx, n_rows, 0, heads, kv_heads, head_dim, kq_scale,
                                                                     alibi, alibi_base_head, total_heads, (half_t *)out, (const AttnRow *)rows_dev);
    }
    IFA_LAUNCH_CHECK();
    return IFA_OK;
}

extern "C" int ifa_attention(const void *q, const void *kcache, const void *vcache, int kv_dtype, int n_ctx,
                             int q_tokens, int prefix_len, int heads, int kv_heads, int head_dim, float kq_scale,
                             int alibi, int alibi_base_head, int alibi_total_heads, void *out, ifa_stream stream)
{
    IFA_REQUIRE(q && kcache && vcache && out, "ifa_attention: null pointer");
    IFA_REQUIRE(kv_dtype == F16 || kv_dtype == Q8_B32T2, "ifa_attention: kv dtype %d", kv_dtype);
    IFA_REQUIRE(heads > 0 && kv_heads > 0 && heads % kv_heads == 0, "ifa_attention: heads %d kv_heads %d", heads, kv_heads);
    IFA_REQUIRE(head_dim > 0 && (kv_heads * head_dim) % 32 == 0, "ifa_attention: head_dim %d", head_dim);
    IFA_REQUIRE(n_ctx > 0 && q_tokens > 0 && prefix_len >= 0, "ifa_attention: n_ctx %d q_tokens %d prefix %d", n_ctx, q_tokens, prefix_len);
    IFA_REQUIRE(n_ctx <= 65536 && q_tokens <= 65535, "ifa_attention: context too long for the op-level kernel");
    IFA_REQUIRE(kq_scale > 0, "ifa_attention: kq_scale must be > 0");
    const int total_heads = alibi_total_heads > 0 ? alibi_total_heads : heads;
    // chunks of >= 64 queries: the two-pass kernel with 64 queries per workgroup and the key blocks split over wave pairs
    if (q_tokens >= g_attn_2pass_min && !(q_tokens >= 128 && n_ctx >= g_attn_2pass_min_keys) && (head_dim == 64 || head_dim == 128)) {
        hipStream_t hs = ifa_s(stream);
        dim3 grid((unsigned)((q_tokens + 63) / 64), (unsigned)heads);
        const size_t smem = (size_t)4 * 32 * head_dim * 2 + (size_t)4 * head_dim * F2_VROW * 2;
#define IFA_F2K(HDV, Q8V) { const auto kern = alibi ? k_attention_2pass_ks<HDV, Q8V, true> : k_attention_2pass_ks<HDV, Q8V, false>; \
        if (smem > 48 * 1024) IFA_HIP_CHECK(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem)); \
        kern<<<grid, dim3(256), smem, hs>>>((const half_t *)q, (const uint8_t *)kcache, (const uint8_t *)vcache, n_ctx, q_tokens, \
                                            prefix_len, heads, kv_heads, kq_scale, alibi_base_head, total_heads, (half_t *)out); }
        if (head_dim == 128) { if (kv_dtype == Q8_B32T2) IFA_F2K(128, true) else IFA_F2K(128, false) }
        else { if (kv_dtype == Q8_B32T2) IFA_F2K(64, true) else IFA_F2K(64, false) }
#undef IFA_F2K
        IFA_LAUNCH_CHECK();
        return IFA_OK;
    }
    // the 128-query variant of it (one wave per 32 queries, every wave walks all key blocks): behind the 64-query one at every
    // length measured (4096 tokens: 519 vs 492 us), selectable through ifa_attention_two_pass_min_keys
    if (q_tokens >= 128 && q_tokens >= g_attn_2pass_min && n_ctx >= g_attn_2pass_min_keys && (head_dim == 64 || head_dim == 128)) {
        hipStream_t hs = ifa_s(stream);
        dim3 grid((unsigned)((q_tokens + F2_QT - 1) / F2_QT), (unsigned)heads);
#define IFA_F2A(HDV, Q8V) k_attention_2pass<HDV, Q8V><<<grid, dim3(256), 0, hs>>>((const half_t *)q, (const uint8_t *)kcache, (const uint8_t *)vcache, n_ctx, q_tokens, \
                                                                                 prefix_len, heads, kv_heads, kq_scale, alibi, alibi_base_head, total_heads, (half_t *)out)
        if (head_dim == 128) { if (kv_dtype == Q8_B32T2) IFA_F2A(128, true); else IFA_F2A(128, false); }
        else { if (kv_dtype == Q8_B32T2) IFA_F2A(64, true); else IFA_F2A(64, false); }
#undef IFA_F2A
        IFA_LAUNCH_CHECK();
        return IFA_OK;
    }
    // prefill: MFMA tiles whenever the [32 x n_keys] score tile fits the 160 KiB LDS (~2300 keys)
    const size_t smem_mfma = (size_t)PF_QT * pf_nkp(n_ctx) * 2 + (size_t)head_dim * PF_VROW * 2 + 64;
    if (q_tokens >= 4 && smem_mfma <= 150 * 1024 && (head_dim == 32 || head_dim == 64 || head_dim == 128)) {
        hipStream_t hs = ifa_s(stream);
        switch (head_dim) {
        case 32: return launch_attention_mfma<32>(q, kcache, vcache, kv_dtype, n_ctx, q_tokens, prefix_len, heads, kv_heads, kq_scale, alibi, alibi_base_head, total_heads, out, smem_mfma, hs);
        case 64: return launch_attention_mfma<64>(q, kcache, vcache, kv_dtype, n_ctx, q_tokens, prefix_len, heads, kv_heads, kq_scale, alibi, alibi_base_head, total_heads, out, smem_mfma, hs);
        default: return launch_attention_mfma<128>(q, kcache, vcache, kv_dtype, n_ctx, q_tokens, prefix_len, heads, kv_heads, kq_scale, alibi, alibi_base_head, total_heads, out, smem_mfma, hs);
        }
    }
    if (q_tokens >= 4 && (head_dim == 32 || head_dim == 64 || head_dim == 128)) {
        // longer contexts: the same kernel with its score tiles in a global workspace (the op-level kernel below takes 131 ms
        // per layer for 2048 queries on 4096 keys)
        const int nkp = pf_nkp(n_ctx);
        const size_t tiles = (size_t)((q_tokens + PF_QT - 1) / PF_QT);
        half_t *ws = nullptr;
        int rc = sg_workspace(ifa_s(stream), (size_t)heads * tiles * PF_QT * (size_t)nkp * 2, &ws);
        if (rc) return rc;
        const size_t smem_v = (size_t)head_dim * PF_VROW * 2 + 64;
        hipStream_t hs = ifa_s(stream);
        switch (head_dim) {
        case 32: return launch_attention_mfma<32>(q, kcache, vcache, kv_dtype, n_ctx, q_tokens, prefix_len, heads, kv_heads, kq_scale, alibi, alibi_base_head, total_heads, out, smem_v, hs, ws, nkp);
        case 64: return launch_attention_mfma<64>(q, kcache, vcache, kv_dtype, n_ctx, q_tokens, prefix_len, heads, kv_heads, kq_scale, alibi, alibi_base_head, total_heads, out, smem_v, hs, ws, nkp);
        default: return launch_attention_mfma<128>(q, kcache, vcache, kv_dtype, n_ctx, q_tokens, prefix_len, heads, kv_heads, kq_scale, alibi, alibi_base_head, total_heads, out, smem_v, hs, ws, nkp);
        }
    }
    size_t smem = (((size_t)n_ctx * 2 + 15) & ~(size_t)15) + 64;
    dim3 grid((unsigned)heads, (unsigned)q_tokens);
    if (kv_dtype == Q8_B32T2) {
        if (smem > 48 * 1024)
            IFA_HIP_CHECK(hipFuncSetAttribute((const void *)k_attention<true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
        k_attention<true><<<grid, dim3(256), smem, ifa_s(stream)>>>((const half_t *)q, (const uint8_t *)kcache, (const uint8_t *)vcache, n_ctx, q_tokens, prefix_len, heads, kv_heads, head_dim, kq_scale, alibi, alibi_base_head, alibi_total_heads > 0 ? alibi_total_heads : heads, (half_t *)out);
    } else {
        if (smem > 48 * 1024)
            IFA_HIP_CHECK(hipFuncSetAttribute((const void *)k_attention<false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
        k_attention<false><<<grid, dim3(256), smem, ifa_s(stream)>>>((const half_t *)q, (const uint8_t *)kcache, (const uint8_t *)vcache, n_ctx, q_tokens, prefix_len, heads, kv_heads, head_dim, kq_scale, alibi, alibi_base_head, alibi_total_heads > 0 ? alibi_total_heads : heads, (half_t *)out);
    }
    IFA_LAUNCH_CHECK();
    return IFA_OK;
}
