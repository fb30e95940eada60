// ifa_decode_attn_keys.h -- attention of a batched decode step (one new token for each of several queries, every query on its own cache), a query's keys split over
// workgroups, in ONE launch.
//
// One workgroup of four waves per (head, query, split).  A key's row is read by LPK lanes, 16 bytes (eight dims) a lane, so that a wave's request covers whole rows; the
// score is eight fma a lane and a sum over the LPK lanes (DPP), and the same lanes hold the same dims of the key's V row: scores, exponentials and P.V stay in registers.
// Every group of LPK lanes keeps its own maximum, sum and output (rescaled when the maximum grows); they meet through LDS at the end.  K and V rows of a pass are requested
// before anything else, K rows of the next pass as soon as the scores are formed, V rows as soon as P.V is.  The workgroup of a (query, head) that is done last (a counter
// each: nobody waits) adds the splits up in split order.
// Rounding points: scores are half (alpha q.k), as in k_dec_attn.  A row that is one pass of one workgroup has k_dec_attn's rounded probabilities too; longer ones keep
// probabilities and partial outputs in fp32 until the output is rounded.  (Single-query steps leave int8 codes of the output, which such differences flip: cosine of the
// logits to the one-workgroup kernel 0.9998.  They stay with k_dec_attn and the two split launches.)
//
// Bound by the bytes from about 16 queries on (5.5 TB/s at 32 x 1000 keys), by one chain of dependent requests a workgroup below.  A workgroup a (head, query) before,
// whatever its keys: Llama-2-7B Q4, us a step, before / now -- 2 queries of 60, 500, 1000 keys 1592 / 1600, 1924 / 1720, 2267 / 1804; 8 queries 1762 / 1743, 2190 / 2116,
// 2572 / 2483; 9 queries (288 workgroups on 256 compute units) 2057 / 2041, 2736 / 2488, 3397 / 2872; 32 queries 2939 / 2821, 4311 / 3999, 5897 / 5435.
// Splits of 64 or 128 keys cost their fixed part more often (8 queries of 250 keys 1866 -> 1995), eight waves a workgroup ran out of step with the places on the chip
// (8 x 1000 keys 2483 -> 2820); the split is the slowest grid dimension: with it in the middle the workgroups without keys unbalanced the others (8 x 250 keys 1866 -> 2030).
#pragma once
#include <algorithm>
#include "ifa_host.h"
#include "ifa_decode_attn.h"

namespace ifa {

constexpr int DEC_KEYS_MAX_SPLITS = 32;      // splits of a query's keys (the last workgroup's lanes hold one each)

struct DecKeysWs {
    float *ml;        // [queries][heads][splits][2]: maximum, sum of exponentials
    float *opart;     // [queries][heads][splits][head_dim]
    unsigned *count;  // [queries][heads]: splits whose values are done; 0 between launches
    int nsplits;      // <= DEC_KEYS_MAX_SPLITS
};

constexpr int DEC_KEYS_WAVES = 4;
constexpr int DEC_KEYS_MAX_QUERIES = 32;     // queries of a fused batched step

// Splits of a query's keys: enough that 1536 workgroups could be at work, none of fewer than 256 keys.  (By what a captured step knows: the number of queries, not their
// contexts.  Up to 2048 workgroups: 32 queries of 1000 keys 5435 -> 5580; up to 1024: 9 of 1000 2872 -> 2924.)
inline int dec_keys_splits(int heads, int queries, int max_ctx)
{
    const int by_chip = 1536 / (heads * queries), by_keys = (max_ctx + 255) / 256;
    return std::max(1, std::min(std::min(by_chip, by_keys), DEC_KEYS_MAX_SPLITS));
}

constexpr int dec_keys_lanes(int head_dim) { return head_dim <= 32 ? 4 : (head_dim <= 64 ? 8 : 16); }

template <int HD, bool Q8>
__global__ void __launch_bounds__(64 * DEC_KEYS_WAVES, 3) k_dec_attn_keys(const DecAttnParams P, const DecKeysWs ws)
{
    static_assert(HD % 8 == 0 && HD <= 128 && (!Q8 || HD % 32 == 0), "head size: multiples of 8 up to 128 (Q8 rows: whole 32-blocks)");
    constexpr int NW = DEC_KEYS_WAVES, DG = HD / 8, LPK = dec_keys_lanes(HD), KPI = 64 / LPK;      // pieces of a row, lanes per row (those beyond DG: idle), rows per request of a wave
    constexpr int U = 8, PK = NW * KPI * U;                                     // requests a wave has under way for K and for V, keys per pass
    constexpr int NG = NW * KPI;                                                // lane groups of the workgroup
    __shared__ __attribute__((aligned(16))) half_t qs[HD], kn[HD], vn[HD];
    __shared__ __attribute__((aligned(16))) float og[NG * HD];
    __shared__ float mls[2 * NG];
    __shared__ int last;
    const int h = blockIdx.x, qb = blockIdx.y, sidx = blockIdx.z, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const DecAttnBatchRow br = reinterpret_cast<const DecAttnBatchRow *>(P.batch_rows)[qb];
    const uint8_t *const kc = br.kc, *const vc = br.vc;
    const int n_ctx = br.n_ctx, pos = n_ctx - 1;
    // (powers of two: no divisions in front of the first request)
    int sh = 8;
    while ((ws.nsplits << sh) < n_ctx) sh++;
    const int nsp = (n_ctx + (1 << sh) - 1) >> sh, j0 = sidx << sh, j1 = min(j0 + (1 << sh), n_ctx);
    if (sidx >= nsp) return;                                                   // (fewer splits than there could be: the counter below counts those with keys)
    const int group = P.heads == P.kv_heads ? 1 : P.heads / P.kv_heads, kvh = group == 1 ? h : h / group;
    const bool one = nsp == 1 && n_ctx <= PK;                                  // the whole row in one pass of this workgroup
    const bool has_new = pos < j1;                                             // (the last split with keys)
    const int kv_dim = P.kv_heads * HD;
    const size_t row_bytes = Q8 ? (size_t)(kv_dim / 32) * 34 : (size_t)kv_dim * 2;
    const size_t head_off = Q8 ? (size_t)((kvh * HD) / 32) * 34 : (size_t)kvh * HD * 2;
    const int dg = min(lane & (LPK - 1), DG - 1), gk = lane / LPK;
    const bool dact = (LPK == DG) || (lane & (LPK - 1)) < DG;
    const int jl = wave * KPI + gk;                                            // this lane's key of request u: jb + jl + NW KPI u
    // ---- requests: the new token's values, the step's (cos, sin) pair, then the first pass of K and V
    const half_t *const q_row = P.q + (size_t)qb * P.q_stride, *const kn_row = P.k_new + (size_t)qb * P.q_stride,
                 *const vn_row = P.v_new + (size_t)qb * P.q_stride;
    const int dq = min(tid, HD - 1);
    const half_t q_in = q_row[(size_t)h * HD + dq], k_in = kn_row[(size_t)kvh * HD + dq], v_in = vn_row[(size_t)kvh * HD + dq];
    float rope_c = 1.0f, rope_s = 0.0f;
    {
        const int c = min(tid < HD / 2 ? tid : tid - HD / 2, HD / 2 - 1);
        const float *rt = P.rope_tab ? P.rope_tab + (size_t)qb * HD : reinterpret_cast<const float *>(P.q);      // (a valid dummy address without RoPE)
        typedef float f32x2 __attribute__((ext_vector_type(2)));
        const f32x2 cs = *IFA_GP(f32x2, rt + 2 * c);
        if (P.rope_order != 0) { rope_c = cs[0]; rope_s = cs[1]; }
    }
    u32x4 kf[Q8 ? 1 : U], vf[Q8 ? 1 : U];
    uint32_t ks8[Q8 ? U : 1], kc8[Q8 ? U : 1][2], vs8[Q8 ? U : 1], vc8[Q8 ? U : 1][2];      // Q8: block scale (half bits) and the lane's eight codes
    auto load = [&](const uint8_t *cache, u32x4 (&f)[Q8 ? 1 : U], uint32_t (&s8)[Q8 ? U : 1], uint32_t (&c8)[Q8 ? U : 1][2], int jb) {
        const uint8_t *const base = cache + (size_t)jb * row_bytes + head_off;     // (uniform; 32-bit offsets within a pass)
#pragma unroll
        for (int u = 0; u < U; u++) {
            const uint32_t off = (uint32_t)min(jl + NW * KPI * u, j1 - 1 - jb) * (uint32_t)row_bytes;      // (rows past the split: clamped, weight 0)
            if constexpr (!Q8) f[u] = *IFA_GP(u32x4, base + (off + (uint32_t)dg * 16u));
            else {
                const auto *blk = IFA_GP(uint16_t, base + (off + (uint32_t)(dg / 4) * 34u));
                typedef uint32_t u32x2_a2 __attribute__((ext_vector_type(2), aligned(2)));
                s8[u] = blk[0];
                const u32x2_a2 cw = *IFA_GP(u32x2_a2, blk + 1 + (dg % 4) * 4);
                c8[u][0] = cw[0]; c8[u][1] = cw[1];
            }
        }
    };
    auto value8 = [&](const u32x4 (&f)[Q8 ? 1 : U], const uint32_t (&s8)[Q8 ? U : 1], const uint32_t (&c8)[Q8 ? U : 1][2], int u) {
        if constexpr (!Q8) return __builtin_bit_cast(half8_t, f[u]);
        else {
            const half_t sc = __builtin_bit_cast(half_t, (uint16_t)s8[u]);
            half2_t a, b, c, d;
            q8x4_dequant_h(c8[u][0], half2_t{sc, sc}, a, b); q8x4_dequant_h(c8[u][1], half2_t{sc, sc}, c, d);
            return half8_t{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
        }
    };
    load(kc, kf, ks8, kc8, j0);
    load(vc, vf, vs8, vc8, j0);
    // (LDS only: the barriers do not wait for the rows under way)
    auto sync_lds = []() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    if (tid < HD) { qs[tid] = q_in; kn[tid] = k_in; vn[tid] = v_in; }
    sync_lds();
    if (P.rope_order != 0) {
        if (tid < HD) rope_apply(tid < HD / 2 ? qs : kn, tid < HD / 2 ? tid : tid - HD / 2, rope_c, rope_s, P.rope_order, P.rope_cols);
        sync_lds();
    }
    if (has_new) {      // KV store of the new row (and its Q8 round trip), as in k_dec_attn
        uint8_t *const kw = const_cast<uint8_t *>(kc), *const vw = const_cast<uint8_t *>(vc);
        const bool writer = (h % group) == 0;
        if constexpr (Q8) {
            constexpr int NB = HD / 32;
            for (int b = wave * 2 + (lane >> 5); b < 2 * NB; b += 2 * NW) {
                half_t *src = b < NB ? kn : vn;
                const int bb = b < NB ? b : b - NB, l32 = lane & 31;
                const float val = h2f(src[bb * 32 + l32]);
                const float mx = half_wave_max(fabsf(val));
                const float sc = mx / 127;
                int qv = sc <= 0.000001f ? 0 : (int)roundf(val / sc);
                qv = min(max(qv, -128), 127);
                const half_t sch = f2h(sc);
                if (writer) {
                    uint8_t *blk = (b < NB ? kw : vw) + (size_t)pos * row_bytes + head_off + (size_t)bb * 34;
                    blk[2 + l32] = (uint8_t)(int8_t)qv;
                    if (l32 == 0) *reinterpret_cast<uint16_t *>(blk) = __builtin_bit_cast(uint16_t, sch);
                }
                src[bb * 32 + l32] = f2h((float)qv * h2f(sch));
            }
            sync_lds();
        } else if (writer && tid < HD) {
            reinterpret_cast<half_t *>(kw + (size_t)pos * row_bytes + head_off)[tid] = kn[tid];
            reinterpret_cast<half_t *>(vw + (size_t)pos * row_bytes + head_off)[tid] = vn[tid];
        }
    }
    const half8_t q8 = *reinterpret_cast<const half8_t *>(qs + dg * 8), kn8 = *reinterpret_cast<const half8_t *>(kn + dg * 8), vn8 = *reinterpret_cast<const half8_t *>(vn + dg * 8);
    const float alpha = 1.0f / sqrtf((float)HD) / P.kq_scale;
    const float mk = P.alibi ? alibi_slope(h + P.alibi_base, P.alibi_total) : 0.0f;
    float m = -INFINITY, l = 0.0f, o[8];
#pragma unroll
    for (int e = 0; e < 8; e++) o[e] = 0.0f;
    for (int jb = j0; jb < j1; jb += PK) {
        const bool tail = jb + PK > j1, fresh = has_new && jb + PK > pos;      // (uniform)
        float p[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int j = jb + jl + NW * KPI * u;
            half8_t k8 = value8(kf, ks8, kc8, u);
            if (fresh) { if (j == pos) k8 = kn8; }
            float c = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; e++) c = __builtin_fmaf((float)q8[e], (float)k8[e], c);
            if (!dact) c = 0.0f;                                               // (an idle lane's 0 * inf)
            c += dpp_xor1(c);
            c += dpp_xor2(c);
            if constexpr (LPK >= 8) c += dpp_half_mirror(c);
            if constexpr (LPK >= 16) c += dpp_mirror(c);
            half_t s = f2h(alpha * c);
            if (P.alibi) { const float a = (float)j * mk; s = f2h(a + h2f(s)); }
            p[u] = j < j1 ? P.kq_scale * h2f(s) : -INFINITY;
        }
        load(kc, kf, ks8, kc8, min(jb + PK, j1 - 1));
        if (one) {          // the row's maximum and sum through LDS, probabilities rounded like k_dec_attn's
            float mx = p[0];
#pragma unroll
            for (int u = 1; u < U; u++) mx = fmaxf(mx, p[u]);
            mx = wave_max(mx);
            if (lane == 0) mls[wave] = mx;
            sync_lds();
#pragma unroll
            for (int i = 0; i < NW; i++) mx = fmaxf(mx, mls[i]);
            float ps = 0.0f;
#pragma unroll
            for (int u = 0; u < U; u++) { p[u] = jb + jl + NW * KPI * u < j1 ? expf(p[u] - mx) : 0.0f; ps += p[u]; }
            ps = wave_sum((lane & (LPK - 1)) == 0 ? ps : 0.0f);
            if (lane == 0) mls[NW + wave] = ps;
            sync_lds();
            ps = mls[NW];
#pragma unroll
            for (int i = 1; i < NW; i++) ps += mls[NW + i];
            const float inv = 1.0f / ps;
#pragma unroll
            for (int u = 0; u < U; u++) p[u] = h2f(f2h(h2f(f2h(p[u])) * inv));
        } else {
        float mn = m;
#pragma unroll
        for (int u = 0; u < U; u++) mn = fmaxf(mn, p[u]);
        const float corr = m == mn ? 1.0f : expf(m - mn);
        m = mn;
        // (a score of -inf -- the half's overflow -- weighs nothing, whatever the maximum is; NaN and +inf leave NaN)
        float ps = 0.0f;
#pragma unroll
        for (int u = 0; u < U; u++) { p[u] = p[u] == -INFINITY ? 0.0f : expf(p[u] - mn); ps += p[u]; }
        l = l * corr + ps;
#pragma unroll
        for (int e = 0; e < 8; e++) o[e] *= corr;
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int j = jb + jl + NW * KPI * u;
            half8_t v8 = value8(vf, vs8, vc8, u);
            if (fresh) { if (j == pos) v8 = vn8; }
            if (tail) { if (j >= j1) v8 = half8_t{0, 0, 0, 0, 0, 0, 0, 0}; }   // (0 * inf of a clamped row)
#pragma unroll
            for (int e = 0; e < 8; e++) o[e] = __builtin_fmaf(p[u], (float)v8[e], o[e]);
        }
        load(vc, vf, vs8, vc8, min(jb + PK, j1 - 1));
    }
    // ---- the lane groups' states through LDS; every wave forms the groups' weights (lane i: group i), thread d < HD adds dim d up in group order
    if (dact) {
        float *w = og + (wave * KPI + gk) * HD + dg * 8;
#pragma unroll
        for (int e = 0; e < 8; e += 4) *reinterpret_cast<float4 *>(w + e) = float4{o[e], o[e + 1], o[e + 2], o[e + 3]};
    }
    if (!one && (lane & (LPK - 1)) == 0) { mls[2 * (wave * KPI + gk)] = m; mls[2 * (wave * KPI + gk) + 1] = l; }
    sync_lds();
    auto weights = [&](float mi, float li, float &M, float &L) {               // weight of this lane's state; the common maximum and sum
        M = wave_max(mi);
        const float w = li == 0.0f ? 0.0f : expf(mi - M);
        L = wave_sum(li == 0.0f ? 0.0f : w * li);
        return w;
    };
    float M = 0.0f, L = 1.0f, wg = 1.0f;
    const int lg = min(lane, NG - 1);
    if (!one) wg = weights(lane < NG ? mls[2 * lg] : -INFINITY, lane < NG ? mls[2 * lg + 1] : 0.0f, M, L);
    auto lane_of = [](float v, int i) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), i)); };
    const int dd = min(tid, HD - 1);
    float acc = 0.0f;
#pragma unroll 16
    for (int i = 0; i < NG; i++) acc = __builtin_fmaf(lane_of(wg, i), og[i * HD + dd], acc);
    const size_t slot = (size_t)qb * P.heads + h;
    half_t *const out = P.out + slot * HD;
    if (nsp == 1) {
        if (tid < HD) out[tid] = f2h(one ? acc : acc / L);
        return;
    }
    float *const op = ws.opart + slot * ws.nsplits * HD, *const ml = ws.ml + slot * ws.nsplits * 2;
    if (tid < HD) __hip_atomic_store(op + (size_t)sidx * HD + tid, acc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);          // (past the caches of this XCD)
    if (tid < 2) __hip_atomic_store(ml + 2 * sidx + tid, tid == 0 ? M : L, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                           // (written: the count says so)
    __syncthreads();
    if (tid == 0) last = __hip_atomic_fetch_add(ws.count + slot, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)(nsp - 1) ? 1 : 0;
    __syncthreads();
    if (!last) return;
    if (tid == 0) __hip_atomic_store(ws.count + slot, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int ls = min(lane, nsp - 1);
    const float ms = __hip_atomic_load(ml + 2 * ls, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), lp = __hip_atomic_load(ml + 2 * ls + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    float ov[DEC_KEYS_MAX_SPLITS];
#pragma unroll
    for (int s = 0; s < DEC_KEYS_MAX_SPLITS; s++) {
        if (s % 8 == 0 && s >= nsp) break;                                     // (eight at a time)
        ov[s] = __hip_atomic_load(op + (size_t)min(s, nsp - 1) * HD + dd, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const float wsp = weights(lane < nsp ? ms : -INFINITY, lane < nsp ? lp : 0.0f, M, L);
    acc = 0.0f;
#pragma unroll
    for (int s = 0; s < DEC_KEYS_MAX_SPLITS; s++) {
        if (s % 8 == 0 && s >= nsp) break;
        if (s < nsp) acc = __builtin_fmaf(lane_of(wsp, s), ov[s], acc);
    }
    if (tid < HD) out[tid] = f2h(acc / L);
}

inline int launch_attn_keys(const DecAttnParams &A, DecKeysWs ws, int head_dim, int nsplits, int queries, hipStream_t s)
{
    ws.nsplits = nsplits;
    const dim3 grid((unsigned)A.heads, (unsigned)queries, (unsigned)nsplits), block(64 * DEC_KEYS_WAVES);
    switch (head_dim) {
#define IFA_KEYS(HDV) case HDV: if (A.kv_q8) k_dec_attn_keys<HDV, true><<<grid, block, 0, s>>>(A, ws); else k_dec_attn_keys<HDV, false><<<grid, block, 0, s>>>(A, ws); break;
#define IFA_KEYS_F16(HDV) case HDV: k_dec_attn_keys<HDV, false><<<grid, block, 0, s>>>(A, ws); break;      // (no whole Q8 blocks: an F16 cache only)
    IFA_KEYS(32) IFA_KEYS(64) IFA_KEYS(96) IFA_KEYS(128) IFA_KEYS_F16(48) IFA_KEYS_F16(80)
#undef IFA_KEYS
#undef IFA_KEYS_F16
    default: return ifa_fail(IFA_ERR_ARG, "fused batched attention: head_dim %d", head_dim);
    }
    IFA_LAUNCH_CHECK();
    return IFA_OK;
}

} // namespace ifa
