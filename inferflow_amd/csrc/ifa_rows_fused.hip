// ifa_rows_fused.hip -- what follows the mixers in a layer of PARALLEL wiring, for a step of one token: the shares of the attention joined, the gated norm of
// the recurrent mixer, the gated feed-forward's activation and the three products that add into the residual, in one launch.
// Such a step is bound by its launches: one that does next to nothing takes 4-6 us here, and these were six of the eleven of a layer (33 us; this one 8.9 at width 1024, of them 2 for its 10 MB of weights; 9.8 with the gates, the shares and the residual asked for behind the
// weights).
// A workgroup forms the whole activation row for itself (10-40 KB of operands out of the L2, behind its own weight requests) and its four waves take an
// output row each; a wave's weights (up to 24 KB a row) are asked for before anything else.
#include "ifa_rows_fused.h"

using namespace ifa32;

namespace {

typedef uint32_t u32x4r __attribute__((ext_vector_type(4)));

template <int NP>
__global__ void __launch_bounds__(256) k_row_out(IfaRowOut P)
{
    extern __shared__ float act[];          // [k0 | k1 | k2]
    __shared__ float red[17];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n = min((int)blockIdx.x * 4 + wave, P.N - 1);
    const int e1 = P.k0 + P.k1, kt = e1 + P.k2;
    // The activations' operands are asked for before the weights (requests come back in order: what is asked for first does not wait for the weights).
    constexpr int NU = (NP + 1) / 2;
    float4 o[4], a0[4], gt[NU], up[NU];
    float ss[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int c = 4 * tid + 1024 * j;
        o[j] = a0[j] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (P.k1) o[j] = *reinterpret_cast<const float4 *>(P.o + min(c, P.k1 - 4));
        if (P.k0 && P.nsplit <= 1) a0[j] = *reinterpret_cast<const float4 *>(P.a0 + min(c, P.k0 - 4));
    }
    if (P.k2)
#pragma unroll
        for (int j = 0; j < NU; j++) {
            const int c = min(4 * tid + 1024 * j, P.k2 - 4);
            gt[j] = *reinterpret_cast<const float4 *>(P.gate_up + c); up[j] = *reinterpret_cast<const float4 *>(P.gate_up + P.k2 + c);
        }
    // ... and so are the gates, the norm's weights, the residual and the first 1024 columns' shares: behind the weights each of them was a further trip to the cache
    float4 gv4[4];
    uint2 nw[4];
    if (P.k1)
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (1024 * j < P.k1) {
                const int c = min(4 * tid + 1024 * j, P.k1 - 4);
                gv4[j] = *reinterpret_cast<const float4 *>(P.gate + c);
                if (P.wlen % 4 == 0) nw[j] = *reinterpret_cast<const uint2 *>(P.norm_w + c % P.wlen);
                else {
                    uint32_t u[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) u[e] = P.norm_w[(c + e) % P.wlen];
                    nw[j] = make_uint2(u[0] | (u[1] << 16), u[2] | (u[3] << 16));
                }
            }
    const bool joined = P.k0 && P.nsplit > 1 && P.vdim % 4 == 0;
    float m8[IFA_ROW_OUT_SPLITS], l8[IFA_ROW_OUT_SPLITS], snk8 = -INFINITY;
    float2 v8[IFA_ROW_OUT_SPLITS][2];
    if (joined) {
        const int c = min(4 * tid, P.k0 - 4), h = c / P.vdim;
        const float *src = P.a0 + (size_t)h * P.nsplit * (P.vdim + 2);
#pragma unroll
        for (int s = 0; s < IFA_ROW_OUT_SPLITS; s++) {
            const float *at = src + (size_t)min(s, P.nsplit - 1) * (P.vdim + 2);
            const float2 ml = *reinterpret_cast<const float2 *>(at);
            m8[s] = ml.x; l8[s] = ml.y;
            v8[s][0] = *reinterpret_cast<const float2 *>(at + 2 + c % P.vdim); v8[s][1] = *reinterpret_cast<const float2 *>(at + 4 + c % P.vdim);
        }
        if (P.sink) snk8 = bf2f(P.sink[h]);
    }
    const float xn = P.x[n], l1 = bf2f(P.ls1[n]), l2 = P.k2 ? bf2f(P.ls2[n]) : 0.0f, b2 = P.k2 ? bf2f(P.bias2[n]) : 0.0f;
    __builtin_amdgcn_sched_barrier(0);
    u32x4r w[NP];
#pragma unroll
    for (int p = 0; p < NP; p++) {
        const int pos = min(512 * p + 8 * lane, kt - 8);          // (a piece of 8 lies in one part; past the end: the last one again, not counted)
        const bf16_t *row = pos < P.k0 ? P.w0 + (size_t)n * P.k0 + pos : (pos < e1 ? P.w1 + (size_t)n * P.k1 + (pos - P.k0) : P.w2 + (size_t)n * P.k2 + (pos - e1));
        w[p] = *reinterpret_cast<const u32x4r *>(row);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (P.k0 && P.nsplit <= 1) {
#pragma unroll
        for (int j = 0; j < 4; j++) if (4 * tid + 1024 * j < P.k0) *reinterpret_cast<float4 *>(act + 4 * tid + 1024 * j) = a0[j];
    } else {
        if (joined && 4 * tid < P.k0) {
            float M = snk8;
#pragma unroll
            for (int s = 0; s < IFA_ROW_OUT_SPLITS; s++) M = fmaxf(M, m8[s]);
            float L = P.sink ? expf(snk8 - M) : 0.0f, a[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s = 0; s < IFA_ROW_OUT_SPLITS; s++)
                if (s < P.nsplit) {
                    const float f = m8[s] == -INFINITY ? 0.0f : expf(m8[s] - M);
                    L = fmaf(l8[s], f, L);
                    a[0] = fmaf(v8[s][0].x, f, a[0]); a[1] = fmaf(v8[s][0].y, f, a[1]); a[2] = fmaf(v8[s][1].x, f, a[2]); a[3] = fmaf(v8[s][1].y, f, a[3]);
                }
            *reinterpret_cast<float4 *>(act + 4 * tid) = make_float4(a[0] / L, a[1] / L, a[2] / L, a[3] / L);
        }
        for (int c = joined ? 1024 + tid : tid; c < P.k0; c += 256) {
            const int h = c / P.vdim, d = c % P.vdim;
            const float *src = P.a0 + (size_t)h * P.nsplit * (P.vdim + 2);
            float m[IFA_ROW_OUT_SPLITS], l[IFA_ROW_OUT_SPLITS], v[IFA_ROW_OUT_SPLITS];
#pragma unroll
            for (int s = 0; s < IFA_ROW_OUT_SPLITS; s++) {
                const float *at = src + (size_t)min(s, P.nsplit - 1) * (P.vdim + 2);
                m[s] = at[0]; l[s] = at[1]; v[s] = at[2 + d];
            }
            const float snk = P.sink ? bf2f(P.sink[h]) : -INFINITY;
            float M = snk;
#pragma unroll
            for (int s = 0; s < IFA_ROW_OUT_SPLITS; s++) M = fmaxf(M, m[s]);
            float L = P.sink ? expf(snk - M) : 0.0f, a = 0.0f;
#pragma unroll
            for (int s = 0; s < IFA_ROW_OUT_SPLITS; s++)
                if (s < P.nsplit) {
                    const float f = m[s] == -INFINITY ? 0.0f : expf(m[s] - M);
                    L = fmaf(l[s], f, L); a = fmaf(v[s], f, a);
                }
            act[c] = a / L;
        }
    }
    if (P.k2)
#pragma unroll
        for (int j = 0; j < NU; j++) {
            const int c = 4 * tid + 1024 * j;
            if (c < P.k2)
                *reinterpret_cast<float4 *>(act + e1 + c) = make_float4(gelu_tanh_f(gt[j].x) * up[j].x, gelu_tanh_f(gt[j].y) * up[j].y, gelu_tanh_f(gt[j].z) * up[j].z,
                                                                        gelu_tanh_f(gt[j].w) * up[j].w);
        }
#pragma unroll
    for (int j = 0; j < 4; j++) ss[j] = 4 * tid + 1024 * j < P.k1 ? (o[j].x * o[j].x + o[j].y * o[j].y) + (o[j].z * o[j].z + o[j].w * o[j].w) : 0.0f;
    if (P.k1) {
        const bool whole = P.group == P.k1;
        float all = 0.0f;
        if (whole) all = block_sum((ss[0] + ss[1]) + (ss[2] + ss[3]), red);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int c = 4 * tid + 1024 * j;
            float s = ss[j];
            if (!whole) for (int x = P.group / 8; x > 0; x >>= 1) s += __shfl_xor(s, x, 64);          // (a group: group / 4 lanes side by side)
            if (c < P.k1) {
                const float r = 1.0f / sqrtf((whole ? all : s) / (float)P.group + P.eps);
                const float gv[4] = {gv4[j].x, gv4[j].y, gv4[j].z, gv4[j].w}, ov[4] = {o[j].x, o[j].y, o[j].z, o[j].w};
#pragma unroll
                for (int e = 0; e < 4; e++) act[P.k0 + c + e] = ov[e] * r * bf2f((bf16_t)((e < 2 ? nw[j].x : nw[j].y) >> (16 * (e & 1)))) * (P.gate_act == 0 ? sigmoid_f(gv[e]) : silu_exact(gv[e]));
            }
        }
    }
    __syncthreads();
    const float c0 = l1 * P.s0, c1 = l1 * P.s1;
    float sum = 0.0f;
#pragma unroll
    for (int p = 0; p < NP; p++) {
        const int pos = 512 * p + 8 * lane;
        const float *a = act + min(pos, kt - 8);
        const float4 a0 = *reinterpret_cast<const float4 *>(a), a1 = *reinterpret_cast<const float4 *>(a + 4);
        const float av[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
        float s = 0.0f;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            s = fmaf(av[2 * e], __uint_as_float(w[p][e] << 16), s);
            s = fmaf(av[2 * e + 1], __uint_as_float(w[p][e] & 0xFFFF0000u), s);
        }
        if (pos < kt) sum = fmaf(s, pos < P.k0 ? c0 : (pos < e1 ? c1 : l2), sum);
    }
    sum = wave_sum(sum);
    if (lane == 0 && (int)blockIdx.x * 4 + wave < P.N) P.x[n] = xn + fmaf(l2, b2, sum);
}

} // namespace

bool ifa_row_out_fits(const IfaRowOut &P)
{
    const int kt = P.k0 + P.k1 + P.k2, g4 = P.group / 4;
    if (P.N <= 0 || P.k0 % 8 || P.k1 % 8 || P.k2 % 8 || kt < 8 || kt > 24 * 512 || P.k1 > 4096 || P.k0 > 4096 || (P.k0 && (P.vdim <= 0 || P.k0 % P.vdim))) return false;
    if (P.k1 && P.group != P.k1 && !(P.group % 4 == 0 && g4 >= 1 && g4 <= 64 && (g4 & (g4 - 1)) == 0 && P.k1 % P.group == 0)) return false;
    uintptr_t al = 0;
    if (P.k0) al |= (uintptr_t)P.w0 | (uintptr_t)P.a0;
    if (P.k1) al |= (uintptr_t)P.w1 | (uintptr_t)P.o | (uintptr_t)P.gate | 2 * (uintptr_t)P.norm_w;          // (8 bytes)
    if (P.k2) al |= (uintptr_t)P.w2 | (uintptr_t)P.gate_up;
    return (al & 15) == 0;
}

int ifa_row_out(const IfaRowOut &P, ifa_stream stream)
{
    IFA_REQUIRE(P.x && P.ls1 && ifa_row_out_fits(P) && P.nsplit <= IFA_ROW_OUT_SPLITS, "row_out: bad arguments (%d + %d + %d columns)", P.k0, P.k1, P.k2);
    const int kt = P.k0 + P.k1 + P.k2;
    const dim3 grid(ifa_cdiv((size_t)P.N, 4));
#define IFA_RO(NP) hipLaunchKernelGGL(k_row_out<NP>, grid, dim3(256), (size_t)kt * 4, ifa_s(stream), P)
    if (kt <= 6 * 512) IFA_RO(6); else if (kt <= 10 * 512) IFA_RO(10); else if (kt <= 14 * 512) IFA_RO(14); else if (kt <= 19 * 512) IFA_RO(19); else IFA_RO(24);
#undef IFA_RO
    IFA_LAUNCH_CHECK();
    return IFA_OK;
}
