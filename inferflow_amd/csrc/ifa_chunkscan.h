// ifa_chunkscan.h -- what the launches of chunked recurrences (ifa_chunkscan.hip, where the form is described) are made of: the decayed linear attention's run beside the windowed
// attention's in launches that both share (ifa_attn_window.hip)
#pragma once
#include "ifa_host.h"
#include "ifa_f32_common.h"

namespace ifachunk {

using namespace ifa32;

constexpr int CL = 64;          // tokens of a chunk
typedef float f32x16c __attribute__((ext_vector_type(16)));
typedef float f32x4c __attribute__((ext_vector_type(4)));
typedef double f64x4c __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(3))) float lds_f32;
typedef const __attribute__((address_space(3))) f32x4c lds_f32x4;

struct ChunkArgs {
    const float *q, *k, *v; size_t ldq, ldk, ldv;
    int heads, qk_heads, dk, dv;
    const float *decay_head, *decay_row, *beta_row;      // kind 0: [heads]; kind 1: [rows][heads] each, decays in (0, 1]
    const SeqDesc *seqs; int n_seqs; float *const *slot_base; size_t state_off;
    float *out; size_t ldo;
    float *st;           // [chunks][heads][dk][dv]: what a chunk adds to the state, then the state before it
    float *u, *w;        // kind 1: [chunks][heads][64][dv], [chunks][heads][64][dk]
    float *dec;          // kind 1: [chunks][heads][CL + 4]: G_last / G_j per position (0 past the end), then G_last
};
constexpr int DEC = CL + 4;

// the step's chunk `id`: its sequence, its number there
__device__ __forceinline__ bool chunk_seq(const ChunkArgs &A, int id, SeqDesc &sd, int &c)
{
    for (int s = 0; s < A.n_seqs; s++) {
        sd = A.seqs[s];
        const int n = (sd.n + CL - 1) / CL;
        if (id < n) { c = id; return true; }
        id -= n;
    }
    return false;
}

// d^n, n <= 64, by squaring in double
__device__ __forceinline__ double power(double d, int n)
{
    double r = 1.0;
#pragma unroll
    for (int b = 0; b < 7; b++) { if (n & (1 << b)) r *= d; d *= d; }
    return r;
}

// e^x for a difference of double sums, within a rounding of the float result (expf's own error, up to two of them, would be in every decay): e^r of the
// remainder |r| <= ln 2 / 2 as its power series up to r^8 / 8! (the rest is below 2.1e-10), in double
__device__ __forceinline__ float exp_of(double x)
{
    const double n = rint(x * 1.4426950408889634), r = fma(n, -0.6931471805599453, x);
    double p = 1.0 / 40320.0;
    p = fma(p, r, 1.0 / 5040.0); p = fma(p, r, 1.0 / 720.0); p = fma(p, r, 1.0 / 120.0); p = fma(p, r, 1.0 / 24.0);
    p = fma(p, r, 1.0 / 6.0); p = fma(p, r, 0.5); p = fma(p, r, 1.0); p = fma(p, r, 1.0);
    return ldexpf((float)p, (int)n);
}

// lane t: the logarithms of the decays of positions 0 .. t of the chunk, summed (none past its end; a decay that has underflowed counts as e^-200, NaN stays)
__device__ __forceinline__ double log_decay_upto(const ChunkArgs &A, const SeqDesc &sd, int t0, int n, int h, int lane)
{
    double l = lane < n ? log((double)A.decay_row[(size_t)(sd.row0 + t0 + lane) * A.heads + h]) : 0.0;
    l = l < -200.0 ? -200.0 : l;
#pragma unroll
    for (int k = 1; k < 64; k <<= 1) { const double x = __shfl_up(l, k, 64); if (lane >= k) l += x; }
    return l;
}

// ---- kind 0, first launch: what the chunk adds, sum_j d^(n - 1 - j) k_j v_j^T.  256 threads for chunk `at` of the step, head h and 64 value columns, a wave per 32 x 32 tiles
__device__ __forceinline__ void linear_chunk(const ChunkArgs &A, int at, int h, int cols)
{
    __shared__ float pw[CL];
    SeqDesc sd; int c;
    if (!chunk_seq(A, at, sd, c)) return;
    const int kh = h / (A.heads / A.qk_heads), tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i = lane & 31, g = lane >> 5;
    const int t0 = c * CL, n = min(CL, sd.n - t0), c0 = cols * 64 + (wave & 1) * 32;
    if (tid < CL) pw[tid] = (float)power((double)A.decay_head[h], tid);
    __syncthreads();
    if (c0 >= A.dv) return;
    const float *kp = A.k + (size_t)(sd.row0 + t0) * A.ldk + (size_t)kh * A.dk, *vp = A.v + (size_t)(sd.row0 + t0) * A.ldv + (size_t)h * A.dv + c0;
    float vr[CL / 2];
#pragma unroll
    for (int s = 0; s < CL / 2; s++) { const float x = vp[(size_t)min(2 * s + g, n - 1) * A.ldv + i]; vr[s] = 2 * s + g < n ? x : 0.0f; }
    for (int kt = (wave >> 1) * 32; kt < A.dk; kt += 64) {
        f32x16c acc;
#pragma unroll
        for (int r = 0; r < 16; r++) acc[r] = 0.0f;
        float kr[CL / 2];
#pragma unroll
        for (int s = 0; s < CL / 2; s++) { const int j = 2 * s + g; const float x = kp[(size_t)min(j, n - 1) * A.ldk + kt + i]; kr[s] = j < n ? x * pw[n - 1 - j] : 0.0f; }
#pragma unroll
        for (int s = 0; s < CL / 2; s++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(kr[s], vr[s], acc, 0, 0, 0);
        float *dst = A.st + (((size_t)at * A.heads + h) * A.dk + kt) * A.dv + c0 + i;
#pragma unroll
        for (int r = 0; r < 16; r++) dst[(size_t)((r & 3) + 8 * (r >> 2) + 4 * g) * A.dv] = acc[r];
    }
}

// ---- kind 0, second launch: the state before every chunk, a thread for element e of head h's in sequence seq
__device__ __forceinline__ void linear_pass(const ChunkArgs &A, int e, int h, int seq)
{
    const size_t per = (size_t)A.dk * A.dv;
    if ((size_t)e >= per) return;
    int first = 0;
    for (int s = 0; s < seq; s++) first += (A.seqs[s].n + CL - 1) / CL;
    const SeqDesc sd = A.seqs[seq];
    const int nc = (sd.n + CL - 1) / CL;
    const double d = (double)A.decay_head[h];
    const float whole = (float)power(d, CL), part = (float)power(d, sd.n - (nc - 1) * CL);
    // (a pointer from a table in memory: unless it is said to be global, its accesses wait for everything under way)
    __attribute__((address_space(1))) float *state = (__attribute__((address_space(1))) float *)(A.slot_base[sd.slot] + A.state_off + (size_t)h * per + e);
    float S = sd.pos0 > 0 ? *state : 0.0f;
    float *p = A.st + ((size_t)first * A.heads + h) * per + e;
    const size_t step = (size_t)A.heads * per;
    for (int c0 = 0; c0 < nc; c0 += 8) {
        float u[8];
#pragma unroll
        for (int x = 0; x < 8; x++) u[x] = p[(size_t)min(c0 + x, nc - 1) * step];
#pragma unroll
        for (int x = 0; x < 8; x++)
            if (c0 + x < nc) { p[(size_t)(c0 + x) * step] = S; S = fmaf(S, c0 + x == nc - 1 ? part : whole, u[x]); }
    }
    *state = S;
}

// ---- third launch: the outputs of a chunk.  256 threads for chunk `id` of the step, head h and 64 value columns, four waves of 16 positions.  The products are transposed: scores K Q^T and
// outputs U^T P^T, so that a lane's accumulators hold four keys of its position and are the second product's operand as they are.  A lane's 16 bytes of a row of S
// or U are columns 4 i .. 4 i + 3: column e of each goes to tile e, so that its outputs are 16 bytes side by side again.
// The scores are summed in 64 bits: q . k of unit vectors is small against its terms, and in 32 bits its rounding was most of the outputs' error.  Everything else
// is summed 16 terms at a time.  (Three workgroups on a compute unit: 168 registers.  Error against 64 bits, rms, and time: see the top.)  VEC: rows of U or v of whole aligned 16 bytes.
constexpr int chunk_out_waves(int kind, int dk) { return kind == 0 && dk == 128 ? 2 : 3; }          // waves a SIMD
template <int KIND, int DK, bool VEC>
__device__ __forceinline__ void chunk_out(const ChunkArgs &A, int id, int h, int cols)
{
    __shared__ double L[4][CL];
    __shared__ float pw[4][CL + 1];
    SeqDesc sd; int c;
    if (!chunk_seq(A, id, sd, c)) return;
    const int kh = h / (A.heads / A.qk_heads), lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), i = lane & 15, g = lane >> 4;
    const int t0 = c * CL, n = min(CL, sd.n - t0), pos = 16 * wave + i, c0 = cols * 64, cl = min(c0 + 4 * i, A.dv - 4);
    if (16 * wave >= n) return;
    // (a table per wave: nothing to wait for but its own writes)
    if (KIND == 0) {
        const double d = (double)A.decay_head[h];
        pw[wave][lane] = (float)power(d, lane);
        if (lane == 0) pw[wave][CL] = (float)power(d, CL);
    } else L[wave][lane] = log_decay_upto(A, sd, t0, n, h, lane);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const float *qp = A.q + (size_t)(sd.row0 + t0 + min(pos, n - 1)) * A.ldq + (size_t)kh * DK + 4 * g, *kp = A.k + (size_t)(sd.row0 + t0) * A.ldk + (size_t)kh * DK + 4 * g;
    const size_t at = (size_t)id * A.heads + h;
    const float *up = KIND == 0 ? A.v + (size_t)(sd.row0 + t0) * A.ldv + (size_t)h * A.dv : A.u + at * CL * A.dv;
    const size_t ldu = KIND == 0 ? A.ldv : (size_t)A.dv;
    auto row4 = [&](const float *p) -> f32x4c {
        if constexpr (VEC) return *(const f32x4c *)p;
        else return f32x4c{p[0], p[1], p[2], p[3]};
    };
    f32x4c q[DK / 16], o[4];
#pragma unroll
    for (int s = 0; s < DK / 16; s++) q[s] = *(const f32x4c *)(qp + 16 * s);
#pragma unroll
    for (int t = 0; t < 4; t++) o[t] = f32x4c{0.f, 0.f, 0.f, 0.f};
    auto add16 = [&](const f32x4c (&a)[4], const f32x4c &b) {          // o += 16 terms, four of them per product
        f32x4c part[4];
#pragma unroll
        for (int t = 0; t < 4; t++) part[t] = f32x4c{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int t = 0; t < 4; t++) part[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e][t], b[e], part[t], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < 4; t++) o[t] += part[t];
    };
    auto not_finite = [&](const f32x4c (&a)[4]) {
        float z = 0.0f;
#pragma unroll
        for (int r = 0; r < 4; r++) z += (a[r][0] * 0.0f + a[r][1] * 0.0f) + (a[r][2] * 0.0f + a[r][3] * 0.0f);
        return z != 0.0f;          // (0, or NaN from any of them)
    };
    const float *st = A.st + at * DK * A.dv + cl;
#pragma unroll
    for (int s = 0; s < DK / 16; s++) {
        f32x4c a[4];
#pragma unroll
        for (int e = 0; e < 4; e++) a[e] = *(const f32x4c *)(st + (size_t)(16 * s + 4 * g + e) * A.dv);
        add16(a, q[s]);
    }
    const double Li = KIND == 1 ? L[wave][pos] : 0.0;
    const float gam = KIND == 0 ? pw[wave][pos + 1] : exp_of(Li);
#pragma unroll
    for (int t = 0; t < 4; t++) o[t] *= gam;
    for (int kt = 0; kt <= wave; kt++) {
        f64x4c p = {0.0, 0.0, 0.0, 0.0};          // keys 16 kt + 4 r + g of the lane's position
        const float *kr = kp + (size_t)min(16 * kt + i, n - 1) * A.ldk;
        f32x4c u[4], w;
#pragma unroll
        for (int r = 0; r < 4; r++) u[r] = row4(up + (size_t)min(16 * kt + 4 * r + g, n - 1) * ldu + cl);
#pragma unroll
        for (int s = 0; s < DK / 16; s++) {
            const f32x4c k = *(const f32x4c *)(kr + 16 * s);
#pragma unroll
            for (int e = 0; e < 4; e++) p = __builtin_amdgcn_mfma_f64_16x16x4f64((double)k[e], (double)q[s][e], p, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int j = 16 * kt + 4 * r + g;
            w[r] = j <= pos ? (float)(p[r] * (double)(KIND == 0 ? pw[wave][max(pos - j, 0)] : exp_of(Li - L[wave][j]))) : 0.0f;
        }
        if (kt == wave && __builtin_amdgcn_ballot_w64(not_finite(u))) {
            // among the wave's own positions a later row has weight 0, which would turn infinities and NaN in it into NaN here: the rows one by one, up to the position's own
#pragma unroll 1
            for (int j = 0; j < 16; j++) {
                const float wj = __shfl(j < 8 ? (j < 4 ? w[0] : w[1]) : (j < 12 ? w[2] : w[3]), i + 16 * (j & 3), 64);
                const float *v = up + (size_t)min(16 * kt + j, n - 1) * ldu;
#pragma unroll
                for (int y = 0; y < 4; y++) {
                    const f32x4c x = row4(v + min(c0 + 16 * g + 4 * y, A.dv - 4));
#pragma unroll
                    for (int t = 0; t < 4; t++) o[t][y] = j <= i ? fmaf(wj, x[t], o[t][y]) : o[t][y];
                }
            }
        } else add16(u, w);
    }
    if (pos >= n) return;
    float *dst = A.out + (size_t)(sd.row0 + t0 + pos) * A.ldo + (size_t)h * A.dv + c0 + 16 * g;
#pragma unroll
    for (int r = 0; r < 4; r++)
        if (c0 + 16 * g + 4 * r < A.dv) *(f32x4c *)(dst + 4 * r) = f32x4c{o[0][r], o[1][r], o[2][r], o[3][r]};
}

} // namespace ifachunk

// ifa_state_chunked_f32's arguments, checked; chunks: of the step.  (seqs: host)
int ifa_chunk_args(ifachunk::ChunkArgs *out, size_t *n_chunks, int kind, const void *q_f32, size_t ldq, const void *k_f32, size_t ldk, const void *v_f32, size_t ldv, int heads, int qk_heads,
                   int dk, int dv, const void *decay_head_f32, const void *decay_row_f32, const void *beta_row_f32, const void *seqs_dev, const void *seqs_host, int n_seqs,
                   void *const *slot_base_dev, size_t state_off, void *ws, size_t ws_bytes, void *out_f32, size_t ldo);
// the second launch of kind 0 by itself
void ifa_linear_pass(const ifachunk::ChunkArgs &A, ifa_stream stream);
