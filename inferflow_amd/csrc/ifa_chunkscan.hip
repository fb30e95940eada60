// ifa_chunkscan.hip -- the state recurrences of the layer-list models over whole prompts, 64 tokens at a time, in 32-bit floats on the matrix cores:
//   kind 0  decayed linear attention   S <- d_h S + k v^T;                                        o = S^T q
//   kind 1  gated delta rule           S <- g S; u = beta (v - S^T k); S <- S + k u^T;            o = S^T q
// Token by token (k_state_scan_reg, ifa_seqmix.hip) a prompt is one chain of dependent steps -- 559 us per 2048 tokens and layer for kind 0 with keys of 64,
// 1033 us for kind 1 with keys of 128 -- on waves that are alone on their SIMDs.  Inside a chunk the recurrence is a set of products
// (positions i, j of the chunk, G_i = product of the decays up to i, S the state before the chunk):
//   kind 0: u = v.   kind 1: u_i + beta_i sum_{j < i} (G_i / G_j)(k_i . k_j) u_j = beta_i (v_i - G_i S^T k_i),
//     a triangular system whose solution is U = U0 - W S with U0, W the solutions for the right hand sides beta V and beta G K: both before S is known
//   o_i = G_i S^T q_i + sum_{j <= i} (G_i / G_j)(q_i . k_j) u_j;     S' = G_last S + sum_j (G_last / G_j) k_j u_j^T
// so three launches do it: what a chunk needs no state for (all chunks at once), the states from chunk to chunk, the outputs (all chunks at once).
// Now 60 us (25 + 10 + 25) and 192 us (33 + 114 + 45) per 2048 tokens and layer of 16 heads; at 601 tokens of 8 heads 27 and 81 (were 159 and 312).  The first and
// third launches wait for their operands (no staging: each is read by one or two waves), the second for its chain.
// Keys of 64 and 128 have instances here; other sizes go token by token.
// fp32 operands; a sum that would leave more error than the token-by-token form's few additions do is formed in 64 bits (scores, states of kind 1), from zero in short
// pieces (the others), and decays are rounded to float once, from double.  Error against 64 bits, rms, 601 tokens: kind 0 1.8e-7 (token by token 3.5e-7), its state 1.7e-7
// (4.2e-7); kind 1 7.8e-8 (1.08e-7), its state 6.0e-8 (8.1e-8).  With one fp32 chain per sum kind 1 had 2.6e-7 and 1.4e-7 (75 us).
#include <utility>
#include "ifa_host.h"
#include "ifa_f32_common.h"
#include "inferflow_amd.h"

using namespace ifa32;

namespace {

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

// ---- kind 0, first launch: what the chunk adds, sum_j d^(n - 1 - j) k_j v_j^T.  grid (chunks, heads, 64 value columns), a wave per 32 x 32 tiles
__global__ void __launch_bounds__(256) k_linear_chunk(ChunkArgs A)
{
    __shared__ float pw[CL];
    SeqDesc sd; int c;
    if (!chunk_seq(A, blockIdx.x, sd, c)) return;
    const int h = blockIdx.y, kh = h / (A.heads / A.qk_heads), tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i = lane & 31, g = lane >> 5;
    const int t0 = c * CL, n = min(CL, sd.n - t0), c0 = blockIdx.z * 64 + (wave & 1) * 32;
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
        float *dst = A.st + (((size_t)blockIdx.x * A.heads + h) * A.dk + kt) * A.dv + c0 + i;
#pragma unroll
        for (int r = 0; r < 16; r++) dst[(size_t)((r & 3) + 8 * (r >> 2) + 4 * g) * A.dv] = acc[r];
    }
}

// ---- kind 0, second launch: the state before every chunk, a thread per element of it; grid (dk dv / 256, heads, sequences)
__global__ void __launch_bounds__(256) k_linear_pass(ChunkArgs A)
{
    const int h = blockIdx.y, e = blockIdx.x * 256 + threadIdx.x;
    const size_t per = (size_t)A.dk * A.dv;
    if ((size_t)e >= per) return;
    int first = 0;
    for (int s = 0; s < (int)blockIdx.z; s++) first += (A.seqs[s].n + CL - 1) / CL;
    const SeqDesc sd = A.seqs[blockIdx.z];
    const int nc = (sd.n + CL - 1) / CL;
    const double d = (double)A.decay_head[h];
    const float whole = (float)power(d, CL), part = (float)power(d, sd.n - (nc - 1) * CL);
    float *state = A.slot_base[sd.slot] + A.state_off + (size_t)h * per + e;
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

// x_T = A_TT (x_T - sum_{j < T} A_Tj x_j), for T = 0, 1, ...: straight-line code, x in registers; `rows`: A's place in LDS
template <int T>
__device__ __forceinline__ void solve_row(float (&x)[CL], uint32_t &rows)
{
    asm volatile("" : "+v"(rows));          // (A's rows are read one by one as they are needed, not all ahead of everything)
    f32x4c s = {0.f, 0.f, 0.f, 0.f};          // (four sums from zero: one chain from x_T on rounded every term to the size of x_T)
    float beta = 0.0f;
#pragma unroll
    for (int j = 0; j <= T; j += 4) {
        const f32x4c a = *(lds_f32x4 *)(uintptr_t)(rows + (T * (CL + 4) + j) * 4);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            if (j + e < T) s[e] = fmaf(a[e], x[j + e], s[e]);
            if (j + e == T) beta = a[e];
        }
    }
    x[T] = beta * (x[T] - ((s[0] + s[1]) + (s[2] + s[3])));
}
template <int... T>
__device__ __forceinline__ void solve_rows(float (&x)[CL], uint32_t rows, std::integer_sequence<int, T...>) { (solve_row<T>(x, rows), ...); }

// ---- kind 1, first launch: U0 and W of a chunk.  grid (chunks, heads).  A_ij = (G_i / G_j)(k_i . k_j), j < i, and A_ii = beta_i in LDS; then a thread per column of
// [V | G K] solves x_i = beta_i (column_i - sum_{j < i} A_ij x_j) forwards, x in registers, A's rows read by all threads alike (2080 multiply-adds per thread)
__global__ void __launch_bounds__(256) k_delta_chunk(ChunkArgs A)
{
    __shared__ __attribute__((aligned(16))) float Am[CL][CL + 4];
    __shared__ double L[CL];
    __shared__ float beta[CL], gam[CL];
    SeqDesc sd; int c;
    if (!chunk_seq(A, blockIdx.x, sd, c)) return;
    const int h = blockIdx.y, kh = h / (A.heads / A.qk_heads), tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i = lane & 31, g = lane >> 5;
    const int t0 = c * CL, n = min(CL, sd.n - t0);
    const float *kp = A.k + (size_t)(sd.row0 + t0) * A.ldk + (size_t)kh * A.dk, *vp = A.v + (size_t)(sd.row0 + t0) * A.ldv + (size_t)h * A.dv;
    if (wave == 0) {
        const double l = log_decay_upto(A, sd, t0, n, h, lane), all = __shfl(l, 63, 64);
        L[lane] = l;
        gam[lane] = exp_of(l);
        beta[lane] = lane < n ? A.beta_row[(size_t)(sd.row0 + t0 + lane) * A.heads + h] : 0.0f;
        float *dec = A.dec + ((size_t)blockIdx.x * A.heads + h) * DEC;
        dec[lane] = lane < n ? exp_of(all - l) : 0.0f;
        if (lane == 0) dec[CL] = exp_of(all);
    }
    __syncthreads();
    const int wi = wave >> 1, wj = wave & 1;          // a 32 x 32 tile of k_i . k_j per wave, 16 columns summed by themselves at a time
    f32x16c acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.0f;
    if (wi >= wj) {
        const float *ri = kp + (size_t)min(32 * wi + i, n - 1) * A.ldk + 4 * g, *rj = kp + (size_t)min(32 * wj + i, n - 1) * A.ldk + 4 * g;
        for (int s0 = 0; s0 < A.dk; s0 += 64)
#pragma unroll
            for (int s = s0; s < s0 + 64; s += 16) {
                f32x16c part;
#pragma unroll
                for (int r = 0; r < 16; r++) part[r] = 0.0f;
#pragma unroll
                for (int u = 0; u < 16; u += 8) {
                    const f32x4c a = *(const f32x4c *)(ri + s + u), b = *(const f32x4c *)(rj + s + u);
#pragma unroll
                    for (int e = 0; e < 4; e++) part = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], b[e], part, 0, 0, 0);
                }
#pragma unroll
                for (int r = 0; r < 16; r++) acc[r] += part[r];
            }
    }
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int row = 32 * wi + (r & 3) + 8 * (r >> 2) + 4 * g, col = 32 * wj + i;
        Am[row][col] = col == row ? beta[row] : (col < row && row < n ? exp_of(L[row] - L[col]) * acc[r] : 0.0f);
    }
    __syncthreads();
    for (int col = tid; col < A.dv + A.dk; col += 256) {
        const bool is_v = col < A.dv;
        const float *src = is_v ? vp + col : kp + col - A.dv;
        const size_t ld = is_v ? A.ldv : A.ldk;
        uint32_t rows = (uint32_t)(uintptr_t)(lds_f32 *)&Am[0][0];
        float x[CL];
#pragma unroll
        for (int t = 0; t < CL; t++) x[t] = src[(size_t)min(t, n - 1) * ld];
#pragma unroll
        for (int t = 0; t < CL; t++) x[t] = t < n ? (is_v ? x[t] : x[t] * gam[t]) : 0.0f;
        solve_rows(x, rows, std::make_integer_sequence<int, CL>());
        const size_t at = (size_t)blockIdx.x * A.heads + h;
        float *dst = is_v ? A.u + at * CL * A.dv + col : A.w + at * CL * A.dk + col - A.dv;
        const size_t lds = is_v ? A.dv : A.dk;
#pragma unroll
        for (int t = 0; t < CL; t++) dst[(size_t)t * lds] = x[t];
    }
}

// LDS written before is read behind it; requests to memory stay in flight across it
__device__ __forceinline__ void lds_barrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// ---- kind 1, second launch: the states from chunk to chunk.  The columns of a state do not meet: a workgroup of four waves per head and 16 of them,
// grid (heads dv / 16, sequences), walks the chunks.  Per chunk U = U0 - W S (a wave: 16 positions) and S' = G_last S + K~^T U (a wave: DK / 4 rows); S
// and U pass through LDS, the next chunk's operands are asked for a chunk ahead.  The chain is two groups of DK / 4 and 16 DK / 64 products long.
template <int DK>
__global__ void __launch_bounds__(256) k_delta_pass(ChunkArgs A)
{
    constexpr int TK = DK / 64, LS = 20;          // 16-row tiles of the state per wave; LDS row of 16 columns (lanes 16 apart read rows 4 apart: distinct banks)
    __shared__ float Sb[DK * LS], Ub[CL * LS];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i = lane & 15, g = lane >> 4;
    const int per_head = A.dv / 16, h = blockIdx.x / per_head, c0 = (blockIdx.x % per_head) * 16, kh = h / (A.heads / A.qk_heads);
    int first = 0;
    for (int s = 0; s < (int)blockIdx.y; s++) first += (A.seqs[s].n + CL - 1) / CL;
    const SeqDesc sd = A.seqs[blockIdx.y];
    const int nc = (sd.n + CL - 1) / CL;
    float *state = A.slot_base[sd.slot] + A.state_off + (size_t)h * DK * A.dv + c0 + i;
    const float *kp = A.k + (size_t)sd.row0 * A.ldk + (size_t)kh * DK + i;
    f32x4c S[TK];
#pragma unroll
    for (int t = 0; t < TK; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) S[t][r] = sd.pos0 > 0 ? state[(size_t)((wave * TK + t) * 16 + 4 * r + g) * A.dv] : 0.0f;
    f32x4c wr[DK / 16], dr[4];
    float kr[TK][16], ur[4], last;
    auto request_w = [&](int c) {
        const size_t at = (size_t)(first + c) * A.heads + h;
        const float *w = A.w + (at * CL + 16 * wave + i) * DK + 4 * g, *u = A.u + (at * CL + 16 * wave + 4 * g) * A.dv + c0 + i;
#pragma unroll
        for (int s = 0; s < DK / 16; s++) wr[s] = *(const f32x4c *)(w + 16 * s);
#pragma unroll
        for (int r = 0; r < 4; r++) ur[r] = u[(size_t)r * A.dv];
    };
    auto request_k = [&](int c) {
        const float *dec = A.dec + ((size_t)(first + c) * A.heads + h) * DEC;
#pragma unroll
        for (int s = 0; s < 4; s++) dr[s] = *(const f32x4c *)(dec + 16 * s + 4 * g);
        last = dec[CL];
#pragma unroll
        for (int t = 0; t < TK; t++)
#pragma unroll
            for (int x = 0; x < 16; x++) kr[t][x] = kp[(size_t)min(c * CL + 16 * (x >> 2) + 4 * g + (x & 3), sd.n - 1) * A.ldk + (wave * TK + t) * 16];
    };
    request_w(0);
    request_k(0);
    for (int c = 0; c < nc; c++) {
        const size_t at = (size_t)(first + c) * A.heads + h;
        float *snap = A.st + at * DK * A.dv + c0 + i;
#pragma unroll
        for (int t = 0; t < TK; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int row = (wave * TK + t) * 16 + 4 * r + g;
                Sb[row * LS + i] = S[t][r];
                snap[(size_t)row * A.dv] = S[t][r];
            }
        lds_barrier();
        f32x4c p0 = {0.f, 0.f, 0.f, 0.f}, p1 = p0;
#pragma unroll
        for (int s = 0; s < DK / 16; s++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                f32x4c &p = e & 1 ? p1 : p0;
                p = __builtin_amdgcn_mfma_f32_16x16x4f32(wr[s][e], Sb[(16 * s + 4 * g + e) * LS + i], p, 0, 0, 0);
            }
        float *u = A.u + (at * CL + 16 * wave + 4 * g) * A.dv + c0 + i;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float x = ur[r] - (p0[r] + p1[r]);
            Ub[(16 * wave + 4 * g + r) * LS + i] = x;
            u[(size_t)r * A.dv] = x;
        }
        if (c + 1 < nc) request_w(c + 1);
        lds_barrier();
        f64x4c add[TK];          // (summed in 64 bits: in 32 the 64 additions left more in the state than the tokens' own updates do)
#pragma unroll
        for (int t = 0; t < TK; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) add[t][r] = (double)S[t][r] * (double)last;
#pragma unroll
        for (int x = 0; x < 16; x++) {
            const double u1 = (double)Ub[(16 * (x >> 2) + 4 * g + (x & 3)) * LS + i];
#pragma unroll
            for (int t = 0; t < TK; t++) add[t] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)(kr[t][x] * dr[x >> 2][x & 3]), u1, add[t], 0, 0, 0);
        }
#pragma unroll
        for (int t = 0; t < TK; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) S[t][r] = (float)add[t][r];
        if (c + 1 < nc) request_k(c + 1);
    }
#pragma unroll
    for (int t = 0; t < TK; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) state[(size_t)((wave * TK + t) * 16 + 4 * r + g) * A.dv] = S[t][r];
}

// ---- third launch: the outputs of a chunk.  grid (chunks, heads, 64 value columns), four waves of 16 positions.  The products are transposed: scores K Q^T and
// outputs U^T P^T, so that a lane's accumulators hold four keys of its position and are the second product's operand as they are.  A lane's 16 bytes of a row of S
// or U are columns 4 i .. 4 i + 3: column e of each goes to tile e, so that its outputs are 16 bytes side by side again.
// The scores are summed in 64 bits: q . k of unit vectors is small against its terms, and in 32 bits its rounding was most of the outputs' error.  Everything else
// is summed 16 terms at a time.  (Three workgroups on a compute unit: 168 registers.  Error against 64 bits, rms, and time: see the top.)  VEC: rows of U or v of whole aligned 16 bytes.
template <int KIND, int DK, bool VEC>
__global__ void __launch_bounds__(256, KIND == 0 && DK == 128 ? 2 : 3) k_chunk_out(ChunkArgs A)
{
    __shared__ double L[4][CL];
    __shared__ float pw[4][CL + 1];
    SeqDesc sd; int c;
    if (!chunk_seq(A, blockIdx.x, sd, c)) return;
    const int h = blockIdx.y, kh = h / (A.heads / A.qk_heads), lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), i = lane & 15, g = lane >> 4;
    const int t0 = c * CL, n = min(CL, sd.n - t0), pos = 16 * wave + i, c0 = blockIdx.z * 64, cl = min(c0 + 4 * i, A.dv - 4);
    if (16 * wave >= n) return;
    // (a table per wave: nothing to wait for but its own writes)
    if (KIND == 0) {
        const double d = (double)A.decay_head[h];
        pw[wave][lane] = (float)power(d, lane);
        if (lane == 0) pw[wave][CL] = (float)power(d, CL);
    } else L[wave][lane] = log_decay_upto(A, sd, t0, n, h, lane);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const float *qp = A.q + (size_t)(sd.row0 + t0 + min(pos, n - 1)) * A.ldq + (size_t)kh * DK + 4 * g, *kp = A.k + (size_t)(sd.row0 + t0) * A.ldk + (size_t)kh * DK + 4 * g;
    const size_t at = (size_t)blockIdx.x * A.heads + h;
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

size_t al16c(size_t n) { return (n + 15) & ~(size_t)15; }

} // namespace

extern "C" {

int ifa_state_chunked_fits(int kind, const void *q_f32, size_t ldq, const void *k_f32, size_t ldk, const void *v_f32, size_t ldv, int dk, int dv, const void *out_f32, size_t ldo)
{
    const bool rows16 = ldq % 4 == 0 && ldk % 4 == 0 && ldo % 4 == 0 && (((uintptr_t)q_f32 | (uintptr_t)k_f32 | (uintptr_t)out_f32) & 15) == 0;
    return (kind == 0 || kind == 1) && (dk == 64 || dk == 128) && dv > 0 && dv % 32 == 0 && dv <= 64 * 65535 && rows16;
}

size_t ifa_state_chunked_workspace_bytes(int kind, size_t chunks, int heads, int dk, int dv)
{
    const size_t at = chunks * heads;
    return al16c(at * dk * dv * 4) + (kind == 1 ? al16c(at * CL * dv * 4) + al16c(at * CL * dk * 4) + al16c(at * DEC * 4) : 0);
}

int ifa_state_chunked_f32(int kind, const void *q_f32, size_t ldq, const void *k_f32, size_t ldk, const void *v_f32, size_t ldv, int heads, int qk_heads, int dk, int dv,
                          const void *decay_head_f32, const void *decay_row_f32, const void *beta_row_f32, const void *seqs_dev, const void *seqs_host, int n_seqs,
                          void *const *slot_base_dev, size_t state_off, void *ws, size_t ws_bytes, void *out_f32, size_t ldo, ifa_stream stream)
{
    IFA_REQUIRE(q_f32 && k_f32 && v_f32 && seqs_dev && seqs_host && slot_base_dev && ws && out_f32, "ifa_state_chunked_f32: null pointer");
    IFA_REQUIRE(heads > 0 && heads < 65536 && qk_heads > 0 && heads % qk_heads == 0 && n_seqs > 0 && n_seqs < 65536
                && ldq >= (size_t)qk_heads * dk && ldk >= (size_t)qk_heads * dk && ldv >= (size_t)heads * dv && ldo >= (size_t)heads * dv, "ifa_state_chunked_f32: bad shape");
    IFA_REQUIRE(ifa_state_chunked_fits(kind, q_f32, ldq, k_f32, ldk, v_f32, ldv, dk, dv, out_f32, ldo), "ifa_state_chunked_f32: kind %d, sizes %d / %d or rows not of whole 16 bytes",
                kind, dk, dv);
    IFA_REQUIRE(kind == 0 ? decay_head_f32 != nullptr : (decay_row_f32 && beta_row_f32), "ifa_state_chunked_f32: the gates of kind %d are missing", kind);
    const ifa_seq_desc *sh = (const ifa_seq_desc *)seqs_host;
    size_t chunks = 0;
    for (int q = 0; q < n_seqs; q++) { IFA_REQUIRE(sh[q].n > 0, "ifa_state_chunked_f32: empty sequence"); chunks += ((size_t)sh[q].n + CL - 1) / CL; }
    IFA_REQUIRE(chunks < (1u << 30) && ws_bytes >= ifa_state_chunked_workspace_bytes(kind, chunks, heads, dk, dv) && ((uintptr_t)ws & 15) == 0,
                "ifa_state_chunked_f32: workspace of %zu bytes, %zu needed", ws_bytes, ifa_state_chunked_workspace_bytes(kind, chunks, heads, dk, dv));
    ChunkArgs A;
    A.q = (const float *)q_f32; A.k = (const float *)k_f32; A.v = (const float *)v_f32; A.ldq = ldq; A.ldk = ldk; A.ldv = ldv;
    A.heads = heads; A.qk_heads = qk_heads; A.dk = dk; A.dv = dv;
    A.decay_head = (const float *)decay_head_f32; A.decay_row = (const float *)decay_row_f32; A.beta_row = (const float *)beta_row_f32;
    A.seqs = (const SeqDesc *)seqs_dev; A.n_seqs = n_seqs; A.slot_base = (float *const *)slot_base_dev; A.state_off = state_off;
    A.out = (float *)out_f32; A.ldo = ldo;
    const size_t at = chunks * heads;
    A.st = (float *)ws;
    A.u = (float *)((char *)ws + al16c(at * dk * dv * 4));
    A.w = (float *)((char *)A.u + al16c(at * CL * dv * 4));
    A.dec = (float *)((char *)A.w + al16c(at * CL * dk * 4));
    const hipStream_t s = ifa_s(stream);
    const dim3 per_chunk((unsigned)chunks, (unsigned)heads, ifa_cdiv((size_t)dv, 64));
    if (kind == 0) {
        hipLaunchKernelGGL(k_linear_chunk, per_chunk, dim3(256), 0, s, A);
        hipLaunchKernelGGL(k_linear_pass, dim3(ifa_cdiv((size_t)dk * dv, 256), (unsigned)heads, (unsigned)n_seqs), dim3(256), 0, s, A);
        const bool vec = ldv % 4 == 0 && ((uintptr_t)v_f32 & 15) == 0;
        if (dk == 64) { if (vec) hipLaunchKernelGGL((k_chunk_out<0, 64, true>), per_chunk, dim3(256), 0, s, A); else hipLaunchKernelGGL((k_chunk_out<0, 64, false>), per_chunk, dim3(256), 0, s, A); }
        else { if (vec) hipLaunchKernelGGL((k_chunk_out<0, 128, true>), per_chunk, dim3(256), 0, s, A); else hipLaunchKernelGGL((k_chunk_out<0, 128, false>), per_chunk, dim3(256), 0, s, A); }
    } else {
        const dim3 pass((unsigned)(heads * (dv / 16)), (unsigned)n_seqs);
        hipLaunchKernelGGL(k_delta_chunk, dim3((unsigned)chunks, (unsigned)heads), dim3(256), 0, s, A);
        if (dk == 64) { hipLaunchKernelGGL(k_delta_pass<64>, pass, dim3(256), 0, s, A); hipLaunchKernelGGL((k_chunk_out<1, 64, true>), per_chunk, dim3(256), 0, s, A); }
        else { hipLaunchKernelGGL(k_delta_pass<128>, pass, dim3(256), 0, s, A); hipLaunchKernelGGL((k_chunk_out<1, 128, true>), per_chunk, dim3(256), 0, s, A); }
    }
    IFA_LAUNCH_CHECK();
    return IFA_OK;
}

} // extern "C"
