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
#include "ifa_chunkscan.h"

using namespace ifa32;
using namespace ifachunk;

namespace {

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

// grids (chunks, heads, 64 value columns), (dk dv / 256, heads, sequences), (chunks, heads, 64 value columns)
__global__ void __launch_bounds__(256) k_linear_chunk(ChunkArgs A) { linear_chunk(A, blockIdx.x, blockIdx.y, blockIdx.z); }
__global__ void __launch_bounds__(256) k_linear_pass(ChunkArgs A) { linear_pass(A, blockIdx.x * 256 + threadIdx.x, blockIdx.y, blockIdx.z); }
template <int KIND, int DK, bool VEC>
__global__ void __launch_bounds__(256, chunk_out_waves(KIND, DK)) k_chunk_out(ChunkArgs A) { chunk_out<KIND, DK, VEC>(A, blockIdx.x, blockIdx.y, blockIdx.z); }

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
    ChunkArgs A;
    size_t chunks;
    const int rc = ifa_chunk_args(&A, &chunks, kind, q_f32, ldq, k_f32, ldk, v_f32, ldv, heads, qk_heads, dk, dv, decay_head_f32, decay_row_f32, beta_row_f32, seqs_dev, seqs_host, n_seqs,
                                  slot_base_dev, state_off, ws, ws_bytes, out_f32, ldo);
    if (rc) return rc;
    const hipStream_t s = ifa_s(stream);
    const dim3 per_chunk((unsigned)chunks, (unsigned)heads, ifa_cdiv((size_t)dv, 64));
    if (kind == 0) {
        hipLaunchKernelGGL(k_linear_chunk, per_chunk, dim3(256), 0, s, A);
        ifa_linear_pass(A, stream);
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

void ifa_linear_pass(const ChunkArgs &A, ifa_stream stream)
{
    hipLaunchKernelGGL(k_linear_pass, dim3(ifa_cdiv((size_t)A.dk * A.dv, 256), (unsigned)A.heads, (unsigned)A.n_seqs), dim3(256), 0, ifa_s(stream), A);
}

int ifa_chunk_args(ChunkArgs *args, size_t *n_chunks, int kind, const void *q_f32, size_t ldq, const void *k_f32, size_t ldk, const void *v_f32, size_t ldv, int heads, int qk_heads,
                   int dk, int dv, const void *decay_head_f32, const void *decay_row_f32, const void *beta_row_f32, const void *seqs_dev, const void *seqs_host, int n_seqs,
                   void *const *slot_base_dev, size_t state_off, void *ws, size_t ws_bytes, void *out_f32, size_t ldo)
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
    ChunkArgs &A = *args;
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
    *n_chunks = chunks;
    return IFA_OK;
}

