// ifa_gemm_few.hip -- the linear layers of 9..192 rows (prompts of some tens of tokens, batched steps of many queries):  Y[T][N] = X[T][K] . W[N][K]^T
//
// Reference: MatrixMultiplication (src/transformer/inference_worker.cc:2364-2432), as in ifa_gemm_mid.hip and ifa_gemm_rows_mfma.hip: every weight is the reference's
// dequantised half, products accumulate in fp32, one F16 rounding, bias / residual / gate as half operations.
//
// What bounds these products is how the rows reach the compute units: 48 rows of 4096 columns are 393 KB, the weights of a 256th of wq | wk | wv 123 KB, and every compute unit needs
// all rows of its range of K (the L2s together deliver some 20 TB/s of them).  Hence:
//   * a wave owns supersteps (128 columns) of K and ALL weight rows of its workgroup: every fragment of X is fetched by one wave, once, straight into its B operands, and multiplied with
//     MT tiles; no barrier and no exchange in the loop.  (k_gemm_mid's waves own weight rows: each reads all rows of X from LDS, behind a barrier a step.)  The waves' sums meet in LDS
//     behind the loop, in wave order;
//   * X comes in fragment order (ifa_gemm_few.h), one KiB a request: 16-byte pieces of 64 rows' bytes took 1.4 to 2 times as long as the whole launch, and through LDS the
//     detour cost 1 us of 14.  The producers write it so: the norm (few_sum_norm) and the gated pair's epilogue; only wo reads rows (the attention's), through LDS;
//   * products of few outputs (wo, w2) share K out instead of rows: 64 outputs and a quarter of K need a quarter of the rows' bytes that 16 outputs and all of K do (w2, 48 rows:
//     18.6 -> 12.6 us).  The parts' sums are added where the next launch, the residual and its norm, reads them anyway: nothing waits inside a launch;
//   * requests behind a wave's last superstep lie outside of their buffers: they return zero, fetch nothing, and the loop has one body without a branch around a request.
//   * from 65 rows on the waves share them out too (TG groups of up to 64 rows): each group dequantises the weights again, which is still faster than one wave on a SIMD with 512 registers
//     (96, 128 rows: a prompt 3.43, 3.82 ms against 3.47, 3.95).
// us a launch, Llama-2-7B, 16, 32, 64, 96, 128, 192 rows, the rows GEMM (16 with its norm inside, 32) and k_gemm_mid -> here: wq | wk | wv 13.6, 15.9, 20.2, 25.3, 25.8, 35.6 -> 10.2, 12.4, 15.2, 20.3,
// 23.0, 33.8; w1 | w3 18.6, 21.3, 30.4, 42.1, 42.4, 68.6 -> 15.2, 17.6, 21.6, 30.5, 34.6, 49.6; wo and w2 together 21.3, 29.8, 34.4, 46.6, 49.4, 56.4 -> 14.8, 17.9, 24.9, 31.2, 34.2, 44.3.  Whole prompts
// of 16, 32, 37, 64, 96, 128, 192 tokens 2.35, 2.91, 3.45, 3.48, 4.54, 4.64, 5.98 -> 2.01, 2.29, 2.48, 2.76, 3.43, 3.82, 5.01 ms; steps of 9, 16, 32 queries 2.45, 2.69, 3.55 -> 2.12, 2.32, 2.96.  Up to
// eight rows the rows GEMM with its norm inside is as fast (8 rows) or faster (2: 1.77 against 1.85 ms); of 256 rows k_gemm_mid's larger tiles are (5.75 against 5.85).
#include <algorithm>
#include <cstring>
#include "ifa_gemm_rows_mfma_body.h"
#include "ifa_gemm_few.h"

namespace ifa {

typedef _Float16 h4m __attribute__((ext_vector_type(4)));
constexpr int FEW_W = 8;           // waves of a workgroup
constexpr int FEW_ROWB = 272;      // X as rows: bytes of a row's 128 halves in LDS (+ 16: the pieces of 16 rows in one column fall on different banks)

// columns of tiles whose waves' sums fit the LDS at once
constexpr int few_cols(int mt, int nt) { return mt * nt * FEW_W <= 144 ? nt : mt * (nt / 2) * FEW_W <= 144 && nt % 2 == 0 ? nt / 2 : 1; }

struct FewLaunch : FewArgs { int ks, tiles, x_tiles; };

// MT tiles of 16 weight rows a workgroup (gated pairs: w1 and w3 by turns), NT tiles of 16 rows of X a wave, TG groups of waves for the rows; DP: supersteps whose weights are under way.  (Two where the registers allow
// it: three or four delay the rows behind them, w1 | w3 of 16 rows 15.9 -> 16.6, 17.2 us.)
template <int OUT, int MT, int NT, int TG, int DP, bool FRAG>
__global__ void __launch_bounds__(512) k_gemm_few(const FewLaunch P)
{
    constexpr bool GLU = OUT == FEW_GLU;
    static_assert((!GLU || MT % 2 == 0) && (OUT == FEW_SUMS || FRAG), "pairs of tiles; rows of X only where parts of K are summed");
    constexpr int NOWHERE = 0x70000000;      // behind every buffer
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, g = lane >> 4;
    constexpr int W = FEW_W, KG = W / TG;
    const int nsup = P.K >> 7, T = P.T, tg = wave % TG, kg = wave / TG, t0 = tg * NT * 16;      // (the waves of one kg: the same weights, other rows of X)
    // (neighbouring workgroups, on different XCDs, take the parts of K: an XCD's L2 holds its parts of X only)
    const int kz = (int)blockIdx.x % P.ks, wg = (int)blockIdx.x / P.ks;
    const int s_lo = kz * nsup / P.ks, s_hi = (kz + 1) * nsup / P.ks;
    const GmSets S = {P.W[0], P.W[1], P.W[2], P.bias[0], P.bias[1], P.bias[2], P.Y[0], P.Y[1], P.Y[2], P.rows[0], P.rows[1], P.rows[2], P.nsets, P.ldy[0], P.ldy[1], P.ldy[2]};
    auto tile_of = [&](int it) { return GLU ? wg * (MT / 2) + (it >> 1) : wg * MT + it; };
    const int mo_tile = (int)mo_tile_bytes(nsup, MO_WORDS), words = (int)mo_words_at(nsup);
    __amdgpu_buffer_rsrc_t wr[MT];
#pragma unroll
    for (int it = 0; it < MT; it++) {
        const GmTile tl = gm_locate(S, min(tile_of(it), P.tiles - 1));
        const uint64_t v = (uint64_t)gm_sel(GLU && (it & 1), P.W1, tl.W0) + (size_t)(tl.row0 >> 4) * mo_tile;
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
        wr[it] = __builtin_amdgcn_make_buffer_rsrc((void *)(((uint64_t)hi << 32) | lo), 0, mo_tile, 0x00020000);
    }
    u32x4 cw[DP][MT]; uint32_t sb[DP][MT];
    auto w_request = [&](int k, int sup) {
        const bool in = sup < s_hi;
#pragma unroll
        for (int it = 0; it < MT; it++) {
            cw[k][it] = __builtin_amdgcn_raw_buffer_load_b128(wr[it], in ? lane * 16 : NOWHERE, in ? sup * 1024 : 0, 2);
            sb[k][it] = __builtin_amdgcn_raw_buffer_load_b32(wr[it], in ? lane * 4 : NOWHERE, in ? words + sup * 256 : 0, 2);
        }
    };
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void *)P.X, 0, FRAG ? nsup * P.x_tiles * 4096 : T * P.ldx * 2, 0x00020000);
    // fragment order: this lane's piece of row 16 n + r; rows: piece r of row 16 n + 4 p + g  (rows that are not there: nowhere)
    int xo[NT][FRAG ? 1 : 4];
#pragma unroll
    for (int n = 0; n < NT; n++) {
        if constexpr (FRAG) xo[n][0] = t0 + 16 * n + r < T ? (tg * NT + n) * 4096 + lane * 16 : NOWHERE;
        else {
#pragma unroll
            for (int p = 0; p < 4; p++) xo[n][p] = t0 + 16 * n + 4 * p + g < T ? (t0 + 16 * n + 4 * p + g) * P.ldx * 2 + r * 16 : NOWHERE;
        }
    }
    h8m x[NT][4];
    auto x_request = [&](int sup, int s4) {
        const bool in = sup < s_hi;
#pragma unroll
        for (int n = 0; n < NT; n++) {
            if constexpr (FRAG) x[n][s4] = __builtin_bit_cast(h8m, __builtin_amdgcn_raw_buffer_load_b128(xr, (in ? xo[n][0] : NOWHERE) + s4 * 1024, in ? sup * P.x_tiles * 4096 : 0, 0));
            else x[n][s4] = __builtin_bit_cast(h8m, __builtin_amdgcn_raw_buffer_load_b128(xr, in ? xo[n][s4] : NOWHERE, in ? sup * 256 : 0, 0));
        }
    };
    char *const xl = smem + wave * (NT * 16 * FEW_ROWB);      // (rows of X: this wave's superstep of them)
    f4m acc[MT][NT];
#pragma unroll
    for (int it = 0; it < MT; it++)
#pragma unroll
        for (int n = 0; n < NT; n++) acc[it][n] = f4m{0.0f, 0.0f, 0.0f, 0.0f};
    auto step = [&](int k, int sup) __attribute__((always_inline)) {
        h8m fb[2][NT];
        auto frags = [&](int s4) {
#pragma unroll
            for (int n = 0; n < NT; n++) fb[s4 & 1][n] = *reinterpret_cast<const h8m *>(xl + (16 * n + r) * FEW_ROWB + (4 * g + s4) * 16);
        };
        if constexpr (!FRAG) {      // (one wave's own LDS: its accesses stay in order, the fences keep the compiler to it)
#pragma unroll
            for (int n = 0; n < NT; n++)
#pragma unroll
                for (int p = 0; p < 4; p++) *reinterpret_cast<h8m *>(xl + (16 * n + 4 * p + g) * FEW_ROWB + r * 16) = x[n][p];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int s4 = 0; s4 < 4; s4++) x_request(sup + KG, s4);
            __builtin_amdgcn_sched_barrier(0);
            frags(0);
        }
#pragma unroll
        for (int s4 = 0; s4 < 4; s4++) {
            if constexpr (!FRAG) { if (s4 < 3) frags(s4 + 1); __builtin_amdgcn_sched_barrier(0); }
#pragma unroll
            for (int it = 0; it < MT; it++) {
                q4_h2 wq[4];
                q4x8_dequant_mo(cw[k][it][s4], q4_scale2(sb[k][it]), q4_base2(sb[k][it]), wq);
                const h8m a = {wq[0][0], wq[0][1], wq[1][0], wq[1][1], wq[2][0], wq[2][1], wq[3][0], wq[3][1]};
#pragma unroll
                for (int n = 0; n < NT; n++) acc[it][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, FRAG ? x[n][s4] : fb[s4 & 1][n], acc[it][n], 0, 0, 0);
            }
            if constexpr (FRAG) x_request(sup + KG, s4);      // (where this group's fragments were)
            __builtin_amdgcn_sched_barrier(0);
        }
        w_request(k, sup + DP * KG);
        if constexpr (!FRAG) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    int sup = s_lo + kg;
#pragma unroll
    for (int s4 = 0; s4 < 4; s4++) x_request(sup, s4);
#pragma unroll
    for (int k = 0; k < DP; k++) w_request(k, sup + k * KG);
    __builtin_amdgcn_sched_barrier(0);
    while (sup < s_hi) {
#pragma unroll
        for (int k = 0; k < DP; k++) { if (sup < s_hi) step(k, sup); sup += KG; }
    }
    // ---- the waves' sums in wave order, as many columns of tiles a round as fit; then a wave finishes whole tiles, a lane four outputs of one row of X
    constexpr int NC = few_cols(MT, NT), STEP = GLU ? 2 : 1;
    float *const part = reinterpret_cast<float *>(smem);
#pragma unroll
    for (int n0 = 0; n0 < NT; n0 += NC) {
        __syncthreads();
#pragma unroll
        for (int it = 0; it < MT; it++)
#pragma unroll
            for (int c = 0; c < NC; c++) *reinterpret_cast<f4m *>(part + ((((size_t)it * NC + c) * TG + tg) * KG + kg) * 256 + lane * 4) = acc[it][n0 + c];
        __syncthreads();
        for (int u = wave; u < MT / STEP * NC * TG; u += W) {
            const int it = u / (NC * TG) * STEP, c = u % (NC * TG), t = 16 * (c % TG * NT + n0 + c / TG) + r, vt = tile_of(it);
            if (vt >= P.tiles) continue;
            auto total = [&](int i) {
                const float *p = part + ((size_t)i * NC * TG + c) * KG * 256 + lane * 4;
                f4m v[KG];
#pragma unroll
                for (int w = 0; w < KG; w++) v[w] = *reinterpret_cast<const f4m *>(p + w * 256);
                f4m s = v[0];
#pragma unroll
                for (int w = 1; w < KG; w++) s = s + v[w];
                return s;
            };
            const f4m s0 = total(it), s1 = GLU ? total(it + 1) : s0;
            if (t >= T) continue;
            const GmTile tl = gm_locate(S, vt);
            const int row = tl.row0 + 4 * g;
            if constexpr (OUT == FEW_SUMS) *reinterpret_cast<f4m *>(P.sums + ((size_t)kz * T + t) * P.rows[0] + row) = s0;
            else {
                h4m o;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    half_t y = f2h(s0[i]);
                    if (tl.b0) y = f2h(h2f(y) + h2f(tl.b0[row + i]));
                    if constexpr (GLU) {
                        half_t y3 = f2h(s1[i]);
                        if (P.bias1) y3 = f2h(h2f(y3) + h2f(P.bias1[row + i]));
                        const half_t act = f2h(act_fn(h2f(y), P.act_kind));
                        y = f2h(h2f(act) * h2f(y3));
                    }
                    o[i] = (_Float16)y;
                }
                if constexpr (GLU) {      // fragment order of the next product, whose columns these outputs are
                    const size_t piece = ((size_t)(row >> 7) * P.x_tiles + (t >> 4)) * 4 + ((row >> 3) & 3);
                    *reinterpret_cast<h4m *>(reinterpret_cast<char *>(P.Y[0]) + piece * 1024 + (((row >> 5) & 3) * 16 + (t & 15)) * 16 + (row & 7) * 2) = o;
                } else *reinterpret_cast<h4m *>(tl.y + (size_t)t * tl.ldy + row) = o;
            }
        }
    }
}

template <int OUT, int MT, int NT, bool FRAG, int TG = 1>
static int few_run(const FewLaunch &P, int wgs, hipStream_t s)
{
    constexpr int W = FEW_W, room = 250 - 45 - MT * NT * 4 - NT * 16, DP = std::max(1, std::min(2, room / (5 * MT)));      // (two waves on a SIMD, 256 registers each)
    constexpr size_t smem = std::max(FRAG ? (size_t)0 : (size_t)W * NT * 16 * FEW_ROWB, (size_t)MT * few_cols(MT, NT) * W * 1024);
    auto kern = k_gemm_few<OUT, MT, NT, TG, DP, FRAG>;
    if (smem > 64 * 1024) IFA_HIP_CHECK(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
    kern<<<dim3((unsigned)wgs * (unsigned)P.ks), dim3(64 * W), smem, s>>>(P);
    IFA_LAUNCH_CHECK();
    return IFA_OK;
}

template <int OUT, int MT, bool FRAG = true>
static int few_rows(const FewLaunch &P, int wgs, hipStream_t s)
{
    if (P.T <= 16) return few_run<OUT, MT, 1, FRAG>(P, wgs, s);
    if (P.T <= 32) return few_run<OUT, MT, 2, FRAG>(P, wgs, s);
    if (P.T <= 48) return few_run<OUT, MT, 3, FRAG>(P, wgs, s);
    if (P.T <= 64) return few_run<OUT, MT, 4, FRAG>(P, wgs, s);
    if (P.T <= 96) return few_run<OUT, MT, 3, FRAG, 2>(P, wgs, s);
    if (P.T <= 128) return few_run<OUT, MT, 4, FRAG, 2>(P, wgs, s);
    return few_run<OUT, MT, 3, FRAG, 4>(P, wgs, s);
}

bool few_ok(size_t rows, size_t cols)
{
    // (a tile's MO copy and the rows in fragment order within a buffer's 32-bit offsets, far below NOWHERE)
    // (fewer than 1024 columns leave waves without a superstep)
    return rows > 0 && rows % 16 == 0 && rows < (1u << 24) && cols >= 1024 && cols % 128 == 0 && cols <= 65536;
}

int few_max_rows(size_t dim, size_t ffn)
{
    // Every workgroup fetches all rows of its range of K: behind 96 rows of wide models k_gemm_mid's 128-token tiles are faster.  Four layers, us, k_gemm_mid / here, 64, 96, 128, 160, 192 rows:
    // 4096 x 11008 431, 513, 528, 694, 698 / 379, 470, 514, 633, 664; 4096 x 14336 432, 523, 529, 717, 719 / 415, 521, 584, 723, 754; 5120 x 13824 502, 619, 630, 915, 919 / 498, 633, 708, 908, 961;
    // 6144 x 16384 546, 677, 687, 1039, 1049 / 556, 738, 828, 1085, 1145; 8192 x 28672 851, 1153, 1171, 1932, 1948 / 886, 1246, 1412, 1963, 2074; narrower ones as the first, 0.75 to 0.97 (3072 x 8192 of
    // 144 to 192 rows 1.02 to 1.08)
    return dim * ffn <= (size_t)4096 * 12288 ? FEW_MAX : 96;
}

// tiles of a workgroup where parts of K are summed
static int few_sum_tiles(size_t rows) { return rows >= 16 * 256 ? 4 : 2; }

int few_parts(size_t rows, size_t cols)
{
    // a workgroup for every compute unit, and a superstep at least for each of its waves
    const int mt = few_sum_tiles(rows), groups = ((int)(rows / 16) + mt - 1) / mt;
    return std::max(1, std::min({256 / groups, (int)(cols / 128) / 8, FEW_PARTS}));
}

int gemm_few(const FewArgs &A, FewOut out, hipStream_t s)
{
    FewLaunch P;
    memset(&P, 0, sizeof(P));
    static_cast<FewArgs &>(P) = A;
    P.ks = 1; P.x_tiles = (A.T + 15) / 16;
    bool ok = A.T >= 1 && A.T <= FEW_MAX && A.nsets >= 1 && A.nsets <= 3 && (out == FEW_ROWS || A.nsets == 1) && A.X && (out != FEW_SUMS || A.sums);
    for (int i = 0; i < A.nsets && ok; i++) { ok = A.W[i] && few_ok((size_t)A.rows[i], (size_t)A.K) && (out == FEW_SUMS || A.Y[i]) && (out != FEW_ROWS || A.ldy[i] % 4 == 0); P.tiles += A.rows[i] / 16; }
    if (!ok || (out == FEW_GLU && (!A.W1 || A.rows[0] % 128 != 0)) || (out == FEW_SUMS ? A.ldx % 8 != 0 || (A.ldx && A.ldx < A.K) : A.ldx != 0))
        return ifa_fail(IFA_ERR_ARG, "rows of a prompt: shape not covered (%d rows, %d x %d)", A.T, A.rows[0], A.K);
    // the tiles a workgroup takes: the least rounds of the 256 compute units times what a workgroup fetches, its weights (a pair's 24 bytes a column, at a compute unit's share of
    // the memory's rate) and its rows (at its share of the L2s').  By rounds of weights alone the pairs of 28672 outputs went one to a workgroup, each with all the rows: a layer of width 8192, 64, 128
    // rows 258, 414 us, so 222, 353; of width 7168 and 20480 outputs 194, 304, so 167, 262; up to 4096 x 14336 the choices are the same.
    const double rows_of = 0.0234 * 16 * P.x_tiles * (out == FEW_GLU ? 1 : 2);
    auto choose = [&](std::initializer_list<int> sizes) {
        int best = 0; double cost = 0;
        for (int n : sizes) {
            const double c = (((long)P.tiles + n - 1) / n + 255) / 256 * (n + rows_of);
            if (!best || c <= cost) { best = n; cost = c; }
        }
        return best;
    };
    auto wgs = [&](int n) { return (P.tiles + n - 1) / n; };
    if (out == FEW_GLU) {
        const int n = choose({1, 2, 3});
        return n == 1 ? few_rows<FEW_GLU, 2>(P, wgs(1), s) : n == 2 ? few_rows<FEW_GLU, 4>(P, wgs(2), s) : few_rows<FEW_GLU, 6>(P, wgs(3), s);
    }
    if (out == FEW_ROWS) {
        const int n = choose({2, 3, 4});
        return n == 2 ? few_rows<FEW_ROWS, 2>(P, wgs(2), s) : n == 3 ? few_rows<FEW_ROWS, 3>(P, wgs(3), s) : few_rows<FEW_ROWS, 4>(P, wgs(4), s);
    }
    P.ks = few_parts((size_t)A.rows[0], (size_t)A.K);
    if (few_sum_tiles((size_t)A.rows[0]) == 4) return A.ldx ? few_rows<FEW_SUMS, 4, false>(P, wgs(4), s) : few_rows<FEW_SUMS, 4>(P, wgs(4), s);
    return A.ldx ? few_rows<FEW_SUMS, 2, false>(P, wgs(2), s) : few_rows<FEW_SUMS, 2>(P, wgs(2), s);
}

// One workgroup a row, a row's 16-byte pieces its threads' (k_rmsnorm_rows' order of sums, so the same values as norm and residual in launches of their own).  The parts' sums are some 30 %
// more bytes than the launch of the norm read, and cost it 1 us of 4.7 where a launch that adds them would cost five.
template <int NC>
__global__ void __launch_bounds__(512) k_few_sum_norm(const float *__restrict__ sums, int parts, const half_t *__restrict__ bias, const half_t *__restrict__ res, half_t *__restrict__ x_out,
                                                      int cols, const half_t *__restrict__ w, const half_t *__restrict__ b, float multi_base, float eps, half_t *__restrict__ y)
{
    __shared__ float part[8 * NC];
    const int t = blockIdx.x, T = gridDim.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63, nw = blockDim.x >> 6, nchunks = cols >> 3, ngroups = (nchunks + 63) >> 6;
    const size_t row = (size_t)t * cols, plane = (size_t)T * cols;
    rms_h8 v[NC], wv[NC], bv[NC];
#pragma unroll
    for (int k = 0; k < NC; k++) {
        const int c = 64 * (wave + nw * k) + lane, at = min(c, nchunks - 1);
        f4m s[FEW_PARTS][2];
#pragma unroll
        for (int z = 0; z < FEW_PARTS; z++)
            if (z < parts) {
#pragma unroll
                for (int h = 0; h < 2; h++) s[z][h] = reinterpret_cast<const f4m *>(sums + z * plane + row)[2 * at + h];
            }
        v[k] = reinterpret_cast<const rms_h8 *>(res + row)[at];
        if (w) wv[k] = reinterpret_cast<const rms_h8 *>(w)[at];
        if (w && b) bv[k] = reinterpret_cast<const rms_h8 *>(b)[at];
        if (parts > 0) {
            rms_h8 pb = {0, 0, 0, 0, 0, 0, 0, 0};
            if (bias) pb = reinterpret_cast<const rms_h8 *>(bias)[at];
#pragma unroll
            for (int z = 1; z < FEW_PARTS; z++)
                if (z < parts) { s[0][0] = s[0][0] + s[z][0]; s[0][1] = s[0][1] + s[z][1]; }
#pragma unroll
            for (int e = 0; e < 8; e++) {
                half_t p = f2h(s[0][e >> 2][e & 3]);
                if (bias) p = f2h(h2f(p) + (float)pb[e]);
                v[k][e] = f2h((float)v[k][e] + h2f(p));
            }
            if (c < nchunks) reinterpret_cast<rms_h8 *>(x_out + row)[c] = v[k];
        }
        if (c >= nchunks) {
#pragma unroll
            for (int e = 0; e < 8; e++) v[k][e] = (half_t)0;
        }
    }
    if (!y) return;
#pragma unroll
    for (int k = 0; k < NC; k++) {
        const float pg = wave_sum(rms_chunk_sq(v[k]));
        if (lane == 0) part[wave + nw * k] = pg;
    }
    __syncthreads();
    const float scale = rms_scale_of(rms_total(part, ngroups), cols, eps);
    const int tiles = (T + 15) >> 4;
#pragma unroll
    for (int k = 0; k < NC; k++) {
        const int c = 64 * (wave + nw * k) + lane;
        rms_h8 o;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            float f = (float)v[k][e] * scale;          // rms_apply
            if (w) {
                const float mlt = multi_base + (float)wv[k][e];
                f = f * mlt;
                if (b) f = f + (float)bv[k][e];
            }
            o[e] = f2h(f);
        }
        if (c < nchunks) *reinterpret_cast<rms_h8 *>(reinterpret_cast<char *>(y) + (((size_t)(c >> 4) * tiles + (t >> 4)) * 4 + (c & 3)) * 1024 + (((c >> 2) & 3) * 16 + (t & 15)) * 16) = o;
    }
}

int few_sum_norm(const float *sums, int parts, const half_t *bias, const half_t *res, half_t *x_out, int T, int cols, const half_t *norm_w, const half_t *norm_b, float multi_base, float eps,
                 half_t *y, hipStream_t s)
{
    IFA_REQUIRE(res && T > 0 && T <= FEW_MAX && cols > 0 && cols % 128 == 0 && cols <= 8192 && parts >= 0 && parts <= FEW_PARTS && (parts == 0 || (sums && x_out)) && (!norm_b || norm_w),
                "sum of parts and norm: %d rows of %d columns, %d parts", T, cols, parts);
    const int waves = (cols / 8 + 63) / 64;
    const dim3 grid((unsigned)T), block(64u * (unsigned)std::min(waves, 8));
    if (waves <= 8) k_few_sum_norm<1><<<grid, block, 0, s>>>(sums, parts, bias, res, x_out, cols, norm_w, norm_b, multi_base, eps, y);
    else k_few_sum_norm<2><<<grid, block, 0, s>>>(sums, parts, bias, res, x_out, cols, norm_w, norm_b, multi_base, eps, y);
    IFA_LAUNCH_CHECK();
    return IFA_OK;
}

} // namespace ifa
