// ifa_gemm_mid.hip -- the linear layers of prompts from 193 tokens on (97 in wide models, 33 where a matrix is not for ifa_gemm_few.hip, which takes the shorter ones):  Y[T][N] = X[T][K] . W[N][K]^T  (+ bias, residual, GLU)
//
// Reference: MatrixMultiplication (src/transformer/inference_worker.cc:2364-2432): Dequantize the weight tensor to F16, F16 x F16
// product with fp32 accumulation (src/tensor/cublas_engine.cu:420-436).  Same values here: every weight is half(fma(q, scale,
// base)) -- the reference's dequantised half -- products accumulate in fp32 in ascending 16-column groups of this workgroup's K
// range, parts of K added in order, one F16 rounding, bias / residual / gate as half operations (k_gemm_big's arithmetic).
//
// Why a second kernel.  k_gemm_big stages the activation tile with direct-to-LDS loads and reads its MFMA operands with
// ordinary LDS loads; hipcc puts `s_waitcnt vmcnt(0)` in front of every LDS read that follows a direct-to-LDS request, so every
// 64-column step ends up waiting for the requests it has just issued: a step is one memory round trip (~1 us; a 128-token prompt's
// w1 | w3 62 us for 64 steps, wq | wk | wv 35 us for 16) however little it multiplies.  Here:
//   * activations go through direct-to-LDS loads into a ring of four stages (128 x 64 halves), requested by four waves that do nothing else, waited for with a
//     COUNTED vmcnt; the raw weight codes, which only one wave reads, go straight to its registers, two steps ahead;
//   * every LDS read of the loop is inline assembly (the compiler sees no LDS access to protect), waited for with lgkmcnt where
//     the values are used;
//   * a wave owns 32 weight rows of the tile and ALL 128 tokens (4 accumulator tiles): it dequantises its rows' codes from the raw
//     bytes straight into the B operand registers (11 VALU per 8 weights, ifa_dequant_q4.h) -- no dequantised tile in LDS, no
//     second barrier -- while the MFMAs of the previous 16-column group run;
//   * one barrier per step (the activation tile is shared by the four waves), and no start of a step: the first groups' fragments and codes of the next step are
//     asked for in this one.  Codes through the ring and a step that began with 19 LDS reads (its conversion and first wait in front of its first product), 140
//     instructions a step, two workgroups on a compute unit to hide that, against 100 instructions and one workgroup, ms a prompt of 193, 300, 512, 600, 768, 2048 tokens,
//     Llama-2-7B: 6.13, 8.78, 9.81, 12.6, 15.0, 33.75 -> 5.74, 8.21, 9.32, 11.5, 13.8, 33.4.
// What bounds it: in the loop power, beside it the ends of the tiles.  Over whole launches the clock is 1.65 - 1.9 GHz (profiles/prompt_products_clock.txt; attention beside
// them 2.2); a step takes 740 - 800 cycles, 512 of them products, 1.25 PFLOP/s in the loop.  So what converts a weight more often to read LDS less or to keep a SIMD busier does not pay: waves of
// 64 rows x 64 tokens (half the fragment reads) took 3 - 7 % longer than the form before, eight computing waves of 32 x 64 8 % longer than this one.  With one workgroup on a compute unit nothing
// runs under a tile's last sums and its output: the gated pair's 7 us an end are 75 of the 379 us of 2048 tokens (2752 tiles, 10.75 rounds) and 20 of the 109 of 512, 0.97 PFLOP/s in all.
// Weights: the MO copy of the rows GEMM (ifa_gemm_rows_mfma.h; Q4_B32T1A / B and the 64-weight nibble formats): a 16-row tile's K range
// is one linear stream of 1 KiB supersteps.
#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <cstring>
#include <cstdio>
#include <type_traits>
#include <vector>
#include "ifa_host.h"
#include "ifa_math.h"
#include "ifa_tiled.h"
#include "ifa_gemm_big.h"
#include "ifa_dequant_q4.h"

namespace ifa {

typedef _Float16 md_h8 __attribute__((ext_vector_type(8)));
typedef float md_f16v __attribute__((ext_vector_type(16)));
typedef uint32_t md_u4 __attribute__((ext_vector_type(4)));
typedef uint32_t md_u2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void md_lds_t;
typedef const __attribute__((address_space(1))) void md_glb_t;

constexpr int MD_BN = 128, MD_BK = 64, MD_NW = 4, MD_NT = 256;      // (token rows of a tile: 32 TA, template parameter)
constexpr int md_a_bytes(int ta) { return 32 * ta * MD_BK * 2; }       // activation tile of a step (TA = 4: 16 KB), rows of 128 bytes, 16-byte chunks swizzled
constexpr int MD_NS = 4;                                               // stages of the ring: one read, one landed, two on their way
constexpr int MD_THREADS = 2 * MD_NT;                                  // launched threads: MD_NT compute and run the tails, as many request the activations

template <int OFF>
__device__ __forceinline__ md_u4 md_lds_b128(uint32_t addr) { md_u4 v; asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF)); return v; }
template <int I, int N, class F>
__device__ __forceinline__ void md_each(F f) { if constexpr (I < N) { f(std::integral_constant<int, I>()); md_each<I + 1, N>(f); } }

// EPI: GM_PLAIN | GM_RESIDUAL | GM_GLU (a weight tile = 64 rows of w1 and the same 64 rows of w3).  KS: parts of K (workgroups per
// tile).  TA: 32-token accumulator tiles of a wave -- the tile is 32 TA tokens x 128 weight rows (TA = 2 up to 64 tokens: half of the products, fragment reads,
// activation requests and exchanged sums of a 128-row tile whose lower half repeats a row, the same bits -- where gemm_few does not take such prompts; TA = 8: md_wide).
template <int EPI, int KS, int TA>
__global__ void __launch_bounds__(MD_THREADS, 2) k_gemm_mid(const GmArgs P, const BigGeo G)
{
    constexpr int BM = 32 * TA, BN = MD_BN, BK = MD_BK, NW = MD_NW, NT = MD_NT, ROWB = BK * 2;
    constexpr int NS = MD_NS, STAGE = md_a_bytes(TA), XP = TA, LEAD = TA == 8 ? 1 : 2;      // XP: activation pieces (8 token rows) a loader wave requests per stage; LEAD: 16-column groups that the fragments are requested ahead
    static_assert(NS * STAGE <= 2 * 65536, "stages that an LDS read's offset reaches from two addresses");
    constexpr bool GLU = EPI == GM_GLU;
    constexpr int BNE = GLU ? BN / 2 : BN;
    auto swz = [](int r) { return (r >> 1) & 7; };
    extern __shared__ __attribute__((aligned(16))) char smem[];
    long long *const trc = (P.trace && threadIdx.x == 0) ? P.trace + (size_t)blockIdx.x * 8 : nullptr;      // (measurement: IFA_MID_TRACE=1)
    if (trc) trc[0] = wall_clock64();
    const int T = P.T, nblk = P.nblk, tiles_m = G.tiles_m;
    const half_t *__restrict__ X = P.X;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave_all = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave = wave_all & (NW - 1);
    const bool loader = wave_all >= NW;
    // XCD-aware tile order, bands of token tiles (k_gemm_big's mapping)
    int wg;
    {
        const int nwg = (int)gridDim.x / KS, orig = (int)blockIdx.x % nwg, xcd = orig & 7, q = nwg >> 3, r = nwg & 7;
        wg = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (orig >> 3);
    }
    const int kz = KS == 1 ? 0 : (int)blockIdx.x / ((int)gridDim.x / KS);
    constexpr int GM = 1024 / BM;
    const int tiles_n = (int)gridDim.x / KS / tiles_m;
    const int band = wg / (GM * tiles_n), within = wg % (GM * tiles_n), band_m = min(GM, tiles_m - band * GM);
    const int t0 = (band * GM + within % band_m) * BM, tn = G.tn0 + within / band_m;
    const int set = (tn >= G.tile0[1] ? 1 : 0) + (tn >= G.tile0[2] ? 1 : 0);
    const int n0 = (tn - (set == 0 ? 0 : (set == 1 ? G.tile0[1] : G.tile0[2]))) * BNE;
    const int N = set == 0 ? P.rows[0] : (set == 1 ? P.rows[1] : P.rows[2]);
    const uint8_t *__restrict__ W = set == 0 ? P.W[0] : (set == 1 ? P.W[1] : P.W[2]);
    const half_t *__restrict__ bias = set == 0 ? P.bias[0] : (set == 1 ? P.bias[1] : P.bias[2]);
    const int ksteps = G.K / BK;
    const int s0 = (int)((long long)kz * ksteps / KS), nsteps = (int)((long long)(kz + 1) * ksteps / KS) - s0;      // (parts of K may differ by one step)

    // ---- sources
    // activations (loader waves): TA pieces of 8 token rows x 128 bytes; lane -> (row, chunk), the swizzle applied to the SOURCE (the load writes LDS linearly)
    const half_t *xsrc[XP];
#pragma unroll
    for (int j = 0; j < XP; j++) {
        const int row = (wave * XP + j) * 8 + lane / 8;
        const int c = (lane % 8) ^ swz(row);
        xsrc[j] = X + (size_t)min(t0 + row, T - 1) * P.ldx + c * 8;
    }
    // weights: this wave's 32 rows = two 16-row tiles of the MO copy (ifa_gemm_rows_mfma.h: per tile, superstep S of 128 columns is ONE
    // contiguous KiB -- lane 16 g + r holds the 16 code bytes of block 4 S + g of row r -- so a tile's K range is one linear stream,
    // like a decode row; the tiled rows fetched 32 bytes per row and step measured 1 TB/s: 32 DRAM pages per request).  A step is
    // half a superstep: lane -> (block l / 32 of the half, tile (l / 16) % 2, row l % 16), 2 x 512 contiguous bytes per request.
    const int nsup = nblk >> 2;
    const size_t mo_tile = mo_tile_bytes(nsup, MO_WORDS);
    __amdgpu_buffer_rsrc_t wres;
    uint32_t woff;
    {
        const int nl0 = wave * 32;
        const uint8_t *Wm = (GLU && nl0 >= BNE) ? P.W1 : W;
        const int first = (n0 + (GLU && nl0 >= BNE ? nl0 - BNE : nl0)) >> 4, last = ((N + 15) >> 4) - 1;
        const int tile0 = min(first, last), two = min(first + 1, last) - tile0;          // (a tile behind the rows: the last one again)
        const uint64_t at = (uint64_t)(Wm + (size_t)tile0 * mo_tile);
        const uint32_t lo = __builtin_amdgcn_readfirstlane((int)(uint32_t)at), hi = __builtin_amdgcn_readfirstlane((int)(uint32_t)(at >> 32));
        wres = __builtin_amdgcn_make_buffer_rsrc((void *)(((uint64_t)hi << 32) | lo), 0, (int)((1 + two) * mo_tile), 0x00020000);
        woff = ((lane >> 4) & 1) && two ? (uint32_t)mo_tile : 0u;
    }
    const uint32_t wc_off = woff + (uint32_t)((lane >> 5) * 256 + (lane & 15) * 16), wb_off = woff + (uint32_t)(mo_words_at(nsup) + (lane >> 5) * 64 + (lane & 15) * 4);
    auto issue = [&](int step, int slot) {          // a loader wave's requests of a stage
        char *st = smem + (size_t)slot * STAGE;
#pragma unroll
        for (int j = 0; j < XP; j++)
            __builtin_amdgcn_global_load_lds((md_glb_t *)(xsrc[j] + (size_t)(s0 + step) * BK), (md_lds_t *)(st + (size_t)(wave * XP + j) * 1024), 16, 0, 0);
    };

    // ---- per-lane LDS offsets: lane (i, g) reads token row i of a 32-row tile, chunk 2 ks + g; weight row i of its wave
    const int i = lane & 31, g = lane >> 5;
    const int lc = g ^ swz(i);
    const uint32_t a_off = (uint32_t)(uintptr_t)(md_lds_t *)smem + (uint32_t)(i * ROWB);
    uint32_t a_at[NS * STAGE > 65536 ? 2 : 1][4];          // by 16-column group; stage and token tile are the reads' offsets
#pragma unroll
    for (int ks = 0; ks < 4; ks++) {
        a_at[0][ks] = a_off + (uint32_t)(((2 * ks) ^ lc) << 4);
        if constexpr (NS * STAGE > 65536) a_at[1][ks] = a_at[0][ks] + 65536;
    }
    auto frag = [&](auto K, auto J, auto A) {          // group, stage, token tile
        constexpr int at = decltype(J)::value * STAGE + decltype(A)::value * 32 * ROWB;
        return md_lds_b128<(at & 65535)>(a_at[at >> 16][decltype(K)::value]);
    };

    md_f16v acc[TA];
#pragma unroll
    for (int a = 0; a < TA; a++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[a][r] = 0.0f;

    if (loader) {
        // the loader wave of a SIMD: a request takes ~70 cycles of the instruction stream that issues it; here they go out while the computing wave multiplies.  It waits
        // for ITS requests of stage `step` + 1 (vmcnt is per wave), every wave meets at the barrier, and it requests stage `step` + 3 into the slot that the computing
        // waves have just left.
#pragma unroll
        for (int p = 0; p < NS - 1; p++) issue(min(p, nsteps - 1), p);
        for (int step = 0, slot = NS - 1; step < nsteps; step++) {
            asm volatile("s_waitcnt vmcnt(%0)" :: "n"((NS - 3) * XP) : "memory");
            __builtin_amdgcn_s_barrier();
            issue(min(step + NS - 1, nsteps - 1), slot);
            slot = slot + 1 == NS ? 0 : slot + 1;
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // the repeats behind the last stage have landed before the ring is reused
        __builtin_amdgcn_s_barrier();                          // (pairs with the computing waves' first barrier behind the loop)
        return;
    }
    if (trc) trc[1] = wall_clock64();
    // The computing waves.  A wave alone on its SIMD issues one instruction in some 8 cycles and a 32 x 32 x 16 product occupies the matrix unit for 32: what is not between
    // products is lost.  So a step has no start and no end: during group G's TA products the fragments of group G + LEAD are requested and the weights of group G + 1
    // converted, whether or not these belong to the next step (whose stage has landed by then), and the codes of the step after next are on their way to registers.
    // sched_barrier pins the order; the loop is unrolled by the ring, so that a read's address is a register of its group and an offset.
    md_u4 raw_c[2], cw; uint32_t raw_b[2]; md_u2 sw;          // codes and (base, scale) words as they come: lane half g holds block g of the step; then by 16-column group / by block
    auto request = [&](int step, int k) {
        const int at = s0 + min(step, nsteps - 1);
        raw_c[k] = __builtin_amdgcn_raw_buffer_load_b128(wres, (int)wc_off, at * 512, 0);
        raw_b[k] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(wres, (int)wb_off, at * 128, 0);
    };
    auto arrange = [&](int k) {          // a lane's chunk of group ks is 2 (ks % 2) + g of block ks / 2
        const uint32_t c0 = raw_c[k][0], c1 = raw_c[k][1], c2 = raw_c[k][2], c3 = raw_c[k][3], w = raw_b[k];
        const auto p = __builtin_amdgcn_permlane32_swap(c0, c1, false, false), q = __builtin_amdgcn_permlane32_swap(c2, c3, false, false), r = __builtin_amdgcn_permlane32_swap(w, w, false, false);
        cw = md_u4{p[0], q[0], p[1], q[1]};
        sw = md_u2{r[0], r[1]};
    };
    // this lane's 8 weights of group ks -- q4x8_dequant_mo's arithmetic (ifa_dequant_q4.h) in four pieces
    uint32_t d_lo = 0, d_hi = 0; q4_h2 d_s2 = {0, 0}, d_b2 = {0, 0}, d_w[4];
    auto dq_a = [&](int ks) {
        const uint32_t code = cw[ks], sbw = sw[ks >> 1];
        d_lo = code & 0x0F0F0F0Fu; d_hi = (code >> 4) & 0x0F0F0F0Fu;
        d_s2 = q4_scale2(sbw); d_b2 = q4_base2(sbw);
    };
    auto dq_b = [&]() { d_w[0] = q4_value2<false>(d_lo, d_s2, d_b2); d_w[1] = q4_value2<true>(d_lo, d_s2, d_b2); };
    auto dq_c = [&]() { d_w[2] = q4_value2<false>(d_hi, d_s2, d_b2); d_w[3] = q4_value2<true>(d_hi, d_s2, d_b2); };
    auto dq_d = [&]() { return md_h8{d_w[0][0], d_w[0][1], d_w[1][0], d_w[1][1], d_w[2][0], d_w[2][1], d_w[3][0], d_w[3][1]}; };
    md_u4 fa[4][TA];          // fragments by 16-column group
    // (a counted wait names the registers it makes valid: later uses depend on the statement)
    auto landed = [&](int k) {
#pragma unroll
        for (int a = 0; a < TA; a++) asm volatile("" : "+v"(fa[k][a]));
    };
    md_h8 fbc, fbn;
    request(0, 0); request(1, 1);
    __builtin_amdgcn_sched_barrier(0);
    // the bare barrier (__syncthreads() is fence + barrier): stages `step` and `step` + 1 have landed, the one read last step may be overwritten
    auto enter = [&]() { __builtin_amdgcn_s_barrier(); asm volatile("" ::: "memory"); };
    auto one = [&](int step, auto J) {          // step % NS == J
        constexpr int j = decltype(J)::value;
        md_each<0, 4>([&](auto K) {
            constexpr int ks = K.value, kf = (ks + LEAD) & 3, jf = ks + LEAD < 4 ? j : (j + 1) % NS;          // the group requested now, its stage
            md_each<0, TA>([&](auto A) {
                constexpr int a = A.value;
                __builtin_amdgcn_sched_barrier(0);
                acc[a] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(md_h8, fa[ks][a]), fbc, acc[a], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (2 * a < TA) {
                    const std::integral_constant<int, kf> kc; const std::integral_constant<int, jf> jc;
                    fa[kf][2 * a] = frag(kc, jc, std::integral_constant<int, 2 * a>());
                    fa[kf][2 * a + 1] = frag(kc, jc, std::integral_constant<int, 2 * a + 1>());
                }
                if constexpr (a == 0) {
                    if constexpr (ks == 3) { arrange((j + 1) & 1); request(step + 3, (j + 1) & 1); }
                    dq_a((ks + 1) & 3);
                }
                if constexpr (a == TA / 4) dq_b();
                if constexpr (a == TA / 2) dq_c();
                if constexpr (a == 3 * TA / 4) fbn = dq_d();
            });
            // group ks + 1 has landed; with two groups of lead the TA requests of group ks + 2 may still be in flight
            asm volatile("s_waitcnt lgkmcnt(%0)" :: "n"(TA * (LEAD - 1)));
            landed((ks + 1) & 3);
            fbc = fbn;
        });
        enter();          // (behind the last step: the loader waves' last barrier, their requests have landed; they end there)
    };
    enter();
    md_each<0, LEAD>([&](auto K) { md_each<0, TA>([&](auto A) { fa[K.value][A.value] = frag(K, std::integral_constant<int, 0>(), A); }); });
    arrange(0); request(2, 0);
    dq_a(0); dq_b(); dq_c(); fbc = dq_d();
    asm volatile("s_waitcnt lgkmcnt(%0)" :: "n"(TA * (LEAD - 1)));
    landed(0);
    int step = 0;
    for (; step + NS <= nsteps; step += NS) {
        one(step, std::integral_constant<int, 0>());
        one(step + 1, std::integral_constant<int, 1>());
        one(step + 2, std::integral_constant<int, 2>());
        one(step + 3, std::integral_constant<int, 3>());
    }
    if (step < nsteps) {
        one(step, std::integral_constant<int, 0>());
        if (step + 1 < nsteps) {
            one(step + 1, std::integral_constant<int, 1>());
            if (step + 2 < nsteps) one(step + 2, std::integral_constant<int, 2>());
        }
    }
    static_assert(NS == 4, "the loop is unrolled by the ring");
    // what was requested behind the last step: in, before its registers and the ring's memory are used for anything else
    asm volatile("s_waitcnt lgkmcnt(0)");
#pragma unroll
    for (int k = 0; k < LEAD; k++) landed(k);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (trc) trc[2] = wall_clock64();
    // ---- parts of K as a REDUCE-SCATTER (KS > 1).  A thread's 16 TA sums are 4 TA units of 16 bytes; unit u = 4 a + q holds the 8 token
    // rows of band u for this lane's weight row.  Part kz OWNS bands [kz UB, (kz + 1) UB), i.e. token rows [8 kz UB, 8 (kz + 1) UB) of the
    // tile: it stores its other units (write-through, 16 bytes per store), arrives at the tile's counter, waits for all KS
    // parts, adds the other parts' values of ITS units in K order (part 0 + part 1 + ... with its own at position kz: the same
    // sequence of additions whichever part performs it) and runs the epilogue for its rows.  k_gemm_big's form -- the last part
    // reads every other part's whole tile -- measured 8 us per launch here (192 KB through one CU) and limits KS; this one reads
    // (KS - 1) / KS x 64 KB per workgroup whatever KS is, so short products can be cut into enough parts to fill the chip twice.
    constexpr int NU = 4 * TA;                           // 8-token-row bands of the tile = 16-byte units of a thread's sums
    static_assert(NU % KS == 0, "parts of K must divide the tile's row bands");
    constexpr int UB = NU / KS;                          // bands a part owns
    const int row_lo = KS == 1 ? 0 : kz * UB * 8, nrows_own = KS == 1 ? BM : UB * 8;
    constexpr int VEC = BNE / 8;
    constexpr int PIECES = (BM / KS * VEC + NT - 1) / NT;  // 16-byte output pieces per thread (its part's rows)
    // GM_RESIDUAL: this thread's pieces of the residual rows are requested NOW: issued from the output loop they were dependent round
    // trips at the very end of the launch (4.6 us of a 25 us launch, IFA_MID_TRACE)
    md_h8 resv[EPI == GM_RESIDUAL ? PIECES : 1];
    if constexpr (EPI == GM_RESIDUAL) {
        const int vr0 = (set >= 1 ? P.rows[0] : 0) + (set >= 2 ? P.rows[1] : 0);
#pragma unroll
        for (int p = 0; p < PIECES; p++) {
            const int idx = tid + p * NT, tl = row_lo + min(idx / VEC, nrows_own - 1), v = idx % VEC;
            const int tok = min(t0 + tl, T - 1), n = min(n0 + v * 8, N - 8);
            resv[p] = *reinterpret_cast<const md_h8 *>(P.res + (size_t)tok * P.ldres + (P.Yset[0] ? 0 : vr0) + n);
        }
    }
    if constexpr (KS > 1) {
        char *pt = reinterpret_cast<char *>(G.part) + (size_t)wg * ((size_t)KS * NU * NT * 16);
        const __amdgpu_buffer_rsrc_t prs = __builtin_amdgcn_make_buffer_rsrc(pt, 0, KS * NU * NT * 16, 0x00020000);
        unsigned *arrive = G.flags + 2 * wg;
#pragma unroll
        for (int u = 0; u < NU; u++) {
            if (u / UB == kz) continue;                  // (wave-uniform)
            md_u4 v;
#pragma unroll
            for (int e = 0; e < 4; e++) { const float f = acc[u >> 2][4 * (u & 3) + e]; v[e] = __builtin_bit_cast(uint32_t, f); }
            __builtin_amdgcn_raw_buffer_store_b128(v, prs, ((kz * NU + u) * NT + tid) * 16, 0, 16);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tid == 0) {
            __hip_atomic_fetch_add(arrive, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const long long t_wait = wall_clock64();
            while (__hip_atomic_load(arrive, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < (unsigned)KS) {
                __builtin_amdgcn_s_sleep(2);
                if (wall_clock64() - t_wait > WAIT_TIMEOUT_TICKS) {      // the other parts are not resident: leave a code and go on (the host fails the call)
                    if (G.err) __hip_atomic_store(G.err, 0x82u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                    break;
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < NU; u++) {
            if (u / UB != kz) continue;
            md_u4 pv[KS];
#pragma unroll
            for (int z = 0; z < KS; z++) pv[z] = md_u4{0, 0, 0, 0};
#pragma unroll
            for (int z = 0; z < KS; z++)
                if (z != kz) pv[z] = __builtin_amdgcn_raw_buffer_load_b128(prs, ((z * NU + u) * NT + tid) * 16, 0, 16);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float own = acc[u >> 2][4 * (u & 3) + e];
                float sf = 0.0f;
#pragma unroll
                for (int z = 0; z < KS; z++) {
                    const uint32_t uz = pv[z][e];            // (scalars first: a bit_cast of a vector ELEMENT reads element 0 every time)
                    const float term = z == kz ? own : __builtin_bit_cast(float, uz);
                    sf = z == 0 ? term : sf + term;
                }
                acc[u >> 2][4 * (u & 3) + e] = sf;
            }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // (the parts' values are in: the count behind the epilogue says so)
    }

    // ---- epilogue (k_gemm_big's arithmetic, this part's rows): products -> F16 (+ bias) -> an LDS tile (rows padded by 64 bytes) ->
    // 16-byte pieces of output rows, residual / GLU applied on the way out
    if (trc) trc[3] = wall_clock64();
    half_t *__restrict__ Yo; int ldo, vrow0 = 0;
    if (P.Yset[0]) { Yo = set == 0 ? P.Yset[0] : (set == 1 ? P.Yset[1] : P.Yset[2]); ldo = set == 0 ? P.ldyset[0] : (set == 1 ? P.ldyset[1] : P.ldyset[2]); }
    else { Yo = P.Y; ldo = P.ldy; vrow0 = (set >= 1 ? P.rows[0] : 0) + (set >= 2 ? P.rows[1] : 0); }
    constexpr int CROW = BN * 2 + 64;
    __syncthreads();                                    // every wave is done with the ring
    {
        const bool odd = i & 1;
        const int cl = wave * 32 + i;
        float bv = 0.0f; bool hb = false;
        if constexpr (GLU) {
            const half_t *bp = cl < BNE ? bias : P.bias1;
            const int n = n0 + (cl < BNE ? cl : cl - BNE);
            if (bp) { hb = true; bv = h2f(bp[min(n, N - 1)]); }
        } else if (bias) { hb = true; bv = h2f(bias[min(n0 + cl, N - 1)]); }
#pragma unroll
        for (int a = 0; a < TA; a++)
#pragma unroll
            for (int rp = 0; rp < 8; rp++) {
                if (KS > 1 && (4 * a + (rp >> 1)) / UB != kz) continue;      // (this part's units only; wave-uniform)
                half_t y0 = f2h(acc[a][2 * rp]), y1 = f2h(acc[a][2 * rp + 1]);
                if (hb) { y0 = f2h(h2f(y0) + bv); y1 = f2h(h2f(y1) + bv); }
                const uint32_t u0 = __builtin_bit_cast(uint16_t, y0), u1 = __builtin_bit_cast(uint16_t, y1);
                const uint32_t send = odd ? u0 : u1;
                const uint32_t recv = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)send, 0xB1, 0xF, 0xF, false);   // quad_perm [1, 0, 3, 2]
                const uint32_t packed = odd ? (recv | (u1 << 16)) : (u0 | (recv << 16));
                const int rr = 2 * rp + (odd ? 1 : 0);
                const int tl = a * 32 + (rr & 3) + 8 * (rr >> 2) + 4 * g;
                *reinterpret_cast<uint32_t *>(smem + (size_t)tl * CROW + (size_t)(cl & ~1) * 2) = packed;
            }
    }
    __syncthreads();
    {
#pragma unroll
        for (int p = 0; p < PIECES; p++) {
            const int idx = tid + p * NT, tr = idx / VEC, v = idx % VEC, tl = row_lo + tr, tok = t0 + tl, n = n0 + v * 8;
            if (tr >= nrows_own) continue;
            md_h8 y = *reinterpret_cast<const md_h8 *>(smem + (size_t)tl * CROW + (size_t)v * 16);
            if constexpr (GLU) {
                const md_h8 u = *reinterpret_cast<const md_h8 *>(smem + (size_t)tl * CROW + (size_t)(BNE + v * 8) * 2);
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const half_t act = f2h(act_fn(h2f(y[e]), P.act_kind));
                    y[e] = f2h(h2f(act) * h2f(u[e]));
                }
            } else if constexpr (EPI == GM_RESIDUAL) {
#pragma unroll
                for (int e = 0; e < 8; e++) y[e] = f2h(h2f(resv[p][e]) + h2f(y[e]));
            }
            if (tok < T && n < N) *reinterpret_cast<md_h8 *>(Yo + (size_t)tok * ldo + vrow0 + n) = y;
        }
    }
    if constexpr (KS > 1) {
        // the part that is last to have read the others' sums puts both counters back to zero (the next launch on this stream finds them clean): behind the output,
        // whose stores do not wait for the counter's way to memory and back
        if (tid == 0) {          // (every thread's reads: the epilogue's barriers)
            unsigned *arrive = G.flags + 2 * wg, *done = arrive + 1;
            const unsigned d = __hip_atomic_fetch_add(done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (d == (unsigned)(KS - 1)) {
                __hip_atomic_store(arrive, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(done, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }
    if (trc) trc[4] = wall_clock64();
}

static int md_num_cus()
{
    static int n = 0;
    if (!n) { int dev = 0; hipDeviceProp_t prop; n = (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess && prop.multiProcessorCount > 0) ? prop.multiProcessorCount : 256; }
    return n;
}

bool gemm_mid_ok(int w_dtype, const GmArgs &P, int epi)
{
    (void)w_dtype;      // (any format the MO copy holds: 4-bit codes with value q * scale + base per 32 weights)
    if (P.mo != MO_WORDS || P.T < 1 || P.nsets < 1 || P.nsets > 3 || P.nblk * 32 < (int)MID_MIN_COLS || P.nblk % 4 != 0) return false;
    for (int i = 0; i < P.nsets; i++) if (P.rows[i] % 16 != 0) return false;
    if (epi == GM_GLU && (P.nsets != 1 || !P.W1 || P.rows[0] % 8 != 0)) return false;
    for (int i = 0; i < P.nsets; i++) if (P.rows[i] % 8 != 0) return false;
    if ((P.Yset[0] ? (P.ldyset[0] | P.ldyset[1] | P.ldyset[2]) : P.ldy) % 8 != 0 || (epi == GM_RESIDUAL && P.ldres % 8 != 0) || P.ldx % 8 != 0) return false;
    return true;
}

template <int EPI, int KS, int TA>
static int md_run(const GmArgs &P, BigGeo G, int tn_count, hipStream_t s)
{
    if constexpr (KS > 1) {
        G.err = wait_err_word();
        const size_t tiles = (size_t)G.tiles_m * tn_count, part_bytes = tiles * (size_t)KS * (32 * TA) * MD_BN * 4;
        void *scratch = nullptr;
        int rcs = gemm_splitk_scratch(s, part_bytes, 2 * tiles, &scratch);      // (two counters per tile)
        if (rcs) return rcs;
        G.flags = (unsigned *)scratch; G.part = (unsigned long long *)((char *)scratch + SPLITK_FLAG_BYTES_H);
    }
    const size_t smem = std::max((size_t)MD_NS * md_a_bytes(TA), (size_t)(32 * TA) * (MD_BN * 2 + 64));
    auto kern = k_gemm_mid<EPI, KS, TA>;
    static std::atomic<uint64_t> attr_set{0};
    int dev = 0;
    (void)hipGetDevice(&dev);
    const uint64_t bit = 1ull << (dev & 63);
    if (!(attr_set.load(std::memory_order_relaxed) & bit)) {
        (void)hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
        attr_set.fetch_or(bit, std::memory_order_relaxed);
    }
    const long long grid = (long long)G.tiles_m * tn_count * KS;
    if constexpr (KS > 1) {
        if (!wait_grid_fits((const void *)kern, MD_THREADS, smem, grid)) return 1;      // (1: not launched -- the caller takes fewer parts)
    }
    static const bool tracing = getenv("IFA_MID_TRACE") != nullptr;
    if (tracing) {      // measurement: per-workgroup phase stamps of this launch on stderr (synchronous)
        static long long *buf = nullptr;
        if (!buf) (void)hipMalloc((void **)&buf, sizeof(long long) * 8 * 4096);
        if (buf && grid <= 4096) {
            (void)hipMemsetAsync(buf, 0, sizeof(long long) * 8 * (size_t)grid, s);
            GmArgs Q = P; Q.trace = buf;
            kern<<<dim3((unsigned)grid), dim3(MD_THREADS), smem, s>>>(Q, G);
            std::vector<long long> h((size_t)grid * 8);
            (void)hipStreamSynchronize(s);
            (void)hipMemcpy(h.data(), buf, h.size() * 8, hipMemcpyDeviceToHost);
            long long t0 = h[0];
            for (long long b = 0; b < grid; b++) t0 = std::min(t0, h[(size_t)b * 8]);
            double mx[5] = {0, 0, 0, 0, 0}, sm[5] = {0, 0, 0, 0, 0};
            for (long long b = 0; b < grid; b++) for (int k = 0; k < 5; k++) { const double v = (h[(size_t)b * 8 + k] - t0) * 0.01; mx[k] = std::max(mx[k], v); sm[k] += v; }
            fprintf(stderr, "k_gemm_mid<%d,%d,%d> grid %lld steps %d | us after the first workgroup's start, mean (max): start %.2f (%.2f) loop begins %.2f (%.2f) loop ends %.2f (%.2f) parts summed %.2f (%.2f) end %.2f (%.2f)\n",
                    EPI, KS, TA, grid, G.K / MD_BK / KS, sm[0] / grid, mx[0], sm[1] / grid, mx[1], sm[2] / grid, mx[2], sm[3] / grid, mx[3], sm[4] / grid, mx[4]);
            return IFA_OK;
        }
    }
    kern<<<dim3((unsigned)grid), dim3(MD_THREADS), smem, s>>>(P, G);
    return IFA_OK;
}

template <int EPI, int TA>
static int md_launch(const GmArgs &P, hipStream_t s)
{
    constexpr int MD_BM = 32 * TA;
    constexpr int BNE = EPI == GM_GLU ? MD_BN / 2 : MD_BN;
    BigGeo G; memset(&G, 0, sizeof(G));
    G.tile0[0] = 0;
    for (int i = 0; i < 3; i++) G.tile0[i + 1] = G.tile0[i] + (i < P.nsets ? (P.rows[i] + BNE - 1) / BNE : 0);
    const int tn_count = G.tile0[P.nsets];
    for (int i = P.nsets; i < 3; i++) G.tile0[i] = 1 << 30;
    G.tiles_m = (P.T + MD_BM - 1) / MD_BM; G.K = P.nblk * 32; G.tn0 = 0;
    const int ksteps = G.K / MD_BK;
    // parts of K: the most that still put ONE workgroup on a CU (150 registers and eight waves: two do not fit).  Every part >= MINS steps
    const long long tiles = (long long)G.tiles_m * tn_count, cap = md_num_cus();
    static const bool no_glu_split = getenv("IFA_MID_NO_GLU_SPLIT") != nullptr;      // (measurement: the gated pair as ONE part of K, like k_gemm_big's -- bit-identical products)
    const bool may = !P.no_waits && waits_enabled() && !(EPI == GM_GLU && no_glu_split);
    int rc = 1;
    static const int force_all = getenv("IFA_MID_KS") ? atoi(getenv("IFA_MID_KS")) : 0;      // (measurement: at most this many parts)
    static const int force_epi = getenv(EPI == GM_PLAIN ? "IFA_MID_KS_PLAIN" : (EPI == GM_GLU ? "IFA_MID_KS_GLU" : "IFA_MID_KS_RES"))
                                     ? atoi(getenv(EPI == GM_PLAIN ? "IFA_MID_KS_PLAIN" : (EPI == GM_GLU ? "IFA_MID_KS_GLU" : "IFA_MID_KS_RES"))) : 0;
    const int force_ks = force_epi ? force_epi : force_all;
    static const int mins = getenv("IFA_MID_MINSTEPS") ? atoi(getenv("IFA_MID_MINSTEPS")) : 4;
    auto fits = [&](int ks) { return may && tiles * ks <= cap && ksteps / ks >= mins && (!force_ks || ks <= force_ks); };
    if constexpr (TA < 8) {
        if (rc == 1 && fits(8)) rc = md_run<EPI, 8, TA>(P, G, tn_count, s);
        if (rc == 1 && fits(4)) rc = md_run<EPI, 4, TA>(P, G, tn_count, s);
        if (rc == 1 && fits(2)) rc = md_run<EPI, 2, TA>(P, G, tn_count, s);
    }
    if (rc == 1) rc = md_run<EPI, 1, TA>(P, G, tn_count, s);
    if (rc) return rc;
    IFA_LAUNCH_CHECK();
    return IFA_OK;
}

// 256-token tiles: a weight is converted once for twice the products.  A round of one tile a compute unit takes 1.9 rounds of 128-token tiles (64 steps: 66 us against 34.5), a last
// round that is not full 0.8 of a full one: the form with the shorter sum.  us a launch, Llama-2-7B, 128 -> 256 tokens a tile: wq | wk | wv of 512, 1536, 2048, 4096 tokens
// 64.6, 162.5, 204.2, 401.3 -> 57.4, 177.3, 198.6, 385.8; the gated pair of 512, 1024, 1536, 4096 109.7, 215.6, 319.8, 784.6 -> 121.2, 198.8, 323.2, 729.8; wo of 1300, 2048, 3000
// 61.7, 72.3, 105.7 -> 59.4, 70.8, 119.1.  No parts of K here: fewer tiles than three quarters of a round are better cut into 128-token tiles' parts (w2 of 1024 tokens 93.3 against 98.1).
static bool md_wide(const GmArgs &P, int epi)
{
    const int bne = epi == GM_GLU ? MD_BN / 2 : MD_BN;
    long long tn = 0;
    for (int i = 0; i < P.nsets; i++) tn += (P.rows[i] + bne - 1) / bne;
    const long long cu = md_num_cus(), n4 = (P.T + 127) / 128 * tn, n8 = (P.T + 255) / 256 * tn;
    auto rounds = [&](long long n) { return (double)(n / cu) + (n % cu ? 0.8 : 0.0); };
    return 4 * n8 >= 3 * cu && 1.9 * rounds(n8) < rounds(n4);
}

int gemm_mid(const GmArgs &P, int epi, hipStream_t s)
{
    if (!gemm_mid_ok(Q4_B32T1A, P, epi)) return ifa_fail(IFA_ERR_ARG, "mid-length GEMM: %d blocks per row / epilogue %d", P.nblk, epi);
    static const int force_ta = getenv("IFA_MID_TA") ? atoi(getenv("IFA_MID_TA")) : 0;      // (measurement)
    if (force_ta == 2 || (!force_ta && P.T <= 64)) {      // (65 .. 192 tokens: the same time either way)
        if (epi == GM_PLAIN) return md_launch<GM_PLAIN, 2>(P, s);
        if (epi == GM_RESIDUAL) return md_launch<GM_RESIDUAL, 2>(P, s);
        return md_launch<GM_GLU, 2>(P, s);
    }
    if (force_ta ? force_ta == 8 : md_wide(P, epi)) {
        if (epi == GM_PLAIN) return md_launch<GM_PLAIN, 8>(P, s);
        if (epi == GM_RESIDUAL) return md_launch<GM_RESIDUAL, 8>(P, s);
        return md_launch<GM_GLU, 8>(P, s);
    }
    if (epi == GM_PLAIN) return md_launch<GM_PLAIN, 4>(P, s);
    if (epi == GM_RESIDUAL) return md_launch<GM_RESIDUAL, 4>(P, s);
    return md_launch<GM_GLU, 4>(P, s);
}

} // namespace ifa
