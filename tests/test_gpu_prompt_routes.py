"""-m gpu: routes of prompts against the routes that they replace (same rows, other kernels: agreement within the F16 rounding of the summation order), mostly on two layers.
A test that compares two settings of an option turns off what would serve both of them alike, and says that their rows differ in some bit: sums of another order, so another route."""
import numpy as np
import pytest
import torch

from inferflow_amd import dtypes as dt, synth
from tests import gpu_util as g

pytestmark = pytest.mark.gpu


def _rows(wk, toks, V):
    lg = torch.empty((len(toks), V), dtype=torch.float16, device="cuda")
    wk.reset()
    tok = wk.forward(toks, 0, lg)
    return int(tok), g.host(lg).astype(np.float32)


def _agree(a, b):
    cos = float((a * b).sum() / (np.linalg.norm(a) * np.linalg.norm(b)))
    return cos >= 0.9999 and float(np.abs(a - b).max()) <= 0.02 * float(b.std()) + 0.01, (cos, float(np.abs(a - b).max()), float(b.std()))


@pytest.mark.parametrize("T", [34, 40, 48])
def test_two_pass_prompt_agrees_with_the_single_pass(T):
    wk, _, s = synth.build("llama2_7b", dt.Q4_B32T1A, dt.F16, max_ctx=64, layers=2, vocab=2000)
    toks = np.random.default_rng(T).integers(3, s["vocab"], T).astype(np.int32)
    out = {}
    wk.set_option("rows_few", 0); wk.set_option("prefill_mid", 0)
    for v in (1, 0):
        wk.set_option("prefill_chunk", v)
        out[v] = _rows(wk, toks, s["vocab"])
    ok, why = _agree(out[1][1], out[0][1])          # ALL rows: the first pass's logits land in rows 0..31, the second's behind them
    assert ok and not np.array_equal(out[1][1], out[0][1]), why
    wk.close()


@pytest.mark.parametrize("T", [48, 64, 128])
def test_short_prompt_large_tile_route_agrees_with_the_op_by_op_layer(T):
    wk, _, s = synth.build("llama2_7b", dt.Q4_B32T1A, dt.F16, max_ctx=160, layers=2, vocab=2000)
    toks = np.random.default_rng(T).integers(3, s["vocab"], T).astype(np.int32)
    out = {}
    for name in ("prefill_chunk", "rows_few", "prefill_mid"):
        wk.set_option(name, 0)
    for v in (47, 128):
        wk.set_option("prefill_big_min", v)
        out[v] = _rows(wk, toks, s["vocab"])
    ok, why = _agree(out[47][1], out[128][1])
    assert ok and not np.array_equal(out[47][1], out[128][1]), why
    wk.close()


@pytest.mark.parametrize("T", [33, 47, 63, 64])
def test_prompts_in_64_token_tiles_agree_with_the_128_token_tiles(T):
    """up to 64 tokens a tile of k_gemm_mid holds 64 rows (rows_few 0: gemm_few serves such prompts otherwise): the products and their sums are those of the 128-row tile, which 65 tokens
    take, so a row is off by no more than one that the other routes (attention and head by prompt length) leave"""
    wk, _, s = synth.build("llama2_7b", dt.Q4_B32T1A, dt.F16, max_ctx=160, layers=2, vocab=2000)
    wk.set_option("prefill_chunk", 0); wk.set_option("rows_few", 0)
    toks = np.random.default_rng(T).integers(3, s["vocab"], 65).astype(np.int32)
    wk.set_option("prefill_mid", 0)
    other = [_rows(wk, toks[:n], s["vocab"])[1] for n in (T, 65)]
    wk.set_option("prefill_mid", 1)
    short, long_ = _rows(wk, toks[:T], s["vocab"])[1], _rows(wk, toks, s["vocab"])[1][:T]
    for a, b in zip(short, long_):
        ok, why = _agree(a, b)
        assert ok, why
    assert not np.array_equal(short, other[0]) and not np.array_equal(long_, other[1][:T])
    print("T=%d rows that differ in a bit: %d" % (T, sum(not np.array_equal(a, b) for a, b in zip(short, long_))))
    wk.close()


@pytest.mark.parametrize("off", [(), ("rows_few",), ("rows_few", "prefill_mid")], ids=["few", "mid", "large"])
@pytest.mark.parametrize("T", [40, 64, 128])
def test_short_prompt_routes_match_the_oracle(T, off):
    """... and against the ORACLE (the reference's T > 1 rule: F16 activations x dequantised weights, fp32 sums), not only against each
    other: two layers of Llama-2-7B width, the model read back from the worker, every row of the prompt.  gemm_few; without it k_gemm_mid; without that two passes of
    the rows GEMM (40 tokens) and the large-tile launches with four parts of K (64, 128).  Measured: worst row 0.006-0.007 x std(logits) at 2 layers; bound 0.03 x std
    on every row (the whole-model law of test_gpu_fullsize_oracle would allow 0.08 sqrt(2) = 0.11), cosine >= 0.9999."""
    from tests import model_util as mu
    wk, _, s = synth.build("llama2_7b", dt.Q4_B32T1A, dt.F16, max_ctx=160, layers=2, vocab=2000)
    om = mu.oracle_model_from_worker(wk, s, 160)
    toks = np.random.default_rng(100 + T).integers(3, s["vocab"], T).astype(np.int32)
    for name in off:
        wk.set_option(name, 0)
    tok, rows = _rows(wk, toks, s["vocab"])
    t_or, l_or = om.forward(toks, 0, nthreads=8)
    ref = l_or.astype(np.float32)
    std = float(ref.std())
    worst = 0.0
    for i in range(T):
        cos = float((rows[i] * ref[i]).sum() / (np.linalg.norm(rows[i]) * np.linalg.norm(ref[i])))
        mad = float(np.abs(rows[i] - ref[i]).max())
        worst = max(worst, mad / std)
        assert cos >= 0.9999 and mad <= 0.03 * std, (i, cos, mad / std)
    top2 = np.sort(ref[-1])[-2:]
    if top2[1] - top2[0] > 0.03 * std:
        assert tok == int(t_or)
    print("T=%d worst row %.4f x std" % (T, worst))
    wk.close()


@pytest.mark.parametrize("shape", ["llama2_7b", "test_gqa"])
def test_short_prompts_leave_the_cache_rows_of_long_ones(shape):
    """up to 768 tokens four workgroups share a token's rotation (head counts that four divide), above one holds it, and the products in front take other kernels: the cache
    rows of the first layer agree to a rounding (the rotation's bits: the test below)"""
    wk, _, s = synth.build(shape, dt.Q4_B32T1A, dt.F16, max_ctx=832, layers=1, vocab=1000)
    toks = np.random.default_rng(3).integers(3, s["vocab"], 800).astype(np.int32)
    rows = {}
    for T in (40, 800):
        wk.reset()
        wk.forward(toks[:T], 0)
        rows[T] = [np.array(wk.read_buffer(n, 0, nbytes=40 * s["kv_heads"] * s["head_dim"] * 2)) for n in ("kcache", "vcache")]
    for a, b in zip(rows[40], rows[800]):
        a, b = a.view(np.float16).astype(np.float32), b.view(np.float16).astype(np.float32)
        assert np.abs(a - b).max() <= 2.0 ** -9 * np.abs(b).max(), np.abs(a - b).max()
    wk.close()


@pytest.mark.parametrize("heads,kv_heads,head_dim,order,part", [(32, 8, 128, 1, 1.0), (8, 4, 64, 2, 1.0), (12, 4, 48, 2, 0.5), (8, 8, 80, 1, 0.5), (6, 6, 48, 1, 1.0), (32, 2, 64, 1, 1.0)])
def test_rotation_by_four_workgroups_a_token_and_by_one_leave_the_same_bits(heads, kv_heads, head_dim, order, part):
    """768 tokens and one more over the same rows: q, k and both caches, head counts that four divides and others"""
    import ctypes as C
    import torch
    import inferflow_amd as ia
    from tests.gpu_util import capi, p
    gen = torch.Generator(device="cuda"); gen.manual_seed(heads + head_dim)
    T, kvd, row = 769, kv_heads * head_dim, kv_heads * head_dim + 8
    rows = [torch.randn(T, n * head_dim, generator=gen, device="cuda").half() for n in (heads, kv_heads, kv_heads)]
    f = capi().ifa_rope_qk_store
    f.argtypes = [C.c_void_p] * 3 + [C.c_int] * 5 + [C.c_float, C.c_int, C.c_float, C.c_void_p, C.c_void_p, C.c_size_t, C.c_void_p]
    out = []
    for n in (T, T - 1):
        q, k, v = (t.clone() for t in rows)
        caches = [torch.zeros(T, row, dtype=torch.float16, device="cuda") for _ in range(2)]
        ia.check(f(p(q), p(k), p(v), head_dim, heads, kv_heads, n, 5, 10000.0, order, part, p(caches[0]), p(caches[1]), row, None))
        torch.cuda.synchronize()
        out.append([q, k] + caches)
    for a, b, src in zip(out[0], out[1], (rows[0], rows[1], None, None)):
        assert torch.equal(a[:T - 1].view(torch.int16), b[:T - 1].view(torch.int16))
        if src is not None:
            assert torch.equal(b[T - 1], src[T - 1]) and not torch.equal(b[:T - 1], src[:T - 1])
        else:
            assert not b[T - 1].any() and not b[:, kvd:].any()
    assert torch.equal(out[0][2][:, :kvd], out[0][1]) and torch.equal(out[0][3][:, :kvd], rows[2])


def _biased(kvd, wd, T, norms=True, **shape):
    """a worker of two layers whose products, and norms, have biases, no two alike"""
    from inferflow_amd import worker as W
    wk, _, s = synth.build("llama2_7b", wd, kvd, max_ctx=T + 16, layers=2, vocab=600, quant_threshold=0, **shape)
    gen = torch.Generator(device="cuda"); gen.manual_seed(1)
    qd, kvdim = s["heads"] * s["head_dim"], s["kv_heads"] * s["head_dim"]
    for l in range(2):
        for tid, n in ((W.T_WQ_B, qd), (W.T_WK_B, kvdim), (W.T_WV_B, kvdim), (W.T_WO_B, s["dim"]), (W.T_W1_B, s["ffn"]), (W.T_W3_B, s["ffn"]), (W.T_W2_B, s["dim"])):
            wk.set_tensor_f16(l, tid, dt.F16, (0.3 * torch.randn(n, generator=gen, device="cuda")).half(), 1, n)
        for tid in (W.T_ATTN_NORM_B, W.T_FFN_NORM_B) if norms else ():
            wk.set_tensor_f16(l, tid, dt.F16, (0.3 * torch.randn(s["dim"], generator=gen, device="cuda")).half(), 1, s["dim"])
    return wk, s


@pytest.mark.parametrize("T", [9, 16, 17, 32, 33, 48, 49, 64, 65, 96, 97, 128, 129, 191, 192])
@pytest.mark.parametrize("wd,shape", [(dt.Q4_B32T1A, {}), (dt.Q3H_B64T1, dict(dim=1024, heads=16, kv_heads=2, head_dim=64, ffn=1408)), (dt.Q4_B32T1B, dict(dim=2176, heads=9, kv_heads=3, ffn=3712))],
                         ids=["7b", "w1024", "w2176"])
def test_products_that_stream_their_weights_over_few_rows_agree_with_the_others(wd, shape, T):
    """9..192 rows (gemm_few) at both ends of every number of 16-row tiles and groups, whole and partial workgroups of tiles, numbers of supersteps that eight waves and the parts of K do not
    divide, biases everywhere: against the products before (rows_few = 0; same halves, other orders of the fp32 sums: the bound of the routes above; up to 32 rows, which no other fused route
    takes with norm biases, the op-by-op layer), from the start and behind a prefix"""
    wk, s = _biased(dt.F16, wd, T, **shape)
    toks = np.random.default_rng(T).integers(3, s["vocab"], T + 5).astype(np.int32)
    out = {}
    for v in (1, 0):
        wk.set_option("rows_few", v)
        out[v] = [_rows(wk, toks[:T], s["vocab"])[1]]
        wk.reset()
        wk.forward(toks[:5], 0)
        lg = torch.empty((T, s["vocab"]), dtype=torch.float16, device="cuda")
        wk.forward(toks[5:], 5, lg)
        out[v].append(g.host(lg).astype(np.float32))
    for a, b in zip(out[1], out[0]):
        ok, why = _agree(a, b)
        assert ok and not np.array_equal(a, b), why
    wk.close()


@pytest.mark.parametrize("T", [9, 20, 32, 33, 60])
@pytest.mark.parametrize("option", ["gemm_rows", "batch_fused", "prefill_mid"])
def test_the_switches_of_the_products_over_few_rows_hold_for_all_that_serve_them(option, T):
    """off, a prompt takes the bits that it has without gemm_few: up to 32 rows by gemm_rows and batch_fused, above by prefill_mid"""
    wk, _, s = synth.build("llama2_7b", dt.Q4_B32T1A, dt.F16, max_ctx=64, layers=2, vocab=600, quant_threshold=0, dim=1024, heads=16, kv_heads=2, head_dim=64, ffn=1408)
    toks, out = np.random.default_rng(T).integers(3, s["vocab"], T).astype(np.int32), []
    wk.set_option("prefill_chunk", 0)
    for sw, few in ((1, 1), (0, 1), (0, 0)):
        wk.set_option(option, sw); wk.set_option("rows_few", few)
        out.append(_rows(wk, toks, s["vocab"])[1])
    off = (T <= 32) != (option == "prefill_mid")
    assert np.array_equal(out[1], out[2]) == off and np.array_equal(out[0], out[1]) != off
    wk.close()


@pytest.mark.parametrize("ffn,most", [(12288, 192), (12416, 96)])
def test_where_wide_models_leave_the_products_over_few_rows(ffn, most):
    """gemm_few sums K in another order, so its rows differ from the other route's in some bits, up to its last row count and no further"""
    wk, _, s = synth.build("llama2_7b", dt.Q4_B32T1A, dt.F16, max_ctx=208, layers=1, vocab=600, ffn=ffn)
    toks = np.random.default_rng(ffn).integers(3, s["vocab"], 193).astype(np.int32)
    for T, same in ((most, False), (most + 1, True)):
        out = []
        for v in (1, 0):
            wk.set_option("rows_few", v)
            out.append(_rows(wk, toks[:T], s["vocab"])[1])
        ok, why = _agree(*out)
        assert ok and np.array_equal(*out) == same, (T, why)
    wk.close()


@pytest.mark.parametrize("T", [193, 257, 385, 2048, 2600, 5003, 8192])
@pytest.mark.parametrize("wd,shape", [(dt.Q4_B32T1A, {}), (dt.Q3H_B64T1, dict(dim=1024, heads=16, kv_heads=2, head_dim=64, ffn=1408)), (dt.Q4_B32T1B, dict(dim=2176, heads=9, kv_heads=3, ffn=3712))],
                         ids=["q4a", "q3h", "q4b"])
def test_products_whose_steps_run_into_each_other_agree_with_the_large_tiles(wd, shape, T):
    """rows that fill no tile, numbers of 64-column steps with every remainder by the ring's four stages (16, 22, 34, 58 steps, whole and in parts), biases everywhere; 256-token
    tiles (three quarters of a tile a compute unit and more, fewer rounds) for wq | wk | wv of 385 and 2048 rows, wo / w2 of 2048 (q4a), the gated pair of 2600 (q3h) and of 2048 (q4b);
    up to the longest prompt that goes this way"""
    wk, s = _biased(dt.F16, wd, T, **shape)
    toks = np.random.default_rng(T).integers(3, s["vocab"], T).astype(np.int32)
    out = []
    for v in (1, 0):
        wk.set_option("prefill_mid", v)
        out.append(_rows(wk, toks, s["vocab"])[1])
        wk.reset()
    ok, why = _agree(out[0], out[1])
    assert ok, why
    wk.close()


@pytest.mark.parametrize("T", [900, 2048, 2600])
def test_a_lowered_border_of_the_mid_length_products_leaves_them_wo_and_w2(T):
    """prefill_mid_max 768: above it the large tiles, wo and w2 of up to prefill_res_mid (2048) tokens through k_gemm_mid with its parts of K"""
    wk, _, s = synth.build("llama2_7b", dt.Q4_B32T1A, dt.F16, max_ctx=T + 16, layers=2, vocab=600, quant_threshold=0, dim=2048, heads=16, kv_heads=16, ffn=5632)
    toks, out = np.random.default_rng(T).integers(3, s["vocab"], T).astype(np.int32), []
    wk.set_option("prefill_mid_max", 768)
    for v in (2048, 0):
        wk.set_option("prefill_res_mid", v)
        out.append(_rows(wk, toks, s["vocab"])[1])
    ok, why = _agree(*out)
    assert ok, why
    print("T=%d the same bits: %s" % (T, np.array_equal(*out)))
    wk.close()


@pytest.mark.parametrize("T", [33, 64, 200, 800, 2100])
@pytest.mark.parametrize("shape", [dict(dim=512, heads=2, kv_heads=2, head_dim=64, ffn=1024), dict(dim=512, heads=8, kv_heads=4, head_dim=64, ffn=128)], ids=["wo", "w2"])
def test_prompts_of_models_with_a_matrix_of_128_columns(shape, T):
    """two steps of 64 columns are fewer than k_gemm_mid takes: such models keep the large tiles at every length, as against the op-by-op layer"""
    wk, _, s = synth.build("llama2_7b", dt.Q4_B32T1A, dt.F16, max_ctx=2112, layers=2, vocab=600, quant_threshold=0, **shape)
    toks, out = np.random.default_rng(T).integers(3, s["vocab"], T).astype(np.int32), []
    for v in (1, 0):
        wk.set_option("prefill_big", v)
        out.append(_rows(wk, toks, s["vocab"])[1])
    ok, why = _agree(*out)
    assert ok, why
    wk.close()


@pytest.mark.parametrize("n", [9, 16, 17, 32])
@pytest.mark.parametrize("kvd", [dt.F16, dt.Q8_B32T2], ids=["f16", "q8"])
def test_batched_steps_of_many_queries_agree_with_the_rows_products_and_replay(kvd, n):
    """the same products in a batched step: against rows_few = 0, and the captured step replayed with other work between the replays gives the eager step's tokens"""
    wk, s = _biased(kvd, dt.Q4_B32T1A, 32, norms=False, dim=1024, heads=8, kv_heads=8, head_dim=128, ffn=2816)
    V = s["vocab"]
    wk.kv_slots(n)
    rng = np.random.default_rng(n)
    for i in range(n):
        wk.select_kv(i); wk.forward(rng.integers(3, V, 3 + i % 7).astype(np.int32), 0)
    new, pos, slots = rng.integers(3, V, n).astype(np.int32), [3 + i % 7 for i in range(n)], list(range(n))
    out, lg = {}, torch.empty((n, V), dtype=torch.float16, device="cuda")
    for v in (0, 1):
        wk.set_option("rows_few", v)
        tok = wk.decode_batch(new, pos, slots, lg)
        out[v] = g.host(lg).astype(np.float32)
    ok, why = _agree(out[1], out[0])
    assert ok and not np.array_equal(out[1], out[0]), why
    for _ in range(4):
        assert [int(t) for t in wk.decode_batch(new, pos, slots)] == [int(t) for t in tok]
        wk.decode_batch(new[:4], pos[:4], slots[:4]); torch.cuda.synchronize()
    wk.close()


@pytest.mark.parametrize("T", [4, 8, 9, 31, 32, 33, 62, 63])
@pytest.mark.parametrize("order,shape", [(2, {}), (1, dict(kv_heads=8)), (2, dict(dim=1024, heads=8, kv_heads=2, head_dim=128, ffn=1408))], ids=["7b", "pairs_kv8", "w1024_kv2"])
def test_rotation_and_attention_of_short_prompts_in_one_launch_leave_the_bits_of_two(order, shape, T):
    """one tile of queries and two, whole and ragged; heads that share keys; both ways of pairing: every row's logits and the last layer's cache rows.  The one launch leaves the step's query rows
    as they came, the two turn them in place (but the first one): which of them ran"""
    wk, _, s = synth.build("llama2_7b", dt.Q4_B32T1A, dt.F16, max_ctx=96, layers=2, vocab=600, quant_threshold=0, rope_order=order, **shape)
    toks = np.random.default_rng(T).integers(3, 600, T).astype(np.int32)
    out, qs = [], []
    for on in (1, 0):
        wk.set_option("attn_fresh", on)
        tok, lg = _rows(wk, toks, 600)
        out.append((tok, lg) + tuple(np.array(wk.read_buffer(n, 1, nbytes=96 * s["kv_heads"] * s["head_dim"] * 2)) for n in ("kcache", "vcache")))
        qs.append(np.array(wk.read_buffer("q", nbytes=T * s["heads"] * s["head_dim"] * 2)).reshape(T, -1))
    wk.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    assert np.array_equal(qs[0][0], qs[1][0]) and (qs[0][1:] != qs[1][1:]).any(axis=1).all()
    assert out[0][2].any() and np.isfinite(out[0][1]).all()


@pytest.mark.parametrize("T,H,G,order,extra", [(4, 2, 2, 2, 0), (31, 4, 1, 1, 8), (32, 6, 2, 2, 0), (33, 3, 3, 1, 0), (63, 4, 2, 2, 16)])
def test_rotation_cache_rows_and_attention_of_one_launch_against_64_bits(T, H, G, order, extra):
    """Queries, keys and values of order 1.  Turned halfs are off by 2^-11 of their size, so a score by about 2^-11 sqrt 2 of its size (at most 6 here), its own rounding 2^-9 at most; a weight by
    as much of itself, its rounding 2^-11; so rows of values up to 4.5: 4.5 (2^-8 + 2^-9 + 2^-11) < 0.03.  Keys in the cache: 2^-11 of values up to 6.5.  Values: the same bits."""
    L, D = g.capi(), 128
    rng = np.random.default_rng(T)
    q, k, v = (torch.from_numpy(rng.standard_normal((T, n, D)).astype(np.float16)).cuda() for n in (H, G, G))
    keep = [t.clone() for t in (q, k, v)]
    a = np.arange(T)[:, None] * 10000.0 ** (-np.arange(D // 2) / (D // 2))
    tab = torch.from_numpy(np.stack([np.cos(a), np.sin(a)], -1).astype(np.float32)).cuda()
    row = G * D + extra
    kc, vc = (torch.full((T + 2, row), 7.0, dtype=torch.float16, device="cuda") for _ in range(2))
    out = torch.full((T + 1, H, D), 7.0, dtype=torch.float16, device="cuda")
    f = L.ifa_attention_fresh
    f.argtypes = [g.C.c_void_p] * 4 + [g.C.c_int] * 4 + [g.C.c_float, g.C.c_int, g.C.c_float] + [g.C.c_void_p] * 2 + [g.C.c_size_t] + [g.C.c_void_p] * 2

    def call(tokens=T, heads=H, dim=D, turn=order, part=1.0, kcache=kc, stride=row):
        return f(g.p(q), g.p(k), g.p(v), g.p(tab), tokens, heads, G, dim, 1.0, turn, part, g.p(kcache), g.p(vc), stride, g.p(out), None)
    # what it leaves to other launches: too few rows and too many, other heads, no turn and a part of one, rows of the cache off 16 bytes (2: IFA_ERR_STATE); nothing is written
    declined = [call(tokens=3), call(tokens=64), call(dim=64), call(turn=0), call(part=0.5), call(stride=row + 4), call(kcache=kc.reshape(-1)[4:])]
    g.sync()
    assert len(set(declined)) == 1 and declined[0] != 0 and all(bool((t == 7.0).all()) for t in (kc, vc, out))
    assert call() == 0
    g.sync()
    assert all(torch.equal(x, y) for x, y in zip((q, k, v), keep))

    def turned(z):
        z = g.host(z).astype(np.float64)
        lo, hi = (z[..., :D // 2], z[..., D // 2:]) if order == 2 else (z[..., 0::2], z[..., 1::2])
        c, s = np.cos(a)[:, None, :], np.sin(a)[:, None, :]
        x, y = lo * c - hi * s, lo * s + hi * c
        return np.concatenate([x, y], -1) if order == 2 else np.stack([x, y], -1).reshape(z.shape)
    qt, kt, vf = turned(q), turned(k), g.host(v).astype(np.float64)
    kgot, vgot = g.host(kc), g.host(vc)
    assert np.abs(kgot[:T, :G * D].reshape(T, G, D) - kt).max() < 2.0 ** -11 * 6.5
    assert np.array_equal(vgot[:T, :G * D].reshape(T, G, D), g.host(v))
    assert (kgot[T:] == 7.0).all() and (vgot[T:] == 7.0).all() and (kgot[:, G * D:] == 7.0).all() and (vgot[:, G * D:] == 7.0).all()
    got = g.host(out)
    assert (got[T] == 7.0).all()
    for h in range(H):
        s = qt[:, h] @ kt[:, h // (H // G)].T / np.sqrt(D)
        assert np.abs(s).max() < 6
        e = np.where(np.tril(np.ones((T, T), bool)), np.exp(s - s.max(1, keepdims=True)), 0.0)
        want = e / e.sum(1, keepdims=True) @ vf[:, h // (H // G)]
        assert np.abs(got[:T, h] - want).max() < 0.03, (h, np.abs(got[:T, h] - want).max())
