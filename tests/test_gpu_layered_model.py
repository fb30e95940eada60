"""The layer-list worker serving Gelarax models through the InferenceEngine (loader registry, slots, scheduler, sampling entry points)
against the float64 oracle of tests/gelarax_oracle.py: whole prompts, token-by-token decoding, portions, mixed batches, slot reuse,
window / kept-first edges, long decoding, other sizes, greedy generation."""
import os
import subprocess
import json

import numpy as np
import pytest
import torch

from tests import gelarax_oracle as orc
from tests import layered_fixtures as fx

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TOL32 = 2e-5        # fp32 operands: rounding of fp32 sums only
TOL16 = 3e-2        # operands of the matrix products rounded to bfloat16


def engine_for(tmp_path, cfg, weights, dtype="float32", ctx=512, queries=6):
    from inferflow_amd.engine import InferenceEngine
    d = fx.write_model_dir(str(tmp_path / ("m%d" % len(os.listdir(tmp_path)))), cfg, weights)
    return InferenceEngine.from_model_dir(d, dtype, ctx, queries, True)


def tokens_for(cfg, n, seed):
    return [int(t) for t in np.random.default_rng(seed).integers(0, cfg["vocab"], n)]


def oracle_logits(cfg, weights, tokens):
    with torch.no_grad():
        return orc.forward(cfg, fx.oracle_weights(weights), tokens).numpy()


def run_whole(eng, tokens):
    q = eng.add_query(tokens)
    assert q > 0
    out = eng.infer()
    assert [i for i, _ in out] == [q]
    lg = eng.last_logits_f32(q)
    eng.remove_query(q)
    return lg, out[0][1]


def run_portions(eng, tokens, sizes):
    """the prompt in portions of the given sizes (the last size repeats); logits of every token"""
    q = eng.add_query(tokens[:sizes[0]])
    rows, at, k = [], sizes[0], 0
    eng.infer(); rows.append(eng.last_logits_f32(q))
    while at < len(tokens):
        k = min(k + 1, len(sizes) - 1)
        n = min(sizes[k], len(tokens) - at)
        for t in tokens[at:at + n]:
            assert eng.commit({q: t})
        eng.infer(); rows.append(eng.last_logits_f32(q))
        at += n
    eng.remove_query(q)
    return np.concatenate(rows, 0)


MIXED = fx.config([fx.parallel_layer(), fx.delta_layer(), fx.parallel_layer(heads=2, kv_heads=1, dim=16, window=9, keep_first=0, lin_heads=3, lin_dim=8, lin_vdim=24,
                                                                           ff=0)], width=64, vocab=97)


@pytest.mark.parametrize("dtype,tol", [("float32", TOL32), ("bfloat16", TOL16)])
def test_whole_prompt_matches_the_oracle(tmp_path, dtype, tol):
    w = fx.random_weights(MIXED, 1)
    toks = tokens_for(MIXED, 71, 2)
    eng = engine_for(tmp_path, MIXED, w, dtype)
    lg, nxt = run_whole(eng, toks)
    want = oracle_logits(MIXED, w, toks)
    assert lg.shape == want.shape
    assert fx.rel_err(lg, want).max() < tol
    if dtype == "float32":
        assert nxt == int(want[-1].argmax())
    eng.close()


def test_residual_after_every_layer_matches_the_oracle(tmp_path):
    import ctypes as C
    import inferflow_amd as ia
    w = fx.random_weights(MIXED, 3)
    toks = tokens_for(MIXED, 40, 4)
    eng = engine_for(tmp_path, MIXED, w)
    L = ia.lib()
    ia.check(L.ifa_model_set_option(eng.worker(), b"tap_layers", 1))
    run_whole(eng, toks)
    res = []
    with torch.no_grad():
        orc.forward(MIXED, fx.oracle_weights(w), toks, res)
    for li, want in enumerate(res):
        p, b = C.c_void_p(), C.c_size_t()
        ia.check(L.ifa_model_get_buffer(eng.worker(), b"layer_taps", li, C.byref(p), C.byref(b)))
        got = np.zeros((len(toks), MIXED["width"]), np.float32)
        ia.check(L.ifa_memcpy_d2h(got.ctypes.data_as(C.c_void_p), p, got.nbytes, None)); ia.check(L.ifa_stream_sync(None))
        assert np.abs(got - want.numpy()).max() < 2e-4 * max(1.0, np.abs(want.numpy()).max()), li
    eng.close()


@pytest.mark.parametrize("sizes", [[1], [2], [5, 3], [30, 1], [7, 2, 1], [64, 4]])
def test_portions_and_token_by_token_equal_the_whole_prompt(tmp_path, sizes):
    w = fx.random_weights(MIXED, 5)
    toks = tokens_for(MIXED, 83, 6)
    eng = engine_for(tmp_path, MIXED, w)
    whole, _ = run_whole(eng, toks)
    parts = run_portions(eng, toks, sizes)
    assert parts.shape == whole.shape
    assert fx.rel_err(parts, whole).max() < TOL32
    assert fx.rel_err(parts, oracle_logits(MIXED, w, toks)).max() < TOL32
    eng.close()


def test_batches_of_unequal_requests_equal_each_alone_and_slots_are_reused(tmp_path):
    w = fx.random_weights(MIXED, 7)
    eng = engine_for(tmp_path, MIXED, w, queries=3)
    prompts = [tokens_for(MIXED, n, 10 + n) for n in (1, 37, 64, 5, 90, 2)]
    tails = [tokens_for(MIXED, 12, 50 + i) for i in range(len(prompts))]
    alone = []
    for p, t in zip(prompts, tails):
        alone.append(oracle_logits(MIXED, w, p + t))
    # two rounds of three queries on three slots: the second round reuses the slots of the first
    for rnd in range(2):
        qs = [eng.add_query(p) for p in prompts[3 * rnd:3 * rnd + 3]]
        assert all(q > 0 for q in qs) and eng.add_query([1, 2]) == 0          # busy: every slot is taken
        got = {q: [] for q in qs}
        assert sorted(i for i, _ in eng.infer()) == sorted(qs)                 # ONE step for the three prompts
        for q in qs:
            got[q].append(eng.last_logits_f32(q))
        for step in range(12):
            live = [q for k, q in enumerate(qs) if not (k == 0 and step >= 6)]  # the first query ends earlier
            if step == 6:
                eng.remove_query(qs[0])
            eng.commit({q: tails[3 * rnd + qs.index(q)][step] for q in live})
            assert sorted(i for i, _ in eng.infer()) == sorted(live)
            for q in live:
                got[q].append(eng.last_logits_f32(q))
        for k, q in enumerate(qs):
            g = np.concatenate(got[q], 0)
            assert fx.rel_err(g, alone[3 * rnd + k][:len(g)]).max() < TOL32, (rnd, k)
            eng.remove_query(q)
    eng.close()


def test_window_and_kept_first_edges_in_prompts_and_decoding(tmp_path):
    """One attention layer whose weights make one key stand out: the token `probe` has a query that matches the key of token `mark`.
    The logits then depend strongly on whether `mark` is visible, so a window or kept-first range that is one token off shows."""
    window, keep = 11, 3
    cfg = fx.config([fx.parallel_layer(heads=2, kv_heads=2, dim=16, window=window, keep_first=keep, scale=1.0, softcap=30.0, lin_heads=1, lin_dim=8, lin_vdim=8,
                                       ff=0)], width=32, vocab=50)
    w = fx.random_weights(cfg, 9, buckets=8)
    mark, probe = 7, 9
    e = w["embed"]
    e[mark] = 0; e[probe] = 0
    e[mark, 0] = 8.0; e[probe, 1] = 8.0
    # keys read feature 0, queries feature 1, both onto head dimension 0
    wq, wk = w["l0.mix.left.q"], w["l0.mix.left.k"]
    wq[:, :2] = 0; wk[:, :2] = 0
    for h in range(2):
        wq[h * 16, 1] = 4.0; wk[h * 16, 0] = 4.0
    w = {k: orc.bf16_round(v) for k, v in w.items()}
    eng = engine_for(tmp_path, cfg, w, ctx=128)
    filler = [t for t in range(10, 50)]
    for mark_at in (0, keep - 1, keep, keep + 1, 20):
        for dist in (1, window - 1, window, window + 1, 40):
            n = mark_at + dist + 1
            toks = [filler[(3 * i + mark_at + dist) % len(filler)] for i in range(n)]
            toks[mark_at] = mark; toks[-1] = probe
            want = oracle_logits(cfg, w, toks)
            whole, _ = run_whole(eng, toks)
            assert fx.rel_err(whole, want).max() < TOL32, ("prompt", mark_at, dist)
            if n > 2:
                dec = run_portions(eng, toks, [max(1, n - 3), 1])
                assert fx.rel_err(dec, want).max() < TOL32, ("decoded", mark_at, dist)
            # the oracle itself must see the edge: with the mark masked out (one past the window, not kept) the last row differs
            seen = mark_at < keep or dist < window
            blind = list(toks); blind[mark_at] = filler[0]
            moved = fx.rel_err(oracle_logits(cfg, w, blind)[-1:], want[-1:]).max()
            assert (moved > 1e-3) == seen or not seen, (mark_at, dist, moved)
    eng.close()


def test_far_key_among_hundreds_and_long_decoding(tmp_path):
    cfg = fx.config([fx.delta_layer(heads=2, kv_heads=1, dim=8, vdim=8, conv=4, ff=32), fx.parallel_layer(heads=2, kv_heads=1, dim=16, window=50, keep_first=4,
                                                                                                          lin_heads=2, lin_dim=8, lin_vdim=16, decay=[0.999, 0.9],
                                                                                                          ff=32)], width=32, vocab=61)
    w = fx.random_weights(cfg, 11, buckets=[0, 10])
    toks = tokens_for(cfg, 330, 12)
    want = oracle_logits(cfg, w, toks)
    eng = engine_for(tmp_path, cfg, w, ctx=400)
    got = run_portions(eng, toks, [200, 1])        # 130 tokens decoded one by one: the window passes over decoded tokens
    assert fx.rel_err(got, want).max() < 5e-5
    # the state reaches far back: another first token changes the last logits (slow decay, kept first tokens)
    other = list(toks); other[0] = (toks[0] + 1) % cfg["vocab"]
    assert fx.rel_err(oracle_logits(cfg, w, other)[-1:], want[-1:]).max() > 1e-4
    eng.close()


@pytest.mark.parametrize("case", ["gqa_1", "mha", "delta_first_taps2", "no_ffn_anywhere", "odd_sizes", "tiny_unaligned", "wide_heads"])
def test_other_sizes(tmp_path, case):
    if case == "gqa_1":
        cfg = fx.config([fx.parallel_layer(heads=4, kv_heads=1, dim=8, window=1, keep_first=1, lin_heads=1, lin_dim=4, lin_vdim=4, ff=16)], width=16, vocab=11)
    elif case == "mha":
        cfg = fx.config([fx.parallel_layer(heads=3, kv_heads=3, dim=12, window=200, keep_first=0, lin_heads=2, lin_dim=20, lin_vdim=70, ff=40),
                         fx.delta_layer(heads=3, kv_heads=3, dim=12, vdim=70, conv=1, ff=40)], width=48, vocab=33)
    elif case == "delta_first_taps2":
        cfg = fx.config([fx.delta_layer(heads=1, kv_heads=1, dim=4, vdim=4, conv=2, ff=8), fx.delta_layer(heads=6, kv_heads=2, dim=24, vdim=8, conv=5, ff=0),
                         fx.parallel_layer()], width=40, vocab=29)
    elif case == "no_ffn_anywhere":
        cfg = fx.config([fx.parallel_layer(ff=0), fx.delta_layer(ff=0)], width=24, vocab=19)
    elif case == "tiny_unaligned":
        cfg = fx.config([fx.parallel_layer(heads=2, kv_heads=1, dim=6, window=5, keep_first=1, lin_heads=1, lin_dim=3, lin_vdim=5, ff=10),
                         fx.delta_layer(heads=2, kv_heads=2, dim=6, vdim=5, conv=3, ff=0)], width=14, vocab=9)
    elif case == "wide_heads":
        cfg = fx.config([fx.parallel_layer(heads=2, kv_heads=1, dim=160, window=30, keep_first=2, lin_heads=1, lin_dim=128, lin_vdim=96, ff=64),
                         fx.delta_layer(heads=2, kv_heads=1, dim=64, vdim=72, conv=4, ff=64), fx.parallel_layer(heads=4, kv_heads=4, dim=32, window=7, keep_first=9,
                                                                                                              lin_heads=2, lin_dim=32, lin_vdim=16, ff=0)],
                        width=128, vocab=50)
    else:
        cfg = fx.config([fx.parallel_layer(heads=5, kv_heads=5, dim=20, window=13, keep_first=2, lin_heads=3, lin_dim=12, lin_vdim=36, ff=52),
                         fx.delta_layer(heads=5, kv_heads=1, dim=12, vdim=20, conv=4, ff=52)], width=36, vocab=23)
    w = fx.random_weights(cfg, 13, buckets=9)
    toks = tokens_for(cfg, 45, 14)
    want = oracle_logits(cfg, w, toks)
    for dtype, tol in (("float32", TOL32), ("bfloat16", TOL16)):
        eng = engine_for(tmp_path, cfg, w, dtype)
        whole, _ = run_whole(eng, toks)
        assert fx.rel_err(whole, want).max() < tol, (case, dtype)
        assert fx.rel_err(run_portions(eng, toks, [20, 9, 1]), want).max() < tol, (case, dtype, "portions")
        eng.close()


def test_greedy_generation_through_the_engine(tmp_path):
    w = fx.random_weights(MIXED, 15)
    prompt = tokens_for(MIXED, 19, 16)
    eng = engine_for(tmp_path, MIXED, w)
    # Generate(): prompt step + decode steps replayed from a captured graph with the token fed back on the device
    q = eng.add_query(prompt)
    gen, _ = eng.generate(q, 24)
    eng.remove_query(q)
    # the serving loop: Infer -> Commit of the greedy token
    q = eng.add_query(prompt)
    loop = []
    for _ in range(24):
        (qq, tok), = eng.infer()
        loop.append(tok); eng.commit({q: tok})
    eng.remove_query(q)
    assert gen == loop
    # the oracle follows the same tokens and agrees wherever its two best logits are clearly apart
    want = oracle_logits(MIXED, w, prompt + gen)
    for i, tok in enumerate(gen):
        row = want[len(prompt) - 1 + i]
        top2 = np.sort(row)[-2:]
        if top2[1] - top2[0] > 1e-3 * np.abs(row).max():
            assert tok == int(row.argmax()), i
    # sampled queries draw from the same logits (top-k with a seed: reproducible)
    a = eng.add_query(prompt, strategy="sample.top_k", seed=5)
    b = eng.add_query(prompt, strategy="sample.top_k", seed=5)
    out = dict(eng.infer())
    assert out[a] == out[b] and 0 <= out[a] < MIXED["vocab"]
    eng.close()


def test_ini_route_and_trace_replay_tool(tmp_path):
    from inferflow_amd.engine import InferenceEngine
    w = fx.random_weights(MIXED, 17)
    d = fx.write_model_dir(str(tmp_path / "model"), MIXED, w)
    ini = tmp_path / "serve.ini"
    ini.write_text("[transformer_engine]\nmodels = m\ndevices = 0\nmax_concurrent_queries = 2\nreturn_output_tensors_f32 = true\n\n"
                   "[model.m]\nmodel_dir = %s/\ncompute_dtype = float32\nmax_context_len = 100\n" % d)
    eng = InferenceEngine.from_ini(str(ini))
    toks = tokens_for(MIXED, 30, 18)
    lg, _ = run_whole(eng, toks)
    want = oracle_logits(MIXED, w, toks)
    assert fx.rel_err(lg, want).max() < TOL32
    assert eng.model_info("vocab_size") == MIXED["vocab"] and eng.model_info("decoder_layers") == 3
    eng.close()
    # the trace tool: two requests start together, go on token by token, one ends earlier
    a, b = tokens_for(MIXED, 26, 19), tokens_for(MIXED, 9, 20)
    steps = [{"step": 0, "entries": [{"id": "a", "tokens": a[:20], "want": [0, 19]}, {"id": "b", "tokens": b[:6], "want": [5]}], "end": []}]
    for s in range(1, 7):
        ent = [{"id": "a", "tokens": [a[19 + s]], "want": [0]}]
        if s <= 3:
            ent.append({"id": "b", "tokens": [b[5 + s]], "want": [0] if s != 2 else []})
        steps.append({"step": s, "entries": ent, "end": (["b"] if s == 3 else []) + (["a"] if s == 6 else [])})
    out = tmp_path / "out"; out.mkdir()
    r = subprocess.run([os.path.join(ROOT, "bin", "trace_run"), "--model", d, "--dtype", "float32", "--out", str(out), "--max-tokens", "64"],
                       input="".join(json.dumps(s) + "\n" for s in steps).encode(), stdout=subprocess.PIPE, stderr=subprocess.PIPE, timeout=900)
    assert r.returncode == 0, r.stderr.decode()[-2000:]
    assert [l for l in r.stdout.decode().split() if l != "done"] == [str(s) for s in range(7)]
    wa, wb = oracle_logits(MIXED, w, a), oracle_logits(MIXED, w, b)
    V = MIXED["vocab"]
    g0 = np.fromfile(out / "0.f32", np.float32).reshape(-1, V)
    assert fx.rel_err(g0, np.stack([wa[0], wa[19], wb[5]])).max() < TOL32
    for s in range(1, 7):
        g = np.fromfile(out / ("%d.f32" % s), np.float32).reshape(-1, V)
        exp = [wa[19 + s]] + ([wb[5 + s]] if s <= 3 and s != 2 else [])
        assert fx.rel_err(g, np.stack(exp)).max() < TOL32, s


CHUNKED = fx.config([fx.parallel_layer(heads=4, kv_heads=2, dim=64, window=200, keep_first=3, lin_heads=3, lin_dim=64, lin_vdim=96, ff=72),
                     fx.delta_layer(heads=4, kv_heads=2, dim=64, vdim=32, conv=3, ff=40)], width=72, vocab=97)


@pytest.mark.parametrize("limit", [4096, 0])
def test_prompts_with_and_without_the_workspaces_of_tiles_and_chunks(tmp_path, limit):
    """a workspace that may not be had (limit 0) costs time, not the step: prompts of growing length, portions on both sides of the chunked form's border"""
    import inferflow_amd as ia
    w = fx.random_weights(CHUNKED, 31)
    toks = tokens_for(CHUNKED, 420, 32)
    want = oracle_logits(CHUNKED, w, toks)
    eng = engine_for(tmp_path, CHUNKED, w)
    ia.check(ia.lib().ifa_model_set_option(eng.worker(), b"workspace_mb", limit))
    for n in (20, 130, 420):
        assert fx.rel_err(run_whole(eng, toks[:n])[0], want[:n]).max() < TOL32, n
    assert fx.rel_err(run_portions(eng, toks, [113, 20, 1, 150]), want).max() < TOL32
    eng.close()


@pytest.mark.parametrize("T", [9, 40, 300])
def test_sums_of_products_with_and_without_the_workspace_of_their_planes(tmp_path, T):
    """K shared out to workgroups, whose sums the next block's norm adds, the last block's an addition by itself; without the workspace (limit 0) a workgroup goes through all of K: sums in
    another order, so some bits differ"""
    import inferflow_amd as ia
    cfg = fx.config([fx.parallel_layer(heads=4, kv_heads=2, dim=64, window=200, keep_first=3, lin_heads=4, lin_dim=64, lin_vdim=128, ff=2816),
                     fx.delta_layer(heads=4, kv_heads=2, dim=64, vdim=64, conv=3, ff=2816)], width=512, vocab=97)
    w, toks, out = fx.random_weights(cfg, 37), tokens_for(cfg, T, 38), []
    for limit in (4096, 0):
        eng = engine_for(tmp_path, cfg, w, "bfloat16", 400, 1)
        for name, value in ((b"attn_tile_min", 1 << 20), (b"scan_chunk_min", 0), (b"workspace_mb", limit)):
            ia.check(ia.lib().ifa_model_set_option(eng.worker(), name, value))
        out.append(run_whole(eng, toks)[0])
        eng.close()
    want = oracle_logits(cfg, w, toks)
    assert all(fx.rel_err(o, want).max() < TOL16 for o in out)
    assert not np.array_equal(*out)


def test_generation_over_bfloat16_rows_of_single_tokens_behind_a_prompt_without_planes(tmp_path):
    """a16_min 1, a launch per operation: the captured step's sums take no planes, which no prompt may have left room for (2048 rows of width 1024: none)"""
    import inferflow_amd as ia
    cfg = fx.config([fx.parallel_layer(heads=8, kv_heads=2, dim=128, window=64, keep_first=0, lin_heads=8, lin_dim=64, lin_vdim=128, ff=2816)], width=1024, vocab=97)
    w, seen = fx.random_weights(cfg, 39), {}
    for graph in (1, 0):
        eng = engine_for(tmp_path, cfg, w, "bfloat16", 2100, 1)
        for name, value in ((b"a16_min", 1), (b"fuse_step", 0), (b"graph", graph)):
            ia.check(ia.lib().ifa_model_set_option(eng.worker(), name, value))
        q = eng.add_query(tokens_for(cfg, 2048, 40))
        seen[graph] = eng.generate(q, 12)[0]
        eng.close()
    assert seen[1] == seen[0]


@pytest.mark.parametrize("T,width", [(9, 520), (16, 520), (17, 520), (130, 520), (601, 520), (1500, 520), (3100, 520), (70, 2056), (300, 72), (130, 128)])
def test_prompts_whose_products_read_bfloat16_rows(tmp_path, T, width):
    """Activations formed in the product's own tiles, outputs of norms and mixers left in bfloat16, a layer's output products in one pass over their columns -- every tile size, few and many
    steps, inner sizes that are no whole step, layers without feed-forward, norm groups of a power of two and others, attention heads that leave 32 bits -- against every operand stored in
    32 bits and rounded on the way into a product of its own (a16_min 0).  Both round the same operands; sums in another order flip such a rounding here and there, which is up to 2^-8 of
    one element: one layer at a time, since flips in one flip more in the next, up to the noise of all roundings"""
    import inferflow_amd as ia
    for layer in (fx.delta_layer(heads=4, kv_heads=2, dim=16, vdim=32, conv=3, ff=72),
                  fx.parallel_layer(heads=2, kv_heads=1, dim=32, window=100, keep_first=0, lin_heads=2, lin_dim=16, lin_vdim=40, ff=1032),
                  fx.parallel_layer(heads=3, kv_heads=1, dim=24, window=50, keep_first=2, lin_heads=2, lin_dim=16, lin_vdim=48, ff=0),
                  fx.delta_layer(heads=2, kv_heads=1, dim=16, vdim=40, conv=3, ff=200)):
        cfg = fx.config([layer], width=width, vocab=97)
        eng = engine_for(tmp_path, cfg, fx.random_weights(cfg, 35), "bfloat16", 3200, 1)
        toks, out = tokens_for(cfg, T, 36), {}
        for border in (0, 9):
            ia.check(ia.lib().ifa_model_set_option(eng.worker(), b"a16_min", border))
            out[border] = run_whole(eng, toks)[0]
        eng.close()
        assert out[9].shape == (T, 97) and np.isfinite(out[9]).all()
        assert fx.rel_err(out[9], out[0]).max() < 2.0 ** -8, layer


def test_chunked_recurrences_are_switched_off_by_0(tmp_path):
    """the bits of the token-by-token form, which a border above every prompt has too; the chunks' differ"""
    import inferflow_amd as ia
    eng = engine_for(tmp_path, CHUNKED, fx.random_weights(CHUNKED, 33))
    toks, out = tokens_for(CHUNKED, 200, 34), {}
    for border in (0, 1 << 30, 112):
        ia.check(ia.lib().ifa_model_set_option(eng.worker(), b"scan_chunk_min", border))
        out[border] = run_whole(eng, toks)[0]
    assert np.array_equal(out[0], out[1 << 30]) and not np.array_equal(out[0], out[112])
    eng.close()


@pytest.mark.parametrize("a16_min", [9, 1])      # (1: the products over bfloat16 rows take steps of a few rows too)
@pytest.mark.parametrize("layer", [fx.parallel_layer(heads=2, kv_heads=1, dim=32, lin_heads=2, lin_dim=16, lin_vdim=40, ff=72), fx.delta_layer(heads=2, kv_heads=1, dim=16, vdim=20, ff=200)],
                         ids=["parallel", "delta"])      # (mixers' outputs of 80 columns, and of 40: fewer than those products take)
def test_norm_and_activation_inside_the_products_of_a_few_rows(tmp_path, layer, a16_min):
    """Every combination of the two (fuse_rows), each operation in a launch of its own otherwise, after a step of other values in the same buffers: one row, two, eight and a step that is too
    large for either, against the oracle"""
    import inferflow_amd as ia
    cfg = fx.config([layer, layer], width=72, vocab=97)
    w, toks = fx.random_weights(cfg, 71), tokens_for(cfg, 40, 72)
    want = oracle_logits(cfg, w, toks)
    eng = engine_for(tmp_path, cfg, w, "bfloat16", 64, 2)
    for name, value in ((b"fuse_step", 0), (b"a16_min", a16_min)):
        ia.check(ia.lib().ifa_model_set_option(eng.worker(), name, value))
    for fused in (0, 1, 2, 3):
        ia.check(ia.lib().ifa_model_set_option(eng.worker(), b"fuse_rows", fused))
        for n in (1, 2, 8, 11):
            run_whole(eng, tokens_for(cfg, 12, 73))
            lg = run_whole(eng, toks[:n])[0]
            assert fx.rel_err(lg, want[:n]).max() < (TOL32 if n <= 8 < a16_min else TOL16), (fused, n)
    eng.close()


@pytest.mark.parametrize("ctx", [340, 60])      # keys of a head by six workgroups whose shares the last launch joins / by one
def test_single_token_steps_in_few_launches(tmp_path, ctx):
    """Steps of one token whose layers' sizes allow the norm inside the input product, both mixers in one launch and everything behind them in another: against the
    oracle and against the same engine with one launch per operation; a layer without feed-forward, windows above and below the context, two norm groups' sizes."""
    import inferflow_amd as ia
    cfg = fx.config([fx.parallel_layer(heads=4, kv_heads=2, dim=64, window=2000, keep_first=0, lin_heads=3, lin_dim=64, lin_vdim=96, ff=200),
                     fx.delta_layer(heads=4, kv_heads=2, dim=16, vdim=32, conv=3, ff=96),
                     fx.parallel_layer(heads=3, kv_heads=1, dim=100, window=50, keep_first=5, lin_heads=2, lin_dim=128, lin_vdim=40, ff=0),
                     fx.delta_layer(heads=2, kv_heads=2, dim=32, vdim=128, conv=1, ff=0)], width=136, vocab=97)
    w = fx.random_weights(cfg, 21)
    n = ctx - 20
    toks = tokens_for(cfg, n + 12, 22)
    want = oracle_logits(cfg, w, toks)
    rows = []
    for fused in (1, 0):
        eng = engine_for(tmp_path, cfg, w, ctx=ctx, queries=2)
        ia.check(ia.lib().ifa_model_set_option(eng.worker(), b"fuse_step", fused))
        eng.add_query(toks[:5]); eng.infer()                  # (another query's slot and cache beside it)
        q = eng.add_query(toks[:n])
        got = []
        for t in toks[n:]:
            eng.infer(); got.append(eng.last_logits_f32(q)[-1])
            assert eng.commit({q: t})
        eng.infer(); got.append(eng.last_logits_f32(q)[-1])
        rows.append(np.stack(got)); eng.close()
    assert fx.rel_err(rows[0], want[n - 1:]).max() < TOL32 and fx.rel_err(rows[1], want[n - 1:]).max() < TOL32
    assert fx.rel_err(rows[0][1:], rows[1][1:]).max() < TOL32


@pytest.mark.parametrize("ctx", [400, 4200])      # (4200: the first layer may have more than 4096 keys in view, for which its steps keep a launch per mixer)
def test_generation_replays_the_single_token_launches(tmp_path, ctx):
    """The captured step (cache rows, states, shares of the keys from the capture on) over the edges of a window and of several shares of 64 keys, with the fused launches and
    with one launch per operation: the oracle's tokens, a prompt in between"""
    import inferflow_amd as ia
    cfg = fx.config([fx.parallel_layer(heads=4, kv_heads=2, dim=64, window=5000, keep_first=0, lin_heads=3, lin_dim=64, lin_vdim=96, ff=72),
                     fx.delta_layer(heads=4, kv_heads=2, dim=64, vdim=32, conv=3, ff=96),
                     fx.parallel_layer(heads=3, kv_heads=1, dim=100, window=150, keep_first=5, lin_heads=2, lin_dim=128, lin_vdim=40, ff=0)], width=136, vocab=97)
    w = fx.random_weights(cfg, 51)
    prompt = tokens_for(cfg, 120, 52)
    for fused in (1, 0):
        eng = engine_for(tmp_path, cfg, w, ctx=ctx, queries=2)
        ia.check(ia.lib().ifa_model_set_option(eng.worker(), b"fuse_step", fused))
        for _ in range(2):
            q = eng.add_query(prompt)
            gen, _ = eng.generate(q, 40)
            eng.remove_query(q)
            want = oracle_logits(cfg, w, prompt + gen)
            for i, tok in enumerate(gen):
                row = want[len(prompt) - 1 + i]
                assert row[tok] > row.max() - 1e-3 * np.abs(row).max(), (fused, i)
            run_whole(eng, tokens_for(cfg, 200, 53))
        eng.close()


def test_capped_logits_of_a_single_row(tmp_path):
    """A model made through the C API with position vectors (stem 0) and a soft cap on its logits: a step of one token, whose head has the norm inside, and the first row of a
    step of three leave the same capped logits"""
    import ctypes as C
    import re
    import inferflow_amd as ia
    text = re.sub(r"/\*.*?\*/", "", open(os.path.join(ROOT, "include", "inferflow_amd.h")).read(), flags=re.S)

    def struct(name):
        body = re.findall(r"typedef struct \{([^}]*)\} %s;" % name, text)[0]
        fields = [(f.strip(), {"int": C.c_int, "float": C.c_float}[t]) for t, names in re.findall(r"(int|float) ([^;]+);", body) for f in names.split(",")]
        return type(name, (C.Structure,), {"_fields_": fields})()
    names = [n.split("=")[0].strip() for n in re.findall(r"enum \{\s*(IFA_LT_NORM1 = 40[^}]*)\}", text)[0].split(",")]
    ids = {n[len("IFA_LT_"):]: 40 + i for i, n in enumerate(names)}
    cfg, L = fx.config([fx.delta_layer(heads=2, kv_heads=1, dim=16, vdim=16, conv=2, ff=0)], width=32, vocab=37), ia.lib()
    w = fx.random_weights(cfg, 61)
    c, sp = struct("ifa_layered_config"), struct("ifa_layer_spec")
    c.width, c.vocab, c.max_ctx, c.n_layers, c.ops32, c.eps, c.pos_base, c.logit_softcap = 32, 37, 64, 1, 1, 1e-5, 10000.0, 0.25
    sp.mixer, sp.d_heads, sp.d_kv_heads, sp.d_dim, sp.d_vdim, sp.d_conv = 2, 2, 1, 16, 16, 2
    m = C.c_void_p()
    ia.check(L.ifa_model_create_layered(C.byref(c), C.byref(sp), C.byref(m)))
    tensors = {(-1, 0): "embed", (-1, 1): "final.norm", (-1, 3): "head"}
    for tid, leaf in (("NORM1", "norm1"), ("LS1", "ls1"), ("D_Q", "mix.q"), ("D_K", "mix.k"), ("D_V", "mix.v"), ("D_QCONV", "mix.q.conv"), ("D_KCONV", "mix.k.conv"),
                      ("D_VCONV", "mix.v.conv"), ("D_B", "mix.b"), ("D_A", "mix.a"), ("D_ALOG", "mix.A_log"), ("D_DTBIAS", "mix.dt_bias"), ("D_G", "mix.g"), ("D_NORM", "mix.norm"),
                      ("D_O", "mix.o")):
        tensors[(0, ids[tid])] = "l0." + leaf
    bf16 = int(re.search(r"IFA_BF16 = (\d+)", text).group(1))
    for (layer, tid), name in tensors.items():
        a = np.atleast_2d(orc.bf16_bits(w[name]))
        ia.check(L.ifa_model_set_tensor_host(m, layer, tid, bf16, a.ctypes.data_as(C.c_void_p), *a.shape))
    ia.check(L.ifa_model_finalize(m))

    def step(tokens):
        ints = lambda *v: (C.c_int * len(v))(*v)
        ia.check(L.ifa_model_step_seqs(m, 1, ints(*tokens), ints(len(tokens)), ints(0), ints(0), 1, ints(0)))
        d, r, k = C.c_void_p(), C.c_size_t(), C.c_size_t()
        ia.check(L.ifa_model_logits_f32(m, C.byref(d), C.byref(r), C.byref(k)))
        out = np.empty((r.value, k.value), np.float32)
        ia.check(L.ifa_memcpy_d2h(out.ctypes.data_as(C.c_void_p), d, out.nbytes, None)); ia.check(L.ifa_stream_sync(None))
        return out
    one, three = step([5]), step([5, 9, 2])
    want = 0.25 * np.tanh(oracle_logits(cfg, w, [5, 9, 2]) / 0.25)
    assert one.shape == (1, 37) and fx.rel_err(one, want[:1]).max() < TOL32 and fx.rel_err(three, want).max() < TOL32
    L.ifa_model_destroy(m)


@pytest.mark.parametrize("K", [8, 120, 512, 520, 1024, 1032, 2048, 2056, 4096])
@pytest.mark.parametrize("N", [1, 5, 4099])
def test_one_row_product_with_the_norm_inside(K, N):
    import inferflow_amd as ia
    from tests.gpu_util import capi, p
    from tests.test_gpu_layered_ops import dev32, devbf
    rng = np.random.default_rng(K + N)
    W, bias, g = orc.bf16_round(rng.standard_normal((N, K)) / K ** 0.5), orc.bf16_round(rng.standard_normal(N)), orc.bf16_round(1 + 0.2 * rng.standard_normal(K))
    x = (2 * rng.standard_normal((1, K)) + 1).astype(np.float32)
    c = torch.full((N + 3,), float("nan"), dtype=torch.float32, device="cuda")
    ia.check(capi().ifa_linear_bf16w_rows(1, p(devbf(g)), 1e-5, p(devbf(W)), N, K, p(dev32(x)), K, 1, p(devbf(bias)), None, 1.0, 0, p(c), N + 3, 2, 4, None))
    want = (orc.layer_norm_nobias(orc.t64(x), orc.t64(g), 1e-5) @ orc.t64(W).T + orc.t64(bias))[0]
    want[2:4] = orc.silu(want[2:4])
    got = c.cpu().numpy()
    assert np.abs(got[:N] - want.numpy()).max() < 1e-5 * max(1.0, float(want.abs().max())) and np.isnan(got[N:]).all()


@pytest.mark.parametrize("start,steps", [(1010, 40), (1000, 25), (1024, 9)])
def test_generation_across_the_end_of_the_ring_of_tokens(tmp_path, start, steps):
    """the ring holds 1024 tokens by position: a call that ends at its last place, one that runs on from its first and one that starts there give the tokens that single steps do"""
    cfg = fx.config([fx.parallel_layer(), fx.delta_layer()])
    eng = engine_for(tmp_path, cfg, fx.random_weights(cfg, 61), ctx=1100, queries=1)
    prompt = tokens_for(cfg, start, 7)
    q = eng.add_query(prompt)
    gen, _ = eng.generate(q, steps)
    eng.remove_query(q)
    q = eng.add_query(prompt)
    one = []
    for _ in range(steps):
        t = eng.infer()[0][1]
        one.append(t)
        assert eng.commit({q: t})
    eng.remove_query(q)
    assert list(gen) == one
    eng.close()
