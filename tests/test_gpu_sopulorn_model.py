"""The layer-list worker serving Sopulorn models through the InferenceEngine (registry, expert stacking, slots, scheduler, sampling entry
points) against the float64 oracle of tests/sopulorn_oracle.py: whole prompts, the residual after every layer, token-by-token decoding,
portions, mixed batches with slots reused, far keys at the edges of key blocks and key shares, the first tokens of a sequence, long
decoding, other sizes, greedy generation, the trace tool."""
import json
import os
import subprocess

import numpy as np
import pytest
import torch

from tests import sopulorn_fixtures as fx
from tests import sopulorn_oracle as orc
from tests.gelarax_oracle import bf16_round

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TOL32 = 2e-5        # fp32 operands: rounding of fp32 sums only
TOL16 = 4e-2        # operands of the matrix products rounded to bfloat16


def assert_close(err, dtype, tol, what=None):
    """fp32: every row within tol.  bfloat16 operands: a router's close call may fall the other way for a row (its experts change, a
    discrete step), so most rows must be within tol and no row far off."""
    if dtype == "float32":
        assert err.max() < tol, (what, err.max())
    else:
        assert np.quantile(err, 0.85) < tol and err.max() < 0.35, (what, np.quantile(err, 0.85), err.max())


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


# a dense layer first, mixtures behind it, two layers on the rows of layer 1, a layer without feed-forward, grouped queries (2 and 3 per
# key head), part of the head rotated, value heads smaller and larger than key heads
MIXED = fx.config([fx.attention_layer(heads=4, kv_heads=2, dim=24, vdim=16, rot_dims=24, mlp=fx.dense()),
                   fx.attention_layer(heads=6, kv_heads=2, dim=16, vdim=40, rot_dims=8, base=500.0),
                   fx.attention_layer(heads=6, kv_heads=2, dim=16, vdim=40, rot_dims=8, base=500.0, kv_from=1, mlp=fx.moe(experts=3, top=1, ff=40, shared=0)),
                   fx.attention_layer(heads=2, kv_heads=2, dim=16, vdim=40, rot_dims=8, base=500.0, kv_from=1, mlp=None),
                   fx.attention_layer(heads=3, kv_heads=1, dim=8, vdim=8, rot_dims=6, mlp=fx.moe(experts=5, top=3, ff=12, shared=20))],
                  width=64, vocab=97)


@pytest.mark.parametrize("dtype,tol", [("float32", TOL32), ("bfloat16", TOL16)])
def test_whole_prompt_matches_the_oracle(tmp_path, dtype, tol):
    w = fx.random_weights(MIXED, 1)
    toks = tokens_for(MIXED, 71, 2)
    eng = engine_for(tmp_path, MIXED, w, dtype)
    lg, nxt = run_whole(eng, toks)
    want = oracle_logits(MIXED, w, toks)
    assert lg.shape == want.shape
    assert_close(fx.rel_err(lg, want), dtype, tol)
    if dtype == "float32":
        assert nxt == int(want[-1].argmax())
    eng.close()


def test_residual_after_every_layer_matches_the_oracle(tmp_path):
    import ctypes as C
    import inferflow_amd as ia
    w = fx.random_weights(MIXED, 3)
    eng = engine_for(tmp_path, MIXED, w)
    L = ia.lib()
    ia.check(L.ifa_model_set_option(eng.worker(), b"tap_layers", 1))
    for n in (40, 5):          # the tiled and the single-row attention, the grouped and the row form of the experts
        toks = tokens_for(MIXED, n, 4)
        run_whole(eng, toks)
        res = []
        with torch.no_grad():
            orc.forward(MIXED, fx.oracle_weights(w), toks, res)
        for li, want in enumerate(res):
            p, b = C.c_void_p(), C.c_size_t()
            ia.check(L.ifa_model_get_buffer(eng.worker(), b"layer_taps", li, C.byref(p), C.byref(b)))
            got = np.zeros((len(toks), MIXED["width"]), np.float32)
            ia.check(L.ifa_memcpy_d2h(got.ctypes.data_as(C.c_void_p), p, got.nbytes, None)); ia.check(L.ifa_stream_sync(None))
            assert np.abs(got - want.numpy()).max() < 2e-4 * max(1.0, np.abs(want.numpy()).max()), (n, li)
    eng.close()


@pytest.mark.parametrize("sizes", [[1], [2], [5, 3], [30, 1], [7, 2, 1], [64, 4], [17, 16, 2]])
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


def test_both_norms_between_sub_layers_as_one_launch_and_as_separate_ops_agree(tmp_path):
    import inferflow_amd as ia
    w = fx.random_weights(MIXED, 25)
    toks = tokens_for(MIXED, 60, 26)
    want = oracle_logits(MIXED, w, toks)
    eng = engine_for(tmp_path, MIXED, w)
    for fuse in (1, 0, 1):
        ia.check(ia.lib().ifa_model_set_option(eng.worker(), b"fuse_post", fuse))
        for sizes in ([33, 1], [3, 2], [8, 7, 1]):
            assert fx.rel_err(run_portions(eng, toks, sizes), want).max() < TOL32, (fuse, sizes)
    eng.close()


@pytest.mark.parametrize("n", [1, 2, 3])
def test_first_tokens_of_a_sequence(tmp_path, n):
    """the shortest prompts, whole and token by token, on a slot that held a longer sequence before (its cache rows and its last token)"""
    cfg = fx.config([fx.attention_layer(mlp=fx.dense()), fx.attention_layer(kv_from=0)])
    w = fx.random_weights(cfg, 21)
    eng = engine_for(tmp_path, cfg, w, queries=1)
    run_whole(eng, tokens_for(cfg, 50, 22))
    toks = tokens_for(cfg, n, 23 + n)
    want = oracle_logits(cfg, w, toks)
    assert fx.rel_err(run_whole(eng, toks)[0], want).max() < TOL32
    assert fx.rel_err(run_portions(eng, toks, [1]), want).max() < TOL32
    eng.close()


def test_batches_of_unequal_requests_equal_each_alone_and_slots_are_reused(tmp_path):
    w = fx.random_weights(MIXED, 7)
    eng = engine_for(tmp_path, MIXED, w, queries=3)
    prompts = [tokens_for(MIXED, n, 10 + n) for n in (1, 37, 64, 5, 90, 2)]
    tails = [tokens_for(MIXED, 12, 50 + i) for i in range(len(prompts))]
    alone = [oracle_logits(MIXED, w, p + t) for p, t in zip(prompts, tails)]
    # three queries on three slots, twice: the second time reuses the slots of the first
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


def marked_model(shared_rows):
    """Attention whose weights make one key stand out: the token `probe` has a query that matches the key of token `mark` in a head
    dimension that does not rotate, so the match holds at any distance.  The last row's logits then depend strongly on whether the
    mark's cache row is read, wherever it lies.  shared_rows: a second layer reads the first layer's rows with the same kind of query."""
    D = 16
    layers = [fx.attention_layer(heads=2, kv_heads=1, dim=D, vdim=24, rot_dims=8, scale=1.0, mlp=None)]
    if shared_rows:
        layers.append(fx.attention_layer(heads=2, kv_heads=1, dim=D, vdim=24, rot_dims=8, scale=1.0, kv_from=0, mlp=None))
    cfg = fx.config(layers, width=32, vocab=50, bigram=None)
    w = fx.random_weights(cfg, 9)
    mark, probe = 7, 9
    e = w["embed"]
    e[mark] = 0; e[probe] = 0
    e[mark, 0] = 8.0; e[probe, 1] = 8.0
    for li in range(len(layers)):
        p = "l%d." % li
        w[p + "norm1"][:2] = 0
        q = w[p + "mix.q"]; q[:, :2] = 0
        for h in range(2):
            q[h * D + D - 1, 1] = 4.0                      # feature 1 (the probe) drives the last dimension of every query head
        w[p + "mix.q.b"][:] = 0
        w[p + "mix.q.norm"][D - 1] = 2.0
        if li == 0:
            k = w[p + "mix.k"]; k[:, :2] = 0
            k[D - 1, 0] = 4.0                              # feature 0 (the mark) drives the last dimension of the key head
            w[p + "mix.k.b"][:] = 0
            w[p + "mix.k.norm"][D - 1] = 2.0
    if shared_rows:
        w["l0.norm1b"][:2] = -1.0                          # the first layer leaves features 0 and 1 as they were
    return cfg, {k_: bf16_round(v) for k_, v in w.items()}, mark, probe


@pytest.mark.parametrize("shared_rows", [False, True])
def test_far_keys_at_block_and_share_edges_in_prompts_and_decoding(tmp_path, shared_rows):
    """the marked key at the borders of the tiled kernel's key blocks (32) and query tiles (128) and of the single-row kernel's
    key shares (16 keys a wave step), hundreds of tokens back"""
    cfg, w, mark, probe = marked_model(shared_rows)
    eng = engine_for(tmp_path, cfg, w, ctx=700)
    filler = [t for t in range(10, 50)]
    for mark_at, n in ((0, 2), (0, 33), (31, 300), (32, 300), (63, 129), (64, 129), (127, 128), (128, 130), (15, 600), (16, 600), (255, 257), (256, 258), (5, 640)):
        toks = [filler[(3 * i + mark_at + n) % len(filler)] for i in range(n)]
        toks[mark_at] = mark; toks[-1] = probe
        want = oracle_logits(cfg, w, toks)
        whole, _ = run_whole(eng, toks)
        assert fx.rel_err(whole, want).max() < TOL32, ("prompt", mark_at, n)
        dec = run_portions(eng, toks, [max(1, n - 3), 1])
        assert fx.rel_err(dec, want).max() < TOL32, ("decoded", mark_at, n)
        # the oracle itself must see the key: without the mark the last row differs clearly
        blind = list(toks); blind[mark_at] = filler[0]
        assert fx.rel_err(oracle_logits(cfg, w, blind)[-1:], want[-1:]).max() > 1e-3, (mark_at, n)
    eng.close()


def test_long_decoding_far_from_the_start(tmp_path):
    cfg = fx.config([fx.attention_layer(heads=2, kv_heads=1, dim=16, vdim=8, rot_dims=16, base=200.0, mlp=fx.moe(experts=4, top=2, ff=16, shared=8)),
                     fx.attention_layer(heads=2, kv_heads=1, dim=16, vdim=8, rot_dims=16, base=200.0, kv_from=0, mlp=fx.dense(ff=24, limit=0.7))], width=32, vocab=61)
    w = fx.random_weights(cfg, 11)
    toks = tokens_for(cfg, 330, 12)
    want = oracle_logits(cfg, w, toks)
    eng = engine_for(tmp_path, cfg, w, ctx=400)
    got = run_portions(eng, toks, [200, 1])        # 130 tokens decoded one by one
    assert fx.rel_err(got, want).max() < 5e-5
    eng.close()


CASES = {
    # one head, one expert of which one is chosen, a pair table of one bucket, two rotated dimensions, value heads of one number
    "ones": lambda: fx.config([fx.attention_layer(heads=1, kv_heads=1, dim=2, vdim=1, rot_dims=2, mlp=fx.moe(experts=1, top=1, ff=4, shared=4)),
                               fx.attention_layer(heads=1, kv_heads=1, dim=4, vdim=4, rot_dims=2, mlp=fx.dense(ff=8, limit=1.0))], width=16, vocab=11, bigram=(1, 1, 1)),
    # no pair table, no rotation, no feed-forward in one layer, every expert chosen, no shared expert
    "plain": lambda: fx.config([fx.attention_layer(rot_dims=0, mlp=None), fx.attention_layer(rot_dims=0, mlp=fx.moe(experts=3, top=3, ff=12, shared=0))],
                               width=48, vocab=33, bigram=None),
    # sizes that keep every 16-byte path off: odd head sizes, width 14
    "unaligned": lambda: fx.config([fx.attention_layer(heads=3, kv_heads=1, dim=5, vdim=7, rot_dims=4, mlp=fx.moe(experts=3, top=2, ff=10, shared=6)),
                                    fx.attention_layer(heads=2, kv_heads=2, dim=7, vdim=3, rot_dims=2, mlp=fx.dense(ff=9, limit=0.5))], width=14, vocab=9, bigram=(7, 3, 2)),
    # the widest heads the tiled kernel takes, all of them rotated
    "wide_heads": lambda: fx.config([fx.attention_layer(heads=2, kv_heads=1, dim=128, vdim=128, rot_dims=128, mlp=fx.moe(experts=4, top=2, ff=64, shared=32)),
                                     fx.attention_layer(heads=4, kv_heads=1, dim=128, vdim=128, rot_dims=64, kv_from=0, mlp=None)], width=128, vocab=50),
    # heads beyond the tiled kernel: prompts take the single-row form too
    "beyond_the_tile": lambda: fx.config([fx.attention_layer(heads=2, kv_heads=2, dim=160, vdim=136, rot_dims=96, mlp=fx.dense(ff=32, limit=2.0))], width=64, vocab=23),
    # many experts, eight chosen
    "many_experts": lambda: fx.config([fx.attention_layer(mlp=fx.moe(experts=70, top=8, ff=16, shared=24))], width=32, vocab=29),
    # every later layer on the rows of the first; as many key heads as query heads; a limit that clamps nearly everything; a large hash
    "one_cache": lambda: fx.config([fx.attention_layer(heads=2, kv_heads=2, dim=32, vdim=32, mlp=fx.dense(ff=40, limit=0.05))]
                                   + [fx.attention_layer(heads=2, kv_heads=2, dim=32, vdim=32, kv_from=0, mlp=fx.dense(ff=40, limit=0.05)) for _ in range(3)],
                                   width=32, vocab=40, bigram=(2039, 40009, 65537)),
}


@pytest.mark.parametrize("case", sorted(CASES))
def test_other_sizes(tmp_path, case):
    cfg = CASES[case]()
    w = fx.random_weights(cfg, 13)
    toks = tokens_for(cfg, 45, 14)
    want = oracle_logits(cfg, w, toks)
    for dtype, tol in (("float32", TOL32), ("bfloat16", TOL16)):
        eng = engine_for(tmp_path, cfg, w, dtype)
        whole, _ = run_whole(eng, toks)
        assert_close(fx.rel_err(whole, want), dtype, tol, (case, dtype))
        assert_close(fx.rel_err(run_portions(eng, toks, [20, 9, 1]), want), dtype, tol, (case, dtype, "portions"))
        eng.close()


def test_router_bias_decides_the_choice(tmp_path):
    """a large bias moves the choice to experts whose logits are small; the weights are the softmax over the chosen values"""
    cfg = fx.config([fx.attention_layer(mlp=fx.moe(experts=5, top=2, ff=16, shared=0))], width=32, vocab=31)
    w = fx.random_weights(cfg, 31)
    b = w["l0.mlp.router.b"]
    b[:] = 0; b[4] = 30.0; b[1] = 29.0
    w = {k: bf16_round(v) for k, v in w.items()}
    toks = tokens_for(cfg, 40, 32)
    eng = engine_for(tmp_path, cfg, w)
    want = oracle_logits(cfg, w, toks)
    assert fx.rel_err(run_whole(eng, toks)[0], want).max() < TOL32
    assert fx.rel_err(run_portions(eng, toks, [1]), want).max() < TOL32
    plain = dict(w); plain["l0.mlp.router.b"] = np.zeros_like(b)
    assert fx.rel_err(oracle_logits(cfg, plain, toks), want).max() > 1e-3
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
    # a second generation on the same slot replays the captured step against a new sequence (and its own previous token)
    q = eng.add_query(prompt[:7])
    gen2, _ = eng.generate(q, 10)
    eng.remove_query(q)
    want2 = oracle_logits(MIXED, w, prompt[:7] + gen2)
    for i, tok in enumerate(gen2):
        row = want2[6 + i]
        top2 = np.sort(row)[-2:]
        if top2[1] - top2[0] > 1e-3 * np.abs(row).max():
            assert tok == int(row.argmax()), i
    # sampled queries draw from the same logits (top-k with a seed: reproducible)
    a = eng.add_query(prompt, strategy="sample.top_k", seed=5)
    b = eng.add_query(prompt, strategy="sample.top_k", seed=5)
    out = dict(eng.infer())
    assert out[a] == out[b] and 0 <= out[a] < MIXED["vocab"]
    eng.close()


@pytest.mark.parametrize("graph", [1, 0])
def test_generation_over_key_block_edges_with_single_rows_sent_to_the_tiles(tmp_path, graph):
    """attn_tile_min 1: the launches of a decode step are shaped once and the position then advances on the device, over the edges of blocks of 32 keys and of the
    shares of a key range (127 -> 128), a longer prompt growing the prompts' workspace in between"""
    import inferflow_amd as ia
    w = fx.random_weights(MIXED, 21)
    prompt, other = tokens_for(MIXED, 100, 22), tokens_for(MIXED, 300, 23)
    eng = engine_for(tmp_path, MIXED, w)
    for name, value in ((b"attn_tile_min", 1), (b"graph", graph)):
        ia.check(ia.lib().ifa_model_set_option(eng.worker(), name, value))
    for _ in range(2):
        q = eng.add_query(prompt)
        gen, _ = eng.generate(q, 70)
        eng.remove_query(q)
        want = oracle_logits(MIXED, w, prompt + gen)
        for i, tok in enumerate(gen):
            row = want[len(prompt) - 1 + i]
            assert row[tok] > row.max() - 1e-3 * np.abs(row).max(), i
        lg, _ = run_whole(eng, other)
        assert fx.rel_err(lg, oracle_logits(MIXED, w, other)).max() < TOL32
    eng.close()


@pytest.mark.parametrize("T", [9, 17, 130, 601, 1500])
def test_experts_over_the_rows_that_the_norm_has_left_in_bfloat16(tmp_path, T):
    """Prompts whose norms leave bfloat16 rows for experts and shared expert, between dense layers whose activations are formed in the tiles of their product, inner sizes of whole and of broken
    steps: the bits of every operand stored in 32 bits and rounded on its way into a product (a16_min 0), and the oracle"""
    import inferflow_amd as ia
    cfg = fx.config([fx.attention_layer(heads=4, kv_heads=2, dim=32, vdim=32, mlp=fx.dense(ff=1032, limit=1.5)),
                     fx.attention_layer(heads=4, kv_heads=2, dim=32, vdim=48, mlp=fx.moe(experts=5, top=2, ff=200, shared=72)),
                     fx.attention_layer(heads=4, kv_heads=2, dim=32, vdim=48, kv_from=1, mlp=fx.moe(experts=3, top=1, ff=264, shared=0)),
                     fx.attention_layer(heads=2, kv_heads=2, dim=32, vdim=40, mlp=fx.dense(ff=72))], width=320, vocab=97)
    w, toks, out = fx.random_weights(cfg, 27), tokens_for(cfg, T, 28), {}
    eng = engine_for(tmp_path, cfg, w, "bfloat16", 1536, 1)
    for border in (0, 9):
        run_whole(eng, tokens_for(cfg, 40, 29))          # (other values in the buffers)
        ia.check(ia.lib().ifa_model_set_option(eng.worker(), b"a16_min", border))
        out[border] = run_whole(eng, toks)[0]
    eng.close()
    assert np.array_equal(out[0], out[9])
    if T <= 601:
        assert_close(fx.rel_err(out[9], oracle_logits(cfg, w, toks)), "bfloat16", TOL16, T)


@pytest.mark.parametrize("T", [9, 130])
def test_experts_of_prompts_that_are_sorted_by_one_workgroup(tmp_path, T):
    """bfloat16 rows for experts whose choice goes through launches of its own: a shared expert too narrow for bfloat16 rows, more than 512 experts; the bits of operands rounded on their way
    (a16_min 0), and the oracle"""
    import inferflow_amd as ia
    cfg = fx.config([fx.attention_layer(heads=2, kv_heads=1, dim=32, vdim=32, mlp=fx.moe(experts=5, top=2, ff=200, shared=40)),
                     fx.attention_layer(heads=2, kv_heads=1, dim=32, vdim=32, mlp=fx.moe(experts=520, top=3, ff=64, shared=72))], width=448, vocab=97)
    w, toks, out = fx.random_weights(cfg, 37), tokens_for(cfg, T, 38), {}
    eng = engine_for(tmp_path, cfg, w, "bfloat16", 192, 1)
    for border in (0, 9):
        run_whole(eng, tokens_for(cfg, 40, 39))
        ia.check(ia.lib().ifa_model_set_option(eng.worker(), b"a16_min", border))
        out[border] = run_whole(eng, toks)[0]
    eng.close()
    assert np.array_equal(out[0], out[9])
    assert_close(fx.rel_err(out[9], oracle_logits(cfg, w, toks)), "bfloat16", TOL16, T)


def test_generation_over_bfloat16_rows_of_single_tokens_beside_longer_and_longer_prompts(tmp_path):
    """a16_min 1: the captured step reads the buffers of rounded activations, which a longer prompt allocates anew: the tokens of uncaptured steps"""
    import inferflow_amd as ia
    cfg = fx.config([fx.attention_layer(heads=2, kv_heads=1, dim=32, vdim=32, mlp=fx.dense(ff=136, limit=1.5)), fx.attention_layer(heads=4, kv_heads=2, dim=32, vdim=32, mlp=fx.dense(ff=72))],
                    width=128, vocab=97)
    w, seen = fx.random_weights(cfg, 25), {}
    for graph in (1, 0):
        eng = engine_for(tmp_path, cfg, w, "bfloat16")
        for name, value in ((b"a16_min", 1), (b"graph", graph)):
            ia.check(ia.lib().ifa_model_set_option(eng.worker(), name, value))
        for n in (20, 90, 400):
            q = eng.add_query(tokens_for(cfg, n, 26))
            seen.setdefault(graph, []).append(eng.generate(q, 30)[0])
            eng.remove_query(q)
        eng.close()
    assert seen[1] == seen[0] and all(len(set(t)) > 5 for t in seen[0])


def test_heads_above_128_share_their_keys_out_in_steps_of_a_few_rows(tmp_path):
    """heads that no tile takes go row by row, a few rows' keys shared out to several workgroups whatever border the tiles have: the same bits"""
    import inferflow_amd as ia
    cfg = fx.config([fx.attention_layer(heads=2, kv_heads=1, dim=160, vdim=144, rot_dims=32)], width=64, vocab=97)
    eng = engine_for(tmp_path, cfg, fx.random_weights(cfg, 41))
    toks, out = tokens_for(cfg, 420, 42), []
    for border in (16, 1 << 30):
        ia.check(ia.lib().ifa_model_set_option(eng.worker(), b"attn_tile_min", border))
        out.append(run_portions(eng, toks, [400, 20]))
    assert np.array_equal(out[0][400:], out[1][400:])
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
    assert eng.model_info("vocab_size") == MIXED["vocab"] and eng.model_info("decoder_layers") == len(MIXED["layers"])
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
