"""-m gpu: the C++ InferenceEngine facade (LoadConfig -> Init -> AddQuery -> Infer -> Commit) on tiny
llama2.c / safetensors / synthetic model directories, against the whole-model oracle."""
import numpy as np
import pytest

import oracle as o
from inferflow_amd import dtypes as dt
from inferflow_amd.engine import InferenceEngine, EngineError
from tests import engine_fixtures as fx
from tests.model_util import oracle_model_from_host

pytestmark = pytest.mark.gpu


def _oracle(w, wd, kvd, rope_order, ctx=64):
    s = fx.SHAPE
    host = fx.host_tensors(w, s, wd)
    return oracle_model_from_host(host, s, ctx, kvd, rope_order=rope_order, unk_id=0)   # the engine excludes the unk id like GetSortedTopK


def _close(a, b):
    a = a.astype(np.float32); b = b.astype(np.float32)
    cos = float((a * b).sum() / (np.linalg.norm(a) * np.linalg.norm(b) + 1e-30))
    return cos, float(np.abs(a - b).max())


@pytest.mark.parametrize("fmt,wd_name,wd,kv_name,kvd,qk", [
    ("llama2.c", "Q4", dt.Q4_B32T1A, "Q8", dt.Q8_B32T2, 0),
    ("llama2.c", "Q3H", dt.Q3H_B64T1, "F16", dt.F16, 0),
    ("safetensors", "Q8", dt.Q8_B32T2, "Q8", dt.Q8_B32T2, 2),
    ("safetensors", "F16", dt.F16, "F16", dt.F16, 2),
], ids=["llama2c_q4_kvq8", "llama2c_q3h_kvf16", "safetensors_q8_kvq8", "safetensors_f16"])
def test_serving_loop_matches_oracle(tmp_path, fmt, wd_name, wd, kv_name, kvd, qk):
    ini, w = fx.write_model_dir(str(tmp_path), fmt=fmt, wd=wd_name, kvd=kv_name, qk_order=qk)
    eng = InferenceEngine.from_ini(ini)
    assert eng.model_info("decoder_kv_heads") == 2 and eng.model_info("vocab_size") == 1000
    assert eng.model_info("device_weight_data_type") == wd and eng.model_info("device_kv_cache_data_type") == kvd
    om = _oracle(w, wd, kvd, rope_order=2 if qk == 2 else 1)
    prompt = np.random.default_rng(3).integers(3, 1000, 9).astype(np.int32)
    qid = eng.add_query(prompt)
    assert qid > 0 and eng.query_count() == 1
    # step 1 = prefill of the whole prompt, with the full logits tensor (return_output_tensors)
    (q, tok), = eng.infer()
    assert q == qid
    tok_o, lg_o = om.forward(prompt, 0, nthreads=4)
    lg = eng.last_logits(qid)
    assert lg.shape == (9, 1000)
    cos, mad = _close(lg, lg_o)
    assert cos >= 0.9995 and mad <= 0.03, (cos, mad)          # same stated tolerance as tests/test_gpu_engine.py
    cur, pos = tok, len(prompt)
    for step in range(10):
        t_or, l_or = om.forward(np.array([cur], np.int32), pos, nthreads=4)
        assert eng.commit({qid: cur})
        (q, tok), = eng.infer()
        top2 = np.sort(l_or[0].astype(np.float32))[-2:]
        if top2[1] - top2[0] > 0.03:
            assert tok == t_or, "step %d" % step
        cur, pos = tok, pos + 1
    assert eng.infer() == []                 # nothing committed since the last step
    assert eng.remove_query(qid) and eng.query_count() == 0 and not eng.remove_query(qid)
    eng.close()


@pytest.mark.parametrize("net,cfg", [
    # data/models/minicpm_2b_dpo_bf16/model_spec.json: scaled embeddings and output scales
    (dict(has_embedding_linear_norm=True, embedding_linear_scale=12, attn_out_scale=0.25, ffn_out_scale=0.25, out_scale=0.111111),
     dict(embd_scale=12.0, attn_out_scale=0.25, ffn_out_scale=0.25, out_scale=0.111111)),
    # data/models/gemma_2b_it/model_spec.json: LinearNorm with the default scale sqrt(dim), RMS weights 1 + w
    (dict(has_embedding_linear_norm=True, attn_pre_norm_base=1.0, ffn_pre_norm_base=1.0, output_norm_base=1.0),
     dict(embd_scale=-1.0, attn_norm_base=1.0, ffn_norm_base=1.0, out_norm_base=1.0)),
], ids=["minicpm_spec", "gemma_spec"])
def test_linear_norm_and_output_scales_from_the_model_spec(tmp_path, net, cfg):
    """has_embedding_linear_norm / embedding_linear_scale (ProcessPreLayer's LinearNorm, inference_worker.cc:447-451) and the
    three output scales (:568-570, 842-843, 928-929) are read from network_structure and run inside the fused decode launches
    (scale folded into the embedding gather and the Wo / W2 epilogues)."""
    ini, w = fx.write_model_dir(str(tmp_path), fmt="llama2.c", wd="Q4", kvd="F16", net_extra=net, std=0.02 if "out_scale" not in net else 0.06)
    eng = InferenceEngine.from_ini(ini)
    host = fx.host_tensors(w, fx.SHAPE, dt.Q4_B32T1A)
    om = oracle_model_from_host(host, fx.SHAPE, 64, dt.F16, rope_order=1, unk_id=0, **cfg)
    prompt = np.random.default_rng(5).integers(3, 1000, 7).astype(np.int32)
    qid = eng.add_query(prompt)
    (q, tok), = eng.infer()
    tok_o, lg_o = om.forward(prompt, 0, nthreads=4)
    cos, mad = _close(eng.last_logits(qid), lg_o)
    assert cos >= 0.9995 and mad <= 0.02 * float(np.abs(lg_o.astype(np.float32)).max()) + 0.02, (cos, mad)
    cur, pos = tok, len(prompt)
    for step in range(8):
        t_or, l_or = om.forward(np.array([cur], np.int32), pos, nthreads=4)
        assert eng.commit({qid: cur})
        (q, tok), = eng.infer()
        row = eng.last_logits(qid)[0]
        cos, mad = _close(row, l_or[0])
        assert cos >= 0.9995 and mad <= 0.02 * float(np.abs(l_or.astype(np.float32)).max()) + 0.02, (step, cos, mad)
        top2 = np.sort(l_or[0].astype(np.float32))[-2:]
        if top2[1] - top2[0] > 0.03:
            assert tok == t_or, "step %d" % step
        cur, pos = tok, pos + 1
    eng.close()


def test_generate_equals_step_loop_and_queries_are_independent(tmp_path):
    ini, _ = fx.write_model_dir(str(tmp_path), fmt="synthetic", wd="Q4", kvd="F16", ret="false", maxq=2)
    eng = InferenceEngine.from_ini(ini)
    rng = np.random.default_rng(11)
    pa, pb = rng.integers(3, 1000, 7), rng.integers(3, 1000, 5)
    qa = eng.add_query(pa)
    gen, ms = eng.generate(qa, 12)
    assert len(gen) == 12 and ms > 0
    # the same prompt through Infer/Commit on a second query: identical tokens (same kernels, step by step)
    qa2 = eng.add_query(pa)
    assert qa2 > 0
    assert eng.add_query(pb) == 0            # busy: max_concurrent_queries = 2
    assert eng.remove_query(qa)
    out_a = []
    for _ in range(12):
        (q, t), = eng.infer()
        out_a.append(t); eng.commit({qa2: t})
    assert out_a == gen
    # two queries at once: after their prefills they advance together in ONE batched step per Infer() (dynamic
    # batching); swapping the order in which they were added must not change anything
    def run_pair(first, second):
        ids = [eng.add_query(first), eng.add_query(second)]
        assert min(ids) > 0
        outs = {ids[0]: [], ids[1]: []}
        for _ in range(10):
            res = dict(eng.infer())
            assert set(res) == set(ids)
            for q, t in res.items():
                outs[q].append(t)
            eng.commit(res)
        for q in ids:
            eng.remove_query(q)
        return outs[ids[0]], outs[ids[1]]
    eng.remove_query(qa2)
    a1, b1 = run_pair(pa, pb)
    b2, a2 = run_pair(pb, pa)
    assert a1 == a2 and b1 == b2
    # a query decoded alone runs the int8-activation GEMV kernels, a batched one the MFMA GEMM (the reference's two
    # MatrixMultiplication branches): same tokens except at near ties
    assert sum(int(x == y) for x, y in zip(a1, gen[:10])) >= 7
    eng.close()


def test_engine_errors_follow_the_reference_conventions(tmp_path):
    ini, _ = fx.write_model_dir(str(tmp_path), fmt="synthetic", wd="Q4", kvd="Q8", ctx=32)
    eng = InferenceEngine.from_ini(ini)
    assert eng.add_query([]) < 0
    assert eng.add_query([5, 1000]) < 0                      # token id out of range
    assert eng.add_query(list(range(3, 40))) < 0             # longer than max_context_len
    q = eng.add_query([5, 6, 7])
    assert q > 0
    assert not eng.commit({q + 1: 5})                        # unknown query
    assert not eng.commit({q: 99999})
    eng.close()
    bad = str(tmp_path / "bad.ini")
    open(bad, "w").write(open(ini).read().replace("device_weight_data_type = Q4", "device_weight_data_type = Q7"))
    with pytest.raises(EngineError, match="device_weight_data_type"):
        InferenceEngine.from_ini(bad)


@pytest.mark.parametrize("qkv_format", [0, 1])
def test_fused_qkv_checkpoints_load_like_separate_tensors(tmp_path, qkv_format):
    """One self_attn.qkv_proj tensor in either ModelSpec::qkv_format must give exactly the model its separate
    q/k/v_proj tensors give (the reference splits the fused product, the loader splits the rows: same numbers)."""
    outs = []
    for sub, fused in (("sep", None), ("fused", qkv_format)):
        ini, _ = fx.write_model_dir(str(tmp_path / sub), fmt="safetensors", wd="Q4", kvd="F16", qk_order=2, fused_qkv=fused)
        eng = InferenceEngine.from_ini(ini)
        qid = eng.add_query([5, 9, 100, 42, 7])
        (q, tok), = eng.infer()
        lg = eng.last_logits(qid).copy()
        assert eng.commit({qid: tok})
        toks, _ = eng.generate(qid, 8)
        outs.append((tok, lg, toks))
        eng.close()
    assert outs[0][0] == outs[1][0] and outs[0][2] == outs[1][2]
    assert np.array_equal(outs[0][1], outs[1][1])


def test_sampled_queries_draw_from_the_engines_logits_with_the_reference_generator(tmp_path):
    """sample.top_p / sample.std / top_k queries: the engine brings the last logits row to the host and draws with the
    query's java.util.Random generator -- same tokens as oracle/sampling.py on the logits the engine returns; a seed
    reproduces the sequence; greedy and sampled queries share batched steps."""
    from oracle import sampling as S
    ini, _ = fx.write_model_dir(str(tmp_path), fmt="llama2.c", wd="Q4", kvd="F16", maxq=6)        # return_output_tensors = true
    eng = InferenceEngine.from_ini(ini)
    assert eng.strategy_id("sample.top_p") == S.TOP_P and eng.strategy_id("greedy") == S.GREEDY and eng.strategy_id("") == S.GREEDY
    prompt = list(np.random.default_rng(5).integers(3, 1000, 7))

    def run(strategy, seed, temperature, steps=8):
        qid = eng.add_query(prompt, strategy=strategy, seed=seed, temperature=temperature)
        assert qid > 0
        rng, toks = S.JavaRandom(seed), []
        for _ in range(steps):
            (q, tok), = eng.infer()
            lg = eng.last_logits(qid)
            (want, _), _ = S.choose_tokens(lg[-1], eng.strategy_id(strategy), rng, temperature=temperature)
            assert tok == want
            toks.append(tok)
            assert eng.commit({qid: tok})
        assert eng.remove_query(qid)
        return toks

    a = run("sample.top_p", 11, 1.0)
    assert run("sample.top_p", 11, 1.0) == a                    # same seed, same text
    b = run("sample.std", 12, 1.3)
    c = run("top_k", 13, 0.8)
    assert len({tuple(a), tuple(b), tuple(c)}) == 3
    # three queries advance together (dynamic batching from 2 queries on in this .ini): two sampled, one greedy
    q1 = eng.add_query(prompt, strategy="sample.std", seed=21, temperature=1.5)
    q2 = eng.add_query(prompt)
    q3 = eng.add_query(prompt, strategy="top_k", seed=23)
    rngs = {q1: (S.JavaRandom(21), S.STD, 1.5), q3: (S.JavaRandom(23), S.TOP_K, 1.0)}
    for _ in range(5):
        res = dict(eng.infer())
        assert set(res) == {q1, q2, q3}
        for q, (rng, sid, temp) in rngs.items():
            (want, _), _ = S.choose_tokens(eng.last_logits(q)[-1], sid, rng, temperature=temp)
            assert res[q] == want
        assert res[q2] == int(np.argmax(eng.last_logits(q2)[-1].astype(np.float32)))
        assert eng.commit(res)
    for q in (q1, q2, q3):
        assert eng.remove_query(q)
    # every other strategy of the reference runs too (host side, tests/test_sampling_cpu.py); ids out of range are refused
    for name in ("fsd", "random_fsd", "min_p", "tfs", "typical", "mirostat"):
        q = eng.add_query(prompt, strategy=name, seed=5)
        assert q > 0, name
        for _ in range(3):
            (qq, tok), = eng.infer()
            assert 0 <= tok < 1000 and eng.commit({q: tok})
        assert eng.remove_query(q)
    assert eng.add_query(prompt, strategy=99) < 0 and "Invalid strategy id" in InferenceEngine._err()
    eng.close()


def test_model_decoding_strategy_from_the_ini(tmp_path):
    ini, _ = fx.write_model_dir(str(tmp_path), fmt="llama2.c", wd="Q4", kvd="F16", ret="false")
    text = open(ini).read().replace("prompt_template =", 'decoding_strategy = {"name":"sample.top_p", "top_p":0.5, "max_k":3}\nprompt_template =')
    open(ini, "w").write(text)
    eng = InferenceEngine.from_ini(ini)
    assert eng.strategy_id("") == 4                               # Auto resolves to the model's strategy
    qid = eng.add_query([1, 5, 9, 200], seed=3)                   # strategy Auto
    seen = set()
    for _ in range(12):
        (q, tok), = eng.infer()
        seen.add(tok)
        assert eng.commit({qid: tok})
    assert len(seen) > 1                                          # not the greedy fixed point of this tiny model
    eng.close()
    open(ini, "w").write(text.replace('{"name":"sample.top_p", "top_p":0.5, "max_k":3}', "sample.nonsense"))
    with pytest.raises(EngineError, match="Invalid decoding_strategy"):
        InferenceEngine.from_ini(ini)


def test_per_tensor_weight_types_from_the_ini(tmp_path):
    """device_weight_data_type.<tensor> (inference_engine.cc:1664-1690, network_builder.cc:1551-1555): the named tensors take their own
    type, every other matrix the global one; element sizes >= 2 mean F16."""
    from inferflow_amd import worker as W
    ini, _ = fx.write_model_dir(str(tmp_path), fmt="llama2.c", wd="Q4", kvd="F16", ret="false")
    text = open(ini).read().replace("device_weight_data_type = Q4", "device_weight_data_type = Q4\ndevice_weight_data_type.ffn_w2 = Q8\ndevice_weight_data_type.attn_wo = F32")
    open(ini, "w").write(text)
    eng = InferenceEngine.from_ini(ini)
    got = {tid: eng.worker_tensor(0, 0, tid)[0] for tid in (W.T_WQ, W.T_WO, W.T_W1, W.T_W2, W.T_W3)}
    assert got[W.T_W2] == dt.Q8_B32T2 and got[W.T_WO] == dt.F16
    assert got[W.T_WQ] == got[W.T_W1] == got[W.T_W3] == dt.Q4_B32T1A
    qid = eng.add_query([1, 5, 9, 200])
    (q, tok), = eng.infer()                                       # the mixed model runs (W2 on the int8 Q8 path, Wo as an F16 GEMV)
    assert q == qid and 0 <= tok < fx.SHAPE["vocab"]
    eng.close()


# ---- mixture of experts through the .ini surface
@pytest.mark.parametrize("devices,tp_merge", [("0", 1), ("0&0", 2)], ids=["one_worker", "tensor_parallel_2"])
def test_moe_safetensors_checkpoint_through_the_engine_matches_oracle(tmp_path, devices, tp_merge):
    """A Mixtral-named safetensors checkpoint (block_sparse_moe.gate / experts.{j}.w1|w2|w3, 4 experts, top-2) loaded by
    host/model_loader.cc: prefill logits and greedy decode against the whole-model oracle -- on one worker and over a
    tensor-parallel device group (every rank holds its slice of every expert; merge restated in the oracle)."""
    s = fx.MOE_SHAPE
    ini, w = fx.write_model_dir(str(tmp_path), fmt="safetensors", wd="Q4", kvd="F16", qk_order=2, s=s, devices=devices)
    eng = InferenceEngine.from_ini(ini)
    host = fx.host_tensors(w, s, dt.Q4_B32T1A)
    om = oracle_model_from_host(host, s, 64, dt.F16, rope_order=2, unk_id=0, **({"tp_merge": tp_merge} if tp_merge > 1 else {}))
    prompt = np.random.default_rng(8).integers(3, 1000, 11).astype(np.int32)
    qid = eng.add_query(prompt)
    (q, tok), = eng.infer()
    tok_o, lg_o = om.forward(prompt, 0, nthreads=4)
    cos, mad = _close(eng.last_logits(qid), lg_o)
    assert cos >= 0.9995 and mad <= 0.03, (cos, mad)
    cur, pos = tok, len(prompt)
    for step in range(8):
        t_or, l_or = om.forward(np.array([cur], np.int32), pos, nthreads=4)
        assert eng.commit({qid: cur})
        (q, tok), = eng.infer()
        top2 = np.sort(l_or[0].astype(np.float32))[-2:]
        if top2[1] - top2[0] > 0.03:
            assert tok == t_or, "step %d" % step
        cur, pos = tok, pos + 1
    eng.close()


def test_moe_synthetic_model_generates_and_batches(tmp_path):
    """model_file_format = synthetic with expert_count: bin/ifa_llm_inference's path; three queries advance together through one
    batched step, each on its own single-query trajectory.  Teacher-forced: every batched step is fed the SOLO run's token, so
    both sides see the same context at every step (a free-running comparison of a small random MoE model ends at the first near-tie:
    the batched rows take the F16 GEMM, the single query the int8 GEMV, and a flipped id changes everything behind it); ids must
    agree wherever the solo logits' top-2 gap exceeds 0.05, and most steps must be such steps."""
    s = fx.MOE_SHAPE
    ini, _ = fx.write_model_dir(str(tmp_path), fmt="synthetic", wd="Q4", kvd="F16", ret="true", maxq=4, s=s)
    eng = InferenceEngine.from_ini(ini)
    rng = np.random.default_rng(5)
    prompts = [rng.integers(3, 1000, n).astype(np.int32) for n in (6, 9, 4)]
    STEPS, TIE = 6, 0.05
    solo, gaps = [], []
    for pr in prompts:
        qid = eng.add_query(pr)
        toks, gap = [], []
        for _ in range(STEPS):
            (q, t), = eng.infer()
            top2 = np.sort(eng.last_logits(qid)[-1].astype(np.float32))[-2:]
            toks.append(int(t)); gap.append(float(top2[1] - top2[0]))
            assert eng.commit({qid: int(t)})
        solo.append(toks); gaps.append(gap)
        assert eng.remove_query(qid)
    qids = [eng.add_query(pr) for pr in prompts]
    checked = 0
    for step in range(STEPS):
        res = {q: int(t) for q, t in eng.infer()}
        assert sorted(res) == sorted(qids)
        for i, q in enumerate(qids):
            if gaps[i][step] > TIE:
                assert res[q] == solo[i][step], (i, step, gaps[i][step])
                checked += 1
        eng.commit({q: solo[i][step] for i, q in enumerate(qids)})
    assert checked >= (len(qids) * STEPS) // 2, (checked, gaps)
    eng.close()
