"""Each mechanism that the Sopulorn layers add to the layer-list worker alone, through its C-ABI op, against the float64 functions of
tests/sopulorn_oracle.py: the token-pair embedding with its carried previous token, the RMS norm with weight (1 + w) (store / accumulate /
both norms between two sub-layers in one launch), the clamped and the row-gated activations, the query / key norm + rotation + cache
writer, attention over rotated caches with values of their own size, a fixed sink and another layer's rows (tiled and single-row forms,
portions, several sequences, slots reused), the router on logits, and the gated experts in the row form and the grouped form."""
import ctypes as C

import numpy as np
import pytest
import torch

import inferflow_amd as ia
from tests import sopulorn_oracle as orc
from tests.gelarax_oracle import bf16_round
from tests.gpu_util import capi, p, sync
from tests.test_gpu_layered_ops import Slots, dev32, devbf, devi, seq_tables

pytestmark = pytest.mark.gpu


def t64(a):
    return orc.t64(a)


def host_seqs(seqs):
    h, r = [], 0
    for n, pos0, slot in seqs:
        h += [r, n, pos0, slot]; r += n
    return (C.c_int * len(h))(*h)


def test_pair_embedding_in_portions_batches_and_reused_slots():
    rng = np.random.default_rng(1)
    V, W, B, mp, mc = 37, 20, 11, 29, 3
    E, P = bf16_round(rng.standard_normal((V, W))), bf16_round(rng.standard_normal((B + 1, W)))
    L = capi()
    slots = Slots(2, 8)
    seqs = {0: [int(t) for t in rng.integers(0, V, 19)], 1: [int(t) for t in rng.integers(0, V, 7)], 2: [int(t) for t in rng.integers(0, V, 5)]}
    want = {k: (t64(E)[v] + t64(P)[orc.pair_rows(v, B, mp, mc)]).numpy() for k, v in seqs.items()}
    at = {0: 0, 1: 0, 2: 0}
    # sequence 2 starts on slot 1 after sequence 1 has ended there; portions of 1, 2 and more tokens; two sequences in a step
    for step in ([(0, 1, 0)], [(0, 2, 0), (1, 4, 1)], [(0, 1, 0), (1, 3, 1)], [(0, 9, 0), (2, 1, 1)], [(2, 4, 1), (0, 6, 0)]):
        sd, rs, rows = seq_tables([(n, at[q], slot) for q, n, slot in step])
        toks = devi(sum([seqs[q][at[q]:at[q] + n] for q, n, _ in step], []))
        x = torch.zeros((rows, W), dtype=torch.float32, device="cuda")
        ia.check(L.ifa_embed_pair_f32(p(devbf(E)), V, W, p(devbf(P)), B, mp, mc, p(toks), p(sd), p(rs), rows, p(slots.table), 4, p(x), None)); sync()
        got, r = x.cpu().numpy(), 0
        for q, n, _ in step:
            assert np.abs(got[r:r + n] - want[q][at[q]:at[q] + n]).max() < 1e-6, (q, at[q], n)
            r += n; at[q] += n
    # without the table: plain embedding rows
    sd, rs, rows = seq_tables([(3, 0, 0)])
    x = torch.zeros((3, W), dtype=torch.float32, device="cuda")
    ia.check(L.ifa_embed_pair_f32(p(devbf(E)), V, W, None, 0, 0, 0, p(devi(seqs[0][:3])), p(sd), p(rs), 3, p(slots.table), 4, p(x), None)); sync()
    assert np.array_equal(x.cpu().numpy(), E[seqs[0][:3]])


@pytest.mark.parametrize("rows,cols", [(1, 64), (5, 96), (33, 40), (3, 14), (2, 1030)])
def test_norm_with_one_plus_weight_store_accumulate_and_both_in_one_launch(rows, cols):
    rng = np.random.default_rng(rows + cols)
    x = rng.standard_normal((rows, cols + 3)).astype(np.float32)
    w, w2 = bf16_round(0.3 * rng.standard_normal(cols)), bf16_round(0.3 * rng.standard_normal(cols))
    y0 = rng.standard_normal((rows, cols + 1)).astype(np.float32)
    want = orc.norm_one_plus(t64(x[:, :cols]), t64(w), 1e-5).numpy()
    L = capi()
    for acc in (0, 1):
        xd, yd = dev32(x), dev32(y0)
        ia.check(L.ifa_rmsnorm_offset_f32(p(xd), cols + 3, rows, cols, p(devbf(w)), 1.0, 1e-5, acc, p(yd), cols + 1, None)); sync()
        got = yd.cpu().numpy()
        ref = want + (y0[:, :cols] if acc else 0)
        assert np.abs(got[:, :cols] - ref).max() < 1e-5 * max(1.0, np.abs(ref).max())
        assert np.array_equal(got[:, cols:], y0[:, cols:])
    # x += norm(m) (1 + w); h = norm(x) (1 + w2)
    for with_h in (1, 0):
        xd, md, hd = dev32(y0), dev32(x), torch.full((rows, cols), 7.0, dtype=torch.float32, device="cuda")
        ia.check(L.ifa_norm_add_norm_f32(p(xd), cols + 1, rows, cols, p(md), cols + 3, p(devbf(w)), p(devbf(w2)) if with_h else None, 1.0, 1e-5, p(hd), cols, None)); sync()
        xs = y0[:, :cols] + want
        assert np.abs(xd.cpu().numpy()[:, :cols] - xs).max() < 1e-5 * max(1.0, np.abs(xs).max())
        if with_h:
            hs = orc.norm_one_plus(t64(xs), t64(w2), 1e-5).numpy()
            assert np.abs(hd.cpu().numpy() - hs).max() < 1e-5 * max(1.0, np.abs(hs).max())
        else:
            assert float(hd.min()) == 7.0


def test_clamped_activation_and_row_gate():
    rng = np.random.default_rng(3)
    T, F = 5, 70
    gu = (3.0 * rng.standard_normal((T, 2 * F + 2))).astype(np.float32)
    gate = rng.standard_normal((T, 3)).astype(np.float32)
    L = capi()
    out = torch.zeros((T, F), dtype=torch.float32, device="cuda")
    ia.check(L.ifa_glu_ex_f32(3, 1.25, p(dev32(gu)), 2 * F + 2, T, F, None, 0, p(out), F, None)); sync()
    g, u = t64(gu[:, :F]).clamp(max=1.25), t64(gu[:, F:2 * F]).clamp(-1.25, 1.25)
    assert np.abs(out.cpu().numpy() - (g * torch.sigmoid(1.702 * g) * (u + 1)).numpy()).max() < 1e-5
    assert (np.abs(gu[:, :F]) > 1.25).any() and (gu[:, F:2 * F] < -1.25).any()          # (the clamps are at work)
    ia.check(L.ifa_glu_ex_f32(0, 0.0, p(dev32(gu)), 2 * F + 2, T, F, p(dev32(gate)), 3, p(out), F, None)); sync()
    g, u = t64(gu[:, :F]), t64(gu[:, F:2 * F])
    want = g * torch.sigmoid(g) * u * torch.sigmoid(t64(gate[:, :1]))
    assert np.abs(out.cpu().numpy() - want.numpy()).max() < 1e-5 * float(want.abs().max())


def attention_case(heads, kv_heads, dim, vdim, rot_dims, L, rng, base=300.0):
    q = rng.standard_normal((L, heads * dim)).astype(np.float32)
    k = rng.standard_normal((L, kv_heads * dim)).astype(np.float32)
    v = rng.standard_normal((L, kv_heads * vdim)).astype(np.float32)
    qw, kw = bf16_round(1 + 0.3 * rng.standard_normal(dim)), bf16_round(1 + 0.3 * rng.standard_normal(dim))
    return q, k, v, qw, kw


def oracle_attention(q, k, v, qw, kw, heads, kv_heads, dim, vdim, rot_dims, base, scale, eps):
    T = q.shape[0]
    pos = list(range(T))
    qq = orc.rotate_half_layout(orc.rms_unit(t64(q).reshape(T, heads, dim), eps) * t64(qw), pos, rot_dims, base)
    kk = orc.rotate_half_layout(orc.rms_unit(t64(k).reshape(T, kv_heads, dim), eps) * t64(kw), pos, rot_dims, base)
    return orc.attention_core(qq, kk, t64(v).reshape(T, kv_heads, vdim), scale).numpy()


def freq_table(rot_dims, base):
    return torch.from_numpy(np.asarray([base ** (-2.0 * i / max(rot_dims, 1)) for i in range(max(rot_dims // 2, 1))], np.float64)).cuda()


@pytest.mark.parametrize("tile_min", [16, 1 << 30])
@pytest.mark.parametrize("heads,kv_heads,dim,vdim,rot_dims", [(4, 2, 24, 16, 24), (2, 2, 8, 40, 4), (3, 1, 68, 36, 30), (6, 3, 32, 32, 0), (2, 1, 128, 128, 128),
                                                              (4, 1, 40, 72, 40), (1, 1, 5, 3, 2), (8, 2, 96, 8, 64), (2, 1, 160, 20, 100), (2, 1, 320, 24, 200)])
def test_rotated_attention_in_portions_and_single_rows(heads, kv_heads, dim, vdim, rot_dims, tile_min):
    rng = np.random.default_rng(heads + dim + vdim)
    L, eps, scale, base, ctx = 150, 1e-5, 0.3, 300.0, 160
    q, k, v, qw, kw = attention_case(heads, kv_heads, dim, vdim, rot_dims, L, rng)
    # one key far back and the very first one get large matching queries at the last rows (before the norm: directions count)
    k[1, :dim] = 5 * rng.standard_normal(dim); q[-1, :dim] = k[1, :dim]
    want = oracle_attention(q, k, v, qw, kw, heads, kv_heads, dim, vdim, rot_dims, base, scale, eps)
    fr = freq_table(rot_dims, base)
    k_off, v_off = 4, 4 + ((ctx * kv_heads * dim + 3) // 4) * 4
    sl = Slots(2, v_off + ctx * kv_heads * vdim)
    ws = torch.full((2 * heads * 32 * (vdim + 2),), float('nan'), dtype=torch.float32, device='cuda')
    Lc = capi()
    at = 0
    for n in (1, 2, 60, 1, 1, 80, 5):
        d, rs, T = seq_tables([(n, at, 1)])
        qd, kd, vd = dev32(q[at:at + n]), dev32(k[at:at + n]), dev32(v[at:at + n])
        ia.check(Lc.ifa_qk_rope_store_f32(p(qd), heads * dim, heads, p(kd), kv_heads * dim, p(vd), kv_heads * vdim, kv_heads, dim, vdim, p(devbf(qw)), p(devbf(kw)), eps,
                                          rot_dims, p(fr), p(d), p(rs), T, p(sl.table), k_off, v_off, None))
        out = torch.empty((T, heads * vdim + 1), dtype=torch.float32, device="cuda")
        ia.check(Lc.ifa_attention_kv_f32(p(qd), heads * dim, heads, kv_heads, dim, vdim, scale, 0, 0, 1, 0.0, p(d), p(rs), T, p(sl.table), k_off, v_off, p(out),
                                         heads * vdim + 1, host_seqs([(n, at, 1)]), 1, tile_min, ctx, p(ws) if n <= 2 else None, ws.numel() * 4, None))
        sync()
        assert np.abs(out.cpu().numpy()[:, :heads * vdim] - want[at:at + n]).max() < 2e-5 * max(1.0, np.abs(want).max()), (at, n)
        at += n
    assert at == L
    # without the one in the denominator the weights sum to one: a different result, so it is really counted; another score counts as exp(score)
    d, rs, T = seq_tables([(1, L - 1, 1)])
    qd = dev32(q[L - 1:])
    ia.check(Lc.ifa_qk_rope_store_f32(p(qd), heads * dim, heads, None, 0, None, 0, kv_heads, dim, vdim, p(devbf(qw)), None, eps, rot_dims, p(fr), p(d), p(rs), T,
                                      p(sl.table), k_off, v_off, None))
    res, flat = [], 0.1 / dim          # (scores so small that no key drowns the sink)
    for sink, score in ((0, 0.0), (1, 0.0), (1, 1.5)):
        out = torch.empty((1, heads * vdim), dtype=torch.float32, device="cuda")
        ia.check(Lc.ifa_attention_kv_f32(p(qd), heads * dim, heads, kv_heads, dim, vdim, flat, 0, 0, sink, score, p(d), p(rs), T, p(sl.table), k_off, v_off, p(out),
                                         heads * vdim, None, 0, 0, ctx, None, 0, None))
        sync(); res.append(out.cpu().numpy())
    want_flat = oracle_attention(q, k, v, qw, kw, heads, kv_heads, dim, vdim, rot_dims, base, flat, eps)
    assert np.abs(res[1] - want_flat[L - 1:]).max() < 2e-5 * max(1.0, np.abs(want_flat).max())
    assert np.abs(res[0] - res[1]).max() > 1e-4 and np.abs(res[2] - res[1]).max() > 1e-4


@pytest.mark.parametrize("heads,kv_heads,dim,vdim,rot_dims", [(2, 2, 40, 72, 40), (4, 1, 100, 100, 50), (2, 1, 16, 200, 8)])
def test_single_rows_over_a_long_context_with_value_heads_that_end_inside_a_group_of_64_columns(heads, kv_heads, dim, vdim, rot_dims):
    """1300 keys: the keys of a (row, head) are shared out to twenty workgroups, and the merge of their partial results walks value
    columns 64 .. vdim - 1 with only some lanes holding a column"""
    rng = np.random.default_rng(dim + vdim)
    L, eps, scale, base, ctx = 1300, 1e-5, 0.3, 10000.0, 2001
    q, k, v, qw, kw = attention_case(heads, kv_heads, dim, vdim, rot_dims, L, rng)
    want = oracle_attention(q, k, v, qw, kw, heads, kv_heads, dim, vdim, rot_dims, base, scale, eps)
    fr = freq_table(rot_dims, base)
    k_off, v_off = 0, ctx * kv_heads * dim
    sl = Slots(1, v_off + ctx * kv_heads * vdim)
    ws = torch.full((heads * 32 * (vdim + 2),), float('nan'), dtype=torch.float32, device='cuda')
    Lc = capi()
    at = 0
    for n in [1290] + [1] * 10:
        d, rs, T = seq_tables([(n, at, 0)])
        qd, kd, vd = dev32(q[at:at + n]), dev32(k[at:at + n]), dev32(v[at:at + n])
        ia.check(Lc.ifa_qk_rope_store_f32(p(qd), heads * dim, heads, p(kd), kv_heads * dim, p(vd), kv_heads * vdim, kv_heads, dim, vdim, p(devbf(qw)), p(devbf(kw)), eps,
                                          rot_dims, p(fr), p(d), p(rs), T, p(sl.table), k_off, v_off, None))
        out = torch.empty((T, heads * vdim), dtype=torch.float32, device="cuda")
        ia.check(Lc.ifa_attention_kv_f32(p(qd), heads * dim, heads, kv_heads, dim, vdim, scale, 0, 0, 1, 0.0, p(d), p(rs), T, p(sl.table), k_off, v_off, p(out),
                                         heads * vdim, host_seqs([(n, at, 0)]), 1, 16, ctx, p(ws), ws.numel() * 4, None))
        sync()
        assert np.abs(out.cpu().numpy() - want[at:at + n]).max() < 2e-5 * max(1.0, np.abs(want).max()), (at, n)
        at += n


def test_rotated_attention_tiles_over_several_sequences():
    """one step holds a 150-token prompt, a single continued token and a 40-token continued portion: tiles must not cross sequences"""
    rng = np.random.default_rng(78)
    heads, kv_heads, dim, vdim, rot_dims, eps, scale, base = 4, 2, 40, 24, 16, 1e-5, 0.4, 1000.0
    L, ctx = 200, 208
    seq = {s_: attention_case(heads, kv_heads, dim, vdim, rot_dims, L, rng) for s_ in (0, 1, 2)}
    fr = freq_table(rot_dims, base)
    k_off, v_off = 0, ctx * kv_heads * dim
    sl = Slots(3, v_off + ctx * kv_heads * vdim)
    Lc = capi()
    at = {0: 0, 1: 0, 2: 0}
    for step in ([(1, 30), (2, 100)], [(0, 150), (1, 1), (2, 40)], [(2, 60), (0, 50), (1, 129)]):
        seqs = [(n, at[s_], s_) for s_, n in step]
        d, rs, T = seq_tables(seqs)
        qd, kd, vd = (dev32(np.concatenate([seq[s_][i][at[s_]:at[s_] + n] for s_, n in step], 0)) for i in range(3))
        qw, kw = seq[0][3], seq[0][4]          # (every sequence shares the norm weights of sequence 0: they are the layer's)
        ia.check(Lc.ifa_qk_rope_store_f32(p(qd), heads * dim, heads, p(kd), kv_heads * dim, p(vd), kv_heads * vdim, kv_heads, dim, vdim, p(devbf(qw)), p(devbf(kw)), eps,
                                          rot_dims, p(fr), p(d), p(rs), T, p(sl.table), k_off, v_off, None))
        out = torch.empty((T, heads * vdim), dtype=torch.float32, device="cuda")
        ia.check(Lc.ifa_attention_kv_f32(p(qd), heads * dim, heads, kv_heads, dim, vdim, scale, 0, 0, 1, 0.0, p(d), p(rs), T, p(sl.table), k_off, v_off, p(out),
                                         heads * vdim, host_seqs(seqs), len(seqs), 16, ctx, None, 0, None))
        sync()
        got, r = out.cpu().numpy(), 0
        for s_, n in step:
            w_ = oracle_attention(seq[s_][0], seq[s_][1], seq[s_][2], qw, kw, heads, kv_heads, dim, vdim, rot_dims, base, scale, eps)
            assert np.abs(got[r:r + n] - w_[at[s_]:at[s_] + n]).max() < 2e-5 * max(1.0, np.abs(w_).max()), (s_, at[s_], n)
            r += n; at[s_] += n


@pytest.mark.parametrize("n_all,top", [(6, 2), (16, 1), (5, 5), (70, 8), (3, 2)])
def test_router_on_logits_with_ties_and_softmax_over_the_chosen(n_all, top):
    rng = np.random.default_rng(n_all + top)
    T = 9
    z = rng.standard_normal((T, n_all + 2)).astype(np.float32)
    z[1, :n_all] = 0.5                      # all equal: the lowest indices win
    if n_all > 2:
        z[2, 2] = z[2, 0] = 3.0             # a tie at the top
    bias = bf16_round(rng.standard_normal(n_all))
    for use_bias in (0, 1):
        zz = t64(z[:, :n_all]) + (t64(bias) if use_bias else 0)
        idx_w = torch.argsort(-zz, dim=-1, stable=True)[:, :top]
        wgt_w = torch.softmax(torch.gather(zz, 1, idx_w), -1).numpy()
        idx = torch.zeros((T, top), dtype=torch.int32, device="cuda"); wgt = torch.zeros((T, top), dtype=torch.float32, device="cuda")
        ia.check(capi().ifa_moe_route_top_f32(p(dev32(z)), n_all + 2, T, n_all, top, p(devbf(bias)) if use_bias else None, p(idx), p(wgt), None)); sync()
        assert np.array_equal(idx.cpu().numpy(), idx_w.numpy())
        assert np.abs(wgt.cpu().numpy() - wgt_w).max() < 1e-6


@pytest.mark.parametrize("T,W,F,E,top", [(1, 64, 24, 6, 2), (8, 40, 10, 3, 3), (8, 128, 64, 16, 4), (7, 64, 16, 256, 9), (2, 16, 8, 1, 1), (5, 14, 6, 70, 8)])
def test_choice_by_the_largest_logits_inside_the_experts_first_launch(T, W, F, E, top):
    """against the choice in a launch of its own and the experts behind it: ties, all equal, some at -inf; a row that has no numbers has experts nevertheless, and the rows beside it
    what they have without it"""
    rng = np.random.default_rng(T + W + E)
    h, z = rng.standard_normal((T, W)).astype(np.float32), rng.standard_normal((T, E + 3)).astype(np.float32)
    z[0, 1:3] = 2.5
    for t, row in ((1, np.zeros(E)), (3, np.where(np.arange(E) % 2, -np.inf, 1.0)), (6, np.full(E, np.nan))):
        if t < T:
            z[t, :E] = row
    gu, dd = devbf(bf16_round(rng.standard_normal((E * 2 * F, W)) / np.sqrt(W))), devbf(bf16_round(rng.standard_normal((E * W, F)) / np.sqrt(F)))
    L, Z, dh, dz = capi(), C.c_size_t, dev32(h), dev32(z)
    nb = L.ifa_moe_workspace_bytes(T, top, W, 3 * F, E)
    ws = torch.zeros((nb + 15) // 4, dtype=torch.float32, device="cuda")
    idx, idx_w = (torch.full((T, top), -1, dtype=torch.int32, device="cuda") for _ in range(2))
    wgt, wgt_w = (torch.zeros((T, top), dtype=torch.float32, device="cuda") for _ in range(2))
    y, y_w = (torch.full((T, W + 1), 0.5, dtype=torch.float32, device="cuda") for _ in range(2))
    ia.check(L.ifa_moe_experts_gated_top_rows_shared(p(dz), Z(E + 3), p(dh), Z(W), Z(T), W, F, E, top, p(gu), p(dd), p(idx), p(wgt), p(ws), Z(nb), p(y), Z(W + 1), 1, None, None)); sync()
    some = [t for t in range(T) if t != 6]
    ia.check(L.ifa_moe_route_top_f32(p(dz), E + 3, T, E, top, None, p(idx_w), p(wgt_w), None))
    got, i, iw = y.cpu().numpy(), idx.cpu().numpy(), idx_w.cpu().numpy()
    assert i.min() >= 0 and i.max() < E and all(len(set(r)) == top for r in i.tolist())
    finite = [t for t in some if np.isfinite(np.take_along_axis(z[t], i[t], 0)).all()]
    assert np.array_equal(i[finite], iw[finite]) and np.abs(wgt.cpu().numpy()[finite] - wgt_w.cpu().numpy()[finite]).max() < 1e-6
    idx_w.copy_(idx); wgt_w.copy_(wgt)
    ia.check(L.ifa_moe_experts_gated_f32(p(dh), W, T, W, F, E, top, p(gu), p(dd), p(idx_w), p(wgt_w), 1, p(ws), nb, p(y_w), W + 1, 1, None)); sync()
    assert np.array_equal(got, y_w.cpu().numpy(), equal_nan=True) and np.isfinite(got[some]).all() and (T <= 6 or np.isnan(got[6, :W]).all())


@pytest.mark.parametrize("W", [1, 4, 7, 1020, 1024, 1028, 1030, 2052])
def test_embedding_rows_in_pieces_of_four_columns_and_one_by_one(W):
    """widths within a round of the threads' pieces and beyond, whole pieces and not; two sequences, one from the start and one behind a token kept in its slot; with a pair table, without, and the
    rows a second time: the values exactly"""
    rng = np.random.default_rng(W)
    V, B, mp, mc, scale = 50, 11, 36313, 27191, 1.7
    E, P = bf16_round(rng.standard_normal((V, W))), bf16_round(rng.standard_normal((B + 1, W)))
    slots = Slots(2, 64)
    toks, L = np.array([3, 49, 0, 7, 8, 60, 12], np.int32), capi()
    sd, rs, rows = seq_tables([(4, 0, 0), (3, 5, 1)])
    for pair in (True, False):
        slots.mem[1].view(torch.int32)[4] = 21
        x, xc = (torch.full((rows, W), float("nan"), dtype=torch.float32, device="cuda") for _ in range(2))
        ia.check(L.ifa_embed_pair_scaled_f32(p(devbf(E)), V, W, scale, p(devbf(P)) if pair else None, B, mp, mc, p(devi(toks)), p(sd), p(rs), rows, p(slots.table), 4, p(x), p(xc), None)); sync()
        prev = [None, 3, 49, 0, 21, 8, 60]
        want = np.zeros((rows, W), np.float32)
        for t in range(rows):
            tok = min(int(toks[t]), V - 1)
            want[t] = E[tok].astype(np.float32) * np.float32(scale)
            if pair:
                want[t] += P[B if prev[t] is None else (prev[t] * mp + tok * mc) % B].astype(np.float32)
        assert np.array_equal(x.cpu().numpy(), want) and torch.equal(x, xc)
        assert int(slots.mem[0].view(torch.int32)[4]) == 7 and int(slots.mem[1].view(torch.int32)[4]) == 12


@pytest.mark.parametrize("T,W,F,SF,E,top", [(1, 64, 24, 8, 6, 2), (6, 128, 64, 1408, 16, 4), (8, 40, 10, 520, 3, 3), (5, 14, 6, 2048, 70, 8), (7, 64, 16, 2056, 16, 9), (2, 16, 8, 4104, 1, 1), (3, 24, 16, 1032, 5, 3), (4, 36, 8, 72, 12, 6),
                                                (1, 20, 8, 520, 9, 7)])
def test_shared_expert_in_the_experts_last_launch_leaves_the_bits_of_its_own(T, W, F, SF, E, top):
    """the output product beside the sum over the experts, in one launch and in two: pieces of 512 columns whole and ragged, more of them than are asked for ahead, rows of activations, gates and
    outputs with strides; the experts' rows onto what is there and in its place; and the norm behind both, which adds them up"""
    class Shared(C.Structure):
        _fields_ = [("down", C.c_void_p), ("act", C.c_void_p), ("lda", C.c_size_t), ("ff", C.c_int), ("gate", C.c_void_p), ("ldg", C.c_size_t), ("out", C.c_void_p), ("ldo", C.c_size_t)]
    rng = np.random.default_rng(T + W + SF)
    L, Z = capi(), C.c_size_t
    dh, dz = dev32(rng.standard_normal((T, W))), dev32(rng.standard_normal((T, E)))
    gu, dd = devbf(bf16_round(rng.standard_normal((E * 2 * F, W)) / np.sqrt(W))), devbf(bf16_round(rng.standard_normal((E * W, F)) / np.sqrt(F)))
    sd, act, gate = devbf(bf16_round(rng.standard_normal((W, SF)) / np.sqrt(SF))), dev32(rng.standard_normal((T, SF + 4))), dev32(rng.standard_normal((T, 3)))
    nb = L.ifa_moe_workspace_bytes(T, top, W, 3 * F, E)
    ws = torch.zeros((nb + 15) // 4, dtype=torch.float32, device="cuda")
    idx, wgt = torch.zeros((T, top), dtype=torch.int32, device="cuda"), torch.zeros((T, top), dtype=torch.float32, device="cuda")
    out, out_w = (torch.full((T, W + 2), 0.25, dtype=torch.float32, device="cuda") for _ in range(2))
    shared = Shared(sd.data_ptr(), act.data_ptr(), SF + 4, SF, gate.data_ptr() + 4, 3, out.data_ptr(), W + 2)
    for acc in (0, 1):
        y, y_w = (torch.full((T, W + 1), 0.5, dtype=torch.float32, device="cuda") for _ in range(2))
        args = [p(dz), Z(E), p(dh), Z(W), Z(T), W, F, E, top, p(gu), p(dd), p(idx), p(wgt), p(ws), Z(nb)]
        ia.check(L.ifa_moe_experts_gated_top_rows_shared(*args, p(y), Z(W + 1), acc, C.byref(shared), None))
        ia.check(L.ifa_moe_experts_gated_top_rows_shared(*args, p(y_w), Z(W + 1), acc, None, None))
        ia.check(L.ifa_linear_bf16w_gated_rows(p(sd), Z(W), Z(SF), p(act), Z(SF + 4), Z(T), C.c_void_p(gate.data_ptr() + 4), Z(3), 0, p(out_w), Z(W + 2), None)); sync()
        assert torch.equal(y, y_w) and torch.equal(out, out_w) and torch.isfinite(y).all() and torch.isfinite(out).all()
    if W % 4:
        return
    L.ifa_norm_add_two_norm_f32.restype = C.c_bool
    a, b = y[:, :W].contiguous(), out[:, :W].contiguous()
    wa, wb, x = devbf(bf16_round(rng.standard_normal(W))), devbf(bf16_round(rng.standard_normal(W))), dev32(rng.standard_normal((T, W)))
    x_w, h, h_w = x.clone(), torch.zeros_like(x), torch.zeros_like(x)
    f1 = C.c_float
    assert L.ifa_norm_add_two_norm_f32(p(x), Z(W), Z(T), Z(W), p(a), p(b), Z(W), p(wa), p(wb), f1(1.0), f1(1e-6), p(h), Z(W), None)
    ia.check(L.ifa_norm_add_norm_f32(p(x_w), W, T, W, p(a + b), W, p(wa), p(wb), 1.0, 1e-6, p(h_w), W, None)); sync()
    assert torch.equal(x, x_w) and torch.equal(h, h_w)


@pytest.mark.parametrize("T,W,F,E,top", [(1, 64, 24, 6, 2), (3, 40, 10, 3, 3), (8, 128, 64, 16, 4), (9, 64, 24, 6, 2), (70, 48, 20, 5, 1), (150, 64, 32, 20, 3), (5, 14, 6, 4, 2)])
def test_gated_experts_in_rows_and_grouped(T, W, F, E, top):
    rng = np.random.default_rng(T + W + F)
    h = rng.standard_normal((T, W + 4)).astype(np.float32)
    gu = bf16_round(rng.standard_normal((E, 2 * F, W)) / np.sqrt(W)); dn = bf16_round(rng.standard_normal((E, W, F)) / np.sqrt(F))
    idx = np.stack([rng.permutation(E)[:top] for _ in range(T)]).astype(np.int32)
    wgt = rng.uniform(0.1, 1.0, (T, top)).astype(np.float32)
    want = np.zeros((T, W))
    for t in range(T):
        for e, a in zip(idx[t], wgt[t]):
            want[t] += a * orc.gated_expert(t64(h[t:t + 1, :W]), t64(gu[e, :F]), t64(gu[e, F:]), t64(dn[e])).numpy()[0]
    L = capi()
    nb = L.ifa_moe_workspace_bytes(T, top, W, 3 * F, E)
    ws = torch.zeros((nb + 15) // 4, dtype=torch.float32, device="cuda")
    y0 = rng.standard_normal((T, W + 1)).astype(np.float32)
    for ops32, tol in ((1, 2e-5), (0, 3e-2)):
        for acc in (0, 1):
            y = dev32(y0)
            ia.check(L.ifa_moe_experts_gated_f32(p(dev32(h)), W + 4, T, W, F, E, top, p(devbf(gu.reshape(E * 2 * F, W))), p(devbf(dn.reshape(E * W, F))), p(devi(idx)),
                                                 p(dev32(wgt)), ops32, p(ws), nb, p(y), W + 1, acc, None)); sync()
            ref = want + (y0[:, :W] if acc else 0)
            t_ = tol if T > 8 else 2e-5          # (steps of at most 8 rows keep fp32 activations in both modes)
            assert np.abs(y.cpu().numpy()[:, :W] - ref).max() < t_ * max(1.0, np.abs(want).max()), (ops32, acc)


@pytest.mark.parametrize("T,W,F,E,top", [(9, 64, 72, 6, 2), (40, 264, 320, 5, 2), (300, 136, 264, 2, 2), (700, 72, 64, 3, 1), (130, 328, 72, 1, 1),
                                         (9, 64, 456, 6, 2), (300, 136, 384, 2, 2), (20, 264, 320, 40, 2), (11, 520, 72, 3, 1), (9000, 520, 72, 2, 1), (130, 440, 72, 1, 1)])
def test_gated_experts_over_bfloat16_rows(T, W, F, E, top):
    """sizes above and below the form's border, row tiles of 64 and 128 (9000 rows), few and many steps, inner sizes that are no multiple of a step, many experts without a row
    (fewer tiles than there may be): h and the activations rounded to bfloat16 once"""
    rng = np.random.default_rng(T + W + F)
    h = bf16_round(rng.standard_normal((T, W)))
    gu = bf16_round(rng.standard_normal((E, 2 * F, W)) / np.sqrt(W)); dn = bf16_round(rng.standard_normal((E, W, F)) / np.sqrt(F))
    idx = np.stack([rng.permutation(E)[:top] for _ in range(T)]).astype(np.int32)
    wgt = rng.uniform(0.1, 1.0, (T, top)).astype(np.float32)
    want, bound = np.zeros((T, W)), np.zeros((T, W))
    for e in range(E):
        g, u = h.astype(np.float64) @ gu[e, :F].astype(np.float64).T, h.astype(np.float64) @ gu[e, F:].astype(np.float64).T
        a, d = g / (1 + np.exp(-g)) * u, dn[e].astype(np.float64).T
        w = np.where(idx == e, wgt, 0).sum(1, keepdims=True)
        want += w * (a @ d)
        bound += w * (np.abs(a) @ np.abs(d) * 2.0 ** -8 + (np.abs(g) + np.abs(u) + 1) @ np.abs(d) * 2.0 ** -18)          # an activation to 8 bits: half a unit is up to 2^-8 of it; the 32-bit sums in front
    L = capi()
    nb = L.ifa_moe_workspace_bytes(T, top, W, 3 * F, E)
    ws = torch.zeros((nb + 15) // 4, dtype=torch.float32, device="cuda")
    y = torch.full((T, W + 1), 7.0, dtype=torch.float32, device="cuda")
    ia.check(L.ifa_moe_experts_gated_f32(p(dev32(h)), W, T, W, F, E, top, p(devbf(gu.reshape(E * 2 * F, W))), p(devbf(dn.reshape(E * W, F))), p(devi(idx)),
                                         p(dev32(wgt)), 0, p(ws), nb, p(y), W + 1, 0, None)); sync()
    got = y.cpu().numpy()
    assert np.all(np.abs(got[:, :W] - want) <= bound) and np.all(got[:, W:] == 7.0)


@pytest.mark.parametrize("T,F,top", [(1, 24, 1), (3, 520, 4), (6, 704, 4), (8, 72, 5), (2, 1032, 9)])
def test_experts_of_a_few_rows_walked_four_and_eight_at_a_time(T, F, top):
    """fewer, as many and more choices than are walked together; inner sizes of one and more passes of 512 columns: against 64 bits"""
    W, E = 40, 12
    rng = np.random.default_rng(F + top)
    h = rng.standard_normal((T, W)).astype(np.float32)
    gu = bf16_round(rng.standard_normal((E, 2 * F, W)) / np.sqrt(W)); dn = bf16_round(rng.standard_normal((E, W, F)) / np.sqrt(F))
    idx = np.stack([rng.permutation(E)[:top] for _ in range(T)]).astype(np.int32)
    wgt = rng.uniform(0.1, 1.0, (T, top)).astype(np.float32)
    want, mag = np.zeros((T, W)), np.zeros((T, W))
    for e in range(E):
        g, u = h.astype(np.float64) @ gu[e, :F].astype(np.float64).T, h.astype(np.float64) @ gu[e, F:].astype(np.float64).T
        a, d, w = g / (1 + np.exp(-g)) * u, dn[e].astype(np.float64).T, np.where(idx == e, wgt, 0).sum(1, keepdims=True)
        want += w * (a @ d); mag += w * ((np.abs(a) + np.abs(g) + np.abs(u) + 1) @ np.abs(d))
    L = capi()
    nb = L.ifa_moe_workspace_bytes(T, top, W, 3 * F, E)
    ws = torch.zeros((nb + 15) // 4, dtype=torch.float32, device="cuda")
    y = torch.full((T, W + 1), 7.0, dtype=torch.float32, device="cuda")
    ia.check(L.ifa_moe_experts_gated_f32(p(dev32(h)), W, T, W, F, E, top, p(devbf(gu.reshape(E * 2 * F, W))), p(devbf(dn.reshape(E * W, F))), p(devi(idx)),
                                         p(dev32(wgt)), 1, p(ws), nb, p(y), W + 1, 0, None)); sync()
    got = y.cpu().numpy()
    # 32-bit sums of W and of F products: at most (W + F / 64 + 16) roundings of half a unit of the magnitudes each
    assert np.all(np.abs(got[:, :W] - want) <= (W + F / 64 + 16) * 2.0 ** -23 * mag) and np.all(got[:, W:] == 7.0)
