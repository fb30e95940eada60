"""Each mechanism of the layer-list worker alone, through its C-ABI op, against the float64 functions of tests/gelarax_oracle.py:
linear layers with bfloat16 weights (row kernel and both matrix-core modes, ragged shapes, every epilogue), embedding + sinusoid,
norms, gated activations, argmax, short convolutions with their carried tail, delta-rule gates, both state recurrences (whole,
continued, several sequences, slots reused), gated group norm, and the windowed attention with sink / soft cap / bucket bias."""
import ctypes as C

import numpy as np
import pytest
import torch

import inferflow_amd as ia
from tests import gelarax_oracle as orc
from tests.gpu_util import capi, p, sync

pytestmark = pytest.mark.gpu


def dev32(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).cuda()


def devbf(a):
    return torch.from_numpy(orc.bf16_bits(a).view(np.int16)).cuda()


def devi(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.int32)).cuda()


def stream():
    return None


class Slots:
    """a slot arena table like the worker's: n slots of `floats` fp32 each, filled with garbage so that stale state shows"""

    def __init__(self, n, floats):
        self.mem = [torch.full((floats,), 1e9, dtype=torch.float32, device="cuda") for _ in range(n)]
        self.table = torch.tensor([m.data_ptr() for m in self.mem], dtype=torch.int64).cuda()


def seq_tables(seqs):
    """seqs: [(n, pos0, slot)] -> device (descs, row_seq), total rows"""
    d, rs, r = [], [], 0
    for i, (n, pos0, slot) in enumerate(seqs):
        d += [r, n, pos0, slot]; rs += [i] * n; r += n
    return devi(d), devi(rs), r


@pytest.mark.parametrize("T", [1, 2, 3, 8, 9, 64, 70, 131])
@pytest.mark.parametrize("N,K", [(64, 64), (5, 36), (130, 200), (48, 7)])
def test_linear_bf16_weights(T, N, K):
    rng = np.random.default_rng(T * 1000 + N + K)
    W = orc.bf16_round(rng.standard_normal((N, K)))
    A = rng.standard_normal((T, K + 4)).astype(np.float32)            # lda > K
    bias, mul = orc.bf16_round(rng.standard_normal(N)), orc.bf16_round(rng.standard_normal(N))
    C0 = rng.standard_normal((T, N + 2)).astype(np.float32)
    prod = A[:, :K].astype(np.float64) @ W.astype(np.float64).T
    for ops32 in (1, 0):
        for use_bias, use_mul, alpha, acc in ((0, 0, 1.0, 0), (1, 0, 1.0, 0), (1, 1, 0.7, 1), (0, 1, 1.3, 1)):
            c = dev32(C0)
            ia.check(capi().ifa_linear_bf16w(p(devbf(W)), N, K, p(dev32(A)), K + 4, T, p(devbf(bias)) if use_bias else None,
                                             p(devbf(mul)) if use_mul else None, alpha, acc, ops32, p(c), N + 2, 2, min(N, 40) if use_mul else 0, stream()))
            sync()
            want = prod + (bias if use_bias else 0)
            if use_mul:                                                 # columns [2, 40) through SiLU after the bias
                want[:, 2:min(N, 40)] = orc.silu(orc.t64(want[:, 2:min(N, 40)])).numpy()
            if use_mul:
                want = want * mul
            want = want * alpha + (C0[:, :N] if acc else 0)
            got = c.cpu().numpy()
            assert np.array_equal(got[:, N:], C0[:, N:])                # columns past N untouched
            tol = 2e-5 if (ops32 or T <= 8) else 2e-2
            assert np.abs(got[:, :N] - want).max() < tol * max(1.0, np.abs(want).max()), (ops32, use_bias, use_mul, acc)


def test_embedding_with_sinusoid_norms_glu_argmax():
    rng = np.random.default_rng(1)
    V, W, T = 37, 50, 9
    E = orc.bf16_round(rng.standard_normal((V, W)))
    toks = rng.integers(0, V, T); pos = np.array([0, 1, 2, 500, 1115, 4095, 7, 8, 100000])
    x = torch.empty((T, W), dtype=torch.float32, device="cuda")
    ia.check(capi().ifa_embed_sinpos_f32(p(devbf(E)), V, W, p(devi(toks)), p(devi(pos)), T, 10000.0, p(x), stream()))
    want = orc.t64(E)[torch.as_tensor(toks)] + orc.sinusoid(pos, W)
    assert np.abs(x.cpu().numpy() - want.numpy()).max() < 2e-6
    g = orc.bf16_round(1 + 0.3 * rng.standard_normal(W))
    xin = (3 * rng.standard_normal((T, W)) + 2).astype(np.float32)
    for kind, f in ((1, lambda a: orc.layer_norm_nobias(a, orc.t64(g), 1e-5)), (0, lambda a: orc.rms_unit(a, 1e-5) * orc.t64(g))):
        y = torch.empty((T, W), dtype=torch.float32, device="cuda")
        ia.check(capi().ifa_layernorm_f32(kind, p(dev32(xin)), W, T, W, p(devbf(g)), 1e-5, p(y), W, stream()))
        assert np.abs(y.cpu().numpy() - f(orc.t64(xin)).numpy()).max() < 1e-5
    F = 21
    gu = rng.standard_normal((T, 2 * F)).astype(np.float32) * 3
    o = torch.empty((T, F), dtype=torch.float32, device="cuda")
    ia.check(capi().ifa_glu_f32(1, p(dev32(gu)), 2 * F, T, F, p(o), F, stream()))
    want = orc.gelu_tanh(orc.t64(gu[:, :F])) * orc.t64(gu[:, F:])
    assert np.abs(o.cpu().numpy() - want.numpy()).max() < 1e-5
    lg = rng.standard_normal((T, 300)).astype(np.float32)
    lg[2, 17] = lg[2, 250] = 9.0
    best = torch.empty(T, dtype=torch.int32, device="cuda")
    excl = devi([2, int(lg[0].argmax()), 17, -1])
    ia.check(capi().ifa_argmax_rows_f32(p(dev32(lg)), 300, 300, T, p(excl), p(best), stream()))
    b = best.cpu().numpy()
    masked = lg.copy(); masked[:, int(lg[0].argmax())] = -np.inf; masked[:, 17] = -np.inf
    assert list(b) == [int(r.argmax()) for r in masked] and b[2] == 250


@pytest.mark.parametrize("C_,gdim,nq,nsc,lens", [(40, 8, 16, 8, [(70, 1, 33), (2, 64, 1), (65, 3, 90)]), (1100, 64, 640, 320, [(3, 90, 1), (61, 2, 2), (1, 1, 100)]),
                                                 (2052, 256, 512, 256, [(1500, 700, 1), (1, 5, 2100)]), (72, 0, 0, 0, [(64, 1, 2)])])
@pytest.mark.parametrize("taps", [2, 3, 4])
def test_short_convolution_of_prompts(taps, C_, gdim, nq, nsc, lens):
    """steps of at least 64 rows: two and eight rows a workgroup, sequences that begin and end inside a workgroup's rows and are shorter than the taps, tails carried from step to step,
    channels in several workgroups and past the last whole one, norm groups of 8 to 256 channels and none"""
    rng = np.random.default_rng(taps + C_)
    w = orc.bf16_round(0.5 * rng.standard_normal((C_, taps)))
    full = {s: rng.standard_normal((sum(l[s] for l in lens), C_ + 4)).astype(np.float32) for s in (0, 1, 2)}
    want = {}
    for s, xs in full.items():
        y = orc.silu(orc.short_conv(orc.t64(xs[:, :C_]), orc.t64(w)))
        if nq:
            y[:, :nq] = orc.unit_vectors(y[:, :nq].reshape(-1, nq // gdim, gdim)).reshape(-1, nq)
        y[:, :nsc] *= 0.25
        want[s] = y.numpy()
    sl, at = Slots(3, (taps - 1) * C_), {0: 0, 1: 0, 2: 0}
    for step in lens:
        seqs = [(n, at[s], s) for s, n in ((2, step[2]), (0, step[0]), (1, step[1]))]
        x = np.concatenate([full[s][at[s]:at[s] + n] for n, _, s in seqs], 0)
        d, rs, T = seq_tables(seqs)
        assert T >= 64
        y, xd = torch.full((T, C_ + 4), 7.0, dtype=torch.float32, device="cuda"), dev32(x)
        ia.check(capi().ifa_shortconv_silu_f32(p(xd), C_ + 4, C_, taps, p(devbf(w)), p(d), p(rs), T, p(sl.table), 0, nq, gdim, 1e-6, nsc, 0.25, p(y), C_ + 4, stream()))
        ia.check(capi().ifa_shortconv_tail_f32(p(xd), C_ + 4, C_, taps, p(d), len(seqs), p(sl.table), 0, stream()))
        sync()
        got, r = y.cpu().numpy(), 0
        for n, a, s in seqs:
            assert np.abs(got[r:r + n, :C_] - want[s][a:a + n]).max() < 1e-5 and np.all(got[r:r + n, C_:] == 7.0), (step, s)
            at[s] += n; r += n


@pytest.mark.parametrize("C_,gdim,nq,nsc", [(40, 8, 16, 8), (1100, 100, 600, 300)])      # (the second: a row's channels in two workgroups)
@pytest.mark.parametrize("taps", [1, 2, 4])
def test_short_convolution_with_carried_tail(taps, C_, gdim, nq, nsc):
    rng = np.random.default_rng(taps)
    # channels [0, nq) unit-normed in groups of gdim, channels [0, nsc) scaled
    w = orc.bf16_round(0.5 * rng.standard_normal((C_, taps)))
    full = {s: rng.standard_normal((23, C_ + 5)).astype(np.float32) for s in (0, 1, 2)}

    def want(xs):
        y = orc.silu(orc.short_conv(orc.t64(xs[:, :C_]), orc.t64(w)))
        y[:, :nq] = orc.unit_vectors(y[:, :nq].reshape(-1, nq // gdim, gdim)).reshape(-1, nq)
        y[:, :nsc] *= 0.25
        return y.numpy()

    sl = Slots(3, max(1, (taps - 1)) * C_)
    at = {0: 0, 1: 0, 2: 0}
    # steps of several sequences with portions shorter than the tail; slot 2 is then reused by a new sequence from position 0
    plan = [[(0, 5), (1, 1), (2, 2)], [(1, 1), (0, 1)], [(2, 9), (1, 2), (0, 3)], [(0, 14), (1, 19)]]
    for step in plan:
        seqs = [(n, at[s], s) for s, n in step]
        x = np.concatenate([full[s][at[s]:at[s] + n] for s, n in step], 0)
        d, rs, T = seq_tables(seqs)
        y = torch.empty((T, C_), dtype=torch.float32, device="cuda")
        xd = dev32(x)
        ia.check(capi().ifa_shortconv_silu_f32(p(xd), C_ + 5, C_, taps, p(devbf(w)), p(d), p(rs), T, p(sl.table), 0, nq, gdim, 1e-6, nsc, 0.25, p(y), C_, stream()))
        ia.check(capi().ifa_shortconv_tail_f32(p(xd), C_ + 5, C_, taps, p(d), len(seqs), p(sl.table), 0, stream()))
        sync()
        got, r = y.cpu().numpy(), 0
        for s, n in step:
            assert np.abs(got[r:r + n] - want(full[s][:at[s] + n])[at[s]:]).max() < 1e-5, (taps, s, at[s])
            r += n; at[s] += n
    # reuse: a new sequence on slot 2 must not see the old tail
    new = rng.standard_normal((4, C_ + 5)).astype(np.float32)
    d, rs, T = seq_tables([(4, 0, 2)])
    y = torch.empty((T, C_), dtype=torch.float32, device="cuda")
    ia.check(capi().ifa_shortconv_silu_f32(p(dev32(new)), C_ + 5, C_, taps, p(devbf(w)), p(d), p(rs), T, p(sl.table), 0, nq, gdim, 1e-6, nsc, 0.25, p(y), C_, stream()))
    assert np.abs(y.cpu().numpy() - want(new)).max() < 1e-5


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("heads,qk_heads,dk,dv", [(2, 2, 8, 8), (4, 2, 24, 70), (3, 1, 130, 33), (2, 1, 32, 40), (4, 2, 64, 64), (2, 2, 128, 100), (2, 1, 16, 17)])
def test_state_recurrences(kind, heads, qk_heads, dk, dv):
    if kind == 0:
        qk_heads = heads
    rng = np.random.default_rng(dk + dv + kind)
    L = 37
    data = {}
    for s in (0, 1):
        q = rng.standard_normal((L, qk_heads * dk)).astype(np.float32) * 0.5
        k = rng.standard_normal((L, qk_heads * dk)).astype(np.float32) * 0.5
        v = rng.standard_normal((L, heads * dv)).astype(np.float32)
        beta = rng.uniform(0, 1, (L, heads)).astype(np.float32)
        g = rng.uniform(0.7, 1, (L, heads)).astype(np.float32)
        if kind == 1:      # unit keys like the design's, one of them far back with a long-lived state
            kk = orc.unit_vectors(orc.t64(k).reshape(L, qk_heads, dk)).reshape(L, -1).numpy().astype(np.float32); k = kk
        data[s] = (q, k, v, beta, g)
    decay = np.array([0.999, 0.5, 0.9, 0.97][:heads], np.float32)

    def want(s, n):
        q, k, v, beta, g = (orc.t64(a[:n]) for a in data[s])
        if kind == 0:
            return orc.decayed_linear_attention(orc.silu(q), orc.silu(k), orc.silu(v), heads, dk, dv, orc.t64(decay)).numpy()
        return orc.gated_delta_rule(q, k, v, beta, g, heads, qk_heads, dk, dv).numpy()

    sl = Slots(2, heads * dk * dv + 8)
    at = {0: 0, 1: 0}
    for step in ([(0, 6), (1, 1)], [(1, 1), (0, 1)], [(0, 2), (1, 30)], [(0, 28)]):
        seqs = [(n, at[s], s) for s, n in step]
        d, rs, T = seq_tables(seqs)
        cat = [np.concatenate([data[s][i][at[s]:at[s] + n] for s, n in step], 0) for i in range(5)]
        out = torch.empty((T, heads * dv), dtype=torch.float32, device="cuda")
        ia.check(capi().ifa_state_scan_f32(kind, 1 if kind == 0 else 0, p(dev32(cat[0])), qk_heads * dk, p(dev32(cat[1])), qk_heads * dk, p(dev32(cat[2])), heads * dv,
                                           heads, qk_heads, dk, dv, p(dev32(decay)) if kind == 0 else None, p(dev32(cat[4])) if kind == 1 else None,
                                           p(dev32(cat[3])) if kind == 1 else None, p(d), len(seqs), p(sl.table), 8, p(out), heads * dv, stream()))
        sync()
        got, r = out.cpu().numpy(), 0
        for s, n in step:
            w_ = want(s, at[s] + n)[at[s]:]
            assert np.abs(got[r:r + n] - w_).max() < 3e-5 * max(1.0, np.abs(w_).max()), (kind, s, at[s], n)
            r += n; at[s] += n


def test_delta_gates_and_gated_group_norm():
    rng = np.random.default_rng(5)
    T, H, dv = 7, 3, 20
    b, a = rng.standard_normal((T, H + 2)).astype(np.float32) * 3, rng.standard_normal((T, H + 1)).astype(np.float32) * 3
    alog, dtb = orc.bf16_round(rng.uniform(-2, 1, H)), orc.bf16_round(rng.uniform(-1, 1, H))
    beta, g = (torch.empty((T, H), dtype=torch.float32, device="cuda") for _ in range(2))
    ia.check(capi().ifa_delta_gates_f32(p(dev32(b)), H + 2, p(dev32(a)), H + 1, H, T, p(devbf(alog)), p(devbf(dtb)), p(beta), p(g), stream()))
    wb, wg = orc.delta_gates(orc.t64(b[:, :H]), orc.t64(a[:, :H]), orc.t64(alog), orc.t64(dtb))
    assert np.abs(beta.cpu().numpy() - wb.numpy()).max() < 1e-6 and np.abs(g.cpu().numpy() - wg.numpy()).max() < 1e-6
    o = rng.standard_normal((T, H * dv)).astype(np.float32) * 4
    gate = rng.standard_normal((T, H * dv + 4)).astype(np.float32) * 2
    for group, wlen, act, f in ((dv, dv, 1, orc.silu), (H * dv, H * dv, 0, torch.sigmoid)):
        w = orc.bf16_round(1 + 0.2 * rng.standard_normal(wlen))
        y = dev32(o)
        ia.check(capi().ifa_gated_groupnorm_f32(p(y), H * dv, T, H * dv, group, p(devbf(w)), wlen, p(dev32(gate)), H * dv + 4, act, 1e-5, p(y), H * dv, stream()))
        want = orc.rms_unit(orc.t64(o).reshape(T, -1, group), 1e-5).reshape(T, -1) * orc.t64(np.tile(w, H * dv // wlen)) * f(orc.t64(gate[:, :H * dv]))
        assert np.abs(y.cpu().numpy() - want.numpy()).max() < 1e-5


@pytest.mark.parametrize("tile_min", [16, 1 << 30])       # prompts through the tiled matrix-core kernel / every row through the per-row kernel
@pytest.mark.parametrize("heads,kv_heads,dim,window,keep,nb,dmax", [(4, 2, 16, 9, 2, 8, 30), (2, 2, 8, 1, 0, 4, 6), (3, 1, 68, 300, 5, 24, 200), (6, 3, 32, 17, 40, 10, 12),
                                                                    (2, 1, 64, 20, 3, 8, 30), (2, 1, 32, 2000, 4, 8, 30), (2, 2, 128, 50, 0, 16, 100), (1, 1, 96, 9, 2, 8, 30), (4, 2, 64, 33, 33, 6, 7), (8, 2, 16, 12, 1, 8, 30), (8, 1, 32, 25, 2, 8, 30)])
def test_windowed_attention_with_sink_cap_and_bucket_bias(heads, kv_heads, dim, window, keep, nb, dmax, tile_min):
    rng = np.random.default_rng(heads + dim + window)
    L, eps, scale, cap = 150, 1e-6, 0.3, 6.0
    q = rng.standard_normal((L, heads * dim + 4)).astype(np.float32)
    k = rng.standard_normal((L, kv_heads * dim + 2)).astype(np.float32)
    # one key far back, one just inside and one just outside the window get large matching queries at the last rows
    k[1, :dim] *= 6; k[max(0, L - window), :dim] *= 6; k[max(0, L - 1 - window), :dim] *= 6
    q[-1, :dim] = k[1, :dim]; q[-2, :dim] = k[max(0, L - 1 - window), :dim]
    rel = orc.bf16_round(rng.standard_normal((nb, heads)))
    sink = orc.bf16_round(rng.standard_normal(heads) * 2)
    want = orc.windowed_attention(orc.t64(q[:, :heads * dim]), orc.t64(k[:, :kv_heads * dim]), heads, kv_heads, dim, scale, cap, window, keep, orc.t64(rel), dmax,
                                  orc.t64(sink), eps).numpy()
    ctx = 160
    bucket_of = devi([orc.distance_bucket(n, nb, dmax) for n in range(ctx)])
    kvd = kv_heads * dim
    sl = Slots(2, 2 * ctx * kvd)
    ws = torch.full((2 * heads * 32 * (dim + 2),), float('nan'), dtype=torch.float32, device='cuda')      # single tokens: the keys shared out over workgroups
    at = 0
    for n in (1, 2, 60, 1, 1, 80, 5):                # prompt portions and single tokens; the same sequence lives on slot 1
        d, rs, T = seq_tables([(n, at, 1)])
        kd = dev32(k[at:at + n])
        ia.check(capi().ifa_kv_store_f32(p(kd), kv_heads * dim + 2, p(kd), kv_heads * dim + 2, kv_heads, dim, 1, eps, p(d), p(rs), T, p(sl.table), 0, ctx * kvd, stream()))
        out = torch.empty((T, heads * dim), dtype=torch.float32, device="cuda")
        ia.check(capi().ifa_attention_window_f32(p(dev32(q[at:at + n])), heads * dim + 4, heads, kv_heads, dim, 1, eps, scale, cap, window, keep, p(devbf(rel)),
                                                 p(bucket_of), nb, p(devbf(sink)), p(d), p(rs), T, p(sl.table), 0, ctx * kvd, p(out), heads * dim,
                                                 (C.c_int * 4)(0, n, at, 1), 1, tile_min, p(ws) if n <= 2 else None, ws.numel() * 4, stream()))
        sync()
        assert np.abs(out.cpu().numpy() - want[at:at + n]).max() < 2e-5 * max(1.0, np.abs(want).max()), (at, n)
        at += n
    assert at == L
    # without the sink the weights sum to one: a different result, so the sink is really counted
    d, rs, T = seq_tables([(1, L - 1, 1)])
    out = torch.empty((1, heads * dim), dtype=torch.float32, device="cuda")
    ia.check(capi().ifa_attention_window_f32(p(dev32(q[L - 1:])), heads * dim + 4, heads, kv_heads, dim, 1, eps, scale, cap, window, keep, p(devbf(rel)),
                                             p(bucket_of), nb, None, p(d), p(rs), T, p(sl.table), 0, ctx * kvd, p(out), heads * dim, None, 0, 0, None, 0, stream()))
    assert np.abs(out.cpu().numpy() - want[L - 1:]).max() > 1e-4


def test_windowed_attention_tiles_over_several_sequences():
    """one step holds a 150-token prompt, a single continued token and a 40-token continued portion: tiles must not cross sequences"""
    rng = np.random.default_rng(77)
    heads, kv_heads, dim, window, keep, nb, dmax, eps, scale, cap = 4, 2, 32, 40, 2, 8, 60, 1e-6, 0.4, 8.0
    L, ctx, kvd = 200, 208, kv_heads * dim
    seq = {s_: (rng.standard_normal((L, heads * dim)).astype(np.float32), rng.standard_normal((L, kvd)).astype(np.float32)) for s_ in (0, 1, 2)}
    rel, sink = orc.bf16_round(rng.standard_normal((nb, heads))), orc.bf16_round(rng.standard_normal(heads))
    want = {s_: orc.windowed_attention(orc.t64(q), orc.t64(k), heads, kv_heads, dim, scale, cap, window, keep, orc.t64(rel), dmax, orc.t64(sink), eps).numpy()
            for s_, (q, k) in seq.items()}
    bucket_of = devi([orc.distance_bucket(n, nb, dmax) for n in range(ctx)])
    sl = Slots(3, 2 * ctx * kvd)
    at = {0: 0, 1: 0, 2: 0}
    for step in ([(1, 30), (2, 100)], [(0, 150), (1, 1), (2, 40)], [(2, 60), (0, 50), (1, 129)]):
        seqs = [(n, at[s_], s_) for s_, n in step]
        d, rs, T = seq_tables(seqs)
        kd = dev32(np.concatenate([seq[s_][1][at[s_]:at[s_] + n] for s_, n in step], 0))
        qd = dev32(np.concatenate([seq[s_][0][at[s_]:at[s_] + n] for s_, n in step], 0))
        ia.check(capi().ifa_kv_store_f32(p(kd), kvd, p(kd), kvd, kv_heads, dim, 1, eps, p(d), p(rs), T, p(sl.table), 0, ctx * kvd, stream()))
        out = torch.empty((T, heads * dim), dtype=torch.float32, device="cuda")
        host, r = [], 0
        for n, pos0, slot in seqs:
            host += [r, n, pos0, slot]; r += n
        ia.check(capi().ifa_attention_window_f32(p(qd), heads * dim, heads, kv_heads, dim, 1, eps, scale, cap, window, keep, p(devbf(rel)), p(bucket_of), nb,
                                                 p(devbf(sink)), p(d), p(rs), T, p(sl.table), 0, ctx * kvd, p(out), heads * dim, (C.c_int * len(host))(*host),
                                                 len(seqs), 16, None, 0, stream()))
        sync()
        got, r = out.cpu().numpy(), 0
        for s_, n in step:
            assert np.abs(got[r:r + n] - want[s_][at[s_]:at[s_] + n]).max() < 2e-5 * max(1.0, np.abs(want[s_]).max()), (s_, at[s_], n)
            r += n; at[s_] += n


def dense_attention_64(q, k, v, pos0, heads, kv_heads, scale, window, keep, cap=0.0, rel=None, bucket_of=None, sink=None, norm_eps=None):
    """rows at positions pos0 .. over all keys, float64; q [n, heads, d], k [T, kv_heads, d], v [T, kv_heads, dv]"""
    n, T = q.shape[0], k.shape[0]
    i, j = torch.arange(pos0, pos0 + n)[:, None], torch.arange(T)[None, :]
    see = (j <= i) & ((i - j < window) | (j < keep))
    if norm_eps is not None:
        q = orc.rms_unit(q, norm_eps)
    out = []
    for h in range(heads):
        g = h // (heads // kv_heads)
        sc = q[:, h] @ k[:, g].T * scale
        if cap:
            sc = cap * torch.tanh(sc / cap)
        if rel is not None:
            sc = sc + rel[:, h][bucket_of[(i - j).clamp(min=0)]]
        sc = sc.masked_fill(~see, -np.inf)
        m = sc.max(-1, keepdim=True).values
        e = torch.exp(sc - m)
        den = e.sum(-1, keepdim=True) + (torch.exp(sink[h] - m) if sink is not None else 0.0)
        out.append(e / den @ v[:, g])
    return torch.stack(out, 1).reshape(n, -1)


# chunks of 64: one token more or less than a chunk, several chunks, sequences that end inside one, continued states, shared q / k heads, one value tile and odd counts of them
@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("heads,qk_heads,dk,dv,steps", [(2, 2, 64, 128, [[(0, 1)], [(0, 63)], [(0, 64)]]), (4, 2, 128, 32, [[(0, 65), (1, 200)], [(1, 64), (0, 1)]]),
                                                        (3, 1, 64, 96, [[(0, 130), (1, 3), (2, 64)], [(2, 66)]]), (2, 1, 128, 160, [[(0, 257)], [(0, 31)]]),
                                                        (4, 2, 64, 64, [[(0, 700)]])])
def test_state_recurrences_in_chunks(kind, heads, qk_heads, dk, dv, steps):
    """Against the float64 recurrence, beside the token-by-token kernel on the same states: no further from it than that kernel is, outputs and states, over all of a case's
    values (a tenth is what the two scatter by; single short sequences by more), and no value off by more than 1e-5 of the largest.  One head's decays reach 0.02
    per token, another's are 1."""
    rng = np.random.default_rng(heads * 10 + dk + kind)
    total = {s_: sum(n for st in steps for q_, n in st if q_ == s_) for s_ in range(3)}
    unit = lambda a: (a / np.linalg.norm(a.reshape(a.shape[0], -1, dk), axis=-1).repeat(dk, -1).reshape(a.shape)).astype(np.float32)
    data = {}
    for s_, L in total.items():
        q, k = rng.standard_normal((L, qk_heads * dk)).astype(np.float32), rng.standard_normal((L, qk_heads * dk)).astype(np.float32)
        v = rng.standard_normal((L, heads * dv)).astype(np.float32)
        g, b = np.exp(-rng.uniform(0, 0.3, (L, heads))).astype(np.float32), rng.uniform(0.05, 1, (L, heads)).astype(np.float32)
        if L:
            g[:, 0] = np.exp(-rng.uniform(0, 4, L)); g[:, -1] = 1.0
        data[s_] = (unit(q) if kind else q, unit(k) if kind else 0.3 * k, v, g, b) if L else None
    dec = np.array([0.02, 1.0, 0.97, 0.999][:heads], np.float32)
    want = {}
    for s_, d in data.items():
        if d is None:
            continue
        q, k, v, g, b = (orc.t64(a) for a in d)
        if kind:
            want[s_] = orc.gated_delta_rule(q, k, v, b, g, heads, qk_heads, dk, dv).numpy()
        else:
            rep = lambda a: a.reshape(-1, qk_heads, dk).repeat_interleave(heads // qk_heads, 1).reshape(a.shape[0], -1)
            want[s_] = orc.decayed_linear_attention(rep(q), rep(k), v, heads, dk, dv, orc.t64(dec)).numpy()
    s_off, off = 8, np.zeros(2)          # (off: squared errors, relative to each sequence's size)
    slots = [Slots(3, s_off + heads * dk * dv + 4) for _ in range(2)]
    at = {0: 0, 1: 0, 2: 0}
    for st in steps:
        seqs = [(n, at[s_], s_) for s_, n in st]
        d, rs, T = seq_tables(seqs)
        host, r = [], 0
        for n, pos0, slot in seqs:
            host += [r, n, pos0, slot]; r += n
        host = (C.c_int * len(host))(*host)
        q, k, v, g, b = (dev32(np.concatenate([data[s_][i][at[s_]:at[s_] + n] for s_, n in st], 0)) for i in range(5))
        chunks = sum((n + 63) // 64 for _, n in st)
        nb = capi().ifa_state_chunked_workspace_bytes(kind, chunks, heads, dk, dv)
        ws = torch.full((nb // 4,), float("nan"), dtype=torch.float32, device="cuda")
        outs = [torch.full((T, heads * dv + 4), float("nan"), dtype=torch.float32, device="cuda") for _ in range(2)]
        gates = (p(dev32(dec)), None, None) if kind == 0 else (None, p(g), p(b))
        assert capi().ifa_state_chunked_fits(kind, p(q), qk_heads * dk, p(k), qk_heads * dk, p(v), heads * dv, dk, dv, p(outs[0]), heads * dv + 4)
        ia.check(capi().ifa_state_chunked_f32(kind, p(q), qk_heads * dk, p(k), qk_heads * dk, p(v), heads * dv, heads, qk_heads, dk, dv, *gates, p(d), host, len(st),
                                              p(slots[0].table), s_off, p(ws), nb, p(outs[0]), heads * dv + 4, None))
        ia.check(capi().ifa_state_scan_f32(kind, 0, p(q), qk_heads * dk, p(k), qk_heads * dk, p(v), heads * dv, heads, qk_heads, dk, dv, *gates, p(d), len(st),
                                           p(slots[1].table), s_off, p(outs[1]), heads * dv + 4, None))
        sync()
        got, r = [o.cpu().numpy()[:, :heads * dv] for o in outs], 0
        for s_, n in st:
            w = want[s_][at[s_]:at[s_] + n]
            err = [np.abs(x[r:r + n] - w).max() / np.abs(w).max() for x in got]
            assert err[0] < 1e-5, (s_, at[s_], n)
            off += np.array([np.square((x[r:r + n] - w) / np.linalg.norm(w) * n ** 0.5).sum() for x in got])
            r += n; at[s_] += n
        assert (slots[0].mem[st[0][0]][s_off + heads * dk * dv:] == 1e9).all() and (slots[0].mem[st[0][0]][:s_off] == 1e9).all()
    print("state", kind, heads, dk, dv, "chunks %.3g tokens %.3g" % tuple(np.sqrt(off / sum(total.values()))))
    assert off[0] < 1.1 ** 2 * off[1], np.sqrt(off / sum(total.values()))
    # the states: the recurrence's own, from the tokens
    off = np.zeros(2)
    for s_, d in data.items():
        if d is None:
            continue
        q, k, v, g, b = (orc.t64(a) for a in d)
        L = len(q)
        kk, vv = k.reshape(L, qk_heads, dk).repeat_interleave(heads // qk_heads, 1), v.reshape(L, heads, dv)
        S = torch.zeros(heads, dk, dv, dtype=torch.float64)
        for t in range(L):
            S = S * (g[t] if kind else orc.t64(dec))[:, None, None]
            u = b[t][:, None] * (vv[t] - torch.einsum("hk,hkv->hv", kk[t], S)) if kind else vv[t]
            S = S + kk[t][:, :, None] * u[:, None]
        for f in range(2):
            off[f] += float((slots[f].mem[s_][s_off:s_off + S.numel()].cpu().double() - S.reshape(-1)).norm() / S.norm()) ** 2 * L
    print("state", kind, heads, dk, dv, "left behind: chunks %.3g tokens %.3g" % tuple(np.sqrt(off / sum(total.values()))))
    assert off[0] < 1.1 ** 2 * off[1], np.sqrt(off / sum(total.values()))


@pytest.mark.parametrize("kind,what,value", [(0, "v", np.inf), (0, "v", np.nan), (0, "k", np.nan), (1, "v", -np.inf), (1, "v", np.nan), (1, "k", np.nan), (1, "g", np.nan), (1, "b", np.nan)])
def test_infinities_and_nan_in_chunks_reach_no_earlier_token_and_no_other_column(kind, what, value):
    """one value of one token not finite, at the edges of chunks and of their 16 positions: finite outputs and states exactly where the token-by-token form has them"""
    rng = np.random.default_rng(kind)
    heads, dk, dv, n = 2, 64, 96, 130
    unit = lambda a: (a / np.linalg.norm(a.reshape(n, heads, dk), axis=-1).repeat(dk, -1)).astype(np.float32)
    base = {"q": unit(rng.standard_normal((n, heads * dk))), "k": unit(rng.standard_normal((n, heads * dk))), "v": rng.standard_normal((n, heads * dv)),
            "g": np.exp(-rng.uniform(0, 0.3, (n, heads))), "b": rng.uniform(0.05, 1, (n, heads))}
    d, rs, _ = seq_tables([(n, 0, 0)])
    host = (C.c_int * 4)(0, n, 0, 0)
    nb = capi().ifa_state_chunked_workspace_bytes(kind, 3, heads, dk, dv)
    for at in (0, 6, 15, 16, 63, 64, 100, 129):
        x = {name: np.array(a, np.float32) for name, a in base.items()}
        x[what][at, x[what].shape[1] - 2] = value
        x = {name: dev32(a) for name, a in x.items()}
        gates = (p(dev32(np.array([0.9, 0.99]))), None, None) if kind == 0 else (None, p(x["g"]), p(x["b"]))
        sl, outs = [Slots(1, heads * dk * dv) for _ in range(2)], [torch.zeros((n, heads * dv), dtype=torch.float32, device="cuda") for _ in range(2)]
        ws = torch.full((nb // 4,), float("nan"), dtype=torch.float32, device="cuda")
        a = (p(x["q"]), heads * dk, p(x["k"]), heads * dk, p(x["v"]), heads * dv)
        ia.check(capi().ifa_state_chunked_f32(kind, *a, heads, heads, dk, dv, *gates, p(d), host, 1, p(sl[0].table), 0, p(ws), nb, p(outs[0]), heads * dv, None))
        ia.check(capi().ifa_state_scan_f32(kind, 0, *a, heads, heads, dk, dv, *gates, p(d), 1, p(sl[1].table), 0, p(outs[1]), heads * dv, None))
        sync()
        for got, want in ((outs[0], outs[1]), (sl[0].mem[0], sl[1].mem[0])):
            fin = torch.isfinite(want)
            assert torch.equal(torch.isfinite(got), fin), (at, int(torch.isfinite(got).sum()), int(fin.sum()))
            assert float((got - want)[fin].abs().max()) < 1e-5 * float(want[fin].abs().max()) if fin.any() else True


# edges of the tiled kernel with a workspace: query tiles of 64 / 128 / 256 (groups of 4, 2, 1 heads), key blocks of 32, windows and kept tokens that begin and end
# inside blocks and meet in one, one chunk and many (short and long key ranges beside each other), continued sequences, four (placed by the launch's arguments) and five, head sizes that are not whole 32s or 4s
TILE_WS = [(4, 1, 128, 128, 1 << 30, 0, [(0, 16)], 1.0), (8, 2, 128, 128, 1 << 30, 0, [(0, 65)], 1.0), (8, 2, 64, 128, 1 << 30, 0, [(0, 700), (0, 3), (610, 90)], 1.0),
           (4, 2, 96, 32, 40, 0, [(0, 257)], 1.0), (3, 3, 32, 96, 33, 31, [(0, 300), (500, 33)], 1.0), (6, 2, 128, 64, 64, 33, [(95, 70), (0, 64)], 1.0),
           (4, 1, 36, 20, 100, 70, [(0, 310)], 1.0), (2, 1, 127, 101, 32, 0, [(0, 129), (31, 32)], 1.0), (8, 2, 128, 128, 1024, 4, [(0, 1300)], 1.0),
           (8, 2, 64, 96, 1 << 30, 0, [(0, 700), (0, 3), (610, 90), (300, 40)], 1.0), (8, 2, 64, 96, 1 << 30, 0, [(0, 700), (0, 3), (610, 90), (300, 40), (900, 1)], 1.0),
           (5, 1, 5, 3, 17, 300, [(200, 150)], 1.0), (8, 2, 128, 128, 1 << 30, 0, [(0, 200)], 1e4), (8, 2, 128, 128, 1 << 30, 0, [(0, 200)], 1e-7)]


@pytest.mark.parametrize("form", ["plain", "capped"])
@pytest.mark.parametrize("heads,kv_heads,dim,vdim,window,keep,seqs,size", TILE_WS)
def test_tiled_attention_with_a_workspace_against_64_bits_and_the_fp32_tiles(heads, kv_heads, dim, vdim, window, keep, seqs, size, form):
    """Three bfloat16 parts per operand leave the results no further from 64 bits than fp32 operands do.  Bound: dim + 2 fp32 roundings of a score, |scores| below
    ~6, weights that sum to one -> 1e-6 of the largest value; measured 2e-7 .. 5e-7 on either side."""
    if form == "capped":
        vdim = dim
    rng = np.random.default_rng(heads * 100 + dim + window % 1000)
    ctx = max(a + n for a, n in seqs) + 3
    k_off, v_off = 4, 4 + (ctx * kv_heads * dim + 3) // 4 * 4
    sl = Slots(len(seqs), v_off + ctx * kv_heads * vdim)
    ks, vs = [], []
    for s_, (pos0, n) in enumerate(seqs):
        k, v = rng.standard_normal((pos0 + n, kv_heads, dim)).astype(np.float32), (size * rng.standard_normal((pos0 + n, kv_heads, vdim))).astype(np.float32)
        if form == "plain":
            k *= np.float32(size)
        sl.mem[s_][k_off:k_off + k.size] = dev32(k.reshape(-1)); sl.mem[s_][v_off:v_off + v.size] = dev32(v.reshape(-1))
        ks.append(k); vs.append(v)
    host, r = [], 0
    for s_, (pos0, n) in enumerate(seqs):
        host += [r, n, pos0, s_]; r += n
    host = (C.c_int * len(host))(*host)
    d, rs, T = seq_tables([(n, pos0, s_) for s_, (pos0, n) in enumerate(seqs)])
    q = rng.standard_normal((T, heads * dim)).astype(np.float32)
    rel, sink, cap = orc.bf16_round(rng.standard_normal((6, heads))), orc.bf16_round(rng.standard_normal(heads)), 5.0
    bucket = rng.integers(0, 6, ctx)
    scale = (1.0 if form == "capped" else 1.0 / size) * dim ** -0.5
    nb = capi().ifa_attention_tile_workspace_bytes(host, len(seqs), heads, kv_heads, dim, vdim, window, keep)
    assert nb > 0
    got = []
    for ws_bytes in (nb, 0):
        ws = torch.full((nb // 4,), float("nan"), dtype=torch.float32, device="cuda")
        out = torch.full((T, heads * vdim + 4), float("nan"), dtype=torch.float32, device="cuda")
        a = (p(d), p(rs), T, p(sl.table), k_off, v_off, p(out), heads * vdim + 4, host, len(seqs), 16)
        w = (p(ws) if ws_bytes else None, ws_bytes, None)
        if form == "capped":
            ia.check(capi().ifa_attention_window_f32(p(dev32(q)), heads * dim, heads, kv_heads, dim, 1, 1e-6, scale, cap, window, keep, p(devbf(rel)), p(devi(bucket)), 6,
                                                     p(devbf(sink)), *a, *w))
        else:
            ia.check(capi().ifa_attention_kv_f32(p(dev32(q)), heads * dim, heads, kv_heads, dim, vdim, scale, 0 if window == 1 << 30 else window, keep, 0, 0.0, *a, 0, *w))
        sync()
        got.append(out.cpu().numpy()[:, :heads * vdim])
    r = 0
    for s_, (pos0, n) in enumerate(seqs):
        extra = dict(cap=cap, rel=orc.t64(rel), bucket_of=torch.from_numpy(bucket), sink=orc.t64(sink), norm_eps=1e-6) if form == "capped" else {}
        want = dense_attention_64(orc.t64(q[r:r + n]).reshape(n, heads, dim), orc.t64(ks[s_]), orc.t64(vs[s_]), pos0, heads, kv_heads, scale, window, keep, **extra).numpy()
        off = [np.abs(g[r:r + n] - want).max() / np.abs(want).max() for g in got]
        print(form, heads, dim, (pos0, n), "parts %.2g fp32 %.2g" % tuple(off), "rms %.3g %.3g" % tuple(np.linalg.norm(g[r:r + n] - want) / np.linalg.norm(want) for g in got))
        assert off[0] < 1e-6 and np.linalg.norm(got[0][r:r + n] - want) < 1.1 * np.linalg.norm(got[1][r:r + n] - want) + 2e-8 * np.linalg.norm(want), (pos0, n)
        r += n


def test_tiled_attention_takes_fewer_chunks_where_the_workspace_is_small():
    """2000 keys: with all the workspace many chunks per tile, with just the operands' bytes and one share more none; both the same sums in another grouping"""
    rng = np.random.default_rng(3)
    heads, kv_heads, dim, T = 4, 1, 32, 2000
    sl = Slots(1, 2 * T * dim)
    sl.mem[0].copy_(dev32(rng.standard_normal(2 * T * dim)))
    host = (C.c_int * 4)(0, T, 0, 0)
    d, rs, _ = seq_tables([(T, 0, 0)])
    q = dev32(rng.standard_normal((T, heads * dim)))
    nb = capi().ifa_attention_tile_workspace_bytes(host, 1, heads, kv_heads, dim, dim, 0, 0)
    ops = (T + 31) // 32 * 3 * 64 * 16 * 4 + ((T + 31) // 32 * 4 + 15) // 16 * 16          # (a mark per block behind them)
    res = []
    for ws_bytes in (nb, nb - 4, ops + 64, ops - 4):          # (the last: the operands do not fit, the fp32 tiles)
        ws, out = torch.empty(nb, dtype=torch.uint8, device="cuda"), torch.empty((T, heads * dim), dtype=torch.float32, device="cuda")
        ia.check(capi().ifa_attention_kv_f32(p(q), heads * dim, heads, kv_heads, dim, dim, dim ** -0.5, 0, 0, 0, 0.0, p(d), p(rs), T, p(sl.table), 0, T * dim, p(out), heads * dim,
                                             host, 1, 16, 0, p(ws), ws_bytes, None))
        sync(); res.append(out.cpu().numpy())
    for r in res[1:]:
        assert np.abs(r - res[0]).max() < 2e-6 * np.abs(res[0]).max()


def test_tiled_attention_of_more_key_blocks_than_a_grid_has():
    """32 queries behind 65600 keys each (2.1 million keys, one slot read by all): the workspace form's launch has a workgroup per block of 32 keys, up to 65535 of
    them; beyond that the step runs as it does without a workspace"""
    rng = np.random.default_rng(4)
    heads, dim, T, ctx = 1, 32, 32, 65600
    sl = Slots(1, 2 * (ctx + 1) * dim)
    sl.mem[0].copy_(dev32(rng.standard_normal(2 * (ctx + 1) * dim)))
    d, rs, _ = seq_tables([(1, ctx, 0)] * T)
    host = (C.c_int * (4 * T))(*sum([[t, 1, ctx, 0] for t in range(T)], []))
    q = dev32(rng.standard_normal((T, dim)))
    nb = capi().ifa_attention_tile_workspace_bytes(host, T, heads, 1, dim, dim, 0, 0)
    assert nb > 65535 * 3 * 64 * 16 * 4
    res = []
    for ws_bytes in (0, nb):
        ws, out = torch.empty(max(ws_bytes, 4), dtype=torch.uint8, device="cuda"), torch.full((T, dim), float("nan"), dtype=torch.float32, device="cuda")
        ia.check(capi().ifa_attention_kv_f32(p(q), dim, heads, 1, dim, dim, dim ** -0.5, 0, 0, 0, 0.0, p(d), p(rs), T, p(sl.table), 0, (ctx + 1) * dim, p(out), dim, host, T, 16, 0,
                                             p(ws) if ws_bytes else None, ws_bytes, None))
        sync(); res.append(out)
    assert torch.equal(res[0], res[1]) and bool(torch.isfinite(res[0]).all())


@pytest.mark.parametrize("where,value", [("k", np.inf), ("k", -np.inf), ("v", np.inf), ("v", -np.inf), ("v", np.nan), ("k", np.nan), ("v", 3.395e38), ("v", -3.402e38), ("k", 3.4e38)])
def test_tiled_attention_with_infinite_and_very_large_keys_and_values(where, value):
    """one element of a key or value that every query sees, in a block of its own and beside others: infinities, NaN and finite outputs where the fp32 tiles have them (an
    infinite key's score is -inf for half of the queries: weight 0), finite ones within 2e-6.  Very large values round to no bfloat16."""
    rng = np.random.default_rng(8)
    heads, kv_heads, dim, pos0, n = 4, 2, 64, 70, 100
    ctx = pos0 + n
    host = (C.c_int * 4)(0, n, pos0, 0)
    d, rs, _ = seq_tables([(n, pos0, 0)])
    q = dev32(rng.standard_normal((n, heads * dim)))
    nb = capi().ifa_attention_tile_workspace_bytes(host, 1, heads, kv_heads, dim, dim, 0, 0)
    for rows in ((5,), (5, 40), (69,)):
        kv = {"k": rng.standard_normal((ctx, kv_heads, dim)).astype(np.float32), "v": rng.standard_normal((ctx, kv_heads, dim)).astype(np.float32)}
        for i, r in enumerate(rows):
            kv[where][r, 1, 17 + i] = value
        sl = Slots(1, 2 * ctx * kv_heads * dim)
        sl.mem[0].copy_(dev32(np.concatenate([kv["k"].reshape(-1), kv["v"].reshape(-1)])))
        out = []
        for ws_bytes in (nb, 0):
            ws, o = torch.full((nb // 4,), float("nan"), dtype=torch.float32, device="cuda"), torch.zeros((n, heads * dim), dtype=torch.float32, device="cuda")
            ia.check(capi().ifa_attention_kv_f32(p(q), heads * dim, heads, kv_heads, dim, dim, dim ** -0.5, 0, 0, 0, 0.0, p(d), p(rs), n, p(sl.table), 0, ctx * kv_heads * dim, p(o),
                                                 heads * dim, host, 1, 16, 0, p(ws) if ws_bytes else None, ws_bytes, None))
            sync(); out.append(o.cpu().numpy())
        got, want = out
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want)) and np.array_equal(got[np.isinf(got)], want[np.isinf(want)]), rows
        fin = np.isfinite(want)
        big = np.abs(want) > 1e30
        for part in (fin & big, fin & ~big):
            assert not part.any() or np.abs(got[part] / 2 - want[part] / 2).max() < 1e-6 * np.abs(want[part]).max(), rows


@pytest.mark.parametrize("value", [3.395e38, -3.402e38, 3.3e38])
def test_tiled_attention_with_very_large_queries(value):
    """one value of two queries that rounds to no bfloat16, or just does, beside ordinary ones, on keys whose column is as small: the fp32 tiles' outputs within 2e-6 (the bound of the test above)"""
    rng = np.random.default_rng(9)
    heads, kv_heads, dim, n = 4, 2, 128, 100
    host = (C.c_int * 4)(0, n, 0, 0)
    d, rs, _ = seq_tables([(n, 0, 0)])
    q = rng.standard_normal((n, heads, dim)).astype(np.float32)
    q[40, 1, 77] = q[99, 3, 77] = value
    k, v = (rng.standard_normal((n, kv_heads, dim)).astype(np.float32) for _ in range(2))
    k[:, :, 77] *= 1e-30
    sl = Slots(1, 2 * n * kv_heads * dim)
    sl.mem[0].copy_(dev32(np.concatenate([k.reshape(-1), v.reshape(-1)])))
    qd = dev32(q.reshape(n, -1))
    nb = capi().ifa_attention_tile_workspace_bytes(host, 1, heads, kv_heads, dim, dim, 0, 0)
    out = []
    for ws_bytes in (nb, 0):
        ws, o = torch.full((nb // 4,), float("nan"), dtype=torch.float32, device="cuda"), torch.zeros((n, heads * dim), dtype=torch.float32, device="cuda")
        ia.check(capi().ifa_attention_kv_f32(p(qd), heads * dim, heads, kv_heads, dim, dim, 1e-8, 0, 0, 0, 0.0, p(d), p(rs), n, p(sl.table), 0, n * kv_heads * dim, p(o), heads * dim, host, 1, 16, 0,
                                             p(ws) if ws_bytes else None, ws_bytes, None))
        sync(); out.append(o.cpu().numpy())
    got, want = out
    assert np.isfinite(want).all() and np.abs(got - want).max() < 2e-6 * np.abs(want).max()
    flat = v[:41, 0].mean(axis=0)          # (the large value counts: its query's weights are not all alike)
    assert np.abs(want[40].reshape(heads, dim)[1] - flat).max() > 0.1


@pytest.mark.parametrize("window,keep", [(1 << 30, 0), (90, 40)])
def test_tiled_attention_over_many_sequences(window, keep):
    """130 sequences, most of one row, some of several and of more than four query tiles, at places that a wave looks at together and one by one: the rows' kernel's
    outputs within the fp32 roundings of 300 keys (the bound of the test above)"""
    rng = np.random.default_rng(6)
    heads, kv_heads, dim, ctx = 4, 1, 32, 420
    seqs = [(1, int(rng.integers(0, 400))) for _ in range(130)]
    for at, one in ((0, (270, 3)), (5, (33, 64)), (63, (330, 31)), (64, (257, 0)), (70, (64, 100)), (127, (300, 100)), (129, (400, 0))):
        seqs[at] = one
    sl = Slots(3, 2 * ctx * dim)
    for m in sl.mem:
        m.copy_(dev32(rng.standard_normal(2 * ctx * dim)))
    d, rs, T = seq_tables([(n, pos0, i % 3) for i, (n, pos0) in enumerate(seqs)])
    host = (C.c_int * (4 * len(seqs)))(*d.cpu().numpy().reshape(-1).tolist())
    q = dev32(rng.standard_normal((T, heads * dim)))
    nb = capi().ifa_attention_tile_workspace_bytes(host, len(seqs), heads, kv_heads, dim, dim, 0 if window == 1 << 30 else window, keep)
    res = []
    for tile_min in (1 << 30, 16):
        ws, out = torch.full((nb // 4,), float("nan"), dtype=torch.float32, device="cuda"), torch.full((T, heads * dim), float("nan"), dtype=torch.float32, device="cuda")
        ia.check(capi().ifa_attention_kv_f32(p(q), heads * dim, heads, kv_heads, dim, dim, dim ** -0.5, 0 if window == 1 << 30 else window, keep, 0, 0.0, p(d), p(rs), T, p(sl.table), 0,
                                             ctx * dim, p(out), heads * dim, host, len(seqs), tile_min, ctx, p(ws) if tile_min == 16 else None, nb, None))
        sync(); res.append(out)
    assert float((res[0] - res[1]).abs().max()) < 2e-6 * float(res[0].abs().max())


@pytest.mark.parametrize("T", [2, 4, 5, 6, 8])
@pytest.mark.parametrize("K", [504, 512, 520, 1024, 1032, 1536, 2048, 2056, 3080])
def test_products_of_a_few_rows_at_the_edges_of_the_weights_pieces(T, K):
    """512 columns a piece, one, two or four pieces asked for together: K fp32 multiply-adds of magnitudes ~1 and weights ~1 / sqrt(K) (bound 1e-5; measured 1e-6)"""
    rng = np.random.default_rng(T + K)
    N = 37
    W, bias = orc.bf16_round(rng.standard_normal((N, K)) / K ** 0.5), orc.bf16_round(rng.standard_normal(N))
    x = rng.standard_normal((T, K + 8)).astype(np.float32)
    c = torch.full((T, N + 1), float("nan"), dtype=torch.float32, device="cuda")
    ia.check(capi().ifa_linear_bf16w_rows(0, None, 0.0, p(devbf(W)), N, K, p(dev32(x)), K + 8, T, p(devbf(bias)), None, 1.0, 0, p(c), N + 1, 0, 0, stream()))
    got = c.cpu().numpy()
    want = (orc.t64(x[:, :K]) @ orc.t64(W).T + orc.t64(bias)).numpy()
    assert np.abs(got[:, :N] - want).max() < 1e-5 * np.abs(want).max() and np.isnan(got[:, N:]).all()


@pytest.mark.parametrize("n", [1, 3, 4, 7, 255, 1024, 4096, 4099, 4100, 8192, 16380, 16384, 16388, 20001, 33000])
def test_argmax_of_rows_of_any_length(n):
    """the largest value first, last, at the edges of rounds of 4 and 16 values a thread, twice (the lower index counts), and excluded"""
    rng = np.random.default_rng(n)
    spots = sorted({0, n - 1, n // 2, (n & ~3) - 1, n & ~3, 4095, 4096, 16383, 16384, 4 * 256 - 1, 4 * 256} & set(range(n)))
    lg = rng.standard_normal((2 * len(spots), (n + 3) // 4 * 4)).astype(np.float32)
    for i, c in enumerate(spots):
        lg[2 * i, c] = 9.0
        lg[2 * i + 1, c] = lg[2 * i + 1, n - 1] = lg[2 * i + 1, n // 3] = 9.0
    lg[:, n:] = 99.0
    for ex in (-1, n - 1):
        best = torch.empty(len(lg), dtype=torch.int32, device="cuda")
        ia.check(capi().ifa_argmax_rows_f32(p(dev32(lg)), n, lg.shape[1], len(lg), p(devi([1, ex, -1, -1])), p(best), stream()))
        masked = lg[:, :n].copy()
        if ex >= 0:
            masked[:, ex] = -np.inf
        assert best.cpu().tolist() == [int(r.argmax()) for r in masked]


@pytest.mark.parametrize("n", [1, 3, 1023, 1024, 1025, 4099, 32000, 40960, 40961, 65535, 65536, 65537, 70001])
def test_argmax_in_parts_takes_what_the_argmax_of_a_row_does(n):
    """the largest value at the edges of parts, twice (the lower index counts), excluded, beside NaN and among infinities; rows that start at odd places; and a decode step's move to its next token"""
    lib = capi()
    lib.ifa_argmax_parts_bytes.restype = C.c_size_t
    f = lib.ifa_argmax_parts_f32
    f.argtypes = [C.c_void_p, C.c_size_t, C.c_size_t, C.c_size_t] + [C.c_void_p] * 5
    part = max(1024, ((n + 63) // 64 + 3) // 4 * 4)
    spots = sorted({0, 3, n - 1, n // 2, part - 1, part, 2 * part - 1, (n - 1) // part * part} & set(range(n)))
    rng = np.random.default_rng(n)
    lg = rng.standard_normal((2 * len(spots) + 2, n + 1)).astype(np.float32)
    for i, c in enumerate(spots):
        lg[2 * i, c] = 9.0
        lg[2 * i + 1, c] = lg[2 * i + 1, n - 1] = lg[2 * i + 1, n // 3] = 9.0
        lg[2 * i, (c + 1) % n] = np.nan if n > 1 else 9.0
    lg[-2] = -np.inf
    lg[-1] = np.nan
    lg[:, n:] = 99.0
    x, ws = dev32(lg), torch.empty(lib.ifa_argmax_parts_bytes(), dtype=torch.uint8, device="cuda")
    for ex in ([0, -1, -1, -1], [1, n - 1, -1, -1], [3, n - 1, 0, n // 3]):
        got, want, rows = (torch.empty(len(lg), dtype=torch.int32, device="cuda") for _ in range(3))
        ia.check(lib.ifa_argmax_rows_f32(p(x), n, lg.shape[1], len(lg), p(devi(ex)), p(want), stream()))
        ia.check(f(p(x), n, lg.shape[1], len(lg), p(devi(ex)), p(rows), p(ws), None, stream()))
        for r in range(len(lg)):
            ia.check(f(C.c_void_p(x.data_ptr() + 4 * r * lg.shape[1]), n, lg.shape[1], 1, p(devi(ex)), C.c_void_p(got.data_ptr() + 4 * r), p(ws), None, stream()))
        assert torch.equal(got, want) and torch.equal(rows, want)

    # (a row that no step follows is left to one launch where that is as fast: nothing lies in the parts' workspace then)
    ws.fill_(77)
    ia.check(f(p(x), n, lg.shape[1], 1, None, p(got), p(ws), None, stream()))
    assert bool((ws == 77).all()) == (n <= 40960)

    class Advance(C.Structure):
        _fields_ = [("tokens", C.c_void_p), ("pos", C.c_void_p), ("seqs", C.c_void_p), ("ring", C.c_void_p), ("ring_size", C.c_int)]
    tokens, pos, seqs, ring, best = devi([7]), devi([1030]), devi([0, 1, 1030, 5]), torch.full((8,), -1, dtype=torch.int32, device="cuda"), devi([-1])
    step = Advance(tokens.data_ptr(), pos.data_ptr(), seqs.data_ptr(), ring.data_ptr(), 8)
    ia.check(f(p(x), n, lg.shape[1], 1, None, p(best), p(ws), C.byref(step), stream()))
    at = int(best.cpu()[0])
    assert tokens.tolist() == [at] and pos.tolist() == [1031] and seqs.tolist() == [0, 1, 1031, 5] and ring.tolist() == [-1] * 6 + [at, -1]


@pytest.mark.parametrize("T", [1, 2, 3, 5, 8])
def test_row_products_with_the_norm_or_the_gated_gelu_folded_in(T):
    rng = np.random.default_rng(40 + T)
    N, K = 77, 96
    W = orc.bf16_round(rng.standard_normal((N, K)) / 8)
    bias, mul, g = (orc.bf16_round(rng.standard_normal(n)) for n in (N, N, K))
    x = (2 * rng.standard_normal((T, K + 4)) + 1).astype(np.float32)
    c0 = rng.standard_normal((T, N)).astype(np.float32)
    c = dev32(c0)
    ia.check(capi().ifa_linear_bf16w_rows(1, p(devbf(g)), 1e-5, p(devbf(W)), N, K, p(dev32(x)), K + 4, T, p(devbf(bias)), p(devbf(mul)), 0.5, 1, p(c), N, 3, 9, stream()))
    h = orc.layer_norm_nobias(orc.t64(x[:, :K]), orc.t64(g), 1e-5)
    want = h @ orc.t64(W).T + orc.t64(bias)
    want[:, 3:9] = orc.silu(want[:, 3:9])
    want = (want * orc.t64(mul) * 0.5 + orc.t64(c0)).numpy()
    assert np.abs(c.cpu().numpy() - want).max() < 2e-5 * max(1.0, np.abs(want).max())
    gu = (2 * rng.standard_normal((T, 2 * K + 4))).astype(np.float32)
    c = torch.empty((T, N), dtype=torch.float32, device="cuda")
    ia.check(capi().ifa_linear_bf16w_rows(2, None, 0.0, p(devbf(W)), N, K, p(dev32(gu)), 2 * K + 4, T, None, None, 1.0, 0, p(c), N, 0, 0, stream()))
    want = ((orc.gelu_tanh(orc.t64(gu[:, :K])) * orc.t64(gu[:, K:2 * K])) @ orc.t64(W).T).numpy()
    assert np.abs(c.cpu().numpy() - want).max() < 2e-5 * max(1.0, np.abs(want).max())
