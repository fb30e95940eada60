"""Prompts' attention that stores the step's keys and values on the way to its operands, turns the queries in the same launch and brings the decayed linear attention of the layer with it
(ifa_attention_kv_to_bf16, ifa_attention_window_to_bf16) against the launches these stand for (ifa_qk_rope_store_f32 / ifa_kv_store_f32, the attention behind them, ifa_state_chunked_f32): the same
values in the same order, so the same bits in the outputs, the cache, the queries and the states."""
import ctypes as C

import numpy as np
import pytest
import torch

import inferflow_amd as ia
from tests.gelarax_oracle import bf16_round
from tests.gpu_util import capi, p, sync
from tests.test_gpu_layered_ops import Slots, dev32, devbf, devi, seq_tables

pytestmark = pytest.mark.gpu
Z, F32 = C.c_size_t, C.c_float


class Fresh(C.Structure):          # IfaFreshKV (csrc/ifa_rows_fused.h)
    _fields_ = [("k", C.c_void_p), ("ldk", Z), ("v", C.c_void_p), ("ldv", Z), ("norm", C.c_int), ("norm_w", C.c_void_p), ("eps", F32), ("rot_dims", C.c_int), ("freq", C.c_void_p),
                ("turn_q", C.c_int), ("q_norm_w", C.c_void_p)]


class Side(C.Structure):           # IfaLinearSide
    _fields_ = [("q", C.c_void_p), ("k", C.c_void_p), ("v", C.c_void_p), ("ldq", Z), ("ldk", Z), ("ldv", Z), ("heads", C.c_int), ("dk", C.c_int), ("dv", C.c_int), ("decay", C.c_void_p),
                ("state_off", Z), ("ws", C.c_void_p), ("ws_bytes", Z), ("out", C.c_void_p), ("ldo", Z)]


def tables(seqs):
    sd, rs, rows = seq_tables(seqs)
    h, r = [], 0
    for n, pos0, slot in seqs:
        h += [r, n, pos0, slot]; r += n
    return sd, rs, rows, (C.c_int * len(h))(*h)


def at(t, col):
    return C.c_void_p(t.data_ptr() + 4 * col)


def same(a, b):
    return np.array_equal(a.cpu().numpy(), b.cpu().numpy(), equal_nan=True)


MAX = 700
ONE, PART, MANY = [[(70, 0, 0)], [(45, 70, 0)]], [[(33, 0, 1), (17, 0, 0), (40, 0, 2)], [(21, 40, 2), (64, 33, 1), (18, 17, 0)]], [[(20 + q, 0, q) for q in range(6)]]
FOUR, FIVE = [[(9 + 15 * q, 0, q) for q in range(4)], [(33 - q, 9 + 15 * q, q) for q in range(4)]], [[(40 - 3 * q, 0, q) for q in range(5)]]          # (as many as a launch's arguments hold, one more)
TWO = [[(9, 0, q) for q in range(64)], [(1, 9, q) for q in range(64)], [(130, 10, q) for q in range(12)], [(1, 140, q) for q in range(12)] + [(40, 10, 20)]]          # (many short ones, single tokens, ...)


# heads a workgroup shares (1, 2, 4) and more of them than a wave turns at once, heads of whole and of ragged 32s, values of their own size, nothing / a part / all of a head turned, windows
# behind kept tokens, up to four sequences and more, portions that begin inside a block, long enough for several chunks, fewer rows than the tiled form takes; steps whose rows a launch in front stores;
# many heads of queries, shared out to the waves of few rows
@pytest.mark.parametrize("H,G,D,DV,rot,window,keep,steps,tile_min", [
    (8, 2, 128, 128, 64, 0, 0, ONE, 16), (4, 1, 128, 64, 128, 0, 0, PART, 16), (12, 3, 64, 96, 32, 40, 5, PART, 16), (6, 3, 96, 32, 0, 33, 70, ONE, 16), (5, 5, 40, 48, 10, 0, 0, PART, 16),
    (20, 5, 32, 128, 32, 0, 0, MANY, 16), (2, 2, 128, 128, 126, 100, 40, [[(650, 0, 0)]], 16), (8, 2, 72, 100, 64, 0, 0, [[(9, 0, 0)], [(6, 9, 0)]], 16), (3, 1, 30, 33, 30, 0, 0, PART, 16),
    (4, 2, 64, 64, 32, 45, 3, FOUR, 16), (4, 2, 64, 64, 32, 45, 3, FIVE, 16),
    (8, 8, 128, 128, 128, 0, 0, TWO, 16), (40, 1, 128, 128, 64, 0, 0, PART, 16), (72, 2, 64, 64, 64, 30, 0, ONE, 16), (33, 3, 96, 128, 96, 0, 0, ONE, 16)])
@pytest.mark.parametrize("own", [True, False])
def test_rows_of_rotated_attention_stored_on_the_way(H, G, D, DV, rot, window, keep, steps, tile_min, own):
    rng = np.random.default_rng(H * D + rot)
    k_off, per = 8, MAX * G * D
    v_off = k_off + per
    L = capi()
    nw, kw = devbf(bf16_round(1 + 0.1 * rng.standard_normal(D))), devbf(bf16_round(1 + 0.1 * rng.standard_normal(D)))
    freq = torch.from_numpy(10000.0 ** -(np.arange(max(rot // 2, 1)) / max(rot // 2, 1))).cuda()
    slots = [Slots(1 + max(q for step in steps for _, _, q in step), v_off + MAX * G * DV) for _ in range(2)]
    if not own:          # another layer's rows
        for a, b in zip(slots[0].mem, slots[1].mem):
            a.copy_(torch.from_numpy(rng.standard_normal(a.numel()).astype(np.float32))); b.copy_(a)
    for step in steps:
        sd, rs, T, hs = tables(step)
        N = H * D + G * D + G * DV + 3
        N += -N % 4 if D % 4 == 0 else 0
        proj = [dev32(rng.standard_normal((T, N)))]
        proj.append(proj[0].clone())
        ck, cv = H * D, H * D + G * D
        args = (T, p(slots[0].table), Z(k_off), Z(v_off))
        nb = L.ifa_attention_tile_workspace_bytes(hs, len(step), H, G, D, DV, window, keep)
        ws = torch.zeros(nb // 4 + 4, dtype=torch.float32, device="cuda")
        out = [torch.zeros((T, H * DV), dtype=torch.float32, device="cuda") for _ in range(2)]
        out16 = torch.zeros((T, H * DV), dtype=torch.bfloat16, device="cuda")
        ia.check(L.ifa_qk_rope_store_f32(p(proj[0]), Z(N), H, at(proj[0], ck) if own else None, Z(N), at(proj[0], cv) if own else None, Z(N), G, D, DV, p(nw), p(kw) if own else None, F32(1e-5), rot,
                                         p(freq), p(sd), p(rs), Z(T), *args[1:], None))
        ia.check(L.ifa_attention_kv_f32(p(proj[0]), Z(N), H, G, D, DV, F32(0.2), window, keep, 1, F32(0.5), p(sd), p(rs), Z(T), *args[1:], p(out[0]), Z(H * DV), hs, len(step), tile_min, MAX,
                                        p(ws), Z(nb), None)); sync()
        ws.fill_(7.0)
        fresh = Fresh(at(proj[1], ck) if own else None, N, at(proj[1], cv) if own else None, N, 1 if own else 0, kw.data_ptr() if own else None, 1e-5, rot, freq.data_ptr(), 1, nw.data_ptr())
        left = C.c_bool(False)
        ia.check(L.ifa_attention_kv_to_bf16(p(proj[1]), Z(N), H, G, D, DV, F32(0.2), window, keep, 1, F32(0.5), p(sd), p(rs), Z(T), p(slots[1].table), Z(k_off), Z(v_off), p(out[1]), Z(H * DV),
                                            p(out16), Z(H * DV), C.byref(left), hs, len(step), tile_min, MAX, p(ws), Z(nb), C.byref(fresh), None)); sync()
        assert left.value == (T >= tile_min)
        got = out16.float() if left.value else out[1]
        assert same(got, out[0].to(torch.bfloat16).float() if left.value else out[0])
        assert same(proj[1][:, :H * D], proj[0][:, :H * D])
        assert all(same(a, b) for a, b in zip(slots[0].mem, slots[1].mem))


# the linear attention's keys of 64 and 128, value columns that are no multiple of 64, rows of v off 16 bytes, one chunk of keys a tile (no shares to join) and several
@pytest.mark.parametrize("H,G,D,LH,dk,dv,pad,window,keep,steps,tile_min", [
    (8, 2, 128, 8, 64, 128, 0, 200, 4, [[(601, 0, 0)], [(65, 601, 0)]], 16), (4, 4, 64, 3, 128, 96, 1, 90, 0, PART, 16), (2, 1, 32, 2, 64, 32, 0, 1 << 20, 0, MANY, 16),
    (4, 2, 96, 2, 64, 64, 0, 50, 0, [[(40, 0, 0)]], 64), (16, 4, 128, 16, 64, 128, 0, 128, 2, [[(130, 0, 3), (64, 0, 1)]], 16),
    (4, 2, 64, 2, 64, 64, 0, 45, 3, FOUR, 16), (4, 2, 64, 2, 64, 64, 0, 45, 3, FIVE, 16)])
def test_linear_attention_in_the_windowed_attentions_launches(H, G, D, LH, dk, dv, pad, window, keep, steps, tile_min):
    rng = np.random.default_rng(H * D + dv)
    NB, k_off = 12, 8
    v_off = k_off + MAX * G * D
    s_off = v_off + MAX * G * D
    L = capi()
    rel, sink = devbf(bf16_round(rng.standard_normal((NB, H)))), devbf(bf16_round(rng.standard_normal(H)))
    bucket = devi(np.minimum(np.arange(MAX), NB - 1))
    decay = dev32(rng.uniform(0.9, 1.0, LH))
    slots = [Slots(6, s_off + LH * dk * dv) for _ in range(2)]
    for step in steps:
        sd, rs, T, hs = tables(step)
        cq, ck, lq = 0, H * D, H * D + G * D
        lk = lq + LH * dk
        lv = lk + LH * dk + pad
        N = lv + LH * dv
        N += -N % 4
        proj = dev32(rng.standard_normal((T, N)))
        nb = L.ifa_attention_tile_workspace_bytes(hs, len(step), H, G, D, D, window, keep)
        ws = torch.zeros(nb // 4 + 4, dtype=torch.float32, device="cuda")
        chunks = sum((n + 63) // 64 for n, _, _ in step)
        sb = L.ifa_state_chunked_workspace_bytes(0, Z(chunks), LH, dk, dv)
        sws = torch.zeros(sb // 4 + 4, dtype=torch.float32, device="cuda")
        out = [torch.zeros((T, H * D), dtype=torch.float32, device="cuda") for _ in range(2)]
        lin = [torch.zeros((T, LH * dv), dtype=torch.float32, device="cuda") for _ in range(2)]
        out16 = torch.zeros((T, H * D), dtype=torch.bfloat16, device="cuda")
        where = [(p(s.table), Z(k_off), Z(v_off)) for s in slots]
        ia.check(L.ifa_kv_store_f32(at(proj, ck), Z(N), at(proj, ck), Z(N), G, D, 1, F32(1e-5), p(sd), p(rs), Z(T), *where[0], None))
        ia.check(L.ifa_attention_window_f32(at(proj, cq), Z(N), H, G, D, 1, F32(1e-5), F32(8.0), F32(20.0), window, keep, p(rel), p(bucket), NB, p(sink), p(sd), p(rs), Z(T), *where[0], p(out[0]),
                                            Z(H * D), hs, len(step), tile_min, p(ws), Z(nb), None))
        ia.check(L.ifa_state_chunked_f32(0, at(proj, lq), Z(N), at(proj, lk), Z(N), at(proj, lv), Z(N), LH, LH, dk, dv, p(decay), None, None, p(sd), hs, len(step), p(slots[0].table), Z(s_off),
                                         p(sws), Z(sb), p(lin[0]), Z(LH * dv), None)); sync()
        ws.fill_(7.0); sws.fill_(7.0)
        fresh = Fresh(at(proj, ck), N, at(proj, ck), N, 1, None, 1e-5, 0, None, 0, None)
        side = Side(at(proj, lq), at(proj, lk), at(proj, lv), N, N, N, LH, dk, dv, decay.data_ptr(), s_off, sws.data_ptr(), sb, lin[1].data_ptr(), LH * dv)
        left, done = C.c_bool(False), C.c_bool(True)
        ia.check(L.ifa_attention_window_to_bf16(at(proj, cq), Z(N), H, G, D, 1, F32(1e-5), F32(8.0), F32(20.0), window, keep, p(rel), p(bucket), NB, p(sink), p(sd), p(rs), Z(T), *where[1],
                                                p(out[1]), Z(H * D), p(out16), Z(H * D), C.byref(left), hs, len(step), tile_min, p(ws), Z(nb), C.byref(fresh), C.byref(side), C.byref(done), None))
        sync()
        assert done.value == left.value == (T >= tile_min)
        got = out16.float() if left.value else out[1]
        assert same(got, out[0].to(torch.bfloat16).float() if left.value else out[0])
        if done.value:
            assert same(lin[1], lin[0])
            assert all(same(a, b) for a, b in zip(slots[0].mem, slots[1].mem))


# no linear attention beside it: rows normed and as they are, heads of one, two and four 32s, portions that begin inside a block, one key block and many, kept tokens, six sequences
@pytest.mark.parametrize("H,G,D,norm,window,keep,steps,tile_min", [
    (8, 2, 128, 1, 200, 4, [[(19, 0, 0)], [(65, 19, 0)]], 16), (4, 4, 64, 0, 90, 0, PART, 16), (2, 1, 32, 1, 1 << 20, 0, MANY, 16), (4, 2, 96, 0, 50, 40, [[(333, 0, 0)]], 16),
    (8, 2, 128, 1, 64, 2, [[(12, 0, 1), (2, 0, 0)]], 2)])
def test_rows_of_windowed_attention_stored_on_the_way(H, G, D, norm, window, keep, steps, tile_min):
    rng = np.random.default_rng(H * D + window % 97)
    NB, k_off = 12, 8
    v_off = k_off + MAX * G * D
    L = capi()
    rel, sink = devbf(bf16_round(rng.standard_normal((NB, H)))), devbf(bf16_round(rng.standard_normal(H)))
    bucket = devi(np.minimum(np.arange(MAX), NB - 1))
    slots = [Slots(6, v_off + MAX * G * D) for _ in range(2)]
    for step in steps:
        sd, rs, T, hs = tables(step)
        ck, cv = H * D, H * D + G * D
        N = cv + G * D
        proj = dev32(rng.standard_normal((T, N)))
        proj[T // 2, ck + 3], proj[T - 1, cv + D - 1] = 1e30, -1e30
        nb = L.ifa_attention_tile_workspace_bytes(hs, len(step), H, G, D, D, window, keep)
        ws = torch.zeros(nb // 4 + 4, dtype=torch.float32, device="cuda")
        out = [torch.zeros((T, H * D), dtype=torch.float32, device="cuda") for _ in range(2)]
        out16 = torch.zeros((T, H * D), dtype=torch.bfloat16, device="cuda")
        where = [(p(s.table), Z(k_off), Z(v_off)) for s in slots]
        ia.check(L.ifa_kv_store_f32(at(proj, ck), Z(N), at(proj, cv), Z(N), G, D, norm, F32(1e-5), p(sd), p(rs), Z(T), *where[0], None))
        ia.check(L.ifa_attention_window_f32(p(proj), Z(N), H, G, D, 1, F32(1e-5), F32(8.0), F32(20.0), window, keep, p(rel), p(bucket), NB, p(sink), p(sd), p(rs), Z(T), *where[0], p(out[0]),
                                            Z(H * D), hs, len(step), tile_min, p(ws), Z(nb), None)); sync()
        ws.fill_(7.0)
        fresh = Fresh(at(proj, ck), N, at(proj, cv), N, norm, None, 1e-5, 0, None, 0, None)
        left, done = C.c_bool(False), C.c_bool(True)
        ia.check(L.ifa_attention_window_to_bf16(p(proj), Z(N), H, G, D, 1, F32(1e-5), F32(8.0), F32(20.0), window, keep, p(rel), p(bucket), NB, p(sink), p(sd), p(rs), Z(T), *where[1],
                                                p(out[1]), Z(H * D), p(out16), Z(H * D), C.byref(left), hs, len(step), tile_min, p(ws), Z(nb), C.byref(fresh), None, C.byref(done), None))
        sync()
        assert left.value == (T >= tile_min) and not done.value
        got = out16.float() if left.value else out[1]
        assert same(got, out[0].to(torch.bfloat16).float() if left.value else out[0])
        assert all(same(a, b) for a, b in zip(slots[0].mem, slots[1].mem))


# as many sequences as go beside the attention, one more, and so many heads and columns that the states are handed on in a launch of their own (more than 2048 workgroups of 512)
@pytest.mark.parametrize("LH,dk,dv,n,beside", [(2, 64, 64, 32, True), (2, 64, 64, 33, False), (8, 128, 96, 10, True), (8, 128, 96, 11, True), (9, 128, 128, 32, True)])
def test_linear_attention_of_many_sequences(LH, dk, dv, n, beside):
    H, G, D, NB, k_off, most = 4, 2, 64, 12, 8, 160
    rng = np.random.default_rng(LH * n + dv)
    v_off = k_off + most * G * D
    s_off = v_off + most * G * D
    L = capi()
    rel, sink = devbf(bf16_round(rng.standard_normal((NB, H)))), devbf(bf16_round(rng.standard_normal(H)))
    bucket = devi(np.minimum(np.arange(most), NB - 1))
    decay = dev32(rng.uniform(0.9, 1.0, LH))
    slots = [Slots(n, s_off + LH * dk * dv) for _ in range(2)]
    lens = [int(k) for k in rng.integers(1, 80, n)]
    for behind in (0, 1):          # (a prompt each, then a portion behind it)
        seqs = [(k, behind * k, q) for q, k in enumerate(lens)]
        sd, rs, T, hs = tables(seqs)
        ck = H * D
        lq = ck + G * D
        lk, lv = lq + LH * dk, lq + 2 * LH * dk
        N = lv + LH * dv
        proj = dev32(rng.standard_normal((T, N)))
        nb = L.ifa_attention_tile_workspace_bytes(hs, n, H, G, D, D, 50, 3)
        ws = torch.full((nb // 4 + 4,), 7.0, dtype=torch.float32, device="cuda")
        sb = L.ifa_state_chunked_workspace_bytes(0, Z(sum((k + 63) // 64 for k, _, _ in seqs)), LH, dk, dv)
        sws = torch.full((sb // 4 + 4,), 7.0, dtype=torch.float32, device="cuda")
        out = [torch.zeros((T, H * D), dtype=torch.float32, device="cuda") for _ in range(2)]
        lin = [torch.zeros((T, LH * dv), dtype=torch.float32, device="cuda") for _ in range(2)]
        out16 = torch.zeros((T, H * D), dtype=torch.bfloat16, device="cuda")
        where = [(p(s.table), Z(k_off), Z(v_off)) for s in slots]

        def alone(i):
            ia.check(L.ifa_state_chunked_f32(0, at(proj, lq), Z(N), at(proj, lk), Z(N), at(proj, lv), Z(N), LH, LH, dk, dv, p(decay), None, None, p(sd), hs, n, p(slots[i].table), Z(s_off),
                                             p(sws), Z(sb), p(lin[i]), Z(LH * dv), None))
        ia.check(L.ifa_kv_store_f32(at(proj, ck), Z(N), at(proj, ck), Z(N), G, D, 1, F32(1e-5), p(sd), p(rs), Z(T), *where[0], None))
        ia.check(L.ifa_attention_window_f32(p(proj), Z(N), H, G, D, 1, F32(1e-5), F32(8.0), F32(20.0), 50, 3, p(rel), p(bucket), NB, p(sink), p(sd), p(rs), Z(T), *where[0], p(out[0]),
                                            Z(H * D), hs, n, 16, p(ws), Z(nb), None))
        alone(0); sync()
        fresh = Fresh(at(proj, ck), N, at(proj, ck), N, 1, None, 1e-5, 0, None, 0, None)
        side = Side(at(proj, lq), at(proj, lk), at(proj, lv), N, N, N, LH, dk, dv, decay.data_ptr(), s_off, sws.data_ptr(), sb, lin[1].data_ptr(), LH * dv)
        left, done = C.c_bool(False), C.c_bool(not beside)
        ia.check(L.ifa_attention_window_to_bf16(p(proj), Z(N), H, G, D, 1, F32(1e-5), F32(8.0), F32(20.0), 50, 3, p(rel), p(bucket), NB, p(sink), p(sd), p(rs), Z(T), *where[1],
                                                p(out[1]), Z(H * D), p(out16), Z(H * D), C.byref(left), hs, n, 16, p(ws), Z(nb), C.byref(fresh), C.byref(side), C.byref(done), None))
        if not done.value:
            alone(1)
        sync()
        assert done.value == beside and left.value
        assert same(out16.float(), out[0].to(torch.bfloat16).float()) and same(lin[0], lin[1])
        assert all(same(a, b) for a, b in zip(slots[0].mem, slots[1].mem))
