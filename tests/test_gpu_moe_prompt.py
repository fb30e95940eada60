"""The mixture of experts of a prompt as run_sandwich_layer runs it -- choice and counts, places of the pairs beside the shared expert's activations, grouped products, the sum of a row's pairs
inside the norm behind them -- against the launches of their own (ifa_moe_route_top_f32, ifa_moe_experts_gated_f32 over the same rows, ifa_norm_add_norm_f32 and its bfloat16 form), bit for bit: the same
products and the same sums in the same order."""
import ctypes as C

import numpy as np
import pytest
import torch

import inferflow_amd as ia
from tests.gelarax_oracle import bf16_round
from tests.gpu_util import capi, p, sync
from tests.test_gpu_layered_ops import dev32, devbf

pytestmark = pytest.mark.gpu


class Prompt(C.Structure):          # IfaMoePrompt (csrc/ifa_rows_fused.h)
    _fields_ = [("logits", C.c_void_p), ("ldl", C.c_size_t), ("rows", C.c_size_t), ("width", C.c_int), ("ff", C.c_int), ("experts", C.c_int), ("top", C.c_int),
                ("gate_up", C.c_void_p), ("down", C.c_void_p), ("h16", C.c_void_p), ("idx", C.c_void_p), ("wgt", C.c_void_p), ("ws", C.c_void_p), ("ws_bytes", C.c_size_t),
                ("sh_gate_up", C.c_void_p), ("sh_ld", C.c_size_t), ("sh_ff", C.c_int), ("sh_gate", C.c_void_p), ("sh_ldg", C.c_size_t), ("sh_act", C.c_void_p), ("sh_ldo", C.c_size_t)]


# rows of one block and of several (16 rows, and 32 of them from 4097 rows on), row tiles of 64 and 128, one expert, experts around a wave's and the ballots' widths, the most there may be, rows of one and of two pieces a thread of the norm
@pytest.mark.parametrize("T,W,F,E,top,SF", [(9, 448, 64, 5, 2, 64), (17, 448, 64, 16, 4, 72), (16, 512, 64, 1, 1, 0), (300, 448, 72, 16, 4, 100), (257, 448, 64, 64, 3, 66), (70, 448, 64, 65, 8, 64),
                                            (40, 448, 64, 512, 9, 0), (4099, 448, 64, 7, 2, 64), (1100, 512, 64, 3, 3, 128), (4500, 1024, 64, 16, 4, 0),
                                            (20, 4096, 64, 5, 2, 64), (20, 4160, 64, 5, 2, 64), (12, 8192, 64, 3, 2, 0)])
def test_experts_of_a_prompt_against_their_launches_one_by_one(T, W, F, E, top, SF):
    rng = np.random.default_rng(T + E)
    g = torch.Generator(device="cuda"); g.manual_seed(T + E)
    N2 = E + 1 + 2 * SF + 3                                     # router | the shared expert's gate | its gate and up (from an odd column on)
    proj = torch.randn((T, N2), generator=g, device="cuda")
    proj[0, :min(2, E)] = 1.5                                   # a tie
    proj[2 % T, :E] = 0.25                                      # all equal
    proj[4, :E:2] = -float("inf")                               # some that are never chosen while others are left
    proj[5, :E] = float("nan")                                  # no numbers at all, and one beside others
    if E > 1:
        proj[6, 1] = float("nan")
    h16 = torch.randn((T, W), generator=g, device="cuda").to(torch.bfloat16).contiguous()
    gu = (torch.randn((E * 2 * F, W), generator=g, device="cuda") * W ** -0.5).to(torch.bfloat16)
    dn = (torch.randn((E * W, F), generator=g, device="cuda") * F ** -0.5).to(torch.bfloat16)
    wa, wb = (devbf(bf16_round(rng.standard_normal(W))) for _ in range(2))
    x = torch.randn((T, W), generator=g, device="cuda"); x_w, x_16 = x.clone(), x.clone()
    m = torch.randn((T, W), generator=g, device="cuda") if SF else None
    L, Z = capi(), C.c_size_t
    nb = L.ifa_moe_workspace_bytes(T, top, W, 3 * F, E)
    ws = torch.zeros((nb + 15) // 4, dtype=torch.float32, device="cuda")
    idx, idx_w = (torch.full((T, top), -1, dtype=torch.int32, device="cuda") for _ in range(2))
    wgt, wgt_w = (torch.zeros((T, top), dtype=torch.float32, device="cuda") for _ in range(2))
    ldo = (SF + 63) // 64 * 64
    act = torch.full((T, max(ldo, 1)), 7.0, dtype=torch.bfloat16, device="cuda")
    ia.check(L.ifa_moe_route_top_f32(p(proj), Z(N2), Z(T), E, top, None, p(idx_w), p(wgt_w), None))
    y = torch.zeros((T, W), dtype=torch.float32, device="cuda")
    h32, h_w = h16.float(), torch.zeros((T, W), dtype=torch.float32, device="cuda")
    # (rounding rows that are bfloat16 already changes nothing: the op that reads 32-bit rows forms the same products)
    ia.check(L.ifa_moe_experts_gated_f32(p(h32), Z(W), Z(T), W, F, E, top, p(gu), p(dn), p(idx_w), p(wgt_w), 0, p(ws), Z(nb), p(y), Z(W), 0, None))
    if m is not None:
        y += m
    ia.check(L.ifa_norm_add_norm_f32(p(x_w), Z(W), Z(T), Z(W), p(y), Z(W), p(wa), p(wb), C.c_float(1.0), C.c_float(1e-5), p(h_w), Z(W), None)); sync()
    P = Prompt(p(proj), N2, T, W, F, E, top, p(gu), p(dn), p(h16), p(idx), p(wgt), p(ws), nb, proj.data_ptr() + 4 * (E + 1) if SF else None, N2, SF,
               proj.data_ptr() + 4 * E if SF else None, N2, p(act) if SF else None, ldo)
    pos, rows = C.c_void_p(), C.c_void_p()
    h = torch.zeros((T, W), dtype=torch.float32, device="cuda")
    ia.check(L.ifa_moe_prompt(C.byref(P), C.byref(pos), C.byref(rows), None))
    ia.check(L.ifa_norm_add_norm_moe(p(x), Z(W), Z(T), Z(W), p(m) if SF else None, Z(W), pos, rows, top, p(wa), p(wb), C.c_float(1.0), C.c_float(1e-5), p(h), None, Z(W), None)); sync()
    assert torch.equal(idx, idx_w) and np.array_equal(wgt.cpu().numpy(), wgt_w.cpu().numpy(), equal_nan=True)
    assert np.array_equal(x.cpu().numpy(), x_w.cpu().numpy(), equal_nan=True) and np.array_equal(h.cpu().numpy(), h_w.cpu().numpy(), equal_nan=True)
    assert torch.isfinite(h[7:]).all()
    # the form that leaves bfloat16 rows, as layers' products read them: those rows rounded
    h_16 = torch.zeros((T, W), dtype=torch.bfloat16, device="cuda")
    ia.check(L.ifa_norm_add_norm_moe(p(x_16), Z(W), Z(T), Z(W), p(m) if SF else None, Z(W), pos, rows, top, p(wa), p(wb), C.c_float(1.0), C.c_float(1e-5), None, p(h_16), Z(W), None)); sync()
    assert np.array_equal(x_16.cpu().numpy(), x_w.cpu().numpy(), equal_nan=True)
    assert np.array_equal(h_16.float().cpu().numpy(), h.to(torch.bfloat16).float().cpu().numpy(), equal_nan=True)
    if SF:          # against the same sum in 64 bits: rounded once to bfloat16, 2^-9 of the value; 32-bit exponentials below that
        s = proj[:, E + 1:].double().cpu()
        want = s[:, :SF] * torch.sigmoid(s[:, :SF]) * s[:, SF:2 * SF] * torch.sigmoid(proj[:, E:E + 1].double().cpu())
        got = act.double().cpu()
        assert ((got[:, :SF] - want).abs() <= 2.0 ** -8 * want.abs() + 1e-30).all() and (got[:, SF:] == 0).all()
