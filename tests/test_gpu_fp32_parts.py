"""fp32 recurrences whose numbers travel and multiply as three bf16 parts (csrc/recurrent_parts.hpp): half k-steps (H = 16 mod 32), every
unit tile and batch tile of the XCD-local and the whole-CU kernels, against float64; numbers that are not finite."""
import ctypes

import numpy as np
import pytest
import torch

import fastlstm_amd.lstm as L
from fastlstm_amd import FastLSTM, _lib
from helpers import nn_lstm_reference
from test_gpu_one_cu import backward, operands, run

pytestmark = pytest.mark.gpu


# (B, H): 16- and 32-row groups, one and two unit tiles, half and whole last k-steps, rows over several launches; 640 on: whole-CU kernels,
# 1280 on with half a unit tile per workgroup, in launches of up to 64 rows
@pytest.mark.parametrize("B,H", [(3, 112), (17, 144), (5, 208), (33, 256), (150, 256), (300, 272), (9, 400), (128, 512), (140, 512), (600, 320),
                                 (3, 640), (90, 640), (33, 768), (20, 896), (70, 1024), (300, 1024), (1, 1280), (66, 1280), (17, 1536), (150, 1792),
                                 (16, 2048), (33, 2048), (64, 2048)])
def test_against_float64(B, H):
    T = 7
    p, g = operands(T, B, H, torch.float32, seed=H + B)
    want = nn_lstm_reference({k: v.double() for k, v in p.items()})
    out, cell, ifgo, d_ifgo, dh, dc = run(g)
    dx = d_ifgo.double().view(T * B, -1) @ g["Wx"].double()
    for name, a, b in (("out", out[1:], want["out"]), ("c_n", cell[-1], want["c_n"]), ("dh0", dh, want["dh0"]), ("dc0", dc, want["dc0"]),
                       ("dx", dx, want["dx"].reshape(T * B, -1))):
        a, b = a.double().cpu().numpy(), b.numpy()
        assert np.linalg.norm(a - b) <= 1e-6 * np.linalg.norm(b), name   # (2-norm: some 2e-7 from the rounding of every step's results)


# 32 units per workgroup, forward: groups of 16 rows and of 32
@pytest.mark.parametrize("B,H,shape", [(520, 256, (8, 2, 2, 8)), (1024, 224, (8, 2, 2, 8)), (600, 192, (8, 2, 1, 8)), (1100, 128, (8, 2, 2, 8)),
                                       (1500, 96, (8, 2, 2, 8))])
def test_32_units_per_workgroup(B, H, shape):
    got = (ctypes.c_int * 5)()
    assert _lib.load().fastlstm_diag_xcd_shape(B, H, 0, 0, 1, got) == 1 and tuple(got)[:4] == shape
    test_against_float64(B, H)


def forward_multi(gs):
    """[(out, cell, gates)] of recurrences in one launch, the inputs' products by torch"""
    lib, n, code = _lib.load(), len(gs), 0
    T, B, H = gs[0]["dout"].shape
    plan = L._plan(gs[0]["x"].device, B, H, code, False)
    size = lib.fastlstm_multi_workspace_bytes(plan, n, T, H, code, 0)
    assert lib.fastlstm_multi_fused(n, T, B, H, code, 0, size) == 1
    ws = torch.zeros(size, dtype=torch.uint8, device="cuda")
    bufs = []
    for g in gs:
        out, cell = (torch.zeros(T + 1, B, H, device="cuda") for _ in range(2))
        out[0], cell[0] = g["h0"], g["c0"]
        bufs.append((out, cell, g["x"] @ g["Wx"].t() + g["bx"] + g["bh"]))
    arr = lambda ts: (ctypes.c_void_p * n)(*[t.data_ptr() for t in ts])
    _lib.check(lib.fastlstm_fwd_persistent_multi(n, arr([b[2] for b in bufs]), arr([b[0] for b in bufs]), arr([b[1] for b in bufs]),
                                                 arr([g["Wh"] for g in gs]), ws.data_ptr(), size, T, B, H, code, 1,
                                                 torch.cuda.current_stream().cuda_stream), "fwd multi")
    return bufs


@pytest.mark.parametrize("B,H,n", [(300, 256, 2), (165, 256, 3), (16, 1024, 3), (32, 1024, 4), (20, 640, 3), (9, 768, 4)])
def test_forward_side_by_side(B, H, n):
    """One launch, the results of calls by themselves to rounding (the inputs' products are torch's here, and H = 256 alone has 16 units per
    workgroup: other sums)."""
    gs = [operands(5, B, H, torch.float32, seed=s)[1] for s in range(n)]
    for g, (out, cell, _) in zip(gs, forward_multi(gs)):
        o, c, _ = L.lstm_persistent_fwd(g["x"], g["h0"], g["c0"], g["Wx"], g["bx"], g["Wh"], g["bh"])
        for a, b in ((out, o), (cell, c)):
            assert float((a.double() - b.double()).norm()) <= 1e-6 * float(b.double().norm())   # (some 2e-7 for either from rounding)


@pytest.mark.parametrize("B,H,n", [(16, 1024, 3), (32, 1024, 4), (20, 640, 3), (9, 768, 4)])
def test_three_and_four_side_by_side_are_the_bits_of_calls_by_themselves(B, H, n):
    lib = _lib.load()
    size = lib.fastlstm_multi_workspace_bytes(L._plan(torch.device("cuda", 0), B, H, 0, True), n, 5, H, 0, 1)
    assert lib.fastlstm_multi_fused(n, 5, B, H, 0, 1, size) == 1
    gs = [operands(5, B, H, torch.float32, seed=s)[1] for s in range(n)]
    alone = [run(g) for g in gs]
    recs = [(g, a[1], a[2], g["dh_n"].clone(), g["dc_n"].clone()) for g, a in zip(gs, alone)]
    for d, r, a in zip(backward(recs), recs, alone):
        assert torch.equal(d, a[3]) and torch.equal(r[3], a[4]) and torch.equal(r[4], a[5])


@pytest.mark.parametrize("B,H", [(19, 640), (40, 1024)])
def test_side_by_side_are_the_bits_of_calls_by_themselves(B, H):
    gs = [operands(5, B, H, torch.float32, seed=s)[1] for s in range(2)]
    alone = [run(g) for g in gs]
    recs = [(g, a[1], a[2], g["dh_n"].clone(), g["dc_n"].clone()) for g, a in zip(gs, alone)]
    for d, r, a in zip(backward(recs), recs, alone):
        assert torch.equal(d, a[3]) and torch.equal(r[3], a[4]) and torch.equal(r[4], a[5])


@pytest.mark.parametrize("B,H", [(9, 112), (40, 512), (40, 768), (40, 1536)])
@pytest.mark.parametrize("weight", [False, True])
def test_numbers_that_are_not_finite(B, H, weight):
    """As test_gpu_one_cu's: the general kernels' entries are infinite, NaN and finite where these are."""
    g = operands(4, B, H, torch.float32, seed=3)[1]
    inf = float("inf")
    g["h0"][2, 5], g["h0"][3, 6], g["h0"][4, 7], g["dh_n"][6, 4] = inf, -inf, float("nan"), inf
    g["Wh"][7, 5], g["Wh"][8, 6] = 0.5, 0.0
    if weight:
        g["Wh"][H + 3, 11] = inf
    lib = _lib.load()
    fast = run(g)
    lib.fastlstm_set_kernel_families(0)
    try:
        slow = run(g)
    finally:
        lib.fastlstm_set_kernel_families(7)
    for a, b in list(zip(fast, slow))[:3 if weight else 6]:
        assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(torch.isinf(a), torch.isinf(b))
        ok = torch.isfinite(b)
        assert bool(ok.any()) and not bool(ok.all()) and float((a - b)[ok].abs().max()) < 1e-4


@pytest.mark.parametrize("T,B,H,padded", [(32, 5, 1100, 1280), (31, 5, 1100, 0), (33, 3, 1800, 2048), (40, 2, 1536, 0)])
def test_module_between_the_sizes(T, B, H, padded):
    """1024 < H < 2048 in the module: padded to a multiple of 256 from 32 steps on; outputs and gradients against float64."""
    assert L._padded_hidden_size(T, B, H, 0, 0, True) == padded
    torch.manual_seed(T + H)
    want = torch.nn.LSTM(24, H).double()
    got = FastLSTM(24, H, device="cuda", dtype=torch.float32)
    got.load_state_dict(want.state_dict())   # (rounds)
    want.load_state_dict(got.state_dict())
    x, d = torch.randn(T, B, 24), torch.randn(T, B, H)
    xg, xw = x.cuda().requires_grad_(), x.double().requires_grad_()
    y, (h, c) = got(xg)
    y.backward(d.cuda())
    yw, (hw, cw) = want(xw)
    yw.backward(d.double())
    pairs = [(y, yw), (h, hw), (c, cw), (xg.grad, xw.grad)] + [(p.grad, q.grad) for p, q in zip(got.parameters(), want.parameters())]
    for i, (a, b) in enumerate(pairs):   # (2-norm: rounding of every step's results and of sums of fp32 products)
        assert a.shape == b.shape and float((a.double().cpu() - b).norm()) <= 2e-6 * float(b.norm()), i


@pytest.mark.parametrize("B,H", [(8, 64), (5, 96), (8, 128), (40, 136), (20, 256), (8, 512), (300, 256), (16, 1024), (8, 1280)])
def test_gradients_that_fade(B, H):
    """A loss on the last step and gates that forget: the gradients of the steps before fade through all magnitudes.  Down to the least normal
    numbers their relative error is that of the sums: an input gradient of step T - n has gone through n products, each 1e-6 off at most."""
    T, I = 60, 16
    torch.manual_seed(H)
    want = torch.nn.LSTM(I, H).double()
    with torch.no_grad():
        want.bias_ih_l0[H:2 * H] = -3.0
    got = FastLSTM(I, H, device="cuda", dtype=torch.float32)
    got.load_state_dict(want.state_dict())   # (rounds)
    want.load_state_dict(got.state_dict())
    x = torch.randn(T, B, I)
    xg, xw = x.cuda().requires_grad_(), x.double().requires_grad_()
    got(xg)[0][-1].sum().backward()
    want(xw)[0][-1].sum().backward()
    a, b, tested = xg.grad.double().cpu(), xw.grad, 0
    for t in range(T):
        size = float(b[t].norm()) / (B * I) ** 0.5
        if size > 1e-37:
            assert float((a[t] - b[t]).norm()) <= (T - t) * 1e-6 * float(b[t].norm()), (t, size)
            tested += size < 1e-33
    assert tested > 2
