"""The one-CU kernels (csrc/recurrent_cu.hpp): every hidden size they take, batches around their four rows, sequences shorter and longer
than their four steps in flight, against float64; several recurrences in a launch; numbers that are not finite."""
import numpy as np
import pytest
import torch

import fastlstm_amd.lstm as L
from fastlstm_amd import _lib
from helpers import make_problem, nn_lstm_reference

pytestmark = pytest.mark.gpu

SIZES = [(torch.float32, H) for H in (64, 80, 96)] + [(torch.float16, H) for H in (80, 96, 112, 128, 144, 160)] + [(torch.bfloat16, 128), (torch.bfloat16, 160)]


def operands(T, B, H, dt, seed, I=32):
    p = make_problem(T, B, I, H, seed=seed)
    return {k: v.to(dt) for k, v in p.items()}, {k: v.to(dt).cuda() for k, v in p.items()}


def run(g):
    """out, cell, ifgo, d_ifgo, dh_0, dc_0"""
    out, cell, ifgo = L.lstm_persistent_fwd(g["x"], g["h0"], g["c0"], g["Wx"], g["bx"], g["Wh"], g["bh"])
    dh, dc = g["dh_n"].clone(), g["dc_n"].clone()
    d_ifgo = backward([(g, cell, ifgo, dh, dc)])[0]
    return out, cell, ifgo, d_ifgo, dh, dc


def backward(recs):
    lib, (g, cell, ifgo, _, _) = _lib.load(), recs[0]
    T, B, H = g["dout"].shape
    code = L._DTYPE_CODE[g["dout"].dtype]
    plan = L._plan(g["dout"].device, B, H, code, True)
    n = lib.fastlstm_multi_workspace_bytes(plan, len(recs), T, H, code, 1)
    ws = torch.zeros(n, dtype=torch.uint8, device="cuda")
    d_ifgo = [torch.empty_like(r[2]) for r in recs]
    st = torch.cuda.current_stream().cuda_stream
    import ctypes
    arr = lambda ts: (ctypes.c_void_p * len(recs))(*[t.data_ptr() for t in ts])
    if len(recs) == 1:
        _lib.check(lib.fastlstm_bwd_persistent(g["dout"].data_ptr(), recs[0][3].data_ptr(), recs[0][4].data_ptr(), ifgo.data_ptr(),
                                               cell.data_ptr(), d_ifgo[0].data_ptr(), g["Wh"].data_ptr(), ws.data_ptr(), n, T, B, H, code, st), "bwd")
    else:
        _lib.check(lib.fastlstm_bwd_persistent_multi(len(recs), arr([r[0]["dout"] for r in recs]), arr([r[3] for r in recs]), arr([r[4] for r in recs]),
                                                     arr([r[2] for r in recs]), arr([r[1] for r in recs]), arr(d_ifgo),
                                                     arr([r[0]["Wh"] for r in recs]), ws.data_ptr(), n, T, B, H, code, st), "bwd multi")
    return d_ifgo


@pytest.mark.parametrize("dt,H", SIZES)
@pytest.mark.parametrize("T,B", [(1, 1), (3, 4), (5, 5), (9, 18), (2, 1024), (2, 1025)])
def test_against_float64(dt, H, T, B):
    p, g = operands(T, B, H, dt, seed=H + B)
    want = nn_lstm_reference({k: v.double() for k, v in p.items()})
    out, cell, ifgo, d_ifgo, dh, dc = run(g)
    dx = d_ifgo.double().view(T * B, -1) @ g["Wx"].double()
    # values, gates and states are rounded to the type at every step; 2-norm over the result
    tol = {torch.float32: 1e-6, torch.float16: 2e-3, torch.bfloat16: 1.5e-2}[dt]
    for name, a, b in (("out", out[1:], want["out"]), ("c_n", cell[-1], want["c_n"]), ("dh0", dh, want["dh0"]), ("dc0", dc, want["dc0"]),
                       ("dx", dx, want["dx"].reshape(T * B, -1))):
        a, b = a.double().cpu().numpy(), b.numpy()
        assert np.linalg.norm(a - b) <= tol * np.linalg.norm(b), name


@pytest.mark.parametrize("dt,H", [(torch.float32, 96), (torch.float16, 144)])
def test_side_by_side_are_the_bits_of_calls_by_themselves(dt, H):
    T, B = 6, 7
    gs = [operands(T, B, H, dt, seed=s)[1] for s in range(3)]
    alone = [run(g) for g in gs]
    recs = [(g, a[1], a[2], g["dh_n"].clone(), g["dc_n"].clone()) for g, a in zip(gs, alone)]
    for d, r, a in zip(backward(recs), recs, alone):
        assert torch.equal(d, a[3]) and torch.equal(r[3], a[4]) and torch.equal(r[4], a[5])


@pytest.mark.parametrize("weight", [False, True])
def test_numbers_that_are_not_finite(weight):
    """fp32: infinities and a NaN in h_0 and dh_n against short numbers and zeros, and an infinite weight (forward: in the reverse pass it
    meets gradients that are zero, and nothing stays finite): the general kernels' entries are infinite, NaN and finite where these are."""
    T, B, H = 4, 9, 96
    g = operands(T, B, H, torch.float32, seed=3)[1]
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


@pytest.mark.parametrize("H,dt", [(80, torch.float16), (112, torch.bfloat16), (144, torch.float16), (80, torch.float32)])
def test_module_leaves_these_sizes_as_they_are(H, dt):
    """... from 32 steps on too, where sizes between those of the fast kernels are padded: outputs and gradients against float64."""
    T, B, I, code = 40, 9, 64, L._DTYPE_CODE[dt]
    assert L._recurrent_form(T, B, H, code, 0) == L._recurrent_form(T, B, H, code, 0, True) == 4
    assert L._padded_hidden_size(T, B, H, code, 0, True) == L._padded_hidden_size(T, B, H, code, 0, False) == 0
    torch.manual_seed(H)
    want = torch.nn.LSTM(I, H).double()
    got = L.FastLSTM(I, H, device="cuda", dtype=dt)
    got.load_state_dict(want.state_dict())   # (rounds)
    want.load_state_dict(got.state_dict())
    x, d = torch.randn(T, B, I).to(dt), torch.randn(T, B, H).to(dt)
    xg, xw = x.cuda().requires_grad_(), x.double().requires_grad_()
    y, (h, c) = got(xg)
    y.backward(d.cuda())
    yw, (hw, cw) = want(xw)
    yw.backward(d.double())
    tol = {torch.float32: 2e-6, torch.float16: 5e-3, torch.bfloat16: 4e-2}[dt]   # (every step's results are rounded to the type)
    for i, (a, b) in enumerate([(y, yw), (h, hw), (c, cw), (xg.grad, xw.grad)] + [(p.grad, q.grad) for p, q in zip(got.parameters(), want.parameters())]):
        a, b = a.detach().double().cpu(), b.detach()
        assert a.shape == b.shape and float((a - b).norm()) <= tol * float(b.norm()), i


def test_padding_goes_by_the_kernels_that_run():
    pad = lambda T, B, H, code, training: L._padded_hidden_size(T, B, H, code, 0, training)
    # 16 bits, more rows than the one-CU kernels hold: sizes that the XCD-local kernels do not take go to those they take
    assert pad(64, 1025, 80, 1, True) == 96 and pad(64, 1024, 80, 1, True) == 0
    # fp32 up to 32 units: as 64 where the one-CU kernels hold the batch, and in training
    assert [pad(128, B, 32, 0, training) for B, training in ((1024, False), (1025, False), (1024, True), (1025, True))] == [64, 0, 64, 64]
    # fp32 between 1024 and 2048: as the next size whose weights stay on the chip, if they do
    lib = _lib.load()
    assert pad(64, 5, 1100, 0, True) == 1280 and L._recurrent_form(64, 5, 1280, 0, 0) == 2
    lib.fastlstm_set_kernel_families(5)
    try:
        assert pad(64, 5, 1100, 0, True) == 0 and L._recurrent_form(64, 5, 1280, 0, 0) == 3
    finally:
        lib.fastlstm_set_kernel_families(7)


def test_form_of_the_kernel_that_runs():
    form = lambda B, H, code, backward=False: L._recurrent_form(5, B, H, code, 0, backward)
    assert form(4, 64, 1) == 0 and form(4, 64, 0) == 4 and form(16, 1024, 0) == 2 and form(16, 1024, 1) == 1
    assert form(16, 576, 0) == 0 and form(16, 2560, 1) == form(16, 2560, 1, True) == 2 and form(16, 2500, 1) == 3 and form(16, 1536, 0, True) == 2
    assert form(1025, 96, 0) == 1 and form(1024, 96, 0) == 4 and form(700, 1024, 1) == 1
    assert _lib.load().fastlstm_recurrent_form(5, 16, 1024, 1, 0, 16) == _lib.ERR_WORKSPACE


def test_stacks_of_sizes_off_a_multiple_of_64():
    """Many rows: padded where that makes the K of the upper layers' projections a multiple of 64."""
    pad = lambda T, B, H, layers, two, training: L._operand_padding_cached(T, B, 128, H, layers, two, True, 1, 0, training, L._families())
    assert pad(128, 32, 112, 3, False, False) == (128, 128) and pad(128, 32, 112, 3, False, True) is None and pad(256, 256, 112, 2, False, True) == (128, 128)
    assert pad(128, 32, 80, 3, False, False) is None and pad(128, 32, 80, 2, True, False) == (96, 128) and pad(128, 32, 112, 1, False, False) is None
    assert pad(128, 32, 128, 3, False, False) is None
