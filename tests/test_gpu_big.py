"""The kernels that keep up to 512 KiB of weights per CU (16-bit, 1280 <= H <= 4096) against the oracle: every number of
k-steps per wave, hidden sizes with padded k-steps and with uneven numbers of teams per XCD, every number of batch tiles, launches
over row ranges, the first steps."""
import pytest
import torch

import fastlstm_amd.lstm as L
from test_gpu_parity import FP32_TOL, FWD_KEYS, HALF_TOL, RM, dev, make_problem, npy, to_np, within
from fastlstm_amd import FastLSTM, _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,B,H,dt", [
    (1, 1, 2112, torch.float16),     # 33 teams: 5 on the first XCDs
    (2, 16, 2560, torch.bfloat16),
    (3, 17, 2624, torch.float16),    # 24 k-steps per wave, the last ones padding
    (4, 48, 3136, torch.bfloat16),   # 28
    (5, 64, 3648, torch.float16),    # 32, padded
    (3, 65, 4096, torch.bfloat16),   # two launches, the second of one row
    (2, 97, 1280, torch.float16),    # 32 units per workgroup: groups of 32 rows, the last one ragged
    (3, 161, 1536, torch.bfloat16),  # ... a launch over 160 rows and one row
    (2, 15, 1792, torch.float16),    # ... one group of 16 rows, the weights' sums four tiles at a time
    (2, 100, 1792, torch.bfloat16),  # ... groups of 32
    (1, 128, 2048, torch.float16),   # ... all CUs
    (3, 33, 2064, torch.float16),    # no multiple of 64: the forward kernel only
    (1, 50, 2304, torch.bfloat16),   # four batch tiles, whose results leave behind the products of the next: one step,
    (2, 36, 2880, torch.float16),    # ... two, with a tile that has no row
])
def test_big_layers_vs_oracle(oracle, T, B, H, dt):
    p = make_problem(T, B, 24, H, seed=T * 1000 + H)
    pr = {k: (v.to(dt).double() if v is not None else None) for k, v in p.items()}
    g = {k: dev(v, dt) for k, v in p.items()}
    o_out, o_cell, o_ifgo = oracle.forward(*to_np(pr, FWD_KEYS), round_mode=RM[dt])
    operands = [g[k] for k in ("x", "h0", "c0", "Wx", "bx", "Wh", "bh")]
    out, cell, ifgo = L.lstm_persistent_fwd(*operands)
    for name, got, want in (("out", out, o_out), ("cell", cell, o_cell), ("ifgo", ifgo, o_ifgo)):
        within(got, want, HALF_TOL, name)
    out_i, cell_i, _ = L.lstm_persistent_fwd(*operands, keep_activations=False)
    assert torch.equal(out_i, out) and torch.equal(cell_i[-1], cell[-1])
    dout, dh_n, dc_n, x, Wx, Wh = to_np(pr, ["dout", "dh_n", "dc_n", "x", "Wx", "Wh"])
    r = oracle.backward(dout, dh_n, dc_n, x, npy(out), npy(cell), npy(ifgo), Wx, Wh, round_mode=RM[dt])
    d_x, dh0, dc0, dWx, dbx, dWh, _ = L.lstm_persistent_bwd(g["dout"], g["dc_n"].clone(), g["dh_n"].clone(), g["x"], out, cell, ifgo,
                                                           g["Wx"], g["Wh"])
    for name, got, want in (("dx", d_x, r["dx"]), ("dh0", dh0, r["dh0"]), ("dc0", dc0, r["dc0"]),
                            ("dWx", dWx, r["dWx"]), ("dWh", dWh, r["dWh"]), ("db", dbx, r["db"])):
        within(got, want, HALF_TOL, name)


def test_module_pads_to_a_multiple_of_64(oracle):
    T, B, H = 16, 3, 2100
    p = make_problem(T, B, 24, H, seed=5)
    m = FastLSTM(24, H, device="cuda", dtype=torch.float16)
    pr = {k: (v.half().double() if v is not None else None) for k, v in p.items()}
    with torch.no_grad():
        for prm, k in zip(m._layer_operands(0), ("Wx", "bx", "Wh", "bh")):
            prm.copy_(p[k].half())
        out, _ = m(p["x"].half().cuda())
    zeros = torch.zeros(B, H, dtype=torch.float64)
    pr["h0"] = pr["c0"] = zeros
    want, _, _ = oracle.forward(*to_np(pr, FWD_KEYS), round_mode=RM[torch.float16])
    within(out, want[1:], HALF_TOL, "out")


@pytest.mark.parametrize("T,B,H,dt,whole", [
    (1, 20, 1280, torch.float16, True),      # two ragged groups of 16 rows each, 20 teams on the XCDs unevenly
    (3, 32, 1792, torch.bfloat16, True),     # ... full groups
    (4, 17, 2048, torch.float16, True),      # all CUs
    (2, 9, 1536, torch.bfloat16, True),      # one partly filled group each
    (3, 32, 2048, torch.bfloat16, False),    # no room for the teams' partial sums: the 16-unit form, alone and as a pair
])
def test_pair_of_reverse_recurrences_equals_two_calls(T, B, H, dt, whole):
    """fastlstm_bwd_persistent_pair on the whole-CU kernel: d_ifgo and the state gradients of both recurrences are the bits of
    two calls of their own (the same kernel adds in the same order, whichever workgroup a group is on)."""
    lib, code = _lib.load(), RM[dt]
    st = torch.cuda.current_stream().cuda_stream
    plan = _lib.Plan()
    _lib.check(lib.fastlstm_plan_device(0, B, H, code, 1, plan), "plan")
    gen = torch.Generator(device="cuda").manual_seed(T * H + B)
    rnd = lambda *shape, s=1.0: (torch.randn(*shape, device="cuda", generator=gen) * s).to(dt)
    sides = [dict(dout=rnd(T, B, H), dh=rnd(B, H), dc=rnd(B, H), ifgo=rnd(T, B, 4 * H), cell=rnd(T + 1, B, H, s=0.5), Wh=rnd(4 * H, H, s=H ** -0.5))
             for _ in range(2)]
    one, two = (lib.fastlstm_recurrent_workspace_bytes(plan, T, H, code, 1), lib.fastlstm_stack2_bwd_workspace_bytes(plan, T, H, code))
    if not whole:
        one, two = plan.ws_bytes, 2 * plan.ws_bytes
    assert lib.fastlstm_pair_fused(T, B, H, code, 1, two) == 1

    def operands(o, d_ifgo):
        return [o[k].data_ptr() for k in ("dout", "dh", "dc", "ifgo", "cell")] + [d_ifgo.data_ptr(), o["Wh"].data_ptr()]

    def fresh():
        return [dict(o, dh=o["dh"].clone(), dc=o["dc"].clone()) for o in sides], [torch.empty(T, B, 4 * H, device="cuda", dtype=dt) for _ in sides]

    got, d_got = fresh()
    ws = torch.zeros(two, dtype=torch.uint8, device="cuda")
    _lib.check(lib.fastlstm_bwd_persistent_pair(*operands(got[0], d_got[0]), *operands(got[1], d_got[1]), ws.data_ptr(), two, T, B, H, code, st), "pair")
    torch.cuda.synchronize()
    assert lib.fastlstm_ws_status(ws[:64].cpu().numpy().tobytes()) == _lib.OK
    want, d_want = fresh()
    for o, d in zip(want, d_want):
        ws = torch.zeros(one, dtype=torch.uint8, device="cuda")
        _lib.check(lib.fastlstm_bwd_persistent(*operands(o, d), ws.data_ptr(), one, T, B, H, code, st), "single")
    torch.cuda.synchronize()
    for g, w, dg, dw in zip(got, want, d_got, d_want):
        assert torch.equal(dg, dw) and torch.equal(g["dh"], w["dh"]) and torch.equal(g["dc"], w["dc"])
        assert torch.isfinite(dg.float()).all()


@pytest.mark.parametrize("B,H,backward", [(1, 1280, True), (4, 2048, True), (17, 1536, True), (3, 2560, True),
                                          (33, 2048, False), (34, 1280, False), (1, 4096, False),
                                          (2, 1280, False), (17, 2048, False)])   # the last two: the 16-unit form
def test_rows_past_the_batch_leave_no_trace(B, H, backward):
    """The gates of rows past the batch are computed on whatever LDS and the exchange blocks hold: a call behind one that left NaN
    in both, on a workspace of NaN, is the same bits as one behind zeros."""
    lib, T, st = _lib.load(), 3, torch.cuda.current_stream().cuda_stream
    results = []
    for fill in (0.0, float("nan")):
        for rows in (64, B):
            plan = _lib.Plan()
            _lib.check(lib.fastlstm_plan_device(0, rows, H, 1, int(backward), plan), "plan")
            n = lib.fastlstm_recurrent_workspace_bytes(plan, T, H, 1, int(backward))
            ws = torch.full((n,), 0xff if fill != fill else 0, dtype=torch.uint8, device="cuda")
            ws[:(n if rows == 64 else plan.ws_zero_bytes)] = 0
            torch.manual_seed(H + rows)
            draw = lambda *shape: torch.full(shape, fill, device="cuda").half() if rows == 64 else torch.randn(*shape, device="cuda").half()
            Wh = (torch.randn(4 * H, H, device="cuda") * H ** -.5).half()
            ifgo, cell = draw(T, rows, 4 * H), draw(T + 1, rows, H)
            if backward:
                d = torch.zeros_like(ifgo)
                moved = [draw(T, rows, H), draw(rows, H), draw(rows, H), ifgo, cell, d, Wh]
                entry, got = lib.fastlstm_bwd_persistent, moved[1:3] + [d]
            else:
                moved = [ifgo, draw(T + 1, rows, H), cell, Wh]
                entry, got = lib.fastlstm_fwd_persistent, moved[:3]
            _lib.check(entry(*(t.data_ptr() for t in moved), ws.data_ptr(), n, T, rows, H, 1, st), "recurrence")
        results.append(got)
    for clean, dirty in zip(*results):
        assert torch.isfinite(clean).all() and torch.equal(clean, dirty)


@pytest.mark.parametrize("T,B,H,dt", [
    (3, 16, 2576, torch.bfloat16),   # one batch tile, half a k-step past H
    (4, 33, 2560, torch.float16),    # three tiles of four
    (3, 64, 4096, torch.bfloat16),
    (4, 128, 2048, torch.float16),   # groups of two tiles
    (4, 192, 1280, torch.bfloat16),  # ... six groups in a launch
    (3, 120, 640, torch.float32),    # two tiles, three words for two numbers
    (4, 9, 1280, torch.float32),     # ... 8 units per workgroup, one tile
    (4, 7, 1536, torch.float32),     # with flags
    (3, 30, 2048, torch.float32),
    (3, 64, 1280, torch.float32),    # with flags
])
def test_rows_that_are_no_numbers(T, B, H, dt):
    """A row of NaN whose bits are all ones, which is what a word that has not been written looks like: the launch ends, the row is NaN from
    its first step on, and no bit of any other row changes."""
    p = make_problem(T, B, 24, H, seed=T * 100 + H)
    g = {k: dev(v, dt) for k, v in p.items() if v is not None}
    bits = torch.int32 if dt == torch.float32 else torch.int16
    row = B - 1 if B % 16 else B // 2
    outs = []
    for h0 in (g["h0"], g["h0"].clone()):
        if outs:
            h0.view(bits)[row] = -1
        outs.append(L.lstm_persistent_fwd(g["x"], h0, g["c0"], g["Wx"], g["bx"], g["Wh"], g["bh"])[:2])
    others = torch.arange(B, device="cuda") != row
    for want, got in zip(*outs):
        assert torch.equal(want[1:, others], got[1:, others])
        assert got[1:, row].isnan().all()


REVERSE = [
    (3, 16, 2560, torch.bfloat16),   # one unit tile per member, one batch tile
    (4, 64, 4096, torch.float16),    # four batch tiles
    (3, 40, 2048, torch.bfloat16),   # two unit tiles per member, groups of 16 rows
    (4, 128, 2048, torch.float16),   # ... of 32, all CUs
    (3, 90, 1280, torch.bfloat16),   # ... a ragged group, teams on the XCDs unevenly
    (4, 64, 1024, torch.float32),    # fp32: teams of four
    (3, 100, 640, torch.float32),
    (4, 7, 1280, torch.float32),     # teams of eight: two members share a unit tile, and the place of its sums
    (3, 50, 2048, torch.float32),
]


def _reverse_call(operands, ws_bytes=None):
    """fastlstm_bwd_persistent on copies: ([d_ifgo, dh_0, dc_0], status of the workspace)."""
    dout, dh, dc, ifgo, cell, Wh = operands
    (T, B, H), code, lib = dout.shape, RM[dout.dtype], _lib.load()
    plan = _lib.Plan()
    _lib.check(lib.fastlstm_plan_device(0, B, H, code, 1, plan), "plan")
    n = ws_bytes or lib.fastlstm_recurrent_workspace_bytes(plan, T, H, code, 1)
    assert lib.fastlstm_recurrent_form(T, B, H, code, 1, n) == 2
    ws = torch.full((n,), 0xff, dtype=torch.uint8, device="cuda")
    ws[:min(n, plan.ws_zero_bytes)] = 0
    dh, dc, d = dh.clone(), dc.clone(), torch.empty_like(ifgo)
    _lib.check(lib.fastlstm_bwd_persistent(dout.data_ptr(), dh.data_ptr(), dc.data_ptr(), ifgo.data_ptr(), cell.data_ptr(), d.data_ptr(),
                                           Wh.data_ptr(), ws.data_ptr(), n, T, B, H, code, torch.cuda.current_stream().cuda_stream), "reverse")
    torch.cuda.synchronize()
    return [d, dh, dc], lib.fastlstm_ws_status(ws[:64].cpu().numpy().tobytes())


def _reverse_operands(T, B, H, dt):
    g = torch.Generator(device="cuda").manual_seed(T * 100 + H)
    n = lambda *s, k=1.0: (torch.randn(*s, device="cuda", generator=g) * k).to(dt)
    return n(T, B, H), n(B, H), n(B, H), n(T, B, 4 * H), n(T + 1, B, H, k=.5), n(4 * H, H, k=H ** -.5)


@pytest.mark.parametrize("T,B,H,dt", REVERSE)
def test_gradients_that_are_no_numbers(T, B, H, dt):
    """A row of NaN whose bits are all ones (what a word of the team's sums that has not been written looks like) in each operand of the
    reverse pass in turn: the launch ends, the row's gradients are NaN from there on, and no bit of any other row changes."""
    clean_operands = _reverse_operands(T, B, H, dt)
    clean, status = _reverse_call(clean_operands)
    assert status == _lib.OK and all(torch.isfinite(t).all() for t in clean)
    bits, row = torch.int32 if dt == torch.float32 else torch.int16, B - 1 if B % 16 else B // 2
    others = torch.arange(B, device="cuda") != row
    for which, name in enumerate(("dout", "dh_n", "dc_n", "ifgo", "cell")):
        operands = [t.clone() for t in clean_operands]
        bad = operands[which].view(bits)
        if bad.dim() == 3:
            bad[T // 2, row] = -1
        else:
            bad[row] = -1
        got, status = _reverse_call(operands)
        assert status == _lib.OK, name
        for a, b in zip(got, clean):
            assert torch.equal(a[..., others, :], b[..., others, :]), name
            assert a[..., row, :].view(-1, a.shape[-1])[0].isnan().all(), name   # (d_ifgo: its first timestep)


@pytest.mark.parametrize("T,B,H,dt", REVERSE)
def test_reverse_launches_drain_on_timeout(T, B, H, dt):
    """A spin limit of one poll, forced from the host: the waits for the group and for the team's sums give up, the grid drains, the
    call reports it and its results are NaN; the next call is healthy."""
    lib, operands = _lib.load(), _reverse_operands(T, B, H, dt)
    want, _ = _reverse_call(operands)
    try:
        lib.fastlstm_set_spin_limit(1)
        got, status = _reverse_call(operands)
    finally:
        lib.fastlstm_set_spin_limit(400000000)
    assert status == _lib.ERR_TIMEOUT and lib.fastlstm_device_status(0, 1) == _lib.ERR_TIMEOUT
    assert got[0][0].isnan().any() and got[1].isnan().all() and got[2].isnan().all()
    again, status = _reverse_call(operands)
    assert status == _lib.OK and all(torch.equal(a, b) for a, b in zip(again, want))


@pytest.mark.parametrize("T,B,H,dt", [
    (3, 128, 1280, torch.float16),    # groups of 64 rows of the 16-unit form: two slots are all there is room for
    (3, 140, 1280, torch.bfloat16),   # ... over row ranges
    (3, 128, 2048, torch.bfloat16),
    (3, 140, 2048, torch.float16),
    (3, 60, 2048, torch.float16),     # one batch tile per group: needs no more than two
    (3, 120, 640, torch.float32),     # two batch tiles, parts of numbers: the general kernel
])
def test_forward_with_the_smallest_workspace(oracle, T, B, H, dt):
    """plan.ws_bytes, the least that is accepted, holds two exchange slots: the forms that take four leave the call to another."""
    lib, code = _lib.load(), RM[dt]
    p = make_problem(T, B, 24, H, seed=T * 1000 + H + B)
    pr = {k: (v.to(dt).double() if v is not None else None) for k, v in p.items()}
    wants = oracle.forward(*to_np(pr, FWD_KEYS), round_mode=RM[dt])
    plan = _lib.Plan()
    _lib.check(lib.fastlstm_plan_device(0, B, H, code, 0, plan), "plan")
    g = {k: dev(v, dt) for k, v in p.items() if v is not None}
    ifgo, out, cell = (torch.empty(s, device="cuda", dtype=dt) for s in ((T, B, 4 * H), (T + 1, B, H), (T + 1, B, H)))
    out[0], cell[0] = g["h0"], g["c0"]
    n = plan.ws_bytes
    ws = torch.zeros(n + (1 << 20), dtype=torch.uint8, device="cuda")
    ws[n:] = 0x5a
    st = torch.cuda.current_stream().cuda_stream
    _lib.check(lib.fastlstm_fwd_layer(*(t.data_ptr() for t in (g["x"], g["Wx"], g["bx"], g["bh"], g["Wh"], ifgo, out, cell, ws)), n, T, B, 24, H,
                                      code, st), "forward")
    torch.cuda.synchronize()
    assert lib.fastlstm_ws_status(ws[:64].cpu().numpy().tobytes()) == _lib.OK and bool((ws[n:] == 0x5a).all())
    for name, got, want in zip(("out", "cell", "ifgo"), (out, cell, ifgo), wants):
        within(got, want, FP32_TOL if dt == torch.float32 else HALF_TOL, name)
