"""The kernels that keep up to 512 KiB of weights per CU (16-bit, 1280 <= H <= 4096) against the oracle: every number of
k-steps per wave, hidden sizes with padded k-steps and with uneven numbers of teams per XCD, every number of batch tiles, launches
over row ranges, the first steps."""
import pytest
import torch

import fastlstm_amd.lstm as L
from test_gpu_parity import FWD_KEYS, HALF_TOL, RM, dev, make_problem, npy, to_np, within
from fastlstm_amd import FastLSTM

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
    (1, 128, 2048, torch.float16),   # ... all CUs
    (3, 33, 2064, torch.float16),    # no multiple of 64: the forward kernel only
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
