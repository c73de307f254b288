"""A few timesteps of inference, one kernel per step (fastlstm_infer_short): against nn.LSTM in float64 with the same
rounded weights and inputs, and the module's choice of it."""
import pytest
import torch

import fastlstm_amd.lstm as L
from fastlstm_amd import FastLSTM, _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,tol", [(torch.float32, 1e-4), (torch.float16, 2e-2), (torch.bfloat16, 2e-2)])
@pytest.mark.parametrize("layers,T,B,I,H,bias,states", [
    (1, 1, 1, 1, 1, True, False),        # the smallest
    (2, 1, 16, 64, 64, True, True),      # one full batch tile, whole pieces in every row
    (1, 3, 17, 33, 70, False, True),     # two batch tiles, rows on odd boundaries, a cut last piece and unit tile
    (3, 2, 33, 50, 129, True, True),     # four batch tiles, H % 4 == 1
    (5, 3, 4, 40, 48, True, False),      # more cells per launch than a launch takes
    (1, 2, 65, 128, 256, True, True),    # two ranges of 64 rows
    (1, 1, 64, 96, 2056, True, True),    # eight units per workgroup
])
def test_short_inference_against_nn_lstm(layers, T, B, I, H, bias, states, dt, tol, monkeypatch):
    lib = _lib.load()
    monkeypatch.setattr(L, "_short_scratch_bytes", lambda l, t, b, i, h, c: lib.fastlstm_infer_short_scratch_bytes(l, t, b, h, c))
    torch.manual_seed(T + B + H)
    m = FastLSTM(I, H, num_layers=layers, bias=bias).to("cuda", dt)
    ref = torch.nn.LSTM(I, H, num_layers=layers, bias=bias).double()
    ref.load_state_dict({k: v.double().cpu() for k, v in m.state_dict().items()})
    x = torch.randn(T, B, I).to(dt)
    s = tuple((torch.randn(layers, B, H) * 0.3).to(dt) for _ in range(2)) if states else None
    with torch.no_grad():
        short = m._forward_short(x.cuda(), None if s is None else tuple(t.cuda() for t in s))
        want = ref(x.double(), None if s is None else tuple(t.double() for t in s))
    assert short is not None
    for got, w in zip((short[0], *short[1]), (want[0], *want[1])):
        torch.testing.assert_close(got.double().cpu(), w, rtol=tol, atol=tol)


def test_module_takes_the_short_form_without_gradients_only():
    m = FastLSTM(64, 128, num_layers=2, device="cuda")
    x = torch.randn(1, 2, 64, device="cuda")
    with torch.no_grad():
        assert m._forward_short(x, None) is not None
        assert m._forward_short(x.half(), None) is None                      # weights of another type
        assert m._forward_short(torch.randn(200, 64, 64, device="cuda"), None) is None   # long
    y, _ = m(x)
    y.sum().backward()
    assert m.weight_hh_l0.grad is not None
