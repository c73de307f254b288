"""16-bit products of few output tiles (csrc/gemm16.hpp, SHORT; tile and split by csrc/gemm.hip gemm_plan): edges of the 64 x 64 and
128 x 128 tiles, one and several k-tiles, sums in parts, against float64; the sums are those of the product's other tiles, bit by bit."""
import pytest
import torch

import fastlstm_amd.lstm as L
from fastlstm_amd import _lib

pytestmark = pytest.mark.gpu
EPS = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}   # unit roundoff: of every result; the fp32 sums add far less


def ptr(t):
    return t.data_ptr() if t is not None else None


def ifgo(x, Wx, b, T, B, I, H):
    y = torch.full((T * B + 2, 4 * H), 7.0, dtype=x.dtype, device="cuda")
    _lib.check(_lib.load().fastlstm_gemm_ifgo(ptr(x), ptr(Wx), ptr(b), ptr(b), ptr(y), T, B, I, H, L._DTYPE_CODE[x.dtype],
                                              torch.cuda.current_stream().cuda_stream), "ifgo")
    assert bool((y[T * B:] == 7).all())
    return y[:T * B]


def dx(g, Wx, T, B, I, H, scratch=None):
    y = torch.full((T * B + 2, I), 7.0, dtype=g.dtype, device="cuda")
    _lib.check(_lib.load().fastlstm_gemm_dx_split(ptr(g), ptr(Wx), ptr(y), T, B, I, H, L._DTYPE_CODE[g.dtype], ptr(scratch),
                                                  scratch.numel() if scratch is not None else 0,
                                                  torch.cuda.current_stream().cuda_stream), "dx")
    assert bool((y[T * B:] == 7).all())
    return y[:T * B]


# (T, B, I, H): M = T B, K = I or 4 H.  One tile and one k-tile; ragged rows and columns; 64 x 64 in two parts and more; 128 x 128 tiles
# below and above 256 of them, whole and in parts
@pytest.mark.parametrize("T,B,I,H", [(1, 1, 64, 80), (1, 65, 192, 136), (3, 43, 72, 96), (35, 20, 704, 704), (2, 33, 64, 1024),
                                     (8, 32, 1024, 1032), (16, 64, 512, 768), (100, 50, 128, 288), (33, 129, 256, 520)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_products(T, B, I, H, dt):
    gen = torch.Generator(device="cuda").manual_seed(T * B + H)
    x, Wx, b, g = (torch.randn(s, generator=gen, device="cuda").mul_(k).to(dt)
                   for s, k in (((T * B, I), 1), ((4 * H, I), I ** -0.5), ((4 * H,), 1), ((T * B, 4 * H), 1)))
    y = ifgo(x, Wx, b, T, B, I, H)
    want = x.double() @ Wx.double().t() + 2 * b.double()
    assert float((y.double() - want).norm()) <= EPS[dt] * float(want.norm())
    want = g.double() @ Wx.double()
    scratch = torch.empty(64 << 20, dtype=torch.uint8, device="cuda")
    whole = dx(g, Wx, T, B, I, H)
    for d in (whole, dx(g, Wx, T, B, I, H, scratch)):
        assert float((d.double() - want).norm()) <= EPS[dt] * float(want.norm())
    m = (T * B + 1) // 2   # other tiles, the same bits
    assert torch.equal(ifgo(x[:m], Wx, b, 1, m, I, H), y[:m]) and torch.equal(dx(g[:m], Wx, 1, m, I, H), whole[:m])


# d.Wx in parts: 64 x 64 tiles in several, 128 x 128 in one round of parts from 257 small tiles and K = 4096 on, and one pass where the parts of a
# large output would cost more
@pytest.mark.parametrize("T,B,I,H", [(10, 100, 64, 512), (151, 19, 408, 1024), (30, 929, 160, 288), (33, 99, 1432, 672)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_parts_of_dx(T, B, I, H, dt):
    test_products(T, B, I, H, dt)


# (rows, I, H) of thin weight gradients: 64 x 64 tiles in one part and in several, 128 x 128 ones from 32768 rows or 2^21 rows x tiles on
@pytest.mark.parametrize("R,I,H", [(500, 80, 96), (16500, 96, 96), (8200, 80, 512), (32767, 192, 64), (32768, 192, 64)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_weight_gradients(R, I, H, dt):
    gen = torch.Generator(device="cuda").manual_seed(R + H)
    d, x, h = (torch.randn(s, generator=gen, device="cuda").mul_(R ** -0.5).to(dt) for s in ((1, R, 4 * H), (1, R, I), (2, R, H)))
    db, _, dWx, dWh = L.Wgrad(d, x, h)
    D = d[0].double()
    # fp32 sums: at most R roundings of a running sum, in practice their square root; the bound of the results' rounding leaves room
    for got, want in ((dWx, D.t() @ x[0].double()), (dWh, D.t() @ h[0].double()), (db, D.sum(0))):
        assert float((got.double() - want).norm()) <= EPS[dt] * float(want.norm())
