"""The fp32 products (csrc/gemm_f32.hpp): edges of their tiles and k-tiles, and operands that are no finite numbers."""
import pytest
import torch

import fastlstm_amd.lstm as L
from fastlstm_amd import _lib

pytestmark = pytest.mark.gpu

# rows T*B, I, H: one element, below and above the tiles of 128 and 256, k-tiles of 16 with a remainder, rows of 4-byte
# alignment, split sums, more tiles than compute units
SHAPES = [(1, 1, 1), (5, 3, 4), (127, 15, 33), (129, 17, 32), (255, 260, 64), (257, 129, 66), (1000, 77, 130), (4099, 256, 256),
          (2048, 513, 1024)]


def products(R, I, H, seed=0, plant=None):
    """((K1, dx, dWx, dWh, db), the same in 64 bits, the same of magnitudes)"""
    g = torch.Generator(device="cuda").manual_seed(seed)
    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    n = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, Wx, bx, bh, d, h = n(1, R, I), n(4 * H, I), n(4 * H), n(4 * H), n(1, R, 4 * H), n(2, R, H)
    if plant is not None:
        plant(x, Wx, d)
    k1, dx = torch.empty(R, 4 * H, device="cuda"), torch.empty(R, I, device="cuda")
    _lib.check(lib.fastlstm_gemm_ifgo(x.data_ptr(), Wx.data_ptr(), bx.data_ptr(), bh.data_ptr(), k1.data_ptr(), 1, R, I, H, 0, st), "k1")
    _lib.check(lib.fastlstm_gemm_dx(d.data_ptr(), Wx.data_ptr(), dx.data_ptr(), 1, R, I, H, 0, st), "dx")
    db, _, dWx, dWh = L.Wgrad(d, x, h)

    def exact(f):
        X, W, D, Hh = f(x[0].double()), f(Wx.double()), f(d[0].double()), f(h[0].double())
        return X @ W.T + f(bx.double()) + f(bh.double()), D @ W, D.T @ X, D.T @ Hh, D.sum(0)
    return (k1, dx, dWx, dWh, db), exact(lambda t: t), exact(torch.abs)


@pytest.mark.parametrize("R,I,H", SHAPES)
def test_products_at_the_edges(R, I, H):
    got, want, magnitude = products(R, I, H, seed=R + I + H)
    for a, b, m, terms in zip(got, want, magnitude, (I + 2, 4 * H, R, R, R)):
        # six roundings of the running sum per 16 terms, the products left out (together 2^-24 of a term) and one of the result; the sums
        # of magnitudes bound the running sums
        bound = m * ((3 + 6 * terms / 16) * 2.0 ** -24 + 2.0 ** -24)
        assert bool(((a.double() - b).abs() <= bound).all())


@pytest.mark.parametrize("I,H,rows", [(40, 64, (1, 63, 65, 4096)), (64, 65, (64, 200)), (65, 96, (31, 129)), (300, 256, (1, 1000)), (1030, 512, (7, 128))])
def test_a_range_of_rows_has_the_bits_of_the_whole(I, H, rows):
    """Tiles of 64 (few rows), 128 and 256 add up in the same order: x.Wx^T and d.Wx of the first rows alone."""
    g = torch.Generator(device="cuda").manual_seed(I + H)
    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    n = lambda *s: torch.randn(*s, generator=g, device="cuda")
    R = 8192
    x, Wx, bx, bh, d = n(R, I), n(4 * H, I), n(4 * H), n(4 * H), n(R, 4 * H)

    def both(r):
        y, dx = torch.empty(r, 4 * H, device="cuda"), torch.empty(r, I, device="cuda")
        _lib.check(lib.fastlstm_gemm_ifgo(x.data_ptr(), Wx.data_ptr(), bx.data_ptr(), bh.data_ptr(), y.data_ptr(), 1, r, I, H, 0, st), "k1")
        _lib.check(lib.fastlstm_gemm_dx(d.data_ptr(), Wx.data_ptr(), dx.data_ptr(), 1, r, I, H, 0, st), "dx")
        return y, dx
    whole = both(R)
    for r in rows:
        for a, b in zip(both(r), whole):
            assert torch.equal(a, b[:r]), r


def test_infinities_and_nans_as_in_the_sum():
    """inf times a number whose lower parts are zero, of either sign, inf times 0, inf - inf and NaN: in an operand of any product."""
    def plant(x, Wx, d):
        inf = float("inf")
        Wx[0, :4] = torch.tensor([1.0, -0.5, 0.0, 3.0])
        x[0, 3, 0], x[0, 4, 1], x[0, 5, 2], x[0, 200, 3] = inf, inf, -inf, float("nan")
        Wx[70, 5] = -inf
        d[0, 10, 9] = inf
        d[0, 11, 40], d[0, 12, 40] = inf, -inf
    got, want, _ = products(300, 40, 130, plant=plant)
    for a, b in zip(got, want):
        assert torch.equal(torch.isnan(a), torch.isnan(b))
        assert torch.equal(torch.isinf(a), torch.isinf(b)) and torch.equal(a[torch.isinf(a)].double(), b[torch.isinf(b)])
        ok = torch.isfinite(b)
        assert float((a.double() - b)[ok].abs().max()) < 1e-3 and bool(ok.any()) and not bool(ok.all())


def chain(A, B):
    """A.B^T as a chain of fp32 multiply-adds (each rounded once; the product in 64 bits is exact)."""
    acc = torch.zeros(A.shape[0], B.shape[0], device=A.device)
    for k in range(A.shape[1]):
        acc = (acc.double() + A[:, k, None].double() * B[None, :, k].double()).float()
    return acc


def each_product(A, B):
    """A[M,K].B[N,K]^T with N a multiple of 4, by every product that has this K: x.Wx^T, d.Wx, the weight gradients."""
    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    (M, K), N = A.shape, B.shape[0]
    y, z = torch.empty(M, N, device="cuda"), torch.zeros(N, device="cuda")
    _lib.check(lib.fastlstm_gemm_ifgo(A.data_ptr(), B.data_ptr(), z.data_ptr(), z.data_ptr(), y.data_ptr(), 1, M, K, N // 4, 0, st), "k1")
    yield "x.Wx^T", y
    if K % 4 == 0:
        dx, W, ws = torch.empty(M, N, device="cuda"), B.t().contiguous(), torch.empty(32 << 20, dtype=torch.uint8, device="cuda")
        _lib.check(lib.fastlstm_gemm_dx_split(A.data_ptr(), W.data_ptr(), dx.data_ptr(), 1, M, N, K // 4, 0, ws.data_ptr(), ws.numel(), st), "dx")
        yield "d.Wx", dx
    d = A.t().contiguous()[None]
    yield "d^T.x", L.Wgrad(d, B.t().contiguous()[None], torch.zeros(2, K, M // 4, device="cuda"))[2]


@pytest.mark.parametrize("K", [1, 2, 3, 4, 5, 8, 16, 17, 64, 65, 128, 4096])
@pytest.mark.parametrize("sign", [False, True])
def test_no_further_off_than_a_chain_of_multiply_adds(K, sign):
    """Short contractions, where every rounding shows, the two sides of the line between nine products and six, and a long sum; terms of
    one sign, whose errors add up if they have one."""
    g = torch.Generator(device="cuda").manual_seed(K)
    A, B = (torch.randn(128, K, generator=g, device="cuda") for _ in range(2))
    if sign:
        A, B = A.abs() + 0.25, B.abs() + 0.25
    want = A.double() @ B.double().t()
    allowed = float((chain(A, B).double() - want).norm())
    for name, got in each_product(A, B):
        # (128 x 128 results: 2-norms of rounding errors differ by less than 1 % from sample to sample, K = 1: the same roundings)
        assert float((got.double() - want).norm()) <= 1.02 * allowed, name
        if sign and K <= 128:   # the mean of 16384 unbiased roundings of up to 6e-8 is some 3e-10; what the MFMA drops below its sum, K / 16 times
            assert abs(float(((got.double() - want) / want).mean())) <= 1e-9 + K / 16 * 1e-9, name


@pytest.mark.parametrize("a,b", [(2.0 ** -107, 1.0), (2.0 ** -113, 1.0), (2.0 ** -126, 1.0), (2.0 ** -126, 2.0 ** 20), (2.0 ** -140, 2.0 ** 30),
                                 (2.0 ** -60, 2.0 ** -60), (2.0 ** 79, 1.0), (2.0 ** 100, 2.0 ** -3), (2.0 ** 120, 2.0 ** -30), (2.0 ** 127, 2.0 ** -10)])
def test_small_and_large_numbers(a, b):
    """Magnitudes over the whole range of fp32, numbers below its least normal one too (exact in the comparison: they are drawn as such)."""
    for K in (8, 100):
        g = torch.Generator(device="cuda").manual_seed(K)
        A, B = ((torch.rand(128, K, generator=g, device="cuda") * 2 - 1) * s for s in (a, b))
        want = A.double() @ B.double().t()
        allowed = float((chain(A, B).double() - want).norm())   # (2-norms of 16384 errors: as above)
        for name, got in each_product(A, B):
            assert float((got.double() - want).norm()) <= 1.05 * allowed, name


@pytest.mark.parametrize("R,I,H", [(9000, 3, 5), (17000, 1, 32), (9000, 40, 16)])
def test_thin_gradients_of_many_rows(R, I, H):
    """One or two output tiles: K in more than 64 parts.  Terms of one sign, whose running sum every rounding is relative to."""
    g = torch.Generator(device="cuda").manual_seed(R + I)
    d, x, h = (torch.rand(*s, generator=g, device="cuda") + 0.25 for s in ((1, R, 4 * H), (1, R, I), (2, R, H)))
    db, _, dWx, dWh = L.Wgrad(d, x, h)
    D = d[0].double()
    for got, want in ((dWx, D.t() @ x[0].double()), (dWh, D.t() @ h[0].double()), (db, D.sum(0))):
        # parts of at most some 200 rows: 2e-7 for the sum of one (its 13 roundings of up to 6e-8 each by their square root), as much for the sum of them
        assert float((got.double() - want).norm()) <= 4e-7 * float(want.norm())


def test_sums_beside_those_that_are_not_finite_keep_their_bits():
    def planted(v):
        def plant(x, Wx, d):
            if v is not None:
                x[0, 7, 3], d[0, 9, 11] = v, v
        return products(300, 40, 130, seed=3, plant=plant)[0]
    clean = planted(None)
    for v in (float("nan"), float("inf"), 3e38, 1e20):
        for i, (a, b) in enumerate(zip(clean, planted(v))):
            if i < 2:     # x.Wx^T and d.Wx: one row of results has it in its sum, the weight gradients one row or column
                row = 7 if i == 0 else 9
                keep = torch.arange(a.shape[0], device="cuda") != row
                assert torch.equal(a[keep], b[keep]), (v, i)
            elif i < 4:
                keep = torch.arange(a.shape[0], device="cuda") != 11
                cols = torch.arange(a.shape[1], device="cuda") != (3 if i == 2 else -1)
                assert torch.equal(a[keep][:, cols], b[keep][:, cols]), (v, i)
