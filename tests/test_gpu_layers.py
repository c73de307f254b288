"""What surrounds the layers of a call: the copy launch (fastlstm_copy_blocks) against torch indexing, and the one-node form of
a call (fastlstm_amd.layers) against the layer loop of the module."""
import pytest
import torch
from torch.nn.utils.rnn import PackedSequence, pack_padded_sequence

import fastlstm_amd.layers as layers
import fastlstm_amd.lstm as L
from fastlstm_amd import FastLSTM

pytestmark = pytest.mark.gpu
CODE = L._DTYPE_CODE


class _Ctx:
    def __init__(self, T=0, B=0, lens=None, offs=None, order=None):
        self.T, self.B, self.stream = T, B, L._stream()
        self.lens, self.offs, self.order = (None if t is None else t.data_ptr() for t in (lens, offs, order))


@pytest.mark.parametrize("src,dst", [(torch.float32, torch.bfloat16), (torch.float16, torch.float32), (torch.float16, torch.float16)])
@pytest.mark.parametrize("G,rs,rd,blocks,cs,cd", [(1, 1, 1, 1, 1, 1), (4, 5, 8, 1, 7, 16), (4, 8, 5, 2, 16, 9), (3, 33, 33, 2, 65, 65), (4, 1, 1, 1, 257, 288)])
def test_padding_cutting_and_converting_copies(G, rs, rd, blocks, cs, cd, src, dst):
    a = torch.randn(G, rs, blocks, cs, device="cuda").to(src)
    out, zero = (torch.full((G, rd, blocks, cd), 7.0, device="cuda", dtype=dst) for _ in range(2))
    c = layers._Copies()
    c.matrix(a.data_ptr(), out.data_ptr(), G, (rs, rd), (cs, cd), CODE[src] + 16 * CODE[dst], blocks=blocks)
    c.matrix(None, zero.data_ptr(), G, (rs, rd), (cs, cd), CODE[src] + 16 * CODE[dst], blocks=blocks)
    c.run(_Ctx())
    want = torch.zeros_like(out)
    r, k = min(rs, rd), min(cs, cd)
    want[:, :r, :, :k] = a[:, :r, :, :k].to(dst)
    assert torch.equal(out, want) and not zero.any()


@pytest.mark.parametrize("n", [1, 40])   # (40 copies: more than one launch)
def test_row_modes_of_the_copies(n):
    T, B, I = 7, 5, 11
    lens = torch.tensor([7, 7, 4, 2, 1])
    sizes = torch.tensor([int((lens > t).sum()) for t in range(T)])
    offs = torch.cumsum(sizes, 0) - sizes
    order = torch.tensor([3, 0, 4, 1, 2], device="cuda")
    packed, padded = torch.randn(int(sizes.sum()), I, device="cuda"), torch.randn(T, B, I, device="cuda")
    ints = torch.cat((lens, offs)).int().cuda()
    ctx = _Ctx(T, B, ints[:B], ints[B:], order)
    f32 = CODE[torch.float32] * 17
    outs = [torch.full((T, B, 16), 7.0, device="cuda") for _ in range(n)]
    back, last, state = torch.zeros_like(packed), torch.zeros(B, I, device="cuda"), torch.zeros(B, I, device="cuda")
    c = layers._Copies()
    for o in outs:
        c.rows(packed.data_ptr(), layers.PACKED_REVERSED, I, o.data_ptr(), layers.PADDED, 16, (I, 16), f32)
    c.rows(padded.data_ptr(), layers.REVERSED, I, back.data_ptr(), layers.PACKED, I, (I, I), f32, packed.data_ptr(), layers.PACKED, I)
    c.rows(padded.data_ptr(), layers.LAST, I, last.data_ptr(), layers.ORDERED, I, (I, I), f32)
    c.run(ctx)
    c = layers._Copies()   # (reads what the first launch wrote)
    c.rows(last.data_ptr(), layers.ORDERED, I, state.data_ptr(), layers.BATCH, I, (I, I), f32)
    c.run(ctx)
    for b in range(B):
        ln = int(lens[b])
        for t in range(T):
            row = packed[int(offs[ln - 1 - t]) + b] if t < ln else torch.zeros(I, device="cuda")
            assert all(torch.equal(o[t, b, :I], row) and not o[t, b, I:].any() for o in outs)
            if t < ln:
                assert torch.equal(back[int(offs[t]) + b], padded[ln - 1 - t, b] + packed[int(offs[t]) + b])
        assert torch.equal(last[int(order[b])], padded[ln - 1, b]) and torch.equal(state[b], padded[ln - 1, b])


@pytest.mark.parametrize("kw,T,B,I,H,dt,autocast,packed", [
    (dict(num_layers=2), 35, 20, 90, 150, torch.float32, torch.bfloat16, False),              # converted and padded parameters
    (dict(num_layers=2, bidirectional=True), 40, 12, 50, 100, torch.float16, None, True),     # both directions between layers, packed
    (dict(num_layers=3, bias=False, batch_first=True), 33, 9, 24, 65, torch.float32, None, False),
    (dict(num_layers=2), 130, 16, 64, 512, torch.float16, None, True),                        # a wavefront of two layers, packed
    (dict(), 12, 5, 16, 48, torch.float32, torch.float16, False),
])
def test_one_node_call_against_the_layer_loop(kw, T, B, I, H, dt, autocast, packed, monkeypatch):
    torch.manual_seed(T)
    m = FastLSTM(I, H, **kw).to("cuda", dt)
    D = 2 if kw.get("bidirectional") else 1
    x = torch.randn(*((B, T) if kw.get("batch_first") else (T, B)), I, device="cuda").to(dt)
    if packed:
        lengths = torch.randint(1, T + 1, (B,))
        lengths[B // 2] = T
        x = pack_padded_sequence(x, lengths, enforce_sorted=False)
    s = tuple((torch.randn(m.num_layers * D, B, H, device="cuda") * 0.3).to(dt) for _ in range(2))
    plan, taken, results = layers.plan, [], []
    for node in (False, True):
        monkeypatch.setattr(layers, "plan", (lambda *a: (taken.append(plan(*a)), taken[-1])[1]) if node else (lambda *a: None))
        m.zero_grad(set_to_none=True)
        leaf = (x.data if packed else x).detach().clone().requires_grad_(True)
        st = tuple(t.clone().requires_grad_(True) for t in s)
        arg = PackedSequence(leaf, x.batch_sizes, x.sorted_indices, x.unsorted_indices) if packed else leaf
        with torch.autocast("cuda", dtype=autocast or torch.float16, enabled=autocast is not None):
            y, (h, c) = m(arg, st)
        y = y.data if packed else y
        w = torch.randn(y.shape, generator=torch.Generator("cuda").manual_seed(3), device="cuda").to(y.dtype)
        loss = (y * w).sum() + (h.float().sum() if packed else 0.0)   # (packed: h_n carries a gradient)
        loss.backward()
        results.append([y, h, c, leaf.grad, st[0].grad, st[1].grad] + [p.grad for p in m.parameters()])
    assert taken and taken[0] is not None
    tol = 2e-5 if (autocast or dt) == torch.float32 else 1.2e-2
    for a, b in zip(*results):
        assert a.shape == b.shape and a.dtype == b.dtype
        assert (a.float() - b.float()).abs().max() <= tol * a.float().abs().max()


def test_backward_passes_over_one_graph_do_not_share_state(monkeypatch):
    """A second backward pass over a retained graph while the first is under way (here: from inside its first layer) leaves the
    first one's tensors alone."""
    torch.manual_seed(0)
    m = FastLSTM(24, 72, num_layers=3, bidirectional=True).cuda()
    x = torch.randn(9, 6, 24, device="cuda", requires_grad=True)
    assert layers.plan(m, x, None) is not None
    y, _ = m(x)
    inputs, dout = [x, *m.parameters()], torch.randn_like(y)
    want = torch.autograd.grad(y, inputs, dout, retain_graph=True)
    names, inner = ("lstm_persistent_bwd", "lstm_persistent_bwd_pair"), []

    def nested(call):
        def run(*args, **kw):
            r = call(*args, **kw)
            if not inner:
                inner.append(None)
                inner[0] = torch.autograd.grad(y, inputs, dout, retain_graph=True)
            return r
        return run

    for name in names:
        monkeypatch.setattr(L, name, nested(getattr(L, name)))
    got = torch.autograd.grad(y, inputs, dout, retain_graph=True)
    assert inner
    for a, b, c in zip(want, got, inner[0]):
        assert torch.equal(a, b) and torch.equal(a, c)


def test_sorted_indices_changed_in_place_after_forward_are_an_error():
    m = FastLSTM(24, 72, num_layers=2).cuda()
    x = pack_padded_sequence(torch.randn(7, 4, 24, device="cuda"), torch.tensor([3, 7, 5, 1]), enforce_sorted=False)
    assert layers.plan(m, x, None) is not None
    y, _ = m(x)
    x.sorted_indices.copy_(torch.arange(4, device="cuda"))
    with pytest.raises(RuntimeError, match="inplace"):
        y.data.sum().backward()


@pytest.mark.parametrize("grads,kw,name", [(False, dict(num_layers=2), "weight_hh_l1"), (False, dict(), "bias_ih_l0"), (True, dict(num_layers=2), "weight_ih_l1"),
                                           (True, dict(num_layers=2, bidirectional=True), "weight_hh_l0_reverse")])
def test_parameters_of_another_shape_are_refused(grads, kw, name):
    """A parameter replaced by one of another shape: no form that takes addresses reads past it."""
    m = FastLSTM(24, 72, **kw).cuda()
    x = torch.randn(2, 3, 24, device="cuda")
    with torch.set_grad_enabled(grads):
        m(x)
        old = getattr(m, name)
        setattr(m, name, torch.nn.Parameter(torch.zeros(*old.shape[:-1], old.shape[-1] // 2, device="cuda")))
        assert layers.plan(m, x, None) is None and (grads or m._forward_short(x, None) is None)
        with pytest.raises((AssertionError, RuntimeError)):
            m(x)
