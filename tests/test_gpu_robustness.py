"""Robustness of the boundary (run with -m gpu): gradients that autograd does not ask for are not computed,
recurrent calls from several streams are ordered by the library, a failed launch shows in its own results,
and the host-side dispatch caches follow the kernel-family switch."""
import ctypes

import pytest
import torch

import fastlstm_amd
import fastlstm_amd.lstm as L
from fastlstm_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _clean_state():
    yield
    lib = _lib.load()
    lib.fastlstm_set_spin_limit(400000000)
    lib.fastlstm_set_kernel_families(7)
    torch.cuda.synchronize()
    lib.fastlstm_device_status(0, 1)


def _module(I, H, layers, dt, seed, **kw):
    torch.manual_seed(seed)
    return fastlstm_amd.FastLSTM(I, H, num_layers=layers, dtype=dt, **kw).cuda()


# T, B, I, H, layers, dtype, keyword arguments:
#   the dx / dW products inside the reverse launch (idle CUs), as launches behind it, fp32 general kernels,
#   two layers in one launch each way, a wavefront of three layers, both directions side by side
PRUNE_CASES = [(96, 64, 1024, 1024, 1, torch.float16, {}),
               (64, 128, 512, 512, 1, torch.bfloat16, {}),
               (20, 16, 48, 160, 1, torch.float32, {}),
               (128, 32, 256, 1024, 2, torch.float16, {}),
               (128, 16, 96, 256, 3, torch.float16, {}),
               (64, 32, 128, 256, 1, torch.float16, {"bidirectional": True})]


@pytest.mark.parametrize("T,B,I,H,layers,dt,kw", PRUNE_CASES)
def test_gradient_of_the_input_is_computed_only_when_asked_for(T, B, I, H, layers, dt, kw):
    """x.requires_grad = False: autograd's needs_input_grad reaches the library as a null dx, the product
    d_ifgo . Wx of the lowest layer is skipped (inside the fused launch and outside it), x.grad stays None and
    every parameter gradient is the same bits as with the product computed."""
    m = _module(I, H, layers, dt, 3, **kw)
    g = torch.Generator().manual_seed(5)
    x0 = torch.randn(T, B, I, generator=g).to(dt).cuda()
    dout = torch.randn(T, B, H * (2 if kw.get("bidirectional") else 1), generator=g).to(dt).cuda()
    grads = []
    for want_dx in (True, False):
        m.zero_grad(set_to_none=True)
        x = x0.clone().requires_grad_(want_dx)
        y, _ = m(x)
        (y * dout).sum().backward()
        torch.cuda.synchronize()
        assert (x.grad is not None) == want_dx
        if want_dx:
            assert torch.isfinite(x.grad.float()).all() and x.grad.abs().max() > 0
        grads.append({n: p.grad.clone() for n, p in m.named_parameters()})
    assert fastlstm_amd.pending_status() == _lib.OK
    for n in grads[0]:
        assert torch.equal(grads[0][n], grads[1][n]), n


def test_null_dx_and_null_weight_gradients_through_the_c_abi():
    """fastlstm_bwd_layer with dx = NULL / with dWx = dWh = db = NULL: the other results are the bits of the full call."""
    T, B, I, H, dt = 96, 64, 1024, 1024, torch.float16
    g = torch.Generator().manual_seed(11)
    k = 1.0 / H ** 0.5
    u = lambda *s: ((torch.rand(*s, generator=g) * 2 - 1) * k).to(dt).cuda()
    x = torch.randn(T, B, I, generator=g).to(dt).cuda()
    Wx, bx, Wh, bh = u(4 * H, I), u(4 * H), u(4 * H, H), u(4 * H)
    dout = torch.randn(T, B, H, generator=g).to(dt).cuda()
    out, cell, ifgo = L.lstm_persistent_fwd(x, None, None, Wx, bx, Wh, bh)
    z = lambda: torch.zeros(B, H, device="cuda", dtype=dt)
    full = L.lstm_persistent_bwd(dout, z(), z(), x, out, cell, ifgo, Wx, Wh)
    no_dx = L.lstm_persistent_bwd(dout, z(), z(), x, out, cell, ifgo, Wx, Wh, need_dx=False)
    no_dw = L.lstm_persistent_bwd(dout, z(), z(), x, out, cell, ifgo, Wx, Wh, need_dw=False)
    torch.cuda.synchronize()
    assert no_dx[0] is None and all(t is None for t in no_dw[3:])
    for k_ in (1, 2, 3, 4, 5):
        assert torch.equal(full[k_], no_dx[k_]), k_
    for k_ in (0, 1, 2):
        assert torch.equal(full[k_], no_dw[k_]), k_
    # a null weight gradient next to the others is an argument error, not a silent skip
    lib = _lib.load()
    t = torch.zeros(64, device="cuda", dtype=dt)
    p = t.data_ptr()
    rc = lib.fastlstm_bwd_layer(p, p, p, p, p, p, p, p, p, p, p, p, None, p, p, 1 << 20, p, 1 << 20, 4, 16, 64, 64, 1,
                                torch.cuda.current_stream().cuda_stream)
    assert rc == _lib.ERR_NULL


def test_recurrent_calls_from_two_streams_are_ordered_by_the_library():
    """Two forward + backward passes of a shape whose time loop holds half the device, issued from two streams
    with nothing between them: the library makes each recurrent call wait for the one before it on the other
    stream (an event per device), so neither starves the other until the time-out, and the results are the bits
    of the same passes run one after the other."""
    T, B, I, H, dt = 128, 64, 512, 1024, torch.float16
    mods = [_module(I, H, 1, dt, 20 + i) for i in range(2)]
    g = torch.Generator().manual_seed(9)
    xs = [torch.randn(T, B, I, generator=g).to(dt).cuda() for _ in range(2)]
    douts = [torch.randn(T, B, H, generator=g).to(dt).cuda() for _ in range(2)]

    def one(i):
        mods[i].zero_grad(set_to_none=True)
        x = xs[i].clone().requires_grad_(True)
        y, (hn, cn) = mods[i](x)
        (y * douts[i]).sum().backward()
        return [y.detach(), hn, cn, x.grad] + [p.grad for p in mods[i].parameters()]

    serial = [[t.clone() for t in one(i)] for i in range(2)]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for s in streams:
        s.wait_stream(torch.cuda.current_stream())
    got = [None, None]
    for rep in range(3):   # several rounds: the passes of the two streams interleave differently each time
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                got[i] = one(i)
    for s in streams:
        s.synchronize()
    torch.cuda.synchronize()
    assert fastlstm_amd.pending_status() == _lib.OK
    for i in range(2):
        for a, b in zip(serial[i], got[i]):
            assert torch.equal(a, b), i


def test_a_failed_launch_shows_in_its_own_results_and_in_pending_status():
    """Failure path forced from the host (a spin limit of one tick; every kernel still exits normally): the
    failing calls return success, their results hold NaN, pending_status reports the failure without a
    synchronisation of its own, and the module raises before it enqueues new work behind it."""
    lib = _lib.load()
    T, B, I, H, dt = 64, 16, 128, 512, torch.float16
    m = _module(I, H, 1, dt, 1)
    x = torch.randn(T, B, I, device="cuda").to(dt).requires_grad_(True)
    y, _ = m(x)
    torch.cuda.synchronize()
    assert torch.isfinite(y.float()).all() and fastlstm_amd.pending_status() == _lib.OK
    try:
        lib.fastlstm_set_spin_limit(1)
        y, (hn, cn) = m(x)           # returns normally: nothing synchronises
        torch.cuda.synchronize()
    finally:
        lib.fastlstm_set_spin_limit(400000000)
    assert torch.isnan(y[-1].float()).all() and torch.isnan(hn.float()).all() and torch.isnan(cn.float()).all()
    assert not torch.isfinite(y.float().sum())          # any loss over the output trips
    assert fastlstm_amd.pending_status() == _lib.ERR_TIMEOUT      # (reading does not clear)
    with pytest.raises(RuntimeError):
        m(x)                          # reported before new work is enqueued; the report is cleared
    assert fastlstm_amd.pending_status() == _lib.OK
    y, _ = m(x)                       # healthy again
    y.float().sum().backward()
    torch.cuda.synchronize()
    assert torch.isfinite(y.float()).all() and torch.isfinite(x.grad.float()).all()
    # the reverse pass: a failed launch poisons dh_0, dc_0, db and the first timestep of dx
    out, cell, ifgo = L.lstm_persistent_fwd(x.detach(), None, None, m.weight_ih_l0.detach(), m.bias_ih_l0.detach(),
                                            m.weight_hh_l0.detach(), m.bias_hh_l0.detach())
    torch.cuda.synchronize()
    z = lambda: torch.zeros(B, H, device="cuda", dtype=dt)
    try:
        lib.fastlstm_set_spin_limit(1)
        r = L.lstm_persistent_bwd(torch.randn(T, B, H, device="cuda").to(dt), z(), z(), x.detach(), out, cell, ifgo,
                                  m.weight_ih_l0.detach(), m.weight_hh_l0.detach())
        torch.cuda.synchronize()
    finally:
        lib.fastlstm_set_spin_limit(400000000)
    assert torch.isnan(r[0][0].float()).all() and torch.isnan(r[1].float()).all() and torch.isnan(r[4].float()).all()
    assert fastlstm_amd.pending_status(clear=True) == _lib.ERR_TIMEOUT
    assert fastlstm_amd.pending_status() == _lib.OK


def test_dispatch_caches_follow_the_kernel_family_switch():
    """The host caches of which kernel a shape gets (and with them the padding and wavefront decisions) are keyed
    on the family mask: a switch changes the answer at once, and switching back restores it."""
    lib = _lib.load()
    code = L._DTYPE_CODE[torch.float16]
    assert lib.fastlstm_get_kernel_families() == 7
    assert L._recurrent_kind(64, 16, 512, code, 0) == 1
    chunks = L.stack_wavefront_chunks(2, 256, 16, 512, torch.float16, "cuda:0")
    assert chunks > 0
    lib.fastlstm_set_kernel_families(0)
    assert L._recurrent_kind(64, 16, 512, code, 0) == 0
    assert L.stack_wavefront_chunks(2, 256, 16, 512, torch.float16, "cuda:0") == 0
    lib.fastlstm_set_kernel_families(7)
    assert L._recurrent_kind(64, 16, 512, code, 0) == 1
    assert L.stack_wavefront_chunks(2, 256, 16, 512, torch.float16, "cuda:0") == chunks


def test_padded_operand_cache_is_opt_in_and_follows_the_version_counters():
    """Inference with a hidden size that runs zero-padded: with cache_padded_operands the padded weights are kept
    across calls and refreshed when a parameter's version counter moves (an optimizer-style in-place update)."""
    T, B, I, H, dt = 40, 16, 300, 300, torch.float16
    m = _module(I, H, 1, dt, 7)
    x = torch.randn(T, B, I, device="cuda").to(dt)
    with torch.no_grad():
        assert m._operand_padding(x) is not None        # this shape is padded
        y0 = m(x)[0].clone()
        assert not m.__dict__.get("_padded_operand_cache")    # off by default: nothing kept
        m.cache_padded_operands = True
        y1 = m(x)[0].clone()
        kept = m._padded_operand_cache
        assert len(kept) == 1 and torch.equal(y0, y1)
        first = next(iter(kept.values()))[1][0]
        y2 = m(x)[0].clone()
        assert next(iter(kept.values()))[1][0] is first and torch.equal(y1, y2)    # reused
        m.weight_hh_l0.mul_(0.5)                          # bumps the version counter
        y3 = m(x)[0].clone()
        assert next(iter(kept.values()))[1][0] is not first
        m.cache_padded_operands = False
        assert torch.equal(y3, m(x)[0]) and not torch.equal(y3, y2)


@pytest.mark.parametrize("dt", [torch.float32, torch.float16])
@pytest.mark.parametrize("T,B,H", [(5, 7, 48), (5, 7, 64), (5, 7, 72), (5, 20, 256), (5, 70, 1024), (3, 5, 2100), (1, 4, 96)])
def test_a_nan_of_the_input_reaches_the_results(T, B, H, dt):
    """x[t, b] = NaN: out of that row is NaN from step t on and so are its last states, on every kernel family (and in the
    gradients of the row); all other rows keep their bits."""
    m = _module(24, H, 1, dt, 4)
    x = torch.randn(T, B, 24, generator=torch.Generator().manual_seed(2)).to(dt).cuda()
    t, b, others = T // 2, B - 2, [r for r in range(B) if r != B - 2]
    bad = x.clone()
    bad[t, b, 5] = float("nan")

    def run(x, grads):
        if not grads:
            with torch.no_grad():
                y, (h, c) = m(x)
            return [y, h, c]
        x = x.clone().requires_grad_(True)
        y, (h, c) = m(x)
        y.sum().backward()
        return [y.detach(), h, c, x.grad]

    for grads in (False, True):
        want, got = run(x, grads), run(bad, grads)
        for w, g in zip(want, got):
            assert torch.equal(w[:, others], g[:, others])
        assert torch.equal(want[0][:t, b], got[0][:t, b])
        assert got[0][t:, b].isnan().all() and all(g[0, b].isnan().all() for g in got[1:3])
        if grads:
            assert got[3][:, b].isnan().all()
    assert fastlstm_amd.pending_status() == _lib.OK


@pytest.mark.parametrize("H", [64, 256])
def test_saturated_fp32_gates(H):
    """Pre-activations from -1e4 to 1e4, where the exponential is 0 or inf: forward and backward against nn.LSTM in 64 bits."""
    m = _module(8, H, 1, torch.float32, 6)
    ref = torch.nn.LSTM(8, H).double()
    ref.load_state_dict({k: v.double().cpu() for k, v in m.state_dict().items()})
    x = torch.randn(6, 5, 8, generator=torch.Generator().manual_seed(1)) * torch.logspace(0, 5, 6)[:, None, None]
    a, b = x.cuda().requires_grad_(True), x.double().requires_grad_(True)
    (y, _), (z, _) = m(a), ref(b)
    y.sum().backward()
    z.sum().backward()
    # fp32 rounding of a sum of eight terms of 1e4 / 3 is about 1e-3, and a gate that is not saturated takes it with a slope of up to 1
    torch.testing.assert_close(y.double().cpu(), z, rtol=2e-3, atol=2e-3)
    torch.testing.assert_close(a.grad.double().cpu(), b.grad, rtol=2e-3, atol=2e-3)


@pytest.mark.parametrize("T,B,I,H,dt", [(6, 20, 32, 256, torch.float32),       # four waves, a ragged second group
                                        (5, 9, 32, 80, torch.float32),
                                        (6, 20, 32, 1024, torch.float16),      # eight waves, K split eight ways
                                        (6, 40, 32, 512, torch.bfloat16),
                                        (5, 300, 32, 256, torch.float16),      # groups of 32 rows
                                        (4, 200, 32, 1024, torch.bfloat16),    # ... LDS-direct tiles
                                        (96, 64, 1024, 1024, torch.float16)])  # products inside the launches
def test_values_that_look_like_an_unwritten_exchange_word(T, B, I, H, dt):
    """The XCD-local kernels mark exchange words as unwritten with all ones, which in h_0 or in a gradient is a NaN like any
    other: it ends no launch and stays in its batch row, whose results are NaN; every other row keeps its bits."""
    g = torch.Generator().manual_seed(H + B)
    k = 1.0 / H ** 0.5
    u = lambda *s: ((torch.rand(*s, generator=g) * 2 - 1) * k).to(dt).cuda()
    n = lambda *s: torch.randn(*s, generator=g).to(dt).cuda()
    x, h0, c0, dout = n(T, B, I), u(B, H), u(B, H), n(T, B, H)
    Wx, bx, Wh, bh = u(4 * H, I), u(4 * H), u(4 * H, H), u(4 * H)
    ones = torch.full((H,), -1, device="cuda", dtype=torch.int32 if dt == torch.float32 else torch.int16).view(dt)
    rows, others = [3, B - 1], [b for b in range(B) if b not in (3, B - 1)]
    z = lambda: torch.zeros(B, H, device="cuda", dtype=dt)
    out, cell, ifgo = L.lstm_persistent_fwd(x, h0, c0, Wx, bx, Wh, bh)
    clean = L.lstm_persistent_bwd(dout, z(), z(), x, out, cell, ifgo, Wx, Wh)
    bad_h, bad_dout, at = h0.clone(), dout.clone(), T // 2
    bad_h[rows], bad_dout[at, rows] = ones, ones
    got = L.lstm_persistent_fwd(x, bad_h, c0, Wx, bx, Wh, bh)
    grads = L.lstm_persistent_bwd(bad_dout, z(), z(), x, out, cell, ifgo, Wx, Wh)
    torch.cuda.synchronize()
    assert fastlstm_amd.pending_status() == _lib.OK
    for a, b in zip(got, (out, cell, ifgo)):
        assert torch.equal(a[:, others], b[:, others])
    assert got[0][1:, rows].isnan().all() and got[1][1:, rows].isnan().all()
    for a, b in zip(grads[:3], clean[:3]):
        assert torch.equal(a.view(-1, B, a.shape[-1])[:, others], b.view(-1, B, b.shape[-1])[:, others])
    assert grads[0][:at + 1, rows].isnan().all() and grads[1][rows].isnan().all() and grads[2][rows].isnan().all()
    assert torch.equal(grads[0][at + 1:], clean[0][at + 1:])


@pytest.mark.parametrize("H,rows,members", [(1024, 16, 32), (2048, 32, 32), (96, 64, 8)])
def test_step_probe_ends_in_every_mode(H, rows, members):
    """fastlstm_diag_step_probe, on a workspace whose exchange slots hold anything: every mode ends and reports no time-out."""
    lib, steps = _lib.load(), 20
    n = lib.fastlstm_diag_step_probe_bytes(steps, H, rows)
    for kind, mode in ((0, 0), (0, 1), (0, 2), (0, 3), (0, 4), (1, 0), (1, 1), (1, 2)):
        ws = torch.randint(0, 256, (n,), dtype=torch.uint8, device="cuda")
        ws[:70000].zero_()
        assert lib.fastlstm_diag_step_probe(kind, mode, members, H, rows, steps, ws.data_ptr(), n, torch.cuda.current_stream().cuda_stream) == _lib.OK
        torch.cuda.synchronize()
        assert lib.fastlstm_ws_status(ws[:64].cpu().numpy().tobytes()) == _lib.OK, (kind, mode)
    assert lib.fastlstm_diag_step_probe(0, 3, 16, 96, 16, steps, ws.data_ptr(), n, None) == _lib.ERR_DIM   # six units per member


class _KernelNode(ctypes.Structure):   # hipKernelNodeParams
    _fields_ = [("block", ctypes.c_uint * 3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p), ("grid", ctypes.c_uint * 3),
                ("args", ctypes.c_void_p), ("shared", ctypes.c_uint)]


def _captured_kernels(call):
    """The functions of the kernels that call() enqueues on the current stream, in order (captured, not run)."""
    hip = _lib.load()   # (its handle finds the functions of the runtime that it is linked with)
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        call()
    raw, n = ctypes.c_void_p(graph.raw_cuda_graph()), ctypes.c_size_t(0)
    assert hip.hipGraphGetNodes(raw, None, ctypes.byref(n)) == 0
    nodes = (ctypes.c_void_p * n.value)()
    assert hip.hipGraphGetNodes(raw, nodes, ctypes.byref(n)) == 0
    funcs = []
    for node in nodes:
        params = _KernelNode()
        assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(params)) == 0   # (kernels only)
        funcs.append(params.func)
    return funcs


@pytest.mark.parametrize("B,H,dt,backward", [(65, 4096, torch.bfloat16, 1),    # teams of whole-CU kernels, two launches
                                             (150, 2560, torch.float16, 1),    # ... three
                                             (65, 1280, torch.float32, 1),     # ... of half unit tiles
                                             (129, 2048, torch.bfloat16, 1),   # ... groups of 32 rows
                                             (300, 1024, torch.float16, 0),    # XCD-local kernels
                                             (300, 1024, torch.float16, 1)])
def test_launches_over_row_ranges_start_from_a_clean_header(B, H, dt, backward):
    """Workgroups of a launch compare the XCD that they run on with what the first one wrote down (check_xcd_placement), which
    is the same within ONE launch: between two that share a workspace something clears it."""
    lib, T, code = _lib.load(), 1, {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}[dt]
    plan = _lib.Plan()
    _lib.check(lib.fastlstm_plan_device(0, B, H, code, backward, plan), "plan")
    n = lib.fastlstm_recurrent_workspace_bytes(plan, T, H, code, backward)
    ws = torch.zeros(n, dtype=torch.uint8, device="cuda")
    z = lambda *shape: torch.zeros(shape, device="cuda", dtype=dt)
    dout, dh, dc, ifgo, cell, d_ifgo, out, Wh = z(T, B, H), z(B, H), z(B, H), z(T, B, 4 * H), z(T + 1, B, H), z(T, B, 4 * H), z(T + 1, B, H), z(4 * H, H)
    operands = (dout, dh, dc, ifgo, cell, d_ifgo, Wh) if backward else (ifgo, out, cell, Wh)
    entry = lib.fastlstm_bwd_persistent if backward else lib.fastlstm_fwd_persistent
    torch.cuda.synchronize()
    kernels = _captured_kernels(lambda: _lib.check(entry(*(t.data_ptr() for t in operands), ws.data_ptr(), n, T, B, H, code,
                                                         torch.cuda.current_stream().cuda_stream), "recurrence"))
    assert len(kernels) >= 4 and len(kernels) % 2 == 0   # launch, (clearing, launch) ..., the status
    clearing = set(kernels[1:-1:2])
    assert len(clearing) == 1 and not clearing & set(kernels[0::2]) and kernels[-1] not in kernels[:-1]
