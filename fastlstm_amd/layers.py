"""All layers of a FastLSTM call as one autograd node, and what surrounds them as one launch per stage.

The layer loop of the reference (fastlstm/lstm.py:685-698) with its casts (:509-515) makes every layer, cast, padding,
reversal and gradient accumulation a node and at least one launch of its own; a short call of a module whose parameters
have to be converted or padded, or whose sequences are packed, was bound by that (2 layers, T = 35, B = 20,
I = H = 650 under bf16 autocast: 78 launches).  Here

    parameters, input and initial states   -> operands in the compute type and the kernels' sizes   one copy launch
    the layers                             -> the host functions of lstm.py, as FastLSTM.forward calls them
    top layer's h, last states             -> results in the caller's sizes, order and packing         one copy launch

and backward the same from the gradient of the result to the gradients of the inputs.  The copies are
fastlstm_copy_blocks descriptors: zero-padding, type conversion, packing, time reversal and addition in one.
"""
import ctypes

import numpy as np
import torch
from torch.nn.utils.rnn import PackedSequence

from . import _lib
from . import lstm as L

# row modes of fastlstm_copy_blocks
PADDED, REVERSED, PACKED, PACKED_REVERSED, LAST, ORDERED, BATCH = range(1, 8)


class _Copies:
    """Descriptors of one fastlstm_copy_blocks call."""

    def __init__(self):
        self.fields, self.n = [], 0

    def matrix(self, src, dst, groups, rows, cols, types, blocks=1):
        """rows / cols: (source, destination) per group / per block; src None: zeros."""
        self.n += 1
        self.fields += (src or 0, 0, dst, 0, 0, 0, groups, rows[0], rows[1], blocks, cols[0], cols[1], blocks * cols[0], 0,
                        blocks * cols[1], types)

    def rows(self, src, mode, ld, dst, dmode, dld, cols, types, src2=0, mode2=0, ld2=0):
        self.n += 1
        self.fields += (src or 0, src2, dst, mode, mode2, dmode, 0, 0, 0, 1, cols[0], cols[1], ld, ld2, dld, types)

    def run(self, at):
        if self.n:
            _lib.check(_lib.load().fastlstm_copy_blocks(
                self.n, (ctypes.c_longlong * len(self.fields))(*self.fields), at.T, at.B, at.lens, at.offs, at.order, at.stream),
                "fastlstm_copy_blocks")


class _Pass:
    """What the copy launches of one pass (forward, or one of several backward passes) take besides their descriptors."""
    __slots__ = ("T", "B", "lens", "offs", "order", "stream")

    def __init__(self, c, order, stream):
        self.T, self.B, self.lens, self.offs, self.stream = c.T, c.B, c.lens, c.offs, stream
        self.order = None if order is None else order.data_ptr()


class _Call:
    """Sizes and options of one call.  Written by plan() and forward() alone: the graph's node keeps it, and several threads may
    run backward over one graph."""
    __slots__ = ("T", "B", "I", "H", "Hp", "Ip", "L", "D", "dt", "code", "es", "device", "packed", "N", "lens", "offs",
                 "index_memory", "copy_weights", "copy_x", "bias", "x_dtype", "held", "states", "groups")

    def view(self, base, offset, shape):
        strides, n = [], 1
        for s in reversed(shape):
            strides.append(n)
            n *= s
        return base.as_strided(shape, strides[::-1], offset)


def plan(module, x, h_c_0):
    """The _Call of FastLSTM.forward(x, h_c_0), or None where the module's own loop handles it: gradients through the
    final states, dropout between layers, kept padded operands, unusual arguments -- and a single plain layer, which is one
    node anyway."""
    packed = isinstance(x, PackedSequence)
    data = x.data if packed else x
    if type(data) is not torch.Tensor or not data.is_cuda or data.dim() != (2 if packed else 3):
        return None
    if module.state_grads or module.cache_padded_operands or (module.training and module.dropout and module.num_layers > 1):
        return None
    autocast, padding = torch.is_autocast_enabled(), module._operand_padding(x)
    if module.num_layers == 1 and padding is None and not (packed or autocast or module.bidirectional):
        p = module._parameters.get("weight_ih_l0")
        if p is not None and p.dtype is data.dtype:
            return None   # (nothing around the layer: before the rest is looked at, 5 of 60 us of the host time of such a call)
    c = _Call()
    c.dt = torch.get_autocast_dtype("cuda") if autocast else data.dtype
    if c.dt not in L._DTYPE_CODE or data.dtype not in L._DTYPE_CODE or data.shape[-1] != module.input_size:
        return None
    params = module._operand_list()
    c.held = params[0].dtype
    idx = data.get_device()
    shapes = L._parameter_shapes(module.num_layers, 2 if module.bidirectional else 1, module.input_size, module.hidden_size, module.bias)
    for p, (_, shape) in zip(params, shapes):
        if p.dtype != c.held or p.get_device() != idx or p.shape != shape or not p.is_contiguous():
            return None
    if c.held not in L._DTYPE_CODE or (c.held != c.dt and not autocast):
        return None
    c.L, c.D, c.H, c.I, c.bias, c.packed = module.num_layers, 2 if module.bidirectional else 1, module.hidden_size, module.input_size, module.bias, packed
    if packed:
        c.T, c.B, c.N = x.batch_sizes.numel(), int(x.batch_sizes[0]), data.shape[0]
        order = x.sorted_indices
        if order is not None and (order.dtype != torch.int64 or order.get_device() != idx or order.numel() != c.B or not order.is_contiguous()):
            return None
    else:
        c.T, c.B = (data.shape[1], data.shape[0]) if module.batch_first else (data.shape[0], data.shape[1])
        c.N = c.T * c.B
    c.states = None
    if h_c_0 is not None:
        h_0, c_0 = h_c_0
        for t in (h_0, c_0):
            if type(t) is not torch.Tensor or t.shape != (c.L * c.D, c.B, c.H) or t.get_device() != idx or t.dtype not in L._DTYPE_CODE:
                return None
        c.states = (h_0.dtype, c_0.dtype)
    c.Hp, c.Ip = padding or (c.H, c.I)
    c.code = L._DTYPE_CODE[c.dt]
    c.copy_weights = c.held != c.dt or c.Hp != c.H or c.Ip != c.I
    if c.copy_weights and c.dt != torch.float32 and not (c.Hp <= 64 and c.I <= 64 and c.I % 16 == 0):
        c.Ip = -(-c.I // 64) * 64   # the weights are rewritten anyway: whole k-tiles for the first layer's products, however few rows
    c.copy_x = packed or c.Ip != c.I or data.dtype != c.dt
    if not (c.copy_weights or c.copy_x or c.D == 2 or c.L > 1):
        return None
    if packed and module._packed_range_rows_of(x, c.Hp):
        return None   # a batch of several launches, each range of rows to its own length
    c.es = 4 if c.dt == torch.float32 else 2
    c.device, c.x_dtype = data.device, data.dtype
    c.lens = c.offs = c.index_memory = None
    return c


def _upload_lengths(c, x, stream):
    """Row lengths and first packed rows on the device, through the arguments of a launch."""
    sizes = x.batch_sizes.numpy()
    ints = np.empty(c.B + c.T, dtype=np.int32)
    ints[:c.B] = np.searchsorted(-sizes, -np.arange(c.B), side="left")   # steps t with sizes[t] > b
    ints[c.B] = 0
    np.cumsum(sizes[:-1], out=ints[c.B + 1:])
    dev = torch.empty(c.B + c.T, dtype=torch.int32, device=c.device)
    _lib.check(_lib.load().fastlstm_upload_ints(ints.ctypes.data, ints.size, dev.data_ptr(), stream), "fastlstm_upload_ints")
    c.lens, c.offs, c.index_memory = dev.data_ptr(), dev.data_ptr() + 4 * c.B, dev


def _weights(c, copies, params):
    """[(Wx, bx, Wh, bh)] per layer and direction in the compute type and padded sizes (converted by `copies`)."""
    H, Hp, D, per = c.H, c.Hp, c.D, 4 if c.bias else 2
    zero = None
    if not c.copy_weights:
        if c.bias:
            return [tuple(params[i:i + 4]) for i in range(0, len(params), 4)]
        zero = torch.zeros(4 * H, dtype=c.dt, device=c.device)
        return [(params[i], zero, params[i + 1], zero) for i in range(0, len(params), 2)]
    up = lambda n: -(-n // 8) * 8                      # every operand on 16 bytes
    sizes = [4 * Hp * (c.Ip if k < D else D * Hp) for k in range(c.L * D)]
    total = sum(up(s) + 2 * up(4 * Hp) + up(4 * Hp * Hp) for s in sizes)
    buf = torch.empty(total, dtype=c.dt, device=c.device)
    base, at, out = buf.data_ptr(), 0, []
    types = L._DTYPE_CODE[c.held] + 16 * c.code
    for k in range(c.L * D):
        Wx, bx, Wh, bh = params[per * k:per * k + 4] if c.bias else (params[2 * k], None, params[2 * k + 1], None)
        K = c.Ip if k < D else D * Hp
        views = []
        for src, n, shape in ((Wx, 4 * Hp * K, (4 * Hp, K)), (bx, 4 * Hp, (4 * Hp,)), (Wh, 4 * Hp * Hp, (4 * Hp, Hp)), (bh, 4 * Hp, (4 * Hp,))):
            dst, ptr = base + at * c.es, src.data_ptr() if src is not None else None
            if src is Wx and k < D:
                copies.matrix(ptr, dst, 4, (H, Hp), (c.I, c.Ip), types)
            elif src is Wx:
                copies.matrix(ptr, dst, 4, (H, Hp), (H, Hp), types, blocks=D)
            elif src is Wh:
                copies.matrix(ptr, dst, 4, (H, Hp), (H, Hp), types)
            else:
                copies.matrix(ptr, dst, 4, (1, 1), (H, Hp), types)
            views.append(c.view(buf, at, shape))
            at += up(n)
        out.append(tuple(views))
    return out


def _states(c, copies, h_0, c_0, order):
    """Per layer and direction (h0 [B,Hp], c0) in the compute type and the kernels' row order, or (None, None)."""
    n = c.L * c.D
    if h_0 is None:
        return [(None, None)] * n
    h_0, c_0 = h_0.contiguous(), c_0.contiguous()
    if c.Hp == c.H and order is None and c.states == (c.dt, c.dt):
        return [(h_0[k], c_0[k]) for k in range(n)]
    buf = torch.empty((2, n, c.B, c.Hp), dtype=c.dt, device=c.device)
    for i, s in enumerate((h_0, c_0)):
        types, src, dst = L._DTYPE_CODE[s.dtype] + 16 * c.code, s.data_ptr(), buf.data_ptr() + i * n * c.B * c.Hp * c.es
        if order is None:
            copies.matrix(src, dst, 1, (n * c.B, n * c.B), (c.H, c.Hp), types)
        else:
            for k in range(n):
                copies.rows(src + k * c.B * c.H * s.element_size(), ORDERED, c.H, dst + k * c.B * c.Hp * c.es, BATCH, c.Hp, (c.H, c.Hp), types)
    return [(buf[0, k], buf[1, k]) for k in range(n)]


def forward(c, x, h_0, c_0, params, keep):
    """(out, h_n, c_n) of the call and, per layer and direction, what the reverse pass reads (with `keep`): the inputs, the
    (out, cell, ifgo), the weights."""
    data, order = (x.data, x.sorted_indices) if c.packed else (x, None)
    stream = L._stream()
    if c.packed:
        _upload_lengths(c, x, stream)
        keep = True   # (a row's last cell state is read out of the history)
    here = _Pass(c, order, stream)
    T, B, H, Hp, D, es = c.T, c.B, c.H, c.Hp, c.D, c.es
    dev, new = c.device, lambda *shape: torch.empty(shape, dtype=c.dt, device=c.device)
    copies = _Copies()
    weights = _weights(c, copies, params)
    states = _states(c, copies, h_0, c_0, order)
    data = data.contiguous()
    types = L._DTYPE_CODE[c.x_dtype] + 16 * c.code
    cur, cur_r = data, None
    if c.packed:
        cur = new(T, B, c.Ip)
        copies.rows(data.data_ptr(), PACKED, c.I, cur.data_ptr(), PADDED, c.Ip, (c.I, c.Ip), types)
    elif c.copy_x:
        cur = new(T, B, c.Ip)
        copies.matrix(data.data_ptr(), cur.data_ptr(), 1, (T * B, T * B), (c.I, c.Ip), types)
    if D == 2:
        cur_r = new(T, B, c.Ip)
        copies.rows(data.data_ptr(), PACKED_REVERSED if c.packed else REVERSED, c.I, cur_r.data_ptr(), PADDED, c.Ip, (c.I, c.Ip), types)
    copies.run(here)

    kw = {} if keep else {"keep_activations": False}
    inputs, kept, c.groups = [], [], []    # groups: (first layer, layers) of a host call
    operands = [states[k] + tuple(weights[k]) for k in range(c.L * D)]
    row, own = B * Hp * es, c.code + 16 * c.code
    layer = 0
    while layer < c.L:
        if D == 1:
            width = min(c.L - layer, 4)
            while width >= 3 and not L.stack_wavefront_chunks(width, T, B, Hp, c.dt, dev):
                width -= 1
            if width >= 3:
                acts = L.lstm_persistent_fwd_stack(cur, operands[layer:layer + width], **kw)
            elif width == 2 and ((L._stack2_overlaps(T, B) and L.stack2_runs_in_one_launch(T, B, cur.shape[2], Hp, c.dt, dev))
                                 or L.stack2_wavefront_chunks(T, B, Hp, c.dt, dev)):
                r = L.lstm_persistent_fwd_stack2(cur, *operands[layer], *operands[layer + 1], **kw)
                acts = [r[:3], r[3:]]
            else:
                width, acts = 1, [L.lstm_persistent_fwd(cur, *operands[layer], **kw)]
            for a in acts:
                inputs.append(cur)
                kept.append(a)
                cur = a[0][1:]
            c.groups.append((layer, width))
            layer += width
            continue
        a, b = operands[2 * layer], operands[2 * layer + 1]
        if L.pair_runs_in_one_launch(T, B, Hp, c.dt, dev):
            r = L.lstm_persistent_fwd_pair(cur, *a, cur_r, *b, **kw)
            acts = [r[:3], r[3:]]
        else:
            acts = [L.lstm_persistent_fwd(cur, *a, **kw), L.lstm_persistent_fwd(cur_r, *b, **kw)]
        inputs += [cur, cur_r]
        kept += acts
        c.groups.append((layer, 1))
        layer += 1
        if layer < c.L:   # both directions' h side by side, in time order and reversed
            cur, cur_r = new(T, B, 2 * Hp), new(T, B, 2 * Hp)
            pa, pb = acts[0][0].data_ptr() + row, acts[1][0].data_ptr() + row
            copies = _Copies()
            for dst, ma, mb in ((cur.data_ptr(), PADDED, REVERSED), (cur_r.data_ptr(), REVERSED, PADDED)):
                copies.rows(pa, ma, Hp, dst, PADDED, 2 * Hp, (Hp, Hp), own)
                copies.rows(pb, mb, Hp, dst + Hp * es, PADDED, 2 * Hp, (Hp, Hp), own)
            copies.run(here)

    copies = _Copies()
    out_mode = PACKED if c.packed else PADDED
    if D == 1 and Hp == H and not c.packed:
        out = cur
    else:
        out = new(c.N, D * H) if c.packed else new(T, B, D * H)
        for d in range(D):
            copies.rows(kept[-D + d][0].data_ptr() + row, REVERSED if d else PADDED, Hp, out.data_ptr() + d * H * es, out_mode, D * H,
                        (H, H), own)
    h_n, c_n = new(c.L * D, B, H), new(c.L * D, B, H)
    for k, a in enumerate(kept):
        for src, dst in ((a[0], h_n), (a[1], c_n)):
            to = dst.data_ptr() + k * B * H * es
            if c.packed:
                copies.rows(src.data_ptr() + row, LAST, Hp, to, ORDERED, H, (H, H), own)
            else:
                copies.matrix(src.data_ptr() + T * row, to, 1, (B, B), (Hp, H), own)
    copies.run(here)
    return (out, h_n, c_n), (inputs, kept, weights)


def backward(c, kept, order, dout, dh_n, need_x, need_states, need_w):
    """Gradients of (x, h_0, c_0, params) for the gradient of out (and, packed input, of h_n; either may be None)."""
    T, B, H, Hp, D, es = c.T, c.B, c.H, c.Hp, c.D, c.es
    inputs, acts_of, weights_of = kept
    here = _Pass(c, order, L._stream())
    new = lambda *shape, dtype=c.dt: torch.empty(shape, dtype=dtype, device=c.device)
    own, row = c.code + 16 * c.code, B * Hp * es
    copies = _Copies()
    if dout is not None:
        dout = dout.contiguous()
    if D == 1 and Hp == H and not c.packed and dout is not None and dout.dtype == c.dt:
        dh = [dout]
    else:
        dh = [new(T, B, Hp) for _ in range(D)]
        for d in range(D):
            mode = (PACKED_REVERSED if d else PACKED) if c.packed else (REVERSED if d else PADDED)
            ptr, types = (0, own) if dout is None else (dout.data_ptr() + d * H * dout.element_size(), L._DTYPE_CODE[dout.dtype] + 16 * c.code)
            copies.rows(ptr, mode, D * H, dh[d].data_ptr(), PADDED, Hp, (H, Hp), types)
    copies.run(here)

    def add_state_gradient(layer):   # packed input: h_n is out at each row's last step
        if dh_n is None:
            return
        g, more = dh_n.contiguous(), _Copies()
        if g.dtype != c.dt:
            g = g.to(c.dt)
        for d in range(D):
            more.rows(g.data_ptr() + (layer * D + d) * B * H * es, ORDERED, H, dh[d].data_ptr(), LAST, Hp, (H, H), own,
                      src2=dh[d].data_ptr(), mode2=LAST, ld2=Hp)
        more.run(here)

    n = c.L * D
    dh0, dc0, dw = [None] * n, [None] * n, [None] * n
    groups = c.groups
    if dh_n is not None:   # (it enters at each row's own last step: layer by layer)
        groups = [(layer, 1) for layer in range(c.L)]
    for layer, width in reversed(groups):
        need_dx = need_x or layer > 0
        k = layer * D
        if D == 1:
            x = inputs[layer]
            add_state_gradient(layer)
            acts, weights = acts_of[layer:layer + width], [(w[0], w[2]) for w in weights_of[layer:layer + width]]
            if width >= 3:
                res = L.lstm_persistent_bwd_stack(dh[0], x, acts, weights, None, need_dx)
            elif width == 2:
                res = L.lstm_persistent_bwd_stack2(dh[0], x, *acts[0], *weights[0], *acts[1], *weights[1], need_dx=need_dx)
            else:
                res = [L.lstm_persistent_bwd(dh[0], None, None, x, *acts[0], *weights[0], need_dx=need_dx, need_dw=need_w)]
            dh = [res[0][0]]
        else:
            add_state_gradient(layer)
            a, b = (inputs[k], *acts_of[k], weights_of[k][0], weights_of[k][2]), (inputs[k + 1], *acts_of[k + 1], weights_of[k + 1][0], weights_of[k + 1][2])
            if L.pair_runs_in_one_launch(T, B, Hp, c.dt, c.device, backward=True):
                res = L.lstm_persistent_bwd_pair(dh[0], None, *a, dh[1], None, *b, need_dx=(need_dx, need_dx))
            else:
                res = [L.lstm_persistent_bwd(dh[d], None, None, *s, need_dx=need_dx, need_dw=need_w) for d, s in enumerate((a, b))]
            dx = [r[0] for r in res]
            if layer > 0:   # the lower layer's h: its own columns of both, the reversed one turned back
                pa, pb = dx[0].data_ptr(), dx[1].data_ptr()
                dh = [new(T, B, Hp), new(T, B, Hp)]
                copies = _Copies()
                copies.rows(pa, PADDED, 2 * Hp, dh[0].data_ptr(), PADDED, Hp, (Hp, Hp), own, pb, REVERSED, 2 * Hp)
                copies.rows(pa + Hp * es, REVERSED, 2 * Hp, dh[1].data_ptr(), PADDED, Hp, (Hp, Hp), own, pb + Hp * es, PADDED, 2 * Hp)
                copies.run(here)
            else:
                dh = dx
        for i, r in enumerate(res):
            dh0[k + i], dc0[k + i], dw[k + i] = r[1], r[2], r[3:]

    copies = _Copies()
    d_x = None
    if need_x:
        if not (c.copy_x or D == 2):
            d_x = dh[0]
        else:
            types = c.code + 16 * L._DTYPE_CODE[c.x_dtype]
            d_x = new(c.N, c.I, dtype=c.x_dtype) if c.packed else new(T, B, c.I, dtype=c.x_dtype)
            second = (dh[1].data_ptr(), REVERSED, c.Ip) if D == 2 else (0, 0, 0)
            copies.rows(dh[0].data_ptr(), PADDED, c.Ip, d_x.data_ptr(), PACKED if c.packed else PADDED, c.I, (c.I, c.I), types, *second)
    d_states = [None, None]
    if c.states is not None:
        for i, parts in enumerate((dh0, dc0)):
            if not need_states[i]:
                continue
            dt = c.states[i]
            d_states[i] = new(n, B, H, dtype=dt)
            step, types = B * H * (4 if dt == torch.float32 else 2), c.code + 16 * L._DTYPE_CODE[dt]
            for k in range(n):
                copies.rows(parts[k].data_ptr(), BATCH, Hp, d_states[i].data_ptr() + k * step, ORDERED, H, (H, H), types)
    d_params = []
    if need_w:
        types = c.code + 16 * L._DTYPE_CODE[c.held]
        for k in range(n):
            dWx, dbx, dWh, dbh = dw[k]
            if not c.copy_weights:
                d_params += (dWx, dbx, dWh, dbh) if c.bias else (dWx, dWh)
                continue
            K = (c.I, c.Ip) if k < D else (H, Hp)
            blocks = 1 if k < D else D
            gx, gh = new(4 * H, blocks * K[0], dtype=c.held), new(4 * H, H, dtype=c.held)
            copies.matrix(dWx.data_ptr(), gx.data_ptr(), 4, (Hp, H), K[::-1], types, blocks=blocks)
            copies.matrix(dWh.data_ptr(), gh.data_ptr(), 4, (Hp, H), (Hp, H), types)
            if c.bias:
                gbx, gbh = new(4 * H, dtype=c.held), new(4 * H, dtype=c.held)
                for g, s in ((gbx, dbx), (gbh, dbh)):
                    copies.matrix(s.data_ptr(), g.data_ptr(), 4, (1, 1), (Hp, H), types)
                d_params += (gx, gbx, gh, gbh)
            else:
                d_params += (gx, gh)
    copies.run(here)
    return d_x, d_states[0], d_states[1], d_params


class Layersfn(torch.autograd.Function):
    """apply(call, packed input | None, x data, h_0 | None, c_0 | None, *params) -> (out, h_n, c_n).  The final states carry no
    gradient, as in the reference (fastlstm/lstm.py:504-538); with packed input h_n does, through out."""

    @staticmethod
    def forward(ctx, c, packed, data, h_0, c_0, *params):
        with torch.cuda.device(data.device):
            (out, h_n, c_n), (inputs, acts, weights) = forward(c, packed if c.packed else data, h_0, c_0, params, True)
        ctx.call, ctx.count = c, (len(inputs), len(acts))
        flat = list(inputs)
        for a in acts:
            flat += a
        for w in weights:
            flat += (w[0], w[2])
        ctx.save_for_backward(packed.sorted_indices if c.packed else None, *flat)   # (the caller's tensor: a change in place is noticed)
        ctx.set_materialize_grads(False)
        ctx.mark_non_differentiable(*((c_n,) if c.packed else (h_n, c_n)))
        return out, h_n, c_n

    @staticmethod
    def backward(ctx, dout, dh_n, _):
        c, need = ctx.call, ctx.needs_input_grad
        if dout is None and dh_n is None:
            return (None,) * len(need)
        L._raise_pending_before_backward(dout if dout is not None else dh_n)   # a failed forward launch is reported before its gradients are computed
        order, *t = ctx.saved_tensors
        ni, na = ctx.count
        acts = [tuple(t[ni + 3 * k:ni + 3 * k + 3]) for k in range(na)]
        w = t[ni + 3 * na:]
        kept = t[:ni], acts, [(w[2 * k], None, w[2 * k + 1], None) for k in range(na)]
        with torch.cuda.device(c.device):
            d_x, d_h, d_c, d_params = backward(c, kept, order, dout, dh_n if c.packed else None, need[2], need[3:5], any(need[5:]))
        if not d_params:
            d_params = [None] * (len(need) - 5)
        return (None, None, d_x, d_h, d_c, *d_params)


def run(module, c, x, h_c_0):
    """FastLSTM.forward through the node (or, without gradients, through its forward part alone)."""
    params = module._operand_list()
    h_0, c_0 = (None, None) if h_c_0 is None else h_c_0
    data = x.data if c.packed else x
    if not c.packed and module.batch_first:
        data = data.transpose(0, 1).contiguous()
    grads = torch.is_grad_enabled() and (data.requires_grad or any(p.requires_grad for p in params)
                                         or (h_0 is not None and (h_0.requires_grad or c_0.requires_grad)))
    if grads:
        out, h_n, c_n = Layersfn.apply(c, x if c.packed else None, data, h_0, c_0, *params)
    else:
        with torch.cuda.device(data.device):
            (out, h_n, c_n), _ = forward(c, x if c.packed else data, h_0, c_0, params, False)
    if c.packed:
        return PackedSequence(out, x.batch_sizes, x.sorted_indices, x.unsorted_indices), (h_n, c_n)
    return (out.transpose(0, 1) if module.batch_first else out), (h_n, c_n)
