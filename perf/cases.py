"""The work whose speed counts: FastLSTM layers as a program runs them, from one step of one stream to a stack of wide layers
in training.

listed()            the cases that are quoted
draw(rng)           one more case of the ranges that they stand for
prepare(case, seed) what a program has in hand: the module, its input, the initial states and, in training, the gradient of its output
run(state)          one call of the module (and of backward(), in training), through the public entry points only
work(case)          bytes and floating-point operations that a pass cannot do without
tolerance(case)     how far another correct implementation of the same precision may be off

A case is a dict:
    mode         "infer": the module under torch.no_grad(); "train": forward and backward()
    dtype        element type of the products and of the results
    autocast     fp32 parameters and input, torch.autocast to dtype (mixed-precision training)
    T, B, I, H   timesteps, batch rows, input size, hidden size
    layers       stacked layers
    bidirectional
    packed       PackedSequence input, lengths spread evenly over T/4 ... T
    states       initial states are handed in (zeros otherwise)
    input_grad   training: the input asks for a gradient (it comes from an embedding or from another layer)
"""
import math

import torch

from fastlstm_amd import FastLSTM

DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}


def _case(name, mode, dtype, T, B, I, H, layers=1, bidirectional=False, packed=False, states=False, input_grad=False, autocast=False):
    c = {"mode": mode, "dtype": dtype, "autocast": autocast, "T": T, "B": B, "I": I, "H": H, "layers": layers,
         "bidirectional": bidirectional, "packed": packed, "states": states, "input_grad": input_grad}
    return dict(c, name=name) if name else c


def listed():
    return [
        # one step of a few streams with the state carried from call to call (sampling, live audio): launches and host time
        _case("step_fp16", "infer", "fp16", 1, 4, 512, 512, layers=2, states=True),
        # a small fp32 model over short windows (sensor data, keyword spotting)
        _case("window_fp32_infer", "infer", "fp32", 64, 8, 80, 96),
        # the single-layer fp32 model of the benchmark's workload A
        _case("small_fp32_train", "train", "fp32", 128, 16, 256, 256),
        # the headline layer (workload B): scoring with initial states, and training in the middle of a model
        _case("headline_fp16_infer", "infer", "fp16", 512, 64, 1024, 1024, states=True),
        _case("headline_fp16_train", "train", "fp16", 512, 64, 1024, 1024, input_grad=True),
        # a wide layer with a full batch, fp32 accumulation of bf16 (workload C: every gradient is wanted)
        _case("wide_bf16_train", "train", "bf16", 256, 128, 2048, 2048, input_grad=True),
        # many long sequences through few units (workload D)
        _case("narrow_fp16_train", "train", "fp16", 1024, 256, 64, 64),
        # long sequences through a stack (workload E)
        _case("stack_fp16_train", "train", "fp16", 2048, 32, 1024, 1024, layers=2, input_grad=True),
        # a word-level language model: short segments, sizes that fit no tile, mixed precision, state carried over
        _case("language_bf16_train", "train", "bf16", 35, 20, 650, 650, layers=2, states=True, input_grad=True, autocast=True),
        # a tagger: sentences of different lengths, packed, both directions
        _case("tagger_fp16_train", "train", "fp16", 199, 50, 123, 257, bidirectional=True, packed=True, input_grad=True),
        # full precision where the products are large
        _case("large_fp32_train", "train", "fp32", 128, 64, 512, 1024, input_grad=True),
        # a layer whose recurrent weights do not fit on the chip
        _case("huge_fp16_infer", "infer", "fp16", 128, 64, 1024, 4096),
    ]


def _log(rng, lo, hi):
    """An integer between lo and hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _size(rng, lo, hi):
    """A layer's size: as often a multiple of 64 as any number."""
    n = _log(rng, lo, hi)
    return max(64, n // 64 * 64) if n >= 64 and rng.random() < 0.5 else n


def _cost(c):
    """Operations with fp32 counted at its matrix rate, one sixteenth of the 16-bit one."""
    return work(c)["flops"] * (16 if c["dtype"] == "fp32" else 1)


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        mode = rng.choice(("infer", "train"))
        dtype = rng.choice(("fp32", "fp16", "bf16"))
        if mode == "infer" and rng.random() < 0.3:   # steps and very short chunks of a stream
            c = _case(None, mode, dtype, _log(rng, 1, 8), _log(rng, 1, 64), _size(rng, 32, 1024), _size(rng, 64, 2048),
                      layers=rng.choice((1, 2, 3)), states=True)
        else:
            bidirectional = rng.random() < 0.2
            c = _case(None, mode, dtype, _log(rng, 16, 2048), _log(rng, 1, 256), _size(rng, 32, 2048),
                      _size(rng, 16, 2048 if dtype == "fp32" else 4096), layers=rng.choice((1, 1, 2, 3)), bidirectional=bidirectional,
                      packed=rng.random() < (0.5 if bidirectional else 0.1), states=rng.random() < 0.3,
                      input_grad=mode == "train" and rng.random() < 0.7,
                      autocast=dtype != "fp32" and mode == "train" and rng.random() < 0.5)
        # no longer chain of steps and no more arithmetic than the largest listed cases (a step touches all of W_h), and
        # tensors that fit in memory with room to spare
        chain = c["T"] * c["layers"] * (2 if c["bidirectional"] else 1)
        if (_cost(c) <= most and chain <= 4096 and chain * c["H"] ** 2 * (4 if dtype == "fp32" else 2) <= 4.5e9
                and c["T"] * c["B"] * c["H"] * c["layers"] <= 1 << 27):
            return c


def _lengths(case):
    """Packed input: B lengths from T down to about T/4."""
    T, B = case["T"], case["B"]
    low = max(1, T // 4)
    return [T - (T - low) * b // max(1, B - 1) for b in range(B)]


def _steps(case):
    """(batch row, timestep) pairs that count."""
    return sum(_lengths(case)) if case["packed"] else case["T"] * case["B"]


def prepare(case, seed):
    device, dtype = torch.device("cuda"), DTYPES[case["dtype"]]
    T, B, I, H, L, D = case["T"], case["B"], case["I"], case["H"], case["layers"], 2 if case["bidirectional"] else 1
    held = torch.float32 if case["autocast"] else dtype      # what the program keeps its tensors in
    g = torch.Generator(device=device).manual_seed(seed)
    module = FastLSTM(I, H, num_layers=L, device=device, dtype=held, bidirectional=case["bidirectional"])
    with torch.no_grad():
        for p in module.parameters():                          # the initialisation of nn.LSTM, from this seed
            p.uniform_(-1 / H ** 0.5, 1 / H ** 0.5, generator=g)

    def normal(*shape):
        return torch.randn(*shape, device=device, dtype=torch.float32, generator=g)

    train = case["mode"] == "train"
    state = {"module": module, "train": train, "autocast": dtype if case["autocast"] else None, "states": None, "dout": None}
    if case["packed"]:
        lengths = torch.tensor(_lengths(case))
        order = torch.randperm(B, generator=torch.Generator().manual_seed(seed))
        alive = (lengths[None, :] > torch.arange(T)[:, None]).sum(1)
        data = normal(int(alive.sum()), I).to(held).requires_grad_(train and case["input_grad"])
        on_device = order.to(device)
        state["x"] = torch.nn.utils.rnn.PackedSequence(data, alive, on_device, torch.argsort(on_device))
        state["leaf"] = data
    else:
        state["leaf"] = state["x"] = normal(T, B, I).to(held).requires_grad_(train and case["input_grad"])
    if case["states"]:
        state["states"] = tuple((normal(L * D, B, H) * 0.1).to(held) for _ in range(2))
    if train:
        shape = (_steps(case), D * H) if case["packed"] else (T, B, D * H)
        state["dout"] = normal(*shape).to(dtype)
    return state


def run(state):
    module, x = state["module"], state["x"]
    if not state["train"]:
        with torch.no_grad():
            out, (h_n, c_n) = module(x, state["states"])
        return {"out": out[0] if isinstance(out, tuple) else out, "h_n": h_n, "c_n": c_n}
    module.zero_grad(set_to_none=True)
    leaf = state["leaf"]
    leaf.grad = None
    if state["autocast"] is not None:
        with torch.autocast("cuda", dtype=state["autocast"]):
            out, (h_n, c_n) = module(x, state["states"])
    else:
        out, (h_n, c_n) = module(x, state["states"])
    y = out.data if isinstance(out, torch.nn.utils.rnn.PackedSequence) else out
    y.backward(state["dout"])
    return {"out": y, "h_n": h_n, "c_n": c_n, "d_x": leaf.grad, "d_w": [p.grad for p in module.parameters()]}


def work(case):
    H, L, D, n = case["H"], case["layers"], 2 if case["bidirectional"] else 1, _steps(case)
    train = case["mode"] == "train"
    es = 4 if case["dtype"] == "fp32" else 2
    held = 4 if case["autocast"] else es
    weights, flops = 0, 0
    for layer in range(L):
        K = case["I"] if layer == 0 else D * H
        weights += D * 4 * H * (K + H + 2)
        products = 8 * n * H * D * (K + H)                     # input projection and recurrence
        flops += products
        if train:                                              # d(input), d(state), dW_x, dW_h
            flops += 2 * products - (8 * n * H * D * K if layer == 0 and not case["input_grad"] else 0)
    states = L * D * case["B"] * H
    moved = n * case["I"] * held + weights * held + n * D * H * es + 2 * states * es       # x, parameters in; out, h_n, c_n out
    if case["states"]:
        moved += 2 * states * held
    if train:
        moved += n * D * H * es + weights * held               # the output's gradient in, the parameters' gradients out
        if case["input_grad"]:
            moved += n * case["I"] * held
    return {"bytes": float(moved), "flops": float(flops)}


def tolerance(case):
    # results, gates and cell states are rounded to the element type at every step: a few units in the last place of the
    # type over the norm; fp32: the order of the sums and the last bits of the gate functions
    return {"fp32": {"rel": 2e-5, "max": 2e-3}, "fp16": {"rel": 2e-3}, "bf16": {"rel": 1e-2}}[case["dtype"]]
