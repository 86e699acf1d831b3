"""The calls by which this package's speed is judged.

``listed()`` names twelve of them, ``draw(rng)`` gives others of the same
ranges, ``prepare`` makes what a user's program holds before the call,
``run`` makes the call through the public entry points and returns its whole
results, ``work`` gives the bytes and operations no implementation can do
without, ``tolerance`` how far two correct implementations of one precision
may be apart, and ``exact`` the same results in 64 bits in plain torch.

Four kinds of call:

* ``fit``      a new batch: ``initialize_batch``, ``steps`` training steps and,
               with ``predict``, the forward pass that scores the batch: one
               turn of the training loop (``lich_amd.train``);
* ``steps``    ``steps`` training steps of a batch already in place: the
               steady state that ``bench.py`` measures;
* ``predict``  the forward pass of a trained net: evaluation and serving;
* ``layer``    one kernel of the operator API (``lich_amd.kernels``) on the
               caller's tensors: prediction + error, inference update, weight
               update by GEMM or by rank-B outer product.

A case is a dict of plain values.  Nets are (classes, hidden x depth,
features); layers are M x K weights at batch B, `storage` the type of the
tensors and `operand` the type the GEMM operands are rounded to.
"""
from __future__ import annotations

import math

import torch

from lich_amd import (HipIPC, IPCConfig, KernelConfig, build_inference_update, build_prediction_error,
                      build_weight_update, build_weight_update_outer)

ALPHA, GAMMA = 1e-4, 0.5  # the trainer's defaults
DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
ACTIVATIONS = ("relu", "tanh", "sigmoid", "silu", "gelu")


def _net(name, kind, classes, hidden, depth, features, batch, operand, activation, steps=0, predict=False):
    return {"name": name, "kind": kind, "classes": classes, "hidden": hidden, "depth": depth, "features": features,
            "batch": batch, "operand": operand, "activation": activation, "steps": steps, "predict": predict}


def _layer(name, op, M, K, B, storage, operand, activation, option=False, workspace=False):
    return {"name": name, "kind": "layer", "op": op, "M": M, "K": K, "batch": B, "storage": storage,
            "operand": operand, "activation": activation, "option": option, "workspace": workspace}


def listed():
    return [
        # Online learning: one sample at a time, eight steps each, everything in fp32.  The smallest work there is.
        _net("online_sample", "fit", 10, 64, 4, 784, 1, "fp32", "tanh", steps=8),
        # One turn of the training loop with the trainer's defaults: two hidden layers of 64 on 28 x 28 images.
        _net("mnist_batch", "fit", 10, 64, 2, 784, 128, "fp16", "relu", steps=4, predict=True),
        # The steady state of the paper's efficiency profile, depth 6 (bench.py's headline).
        _net("paper_steady", "steps", 10, 64, 6, 784, 128, "fp16", "tanh", steps=4),
        # The same images with twice the width and a large batch, as a longer training run would take them.
        _net("broad_batch", "fit", 10, 128, 3, 784, 512, "fp16", "tanh", steps=4),
        # An ordinary image MLP: three hidden layers of 512.
        _net("mlp_batch", "fit", 10, 512, 3, 784, 256, "fp16", "tanh", steps=4),
        # One step of the wide, MFMA-bound net (bench.py's wide configuration).  The largest work there is.
        _net("wide_step", "steps", 1000, 4096, 4, 4096, 1024, "bf16", "tanh", steps=1),
        # Scoring a part of a test set with the ordinary MLP; 2000 columns fill no tile evenly.
        _net("evaluate", "predict", 10, 512, 3, 784, 2000, "fp16", "tanh"),
        # The reference's own kernel shape: the first layer of the image nets in 16-bit storage.  Latency and launches.
        _layer("first_layer", "pred", 64, 784, 128, "fp16", "fp16", "relu"),
        # A large layer's prediction error as a drop-in caller makes it, f(X) evaluated in the call.
        _layer("large_pred", "pred", 4096, 4096, 2048, "bf16", "bf16", "tanh"),
        # The inference update of the same layer, keeping f(X) for the weight update.
        _layer("large_infer", "infer", 4096, 4096, 2048, "bf16", "bf16", "tanh", option=True),
        # A weight update at odd sizes over fp32 master data with 16-bit operands.
        _layer("ragged_weight", "weight", 1000, 1531, 300, "fp32", "bf16", "silu", option=True),
        # The small-batch weight update of a wide layer: W streams once.
        _layer("outer_weight", "outer", 2048, 2048, 8, "fp32", "fp32", "relu", option=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_net(rng):
    kind = rng.choice(("fit", "fit", "fit", "steps", "predict", "predict"))
    size = rng.choice(("narrow", "narrow", "broad", "mlp", "mlp", "wide"))
    hidden = {"narrow": (16, 64), "broad": (65, 128), "mlp": (129, 1024), "wide": (1025, 4096)}[size]
    depth = rng.randint(1, 6 if size in ("narrow", "broad") else 4)
    width = _log_int(rng, *hidden)
    if rng.random() < 0.5:
        width = max(hidden[0], width // 16 * 16)
    features = rng.choice((784, _log_int(rng, 64, 4096)))
    classes = rng.choice((10, 10, 100, 1000)) if size in ("mlp", "wide") else 10
    operand = rng.choice(("fp16", "fp16", "bf16", "bf16", "fp32"))
    batch = _log_int(rng, 1, 4096 if kind == "predict" else 1024)
    if rng.random() < 0.4:
        batch = max(1, batch // 32 * 32)
    # without a new batch the states keep evolving, which only the bounded activations keep tame
    activation = rng.choice(("tanh", "sigmoid") if kind == "steps" else ACTIVATIONS)
    steps = 0 if kind == "predict" else rng.randint(1, 4)
    return _net("", kind, classes, width, depth, features, batch, operand, activation, steps,
                kind == "fit" and rng.random() < 0.5)


def _draw_layer(rng):
    op = rng.choice(("pred", "pred", "infer", "infer", "weight", "weight", "outer"))
    storage, operand = rng.choice((("fp16", "fp16"), ("bf16", "bf16"), ("bf16", "bf16"), ("fp32", "fp16"),
                                   ("fp32", "bf16"), ("fp32", "fp32")))
    if op == "outer":
        operand = storage
    M, K = _log_int(rng, 16, 8192), _log_int(rng, 16, 8192)
    batch = _log_int(rng, 1, 16) if op == "outer" else _log_int(rng, 16, 4096)
    if rng.random() < 0.5:  # half of the layers are as even as real nets are
        M, K = (max(16, v // 64 * 64) for v in (M, K))
        batch = max(1, batch // 64 * 64) if op != "outer" else batch
    return _layer("", op, M, K, batch, storage, operand, rng.choice(ACTIVATIONS), rng.random() < 0.6,
                  op != "outer" and storage != "fp32" and rng.random() < 0.4)


def draw(rng):
    limit = work(next(c for c in listed() if c["name"] == "wide_step"))["flops"]
    while True:
        case = _draw_net(rng) if rng.random() < 0.55 else _draw_layer(rng)
        # fp32 operands run at a sixteenth of the 16-bit matrix rate
        cost = work(case)["flops"] * (16 if case["operand"] == "fp32" else 1)
        if cost <= limit / 2:
            del case["name"]
            return case


# ------------------------------------------------------------------ inputs
def _dims(case):
    return (case["classes"],) + (case["hidden"],) * case["depth"] + (case["features"],)


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _net_inputs(case, seed):
    """Xavier-uniform weights, pixels in [0, 1) and one-hot targets, fp32."""
    g, dims, B = _generator(seed), _dims(case), case["batch"]
    w = []
    for m, k in zip(dims[:-1], dims[1:]):
        bound = math.sqrt(6.0 / (m + k))
        w.append((torch.rand((m, k), generator=g, device="cuda") * 2 - 1) * bound)
    x = torch.rand((dims[-1], B), generator=g, device="cuda")
    labels = torch.randint(0, dims[0], (B,), generator=g, device="cuda")
    y = torch.nn.functional.one_hot(labels, dims[0]).float().T.contiguous()
    return w, x, y


def _layer_inputs(case, seed):
    """States of unit size, Xavier-uniform weights and errors a tenth of the states, rounded to the storage type."""
    g, M, K, B = _generator(seed), case["M"], case["K"], case["batch"]
    dt = DTYPES[case["storage"]]

    def normal(rows, cols, size):
        return (torch.randn((rows, cols), generator=g, device="cuda") * size).to(dt)

    def weights(rows, cols):
        bound = math.sqrt(6.0 / (M + K))
        return ((torch.rand((rows, cols), generator=g, device="cuda") * 2 - 1) * bound).to(dt)

    if case["op"] == "pred":
        return {"x_upper": normal(K, B, 1.0), "w": weights(M, K), "x_lower": normal(M, B, 1.0)}
    if case["op"] == "infer":
        return {"x": normal(M, B, 1.0), "e": normal(M, B, 0.1), "w_lower": weights(K, M), "e_lower": normal(K, B, 0.1)}
    return {"w": weights(M, K), "e": normal(M, B, 0.1), "x_upper": normal(K, B, 1.0)}


# ------------------------------------------------------------------ the calls
def prepare(case, seed):
    if case["kind"] == "layer":
        state = _layer_inputs(case, seed)
        M, K, B, act, dt = case["M"], case["K"], case["batch"], case["activation"], DTYPES[case["storage"]]
        operand = DTYPES[case["operand"]]
        if case["op"] == "pred":
            state["kernel"] = build_prediction_error(M, K, B, act, dt, KernelConfig(), operand_dtype=operand)
            state["out"] = torch.empty_like(state["x_lower"])
        elif case["op"] == "infer":  # option: keep f(X)
            state["kernel"] = build_inference_update(M, K, B, act, dt, KernelConfig(), GAMMA, case["option"],
                                                     operand_dtype=operand)
            state["a"] = torch.empty_like(state["x"]) if case["option"] else None
        elif case["op"] == "weight":  # option: f evaluated in the call, else X_upper is f(X) already
            state["kernel"] = build_weight_update(M, K, B, act, dt, KernelConfig(), ALPHA, case["option"],
                                                  operand_dtype=operand)
        else:
            state["kernel"] = build_weight_update_outer(M, K, B, act, dt, ALPHA, case["option"])
        state["case"] = case
        state["kw"] = {"workspace": state["kernel"].new_workspace()} if case["workspace"] else {}
        return state
    w, x, y = _net_inputs(case, seed)
    model = HipIPC(IPCConfig(dims=_dims(case), alpha=ALPHA, gamma=GAMMA, activation=case["activation"],
                             dtype=DTYPES[case["operand"]]), device="cuda", weights=w)
    if case["kind"] != "predict":
        model.initialize_batch(x, y)
    return {"case": case, "model": model, "x": x, "y": y}


def run(state):
    case = state["case"]
    if case["kind"] == "layer":
        kernel, kw = state["kernel"], state["kw"]
        if case["op"] == "pred":
            kernel(state["x_upper"], state["w"], state["x_lower"], state["out"], **kw)
            return state["out"]
        if case["op"] == "infer":
            if case["option"]:
                kernel(state["x"], state["e"], state["w_lower"], state["e_lower"], state["a"], **kw)
                return [state["x"], state["a"]]
            kernel(state["x"], state["e"], state["w_lower"], state["e_lower"], **kw)
            return state["x"]
        kernel(state["w"], state["e"], state["x_upper"], **kw)
        return state["w"]
    model = state["model"]
    if case["kind"] == "predict":
        return model.predict(state["x"])
    if case["kind"] == "fit":
        model.initialize_batch(state["x"], state["y"])
    model.run_steps(case["steps"])
    out = {"w": model.w, "x": model.x[1:-1], "e0": model.e[0]}
    if case["predict"]:
        out["logits"] = model.predict(state["x"])
    return out


# ------------------------------------------------------------------ what they cost
def work(case):
    B = case["batch"]
    if case["kind"] == "layer":
        M, K, s = case["M"], case["K"], 4 if case["storage"] == "fp32" else 2
        values = {"pred": M * K + K * B + 2 * M * B,
                  "infer": M * K + K * B + (3 + bool(case["option"])) * M * B,
                  "weight": 2 * M * K + M * B + K * B, "outer": 2 * M * K + M * B + K * B}[case["op"]]
        return {"bytes": s * values, "flops": 2.0 * M * K * B}
    dims = _dims(case)
    edges = [m * k for m, k in zip(dims[:-1], dims[1:])]
    S, hidden = sum(edges), sum(dims[1:-1])
    if case["kind"] == "predict":
        return {"bytes": 4 * (S + (dims[0] + dims[-1]) * B), "flops": 2.0 * S * B}
    # a step: prediction and weight update of every layer, inference of every layer but the top one
    flops = 2.0 * B * case["steps"] * (2 * S + S - edges[-1])
    nbytes = 4 * (2 * S + (dims[0] + dims[-1]) * B + hidden * B + dims[0] * B)
    if case["kind"] == "fit":
        flops += 2.0 * B * (S - edges[0])
        if case["predict"]:
            flops += 2.0 * B * S
            nbytes += 4 * dims[0] * B
    else:
        nbytes += 4 * hidden * B  # the states come in as well
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times what the same call shows with its sums in another order
    (auto path against phased path, one and two passes, MI355X): fp32 nets 8e-7
    (relu's step can turn on one state: its bound is ten times wider), fp16 nets
    1e-3, bf16 nets 3e-4 where the operands are split and eight times fp16's
    rounding where they are not.  Layers differ by the rounding of their outputs
    (16-bit storage: a share of elements by one unit) or by single operands
    whose rounding an activation's last bit turns (fp32 storage)."""
    if case["kind"] == "layer":
        if case["storage"] == "fp32":
            return {"rel": 1e-5 if case["operand"] == "fp32" else 1e-4}
        return {"rel": 1e-3 if case["storage"] == "fp16" else 5e-3}
    if case["operand"] == "fp32":
        return {"rel": 1e-4 if case["activation"] == "relu" else 1e-5}
    return {"rel": 4e-3 if case["operand"] == "fp16" else 1e-2}


# ------------------------------------------------------------------ the same in 64 bits
def _f(name, x):
    if name == "relu":
        return torch.relu(x)
    if name == "tanh":
        return torch.tanh(x)
    if name == "sigmoid":
        return torch.sigmoid(x)
    if name == "silu":
        return x * torch.sigmoid(x)
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def _df(name, x):
    if name == "relu":
        return (x > 0).to(x.dtype)
    if name == "tanh":
        return 1 - torch.tanh(x) ** 2
    if name == "sigmoid":
        s = torch.sigmoid(x)
        return s * (1 - s)
    if name == "silu":
        s = torch.sigmoid(x)
        return s * (1 + x * (1 - s))
    k = math.sqrt(2 / math.pi)
    t = torch.tanh(k * (x + 0.044715 * x ** 3))
    return 0.5 * (1 + t) + 0.5 * x * (1 - t * t) * k * (1 + 3 * 0.044715 * x * x)


def exact(case, seed):
    act = case["activation"]
    if case["kind"] == "layer":
        v = {k: t.double() for k, t in _layer_inputs(case, seed).items()}
        if case["op"] == "pred":
            return v["x_lower"] - v["w"] @ _f(act, v["x_upper"])
        if case["op"] == "infer":
            x = v["x"] + GAMMA * (-v["e"] + _df(act, v["x"]) * (v["w_lower"].T.contiguous() @ v["e_lower"]))
            return [x, _f(act, x)] if case["option"] else x
        a = _f(act, v["x_upper"]) if case["option"] else v["x_upper"]
        return v["w"] + ALPHA * (v["e"] @ a.T.contiguous())
    w, x_in, y = _net_inputs(case, seed)
    w, x_in, y = [t.double() for t in w], x_in.double(), y.double()
    L = len(w)

    def forward(h):
        states = [h]
        for l in range(L - 1, -1, -1):
            states.insert(0, w[l] @ _f(act, states[0]))
        return states

    if case["kind"] == "predict":
        return forward(x_in)[0]
    x = [y] + forward(x_in)[1:]
    for _ in range(case["steps"]):
        e = [x[l] - w[l] @ _f(act, x[l + 1]) for l in range(L)]
        back = [w[l - 1].T.contiguous() @ e[l - 1] for l in range(1, L)]
        for l in range(1, L):
            x[l] = x[l] + GAMMA * (-e[l] + _df(act, x[l]) * back[l - 1])
        w = [w[l] + ALPHA * (e[l] @ _f(act, x[l + 1]).T.contiguous()) for l in range(L)]
    out = {"w": w, "x": x[1:-1], "e0": e[0]}
    if case["predict"]:
        out["logits"] = forward(x_in)[0]
    return out
