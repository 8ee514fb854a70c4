"""The work a program on this package has it do, as cases that can be timed and compared.

A case is a dict of plain values; its "kind" names the public entry point and the direction:

    train        scan() and its backward: dx, da, db, dc from a given dy
    pieces       scan_chunk() and its backward, a state carried in and its gradient carried out
    generate     scan_chunk() without gradients: one token (L = 1) or one piece of a prompt, state in and out
    layer_train  SSM.forward and backward: gradients of the input and of every parameter
    layer_infer  SSM.forward under no_grad
    copy_step    copy_task.train_step: forward, loss, backward, gradient clipping, AdamW over a stack of layers

`listed()` gives the fixed cases, `draw(rng)` one more of the same ranges, `prepare` what a program has in hand
before the call, `run` one pass, `work` the bytes and operations a pass cannot do without and `tolerance` how far
the results of two correct implementations may lie apart.
"""
import math

import torch

from quick_ssm_amd import SSM, copy_task, scan, scan_chunk

_DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
_BYTES = {"float32": 4, "float16": 2, "bfloat16": 2}


def _scan_case(name, kind, B, L, D, dtype, out_dtype=None, a_lo=0.9, block_l=256, checkpoint=True):
    case = {"kind": kind, "B": B, "L": L, "D": D, "dtype": dtype, "out_dtype": out_dtype or dtype, "a_lo": a_lo,
            "block_l": block_l, "checkpoint": checkpoint}
    return dict(case, name=name) if name else case


def _layer_case(name, kind, B, L, hidden, mult, params, compute):
    case = {"kind": kind, "B": B, "L": L, "hidden": hidden, "mult": mult, "params": params, "compute": compute}
    return dict(case, name=name) if name else case


def listed():
    return [
        # One token of generation for a batch of 32 sequences at the layer's state width (4 x hidden 1024): the
        # smallest call there is, made once per token and layer.
        _scan_case("generate_token", "generate", 32, 1, 4096, "bfloat16"),
        # A prompt read in pieces of 512 steps in front of the generation.
        _scan_case("generate_prompt_piece", "generate", 4, 512, 4096, "bfloat16"),
        # The reference's own test size: many steps of a narrow fp32 state (what a first experiment looks like).
        _scan_case("train_narrow_fp32", "train", 4, 2048, 16, "float32"),
        # The headline shape of the benchmark.
        _scan_case("train_headline_bf16", "train", 8, 4096, 2048, "bfloat16"),
        # The largest: one long sequence, decay close to one.
        _scan_case("train_long_fp16", "train", 1, 65536, 4096, "float16", a_lo=0.99, block_l=1024),
        # fp32 training without mixed precision at an ordinary size.
        _scan_case("train_fp32", "train", 4, 4096, 1024, "float32"),
        # Sizes nobody rounded: an odd width (rows that start at any 2-byte address) and an odd length.
        _scan_case("train_odd_bf16", "train", 5, 1537, 777, "bfloat16"),
        # A document trained on in pieces (truncated back-propagation with the state's gradient): few, long chains.
        _scan_case("pieces_fp16", "pieces", 2, 8192, 512, "float16"),
        # The layer the reference's scripts build: fp32 parameters, fp16 compute, state = 4 x hidden.
        _layer_case("layer_train_fp32_params", "layer_train", 16, 2048, 1024, 4, "float32", "float16"),
        # The same layer with everything in bf16, the way a large model trains it, at half the batch.
        _layer_case("layer_train_bf16", "layer_train", 8, 2048, 1024, 4, "bfloat16", "bfloat16"),
        # That layer reading one prompt.
        _layer_case("layer_infer_bf16", "layer_infer", 1, 2048, 1024, 4, "bfloat16", "bfloat16"),
        # Half the depth of the copy task's stack (hidden 256, state 1024, 32 strings of 64 + 64 symbols).
        {"name": "copy_step_bf16", "kind": "copy_step", "layers": 6, "hidden": 256, "batch": 32, "seq": 64,
         "compute": "bfloat16"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A state width: mostly whole multiples of 64, sometimes of 8, now and then any number."""
    w = _log_int(rng, lo, hi)
    u = rng.random()
    unit = 64 if u < 0.6 and w >= 64 else 8 if u < 0.8 and w >= 8 else 1
    return max(unit, w // unit * unit)


def _length(rng, lo, hi):
    n = _log_int(rng, lo, hi)
    return 1 << (n.bit_length() - 1) if rng.random() < 0.4 else n


def draw(rng):
    kind = rng.choice(("train", "train", "train", "pieces", "generate", "layer_train", "layer_infer", "copy_step"))
    if kind in ("train", "pieces"):
        dtype = rng.choice(("bfloat16", "bfloat16", "float16", "float32"))
        out = "float32" if rng.random() < 0.25 else dtype
        D, L = _width(rng, 16, 4096), _length(rng, 64, 32768)
        n = _log_int(rng, 1 << 17, 1 << 26)
        B = max(1, min(64, n // (L * D)))
        L = max(1, min(L, (1 << 27) // (B * D)))
        return _scan_case(None, kind, B, L, D, dtype, out, a_lo=rng.choice((0.9, 0.99)),
                          checkpoint=rng.random() < 0.85)
    if kind == "generate":
        L = 1 if rng.random() < 0.5 else _length(rng, 2, 2048)
        return _scan_case(None, kind, _log_int(rng, 1, 64), L, _width(rng, 256, 8192),
                          rng.choice(("bfloat16", "float16", "float32")))
    if kind in ("layer_train", "layer_infer"):
        params, compute = rng.choice((("bfloat16", "bfloat16"), ("float16", "float16"), ("float32", "float16"),
                                      ("float32", "bfloat16")))
        hidden = max(64, _width(rng, 128, 1024) // 8 * 8)
        rows = _log_int(rng, 512, 16384)
        L = max(1, min(rows, _length(rng, 64, 4096)))
        return _layer_case(None, kind, max(1, rows // L), L, hidden, rng.choice((1, 2, 4)), params, compute)
    return {"kind": kind, "layers": rng.randint(1, 6), "hidden": rng.choice((128, 256)), "batch": _log_int(rng, 4, 32),
            "seq": _log_int(rng, 8, 64), "compute": rng.choice(("float32", "float16", "bfloat16"))}


# ---- inputs ------------------------------------------------------------------------------------------------------


def _operands(case, gen):
    """x ~ N(0, 1), decays just below one, small input gates, output gates between 0 and 1, dy ~ N(0, 1)."""
    shape = (case["B"], case["L"], case["D"])
    dtype, out = _DTYPES[case["dtype"]], _DTYPES[case["out_dtype"]]
    new = lambda: torch.empty(shape, dtype=torch.float32, device="cuda")  # noqa: E731
    x = new().normal_(generator=gen).to(dtype)
    a = new().uniform_(case["a_lo"], 1.0, generator=gen).to(dtype)
    b = new().normal_(0.0, 0.1, generator=gen).to(dtype)
    c = new().normal_(generator=gen).sigmoid_().to(dtype)
    dy = new().normal_(generator=gen).to(out)
    return x, a, b, c, dy


def _seed_parameters(module, gen):
    """Linear weights as torch initialises them (uniform within 1 / sqrt(fan in)), from the case's own generator."""
    with torch.no_grad():
        for name, p in module.named_parameters():
            if name.endswith("embed.weight"):
                p.normal_(generator=gen)
            elif name.endswith("norm.weight"):
                p.uniform_(0.8, 1.2, generator=gen)
            else:
                bound = 1.0 / math.sqrt(p.shape[-1])
                p.uniform_(-bound, bound, generator=gen)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind in ("train", "pieces", "generate"):
        x, a, b, c, dy = _operands(case, gen)
        state = {"case": case, "ops": [x, a, b, c]}
        if kind != "train":
            h = torch.empty((case["B"], case["D"]), dtype=torch.float32, device="cuda")
            state["h"] = h.normal_(generator=gen)
        if kind != "generate":
            state["dy"] = dy
            leaves = state["ops"] + ([state["h"]] if kind == "pieces" else [])
            state["leaves"] = [t.requires_grad_(True) for t in leaves]
        if kind == "pieces":
            state["dh"] = torch.empty_like(state["h"]).detach().normal_(generator=gen)
        return state
    if kind in ("layer_train", "layer_infer"):
        dtype = _DTYPES[case["params"]]
        layer = SSM(case["hidden"], case["mult"], dtype=dtype, device="cuda", compute_dtype=_DTYPES[case["compute"]])
        _seed_parameters(layer, gen)
        shape = (case["B"], case["L"], case["hidden"])
        new = lambda: torch.empty(shape, dtype=torch.float32, device="cuda").normal_(generator=gen).to(dtype)  # noqa: E731
        state = {"case": case, "layer": layer, "x": new()}
        if kind == "layer_train":
            state["x"].requires_grad_(True)
            state["dy"] = new()
        return state
    model = copy_task.CopyStack(case["hidden"], case["layers"], _DTYPES[case["compute"]], torch.device("cuda"))
    _seed_parameters(model, gen)
    # the learning rate the schedule of the copy task starts its warm-up of 500 steps with
    opt = torch.optim.AdamW(model.parameters(), lr=1e-3 / 500, weight_decay=0.0)
    host = torch.Generator(device="cpu").manual_seed(seed)
    tokens, labels = copy_task.build_teacher_batch(case["batch"], case["seq"], torch.device("cuda"), generator=host)
    return {"case": case, "model": model, "opt": opt, "tokens": tokens, "labels": labels}


# ---- one pass ----------------------------------------------------------------------------------------------------


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "generate":
        with torch.no_grad():
            return scan_chunk(*state["ops"], state["h"], out_dtype=_DTYPES[case["out_dtype"]])
    if kind == "train":
        leaves = state["leaves"]
        for t in leaves:
            t.grad = None
        y = scan(*leaves, block_l=case["block_l"], checkpoint=case["checkpoint"], out_dtype=_DTYPES[case["out_dtype"]])
        y.backward(state["dy"])
        return [y.detach()] + [t.grad for t in leaves]
    if kind == "pieces":
        leaves = state["leaves"]
        for t in leaves:
            t.grad = None
        y, h = scan_chunk(*leaves, checkpoint=case["checkpoint"], out_dtype=_DTYPES[case["out_dtype"]])
        torch.autograd.backward((y, h), (state["dy"], state["dh"]))
        return [y.detach(), h.detach()] + [t.grad for t in leaves]
    if kind == "layer_infer":
        with torch.no_grad():
            return state["layer"](state["x"])
    if kind == "layer_train":
        layer, x = state["layer"], state["x"]
        x.grad = None
        layer.zero_grad(set_to_none=True)
        y = layer(x)
        y.backward(state["dy"])
        return [y.detach(), x.grad] + [p.grad for p in layer.parameters()]
    model = state["model"]
    loss, logits = copy_task.train_step(model, state["opt"], state["tokens"], state["labels"])
    return [loss, logits] + [p.grad for p in model.parameters()]


# ---- what a pass cannot do without ---------------------------------------------------------------------------------


def work(case):
    kind = case["kind"]
    if kind in ("train", "pieces", "generate"):
        n = case["B"] * case["L"] * case["D"]
        es, os_ = _BYTES[case["dtype"]], _BYTES[case["out_dtype"]]
        states = case["B"] * case["D"] * 4
        forward = n * (4 * es + os_)               # x, a, b, c in, y out
        backward = n * (8 * es + os_)              # x, a, b, c, dy in, dx, da, db, dc out
        if kind == "generate":
            return {"bytes": forward + 2 * states, "flops": 4 * n}
        return {"bytes": forward + backward + (5 * states if kind == "pieces" else 0), "flops": 14 * n}
    if kind in ("layer_train", "layer_infer"):
        rows, H = case["B"] * case["L"], case["hidden"]
        S = int(H * case["mult"])
        ps = _BYTES[case["params"]]
        weights = 6 * S * H + S + 2 * H
        if kind == "layer_infer":
            return {"bytes": (2 * rows * H + weights) * ps, "flops": 12 * rows * S * H}
        return {"bytes": (5 * rows * H + 3 * weights) * ps, "flops": 36 * rows * S * H}
    rows, H = case["batch"] * case["seq"] * 2, case["hidden"]
    S, V = 4 * H, copy_task.VOCAB_SIZE
    weights = case["layers"] * (6 * S * H + S + 2 * H) + 2 * V * H + V
    # weights read by both passes, gradients written and read, two moments and the weights read and written
    return {"bytes": 4 * (10 * weights + 3 * rows * V), "flops": rows * (36 * S * H * case["layers"] + 6 * V * H)}


# (rel, max) about four times what each path was seen to differ by from the same path in float64 on the same inputs.
_SCAN_TOL = {"float32": (1.2e-6, 1.5e-5), "float16": (8.4e-4, 2e-3), "bfloat16": (6.8e-3, 1.6e-2)}
_INFER_TOL = {("float32", "float16"): (6e-5, 4.2e-4), ("float32", "bfloat16"): (4.8e-4, 3.3e-3),
              ("float16", "float16"): (8.4e-4, 2.4e-3), ("bfloat16", "bfloat16"): (6.8e-3, 1.9e-2)}
_TRAIN_TOL = {("float32", "float16"): (1.9e-3, 1.3e-2), ("float32", "bfloat16"): (1.5e-2, 0.1),
              ("float16", "float16"): (3.2e-3, 2.1e-2), ("bfloat16", "bfloat16"): (2.6e-2, 0.17)}
_COPY_TOL = {"float32": (6e-6, 6.4e-5), "float16": (1.9e-3, 2.4e-2), "bfloat16": (1.5e-2, 0.2)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("train", "pieces", "generate"):
        rel, top = _SCAN_TOL[case["dtype"]]
    elif kind == "copy_step":
        rel, top = _COPY_TOL[case["compute"]]
    else:
        rel, top = (_INFER_TOL if kind == "layer_infer" else _TRAIN_TOL)[case["params"], case["compute"]]
    return {"rel": rel, "max": top}
