"""The work that users of this package have it do, as cases that can be timed and compared.

Every case goes through the modules and operators that the package exports, with the default ``scan_mode="auto"``,
in eager mode, as a program calls them.  The kinds:

``lru_train``      RG_LRU forward and backward: the recurrent layer inside somebody's own block.
``lru_forward``    RG_LRU without gradients over whole sequences, final state returned: evaluation and prefill.
``lru_step``       RG_LRU on one token per row with the carried state: a decode loop around the bare layer.
``block_train``    RMSNorm + RecurrentBlock forward and backward: one residual branch of a training step.
``block_forward``  RMSNorm + RecurrentBlock without gradients, cache in and out: (chunked) prefill.
``block_step``     RMSNorm + RecurrentBlock on one token per row with the carried cache: generation.
``scan``           the bare linear recurrence h = a h + z (fp32), forward and backward.

``tokens`` says which tokens count: "all" (every row is one document), "packed" (several documents to a row, marked
by a reset mask or by segment positions) or "padded" (rows of different lengths with padding behind them).
"""

import math

import torch

from griffin_amd import RG_LRU, RMSNorm, RecurrentBlock, RecurrentBlockCache, hip_rglru_scan

DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}
TAPS = 4


def _case(kind, batch, steps, width, blocks=16, dtype="bf16", tokens="all", carried=False, dim=0, slow=False):
    return {"kind": kind, "batch": batch, "steps": steps, "dim": dim, "width": width, "blocks": blocks, "dtype": dtype,
            "tokens": tokens, "carried": carried, "slow": slow}


def listed():
    named = {
        # the layer at the training shape of a 100M-parameter model: the shape of the package's headline figure
        "layer train B8 T2048 W1024": _case("lru_train", 8, 2048, 1024, blocks=8),
        # a small layer in full precision: unit-test and toy-model sized training, bound by launches and the host
        "layer train small f32": _case("lru_train", 2, 256, 256, blocks=8, dtype="f32"),
        # one long document, wide layer, slow decay: the state crosses the whole sequence
        "layer train long B1 T32768 W2560": _case("lru_train", 1, 32768, 2560, blocks=8, slow=True),
        # full-precision training at a real width, with the default number of gate blocks
        "layer train f32 B4 T1024 W1024": _case("lru_train", 4, 1024, 1024, dtype="f32"),
        # packed documents, odd batch and length, rnn width = model width with the default number of gate blocks
        "layer train packed B3 T1537 W768": _case("lru_train", 3, 1537, 768, tokens="packed", carried=True),
        # prompts of a large serving batch in front of the decode loop
        "layer prefill B256 T2048 W1024": _case("lru_forward", 256, 2048, 1024, blocks=8),
        # one token for each sequence of that batch
        "layer decode B256 W1024": _case("lru_step", 256, 1, 1024, blocks=8, carried=True),
        # the residual branch (norm, projections, convolution, recurrence, gate, projection) at the training shape
        "block train B8 T2048 W1024": _case("block_train", 8, 2048, 1024, dim=768),
        # the same branch on a batch of sequences of different lengths
        "block train padded B8 T2048 W1024": _case("block_train", 8, 2048, 1024, dim=768, tokens="padded"),
        # the next chunk of a few prompts, of ragged length, behind a cache
        "block prefill B3 T777 W1024": _case("block_forward", 3, 777, 1024, dim=768, carried=True),
        # generation for a single user: the smallest call there is
        "block decode B1 W1024": _case("block_step", 1, 1, 1024, dim=768, carried=True),
        # the bare recurrence for callers that compute their own gates
        "scan B8 T2048 W1024 f32": _case("scan", 8, 2048, 1024, dtype="f32", carried=True),
    }
    return [dict(c, name=name) for name, c in named.items()]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """One more case: batch and length spread over their logarithms and not rounded, so most of them are odd."""
    kind = rng.choice(("lru_train", "lru_train", "lru_forward", "lru_step", "block_train", "block_forward", "block_step", "scan"))
    dtype = "f32" if kind == "scan" or rng.random() < 0.25 else "bf16"
    # widths that people choose are multiples of 128; a few are anything
    width = 128 * _log(rng, 2, 20) if rng.random() < 0.85 else 8 * _log(rng, 16, 160)
    dim = 0
    if kind.startswith("block"):
        dim = width if rng.random() < 0.5 else 64 * max(2, round(width * 0.75 / 64))
    blocks = rng.choice((8, 16))
    if kind.endswith("step"):
        return _case(kind, _log(rng, 1, 512), 1, width, blocks, dtype, "all", True, dim)
    # elements of one activation tensor: no case is larger than the largest listed one of its sort
    most = {"lru_forward": 1 << 27, "block_forward": 1 << 25, "lru_train": 1 << 24, "block_train": 1 << 24, "scan": 1 << 25}[kind]
    if dtype == "f32" and kind != "scan":
        most //= 4
    if kind == "block_train":
        most = min(most, (1 << 33) // dim)                          # the projections grow with the model width as well
    elements = _log(rng, 1 << 17, most)
    steps = min(_log(rng, 32, 8192), max(16, elements // width))
    batch = max(1, elements // (width * steps))
    tokens = rng.choice(("all", "packed", "padded")) if kind != "scan" else "all"
    carried = kind == "scan" or (kind != "block_train" and rng.random() < 0.5)
    return _case(kind, batch, steps, width, blocks, dtype, tokens, carried, dim, rng.random() < 0.25)


# ---- what a program holds before the call ------------------------------------------------------------------------

def _normal(*shape, dtype=torch.float32, std=1.0, leaf=False):
    t = torch.randn(*shape, device="cuda", dtype=dtype)
    if std != 1.0:
        t *= std
    return t.requires_grad_(leaf)


def _lengths(case):
    """Active tokens of each row of a padded batch: evenly spread from a 26th of the length to all of it."""
    batch, steps = case["batch"], case["steps"]
    least = max(1, steps // 26)
    return [steps if batch == 1 else least + (steps - least) * i // (batch - 1) for i in range(batch)]


def _spread(parameters):
    """Biases as training leaves them: not at the zeros they are initialised with."""
    with torch.no_grad():
        for name, p in parameters:
            if name.endswith("bias"):
                p.normal_(std=0.1)


def _decays(layer, slow):
    """sigmoid(Lambda)^c uniform on [0.9, 0.999], or on [0.99, 0.9999] for long memories."""
    low, high = (0.99, 0.9999) if slow else (0.9, 0.999)
    with torch.no_grad():
        layer.Lambda.copy_(torch.logit(torch.empty_like(layer.Lambda).uniform_(low, high).pow(1.0 / layer.c)))


def prepare(case, seed):
    torch.manual_seed(seed)
    kind, dtype = case["kind"], DTYPES[case["dtype"]]
    batch, steps, width, dim = case["batch"], case["steps"], case["width"], case["dim"]
    train = kind.endswith("train") or kind == "scan"
    s = {"kind": kind}
    if kind == "scan":
        s["a"] = torch.sigmoid(_normal(batch, steps, width) + 2.0).requires_grad_(True)
        s["z"] = _normal(batch, steps, width, leaf=True)
        s["h"] = _normal(batch, width, leaf=True)
        s["dy"] = _normal(batch, steps, width)
        return s

    with torch.device("cuda"):
        if dim:
            norm, block = RMSNorm(dim), RecurrentBlock(dim, width, conv_kernel_size=TAPS, gate_blocks=case["blocks"])
            layer = block.rg_lru
            with torch.no_grad():
                norm.g.normal_(std=0.1)
            modules = [norm, block]
        else:
            layer = RG_LRU(width, gate_blocks=case["blocks"])
            modules = [layer]
    for m in modules:
        _spread(m.named_parameters())
    _decays(layer, case["slow"])
    modules = [m.to(dtype).train(train) for m in modules]
    s["layer"] = modules[-1]
    s["norm"] = modules[0] if dim else None
    s["parameters"] = [p for m in modules for p in m.parameters()]

    features = dim or width
    s["x"] = _normal(batch, steps, features, dtype=dtype, leaf=train)
    s["dy"] = _normal(batch, steps, features, dtype=dtype) if train else None

    s["reset"] = s["active"] = s["positions"] = None
    token = torch.arange(steps, device="cuda")
    if case["tokens"] == "packed":
        # documents of about a fifth of the row, another cut in every row
        starts = torch.rand(batch, steps, device="cuda") < 5.0 / steps
        starts[:, 0] = True
        begin = torch.where(starts, token, 0).cummax(dim=1).values
        s["reset"], s["positions"] = starts, token - begin
    elif case["tokens"] == "padded":
        lengths = torch.tensor(_lengths(case), device="cuda")[torch.randperm(batch, device="cuda")]
        s["active"] = token[None, :] < lengths[:, None]

    s["h"] = s["cache"] = None
    if case["carried"]:
        state = _normal(batch, width, std=0.5, leaf=train)
        if dim:
            # a cache as an earlier chunk of 100 tokens leaves it
            s["cache"] = RecurrentBlockCache(state, _normal(batch, TAPS - 1, width, dtype=dtype),
                                             torch.full((batch,), 99, device="cuda", dtype=torch.long))
        else:
            s["h"] = state
    return s


# ---- one pass ------------------------------------------------------------------------------------------------------

def run(s):
    kind = s["kind"]
    if kind == "scan":
        y = hip_rglru_scan(s["a"], s["z"], s["h"])
        return [y, *torch.autograd.grad(y, [s["a"], s["z"], s["h"]], s["dy"])]

    layer = s["layer"]
    if kind == "lru_train":
        y, h = layer(s["x"], s["h"], reset_mask=s["reset"], active_mask=s["active"], return_state=True)
        leaves = [s["x"], *s["parameters"]] + ([] if s["h"] is None else [s["h"]])
        return [y, h, *torch.autograd.grad(y, leaves, s["dy"])]
    if kind == "block_train":
        y = layer(s["norm"](s["x"]), segment_pos=s["positions"], active_mask=s["active"])
        return [y, *torch.autograd.grad(y, [s["x"], *s["parameters"]], s["dy"])]
    with torch.no_grad():
        if kind == "lru_forward":
            return layer(s["x"], s["h"], reset_mask=s["reset"], active_mask=s["active"], return_state=True)
        if kind == "lru_step":
            y, s["h"] = layer(s["x"], s["h"], return_state=True)   # the loop's next pass goes on from this state
            return y, s["h"]
        y, cache = layer(s["norm"](s["x"]), s["cache"], s["positions"], active_mask=s["active"], return_cache=True)
        if kind == "block_step":
            s["cache"] = cache
        return y, cache.rnn_state, cache.conv_state, cache.segment_position


# ---- what a pass cannot do without ---------------------------------------------------------------------------------

def work(case):
    """Bytes: inputs and parameters read once, outputs and gradients written once, for the tokens that count (padding
    is only written).  Operations: the matrix products, two per multiply-add, and about as many elementwise ones as
    the formulas of the gates and of the recurrence have."""
    kind, size = case["kind"], DTYPES[case["dtype"]].itemsize
    batch, steps, width, dim = case["batch"], case["steps"], case["width"], case["dim"]
    tokens = batch * steps
    n = tokens * width
    if kind == "scan":
        return {"bytes": 4 * (6 * n + 2 * batch * width), "flops": 5 * n}

    live = sum(_lengths(case)) if case["tokens"] == "padded" else tokens
    blocks = case["blocks"]
    while width % blocks:
        blocks -= 1
    block_width = width // blocks
    train = kind.endswith("train")
    features = dim or width
    parameters = 2 * width * block_width + 3 * width
    products = 2 * width * block_width                              # multiply-adds a token
    elementwise = 20 * width
    if dim:
        parameters += 3 * width * dim + 2 * width + dim + width * (TAPS + 1) + dim
        products += 3 * width * dim
        elementwise += (2 * TAPS + 10) * width + 4 * dim
    activations = (live + tokens) * features                        # x in, y out
    if train:
        activations *= 2                                            # dy in, dx out
        parameters *= 2
        products *= 3
        elementwise *= 3
    total = size * (activations + parameters)
    if case["carried"]:
        total += 2 * 4 * batch * width
        if dim:
            total += 2 * size * batch * (TAPS - 1) * width
    return {"bytes": total, "flops": live * (2 * products + elementwise)}


def tolerance(case):
    """bf16 storage rounds every activation to 8 bits; fp32 leaves the rounding of long sums."""
    return {"rel": 1e-2} if case["dtype"] == "bf16" else {"rel": 2e-5}
