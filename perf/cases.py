"""The work a user of this package has it do, through its public entry points: what a change to the kernels or to the
host path is timed on.

Twelve listed cases stand for the range; ``draw`` gives further ones of the same kinds, sizes and options. Attention cases
run ``function.scaled_dot_product_attention`` and, where they train, the gradients of query, key, value and of a mask that
asks for one; row cases run ``function.masked_softmax`` / ``function.softmax`` and ``function.dropout`` the same way.

Fields of an attention case: ``dtype``, ``B``, ``H``, ``S``, ``D``, ``causal``, ``dropout``, ``train`` (forward only, or
forward and backward), ``layout`` ("bhsd": dense [B,H,S,D]; "bshd": the [B,S,H,D] result of a projection, seen as
[B,H,S,D]) and ``mask``:
  none
  length    additive fp32 [B,1,S,S], keys behind the sequence's length at -inf (lengths in [S/2, S])
  padding   boolean [B,1,1,S], True where the key exists (same lengths)
  dense     additive fp32 [B,1,S,S], N(0, 0.5) in every entry
  bias      additive [1,H,S,S] in the operand type, learned: it has a gradient
Fields of a row case: ``dtype``, ``rows``, ``cols``, ``dim`` (0 or 1), ``masked`` (a uint8 mask, a quarter of it set),
``dropout``, ``train``.
"""
import math

import torch

import trident_amd as trident

# any sequence length and boolean masks, as torch's own attention takes them
trident.config.reference_limits = False

_DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}


def _attention(dtype, B, H, S, D, causal=False, mask="none", dropout=0.0, train=True, layout="bhsd", name=None):
    case = {"op": "attention", "dtype": dtype, "B": B, "H": H, "S": S, "D": D, "causal": causal, "mask": mask,
            "dropout": dropout, "train": train, "layout": layout}
    return case if name is None else dict(case, name=name)


def _rows(dtype, rows, cols, dim=1, masked=False, dropout=0.0, train=True, name=None):
    case = {"op": "rows", "dtype": dtype, "rows": rows, "cols": cols, "dim": dim, "masked": masked, "dropout": dropout,
            "train": train}
    return case if name is None else dict(case, name=name)


def listed():
    return [
        # the smallest call of the benchmark configurations (C1): one launch, all latency
        _attention("float32", 2, 4, 64, 32, train=False, name="tiny_fp32_fwd"),
        # the reference's attention benchmark at a short length, forward and backward: launches and host work count
        _attention("float16", 32, 8, 128, 64, name="short_fp16_train"),
        # an encoder's forward pass in fp16 (C2)
        _attention("float16", 4, 16, 1024, 64, train=False, name="encoder_fp16_fwd"),
        # the reference's benchmark as it runs by default: fp32, its longest length
        _attention("float32", 32, 8, 512, 64, name="bench_fp32_train"),
        # the headline workload (C3): a decoder's training step in bf16
        _attention("bfloat16", 2, 16, 4096, 128, causal=True, name="causal_bf16_train"),
        # the same kind of step on a batch whose length is what the text gave, straight from the projections
        _attention("bfloat16", 4, 16, 1531, 128, causal=True, layout="bshd", name="ragged_causal_bf16_train"),
        # an encoder's training step with a length mask as an additive matrix (C4)
        _attention("bfloat16", 8, 12, 2048, 64, mask="length", name="length_mask_bf16_train"),
        # an encoder's training step on a padded batch: boolean key-padding mask, an odd length
        _attention("float16", 16, 12, 777, 64, mask="padding", layout="bshd", name="padding_fp16_train"),
        # attention with a learned additive bias per head, shared by the batch: the mask has a gradient
        _attention("bfloat16", 8, 12, 512, 64, mask="bias", name="bias_bf16_train"),
        # the longest sequence (C5): causal with dropout
        _attention("bfloat16", 1, 32, 16384, 128, causal=True, dropout=0.1, name="long_dropout_bf16_train"),
        # attention probabilities written out: masked softmax along odd-length rows, then dropout
        _rows("bfloat16", 12288, 2047, masked=True, dropout=0.1, name="probabilities_bf16_train"),
        # softmax down the columns of a matrix
        _rows("float32", 4096, 4096, dim=0, name="columns_fp32_train"),
    ]


def _spread(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _length(rng, low, high):
    """Over the logarithm of the range: a power of two, a multiple of 64, or any length."""
    s = _spread(rng, low, high)
    kind = rng.randrange(3)
    if kind == 0:
        return min(high, 1 << max(4, round(math.log2(s))))
    return max(64, s // 64 * 64) if kind == 1 and s >= 64 else s


def draw(rng):
    if rng.random() < 0.2:
        dtype = rng.choice(["float32", "float16", "bfloat16"])
        cols = _spread(rng, 64, 16384)
        if rng.random() < 0.5:
            cols = max(8, cols // 8 * 8)
        rows = max(16, min(65536, _spread(rng, 1 << 14, 1 << 26) // cols))
        masked = rng.random() < 0.5
        return _rows(dtype, rows, cols, dim=0 if rng.random() < 0.25 else 1, masked=masked,
                     dropout=0.1 if rng.random() < 0.4 else 0.0, train=rng.random() < 0.7)
    dtype = rng.choice(["float32", "float16", "float16", "bfloat16", "bfloat16", "bfloat16"])
    D = rng.choice([16, 32, 64, 64, 64, 128, 128, 128])
    kind = rng.choice(["plain", "causal", "causal", "causal", "length", "padding", "padding", "dense", "bias"])
    mask = kind if kind not in ("plain", "causal") else "none"
    S = _length(rng, 32, 2048 if mask in ("length", "dense", "bias") else (4096 if dtype == "float32" else 16384))
    # scores of the pass: up to 1/8 of the longest case's, 1/32 in fp32; at least what a call of a few heads has
    limit = (1 << 33) // (32 if dtype == "float32" else 8)
    heads = max(4, min(1024, _spread(rng, 1 << 16, limit) // (S * S)))
    H = rng.choice([h for h in (4, 8, 12, 16, 32) if h <= heads])
    B = max(1, heads // H)
    if mask in ("length", "dense"):
        B = min(B, max(1, (1 << 27) // (S * S)))  # (the mask matrix: at most 512 MiB)
    return _attention(dtype, B, H, S, D, causal=kind == "causal", mask=mask,
                      dropout=rng.choice([0.0, 0.0, 0.0, 0.1]), train=rng.random() < 0.7,
                      layout=rng.choice(["bhsd", "bshd"]))


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    dtype = _DTYPES[case["dtype"]]
    train = case["train"]
    state = {"case": case, "seed": seed}
    if case["op"] == "rows":
        shape = (case["rows"], case["cols"])
        state["x"] = torch.randn(shape, generator=g, device="cuda").mul_(3.0).to(dtype).requires_grad_(train)
        if case["masked"]:
            state["mask"] = (torch.rand(shape, generator=g, device="cuda") < 0.25).to(torch.uint8)
            state["mask"][:, 0] = 0  # (no row or column is masked out altogether)
            state["mask"][0, :] = 0
        if train:
            state["grad"] = torch.randn(shape, generator=g, device="cuda").to(dtype)
        return state

    B, H, S, D = case["B"], case["H"], case["S"], case["D"]

    def tensor():
        if case["layout"] == "bshd":
            return torch.randn((B, S, H, D), generator=g, device="cuda").to(dtype).transpose(1, 2)
        return torch.randn((B, H, S, D), generator=g, device="cuda").to(dtype)

    state["q"], state["k"], state["v"] = (tensor().requires_grad_(train) for _ in range(3))
    if train:
        state["grad"] = tensor()
    mask = None
    if case["mask"] in ("length", "padding"):
        lengths = torch.randint((S + 1) // 2, S + 1, (B,), generator=g, device="cuda")
        exists = torch.arange(S, device="cuda")[None, :] < lengths[:, None]
        if case["mask"] == "padding":
            mask = exists[:, None, None, :].contiguous()
        else:
            mask = torch.zeros((B, 1, S, S), device="cuda").masked_fill_(~exists[:, None, None, :], float("-inf"))
    elif case["mask"] == "dense":
        mask = torch.randn((B, 1, S, S), generator=g, device="cuda").mul_(0.5)
    elif case["mask"] == "bias":
        mask = torch.randn((1, H, S, S), generator=g, device="cuda").mul_(0.5).to(dtype).requires_grad_(train)
    state["mask"] = mask
    return state


def run(state):
    case = state["case"]
    if case["dropout"] > 0.0:
        trident.config.dropout_seed = (state["seed"], 0)  # (a fixed dropout stream: the same decisions in every pass)
    if case["op"] == "rows":
        x = state["x"]
        if case["masked"]:
            probabilities = trident.function.masked_softmax(x, state["mask"], case["dim"])
        else:
            probabilities = trident.function.softmax(x, case["dim"])
        out = trident.function.dropout(probabilities, case["dropout"]) if case["dropout"] > 0.0 else probabilities
        if not case["train"]:
            return out
        (grad,) = torch.autograd.grad(out, (x,), state["grad"])
        return {"out": out.detach(), "grad": grad}

    q, k, v, mask = state["q"], state["k"], state["v"], state["mask"]
    out = trident.function.scaled_dot_product_attention(q, k, v, mask, case["dropout"], case["causal"])
    if not case["train"]:
        return out
    names = ["grad_query", "grad_key", "grad_value"]
    inputs = [q, k, v]
    if mask is not None and mask.requires_grad:
        names.append("grad_mask")
        inputs.append(mask)
    return {"out": out.detach(), **dict(zip(names, torch.autograd.grad(out, inputs, state["grad"])))}


def work(case):
    size = 4 if case["dtype"] == "float32" else 2
    if case["op"] == "rows":
        n = case["rows"] * case["cols"]
        tensors = 4 if case["train"] else 2  # input, output, output's gradient, input's gradient
        return {"bytes": tensors * n * size + (n if case["masked"] else 0), "flops": n * (12 if case["train"] else 6)}
    B, H, S, D = case["B"], case["H"], case["S"], case["D"]
    visible = S * (S + 1) / 2 if case["causal"] else float(S * S)
    if case["mask"] in ("length", "padding"):
        visible *= 0.75  # (the average length is 3 S / 4)
    tensors = 8 if case["train"] else 4
    mask_bytes = {"none": 0, "length": 4 * B * S * S, "dense": 4 * B * S * S, "padding": B * S,
                  "bias": (2 if case["train"] else 1) * size * H * S * S}[case["mask"]]
    return {"bytes": tensors * B * H * S * D * size + mask_bytes, "flops": (14 if case["train"] else 4) * B * H * visible * D}


def tolerance(case):
    # About four times the largest error measured against the same computation in 64 bits, over head sizes, masks, dropout
    # and lengths ("rel"; "max" in brackets):
    #   attention  fp32 1.2e-6 (4.6e-5)   fp16 3.5e-4 (1.5e-2)   bf16 2.8e-3 (0.12)
    #   rows       fp32 7.2e-7 (3.0e-5)   fp16 3.1e-4 (3.1e-2)   bf16 2.4e-3 (0.28); dropout rounds 16 bits once more
    #   columns in fp32: a sum in plain order down the column is off in proportion to its length, 2.6e-6 at 4096 elements
    #   and 7.5e-5 (2.0e-3) at 65536
    dtype = case["dtype"]
    if case["op"] == "rows":
        limits = {"float32": {"rel": 3e-6, "max": 1.2e-4}, "float16": {"rel": 1.4e-3, "max": 0.13}, "bfloat16": {"rel": 1.1e-2, "max": 0.95}}
        if dtype == "float32" and case["dim"] == 0:
            rel = max(3e-6, 4.8e-9 * case["rows"])
            return {"rel": rel, "max": 40 * rel}
        return limits[dtype]
    return {"float32": {"rel": 5e-6, "max": 2e-4}, "float16": {"rel": 1.4e-3, "max": 6e-2}, "bfloat16": {"rel": 1.1e-2, "max": 0.5}}[dtype]
