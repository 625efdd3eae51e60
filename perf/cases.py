"""The calls that a user of the package makes, as measurable cases.

Each case is one pass of a differentially private training step's
clip -> sum -> noise path, through a public entry point:

``linear``   ``ghost_clip_sum``: one linear layer from its inputs and output gradients
``block``    ``ghost_clip_captured``: a Llama-style block's projections and norm weights
``lora``     ``ghost_clip_captured``: the 14 adapter layers of a LoRA block
``moe``      ``ghost_clip_captured``: the experts of a top-2 MoE FFN, clipped per expert
``mlp``      ``ghost_clipped_grad``: a whole step (forward, backward, clip, noise)
``leaves``   ``clipped_fun``: per-example gradients that already exist, any model
``noise``    ``gaussian_noise``: the noise alone, on a model's parameter tree

``listed()`` names twelve of them, ``draw(rng)`` gives more of the same
ranges.  ``exact`` restates each pass in 64 bits with plain torch.
"""

from __future__ import annotations

import hashlib
import math

import opake_amd  # noqa: F401  (first: it sets HIP's options before the GPU is used)
import torch

from opake_amd.clipping import (
    DirectCapture,
    LinearCapture,
    clipped_fun,
    ghost_clip_captured,
    ghost_clip_sum,
    ghost_clipped_grad,
)
from opake_amd.noise import gaussian_noise
from opake_amd.random import key
from opake_amd.types import PerGroup, clipped

C = 1.0  # clipping norm
GAMMA = 0.01  # AUTO-S
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}


# --------------------------------------------------------------------------
# Cases
# --------------------------------------------------------------------------


def _linear(name, B, T, din, dout, dtype="bf16", bias=False, noise=True, auto=False, out="same"):
    """``out``: "same" (the operand dtype) or "fp32" (sums that are accumulated
    over microbatches before the noise)."""
    return dict(name=name, kind="linear", B=B, T=T, din=din, dout=dout, dtype=dtype, bias=bias,
                noise=noise, auto=auto, out=out)


def listed():
    return [
        # The smallest call: a narrow layer on a short batch, where launches and host
        # time are all there is.
        _linear("linear_tiny", 4, 24, 64, 96),
        # The headline workload: one 4096 x 4096 projection of a sequence model.
        _linear("linear_headline", 32, 512, 4096, 4096),
        # A vision or speech encoder's feed-forward layer: a bias, a sequence length that no
        # tile divides, sums kept in float32 for accumulation over microbatches.
        _linear("linear_ragged_bias", 24, 197, 768, 3072, bias=True, noise=False, out="fp32"),
        # A classification or token head: an odd number of outputs.
        _linear("linear_odd_head", 16, 384, 1024, 1001, bias=True),
        # Training in float32, AUTO-S scaling.
        _linear("linear_fp32", 16, 256, 1024, 1024, dtype="fp32", bias=True, noise=False,
                auto=True),
        # A Llama-style block: the largest dense case.
        dict(name="block", kind="block", B=16, T=1024, d=2048, ffn=8192, noise=True),
        # LoRA fine-tuning of an 8B-shaped block.
        dict(name="lora", kind="lora", B=8, T=2048, d=4096, kv=1024, ffn=14336, r=16, noise=True),
        # Top-2 MoE FFN, per-expert clipping: the largest case.
        dict(name="moe", kind="moe", B=16, T=1024, d=2048, ffn=5632, experts=8, noise=True),
        # The MLP step of the parity configuration, whole.
        dict(name="mlp_step", kind="mlp", B=256, din=784, hidden=512, classes=10, noise=True),
        # Materialised per-example gradients of one big bf16 layer: two passes over memory.
        dict(name="leaves_one_bf16", kind="leaves", B=32, net="one", width=4096, odd=0,
             dtype="bf16", groups=1, aux=False, second=False, noise=True),
        # A small convolutional net's per-example gradients: many leaves of all sizes (rows
        # that start at any alignment), per-layer groups, diagnostics and the second moment.
        dict(name="leaves_conv_fp32", kind="leaves", B=64, net="conv", width=48, odd=1,
             dtype="fp32", groups=4, aux=True, second=True, noise=False),
        # Noise on a block's parameter tree (the step after an accumulated sum).
        dict(name="noise_block", kind="noise", d=2048, ffn=8192, odd=0, dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A layer width: a multiple of 64 or 8 as most are, or any number."""
    w = _log(rng, lo, hi)
    step = rng.choice((64, 64, 8, 1))
    return max(lo, w // step * step)


def _draw(rng):
    kind = rng.choice(("linear",) * 4 + ("leaves",) * 2 + ("block", "lora", "moe", "mlp", "noise"))
    if kind == "linear":
        dtype = rng.choice(("bf16", "bf16", "bf16", "fp32"))
        top = 4096 if dtype == "bf16" else 1536
        T = rng.choice((_log(rng, 2, 1024), 64 * rng.randint(1, 16)))
        noise = rng.random() < 0.5
        return _linear("", _log(rng, 1, 48), T, _width(rng, 32, top), _width(rng, 32, top), dtype,
                       bias=rng.random() < 0.5, noise=noise, auto=rng.random() < 0.25,
                       out="same" if noise else rng.choice(("same", "fp32")))
    if kind == "block":
        d = 64 * rng.randint(4, 32)
        return dict(kind=kind, B=_log(rng, 1, 24),
                    T=rng.choice((_log(rng, 16, 1024), 128 * rng.randint(1, 8))), d=d,
                    ffn=8 * _log(rng, d // 4, d // 2), noise=rng.random() < 0.5)
    if kind == "lora":
        d = 128 * rng.randint(2, 32)
        return dict(kind=kind, B=_log(rng, 1, 8), T=_log(rng, 64, 2048), d=d,
                    kv=d // rng.choice((1, 2, 4)), ffn=8 * _log(rng, d // 4, int(d * 0.4375)),
                    r=rng.choice((4, 8, 16, 32)), noise=rng.random() < 0.5)
    if kind == "moe":
        return dict(kind=kind, B=_log(rng, 2, 16), T=_log(rng, 64, 1024), d=64 * rng.randint(4, 32),
                    ffn=8 * _log(rng, 64, 704), experts=rng.choice((4, 8)),
                    noise=rng.random() < 0.5)
    if kind == "mlp":
        return dict(kind=kind, B=_log(rng, 16, 1024), din=_log(rng, 64, 1024),
                    hidden=_log(rng, 64, 1024), classes=rng.choice((2, 10, 100)),
                    noise=rng.random() < 0.5)
    if kind == "leaves":
        net = rng.choice(("one", "conv"))
        top = 4096 if net == "one" else 64
        return dict(kind=kind, B=_log(rng, 2, 64), net=net, width=_log(rng, top // 16, top),
                    odd=rng.randint(0, 1), dtype=rng.choice(("bf16", "fp32", "fp16")),
                    groups=1 if net == "one" else rng.choice((1, 4)), aux=rng.random() < 0.5,
                    second=rng.random() < 0.25, noise=rng.random() < 0.5)
    return dict(kind="noise", d=_log(rng, 64, 2048), ffn=_log(rng, 128, 8192),
                odd=rng.randint(0, 1), dtype=rng.choice(("bf16", "fp32")))


def draw(rng):
    """A case of the listed ranges that costs no more than the largest listed one."""
    top = [work(c) for c in listed()]
    flops, nbytes = (max(w[k] for w in top) for k in ("flops", "bytes"))
    while True:
        case = _draw(rng)
        case.pop("name", None)
        w = work(case)
        # float32 runs at a sixteenth of the bf16 matrix rate.
        cost = w["flops"] * (16 if case.get("dtype") == "fp32" else 1)
        if cost <= flops and w["bytes"] <= nbytes:
            return case


# --------------------------------------------------------------------------
# Shapes and work
# --------------------------------------------------------------------------


def _block_layers(case):
    d, f = case["d"], case["ffn"]
    return [("qkv", d, 3 * d), ("o", d, d), ("gate_up", d, 2 * f), ("down", f, d)]


def _lora_layers(case):
    """(name, input it reads, din, dout): the projections an adapter pair sits on."""
    d, kv, f = case["d"], case["kv"], case["ffn"]
    return [("q", "attn", d, d), ("k", "attn", d, kv), ("v", "attn", d, kv), ("o", "att", d, d),
            ("gate", "mlp", d, f), ("up", "mlp", d, f), ("down", "act", f, d)]


def _moe_layers(case):
    return [("gate_up", case["d"], 2 * case["ffn"]), ("down", case["ffn"], case["d"])]


def _leaf_shapes(case):
    """Parameter shapes: one square layer, or a convolutional net (3 x 3 kernels, norm
    scales and biases, a linear head)."""
    w, odd = case["width"], case["odd"]
    if case["net"] == "one":
        return {"weight": (w, w + odd)}
    shapes, cin = {}, 3
    for i, cout in enumerate((w, w, 2 * w, 2 * w, 4 * w, 4 * w)):
        cout += odd
        shapes[f"conv{i}.weight"] = (cout, cin, 3, 3)
        shapes[f"norm{i}.weight"] = (cout,)
        shapes[f"norm{i}.bias"] = (cout,)
        cin = cout
    shapes["head.weight"] = (10, cin)
    shapes["head.bias"] = (10,)
    return shapes


def _noise_shapes(case):
    d, f, odd = case["d"] + case["odd"], case["ffn"], case["odd"]
    return {"block.attn_norm.weight": (d,), "block.qkv.weight": (3 * d, d),
            "block.o.weight": (d, d), "block.mlp_norm.weight": (d,),
            "block.gate_up.weight": (2 * f, d), "block.down.weight": (d, f + odd)}


def work(case):
    """Bytes: each input read once, each output written once.  Flops: per-example norms
    through the smaller of the Gram matrix and the gradient itself, and the clipped sum."""
    k = case["kind"]
    if k == "noise":
        n = sum(math.prod(s) for s in _noise_shapes(case).values())
        return {"bytes": 2 * n * BYTES[case["dtype"]], "flops": 2 * n}
    if k == "leaves":
        n = sum(math.prod(s) for s in _leaf_shapes(case).values())
        outs = 2 if case["second"] else 1
        return {"bytes": (case["B"] + outs) * n * BYTES[case["dtype"]],
                "flops": (4 + 2 * (outs - 1)) * case["B"] * n}
    B = case["B"]
    if k == "mlp":
        i, h, c = case["din"], case["hidden"], case["classes"]
        params = i * h + h + h * c + c
        # Forward, backward to the hidden layer, the two clipped sums.
        return {"bytes": 4 * (B * i + 2 * params),
                "flops": 2 * B * (2 * i * h + 3 * h * c)}
    if k == "lora":
        T, r, flops, ins, outs = case["T"], case["r"], 0, {}, 0
        for n, src, i, o in _lora_layers(case):
            flops += 2 * B * T * r * (i + o)
            ins[src] = i
            ins[n] = 2 * r + o
            outs += r * (i + o)
        return {"bytes": 2 * (B * T * sum(ins.values()) + outs), "flops": flops}
    if k == "linear":
        layers = [(case["din"], case["dout"], [case["T"]] * B)]
        in_bytes, out_bytes = BYTES[case["dtype"]], 4 if case["out"] == "fp32" else None
    elif k == "block":
        layers = [(i, o, [case["T"]] * B) for _, i, o in _block_layers(case)]
        in_bytes, out_bytes = 2, None
    else:  # moe: every expert takes its even share of each example's tokens
        seg = max(1, case["T"] * 2 // case["experts"])
        layers = [(i, o, [seg] * B) for _, i, o in _moe_layers(case)] * case["experts"]
        in_bytes, out_bytes = 2, None
    nbytes = flops = 0
    for i, o, rows in layers:
        n = sum(rows)
        nbytes += n * (i + o) * in_bytes + i * o * (out_bytes or in_bytes)
        flops += 2 * n * i * o
        flops += sum(min(t * (t + 1) * (i + o) + 2 * t * t, 2 * t * i * o) for t in rows)
    return {"bytes": nbytes, "flops": flops}


# --------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------


def _device():
    return torch.device("cuda:0")


def _gen(seed, tag):
    digest = hashlib.blake2b(f"{tag}/{seed}".encode(), digest_size=7).digest()
    return torch.Generator(device=_device()).manual_seed(int.from_bytes(digest, "little"))


def _randn(g, shape, scale=1.0, dtype=torch.bfloat16):
    x = torch.randn(shape, generator=g, device=_device())
    return (x * scale).to(dtype)


def _factors(g, B):
    """Per-example gradient scales: lognormal, so that about half are clipped."""
    return torch.exp(torch.randn(B, generator=g, device=_device()))


def _operands(g, B, T, din, dout, factor, n_layers=1, dtype=torch.bfloat16):
    """Activations N(0, 1) and output gradients whose per-example weight gradient has norm
    ``factor * C / sqrt(n_layers)``."""
    sigma = C / math.sqrt(n_layers * T * din * dout)
    A = _randn(g, (B, T, din), dtype=dtype)
    G = _randn(g, (B, T, dout), factor[:, None, None] * sigma, dtype)
    return A, G


def _linear_inputs(case, seed):
    g = _gen(seed, "linear")
    A, G = _operands(g, case["B"], case["T"], case["din"], case["dout"], _factors(g, case["B"]),
                     dtype=DTYPES[case["dtype"]])
    return {"A": A, "G": G}


def _block_inputs(case, seed):
    g = _gen(seed, "block")
    B, T = case["B"], case["T"]
    factor = _factors(g, B)
    layers = [(n, *_operands(g, B, T, i, o, factor, 4)) for n, i, o in _block_layers(case)]
    scale = factor[:, None] * (0.01 / math.sqrt(case["d"]))
    norms = {f"{n}.weight": _randn(g, (B, case["d"]), scale) for n in ("attn_norm", "mlp_norm")}
    return {"layers": layers, "norms": norms}


def _lora_inputs(case, seed):
    g = _gen(seed, "lora")
    B, T, r = case["B"], case["T"], case["r"]
    factor = _factors(g, B)
    x, layers = {}, []
    for n, src, i, o in _lora_layers(case):
        if src not in x:
            x[src] = _randn(g, (B, T, i))
        sa, sb = (C / math.sqrt(14 * T * r * w) for w in (i, o))
        layers.append((f"{n}.lora_A", x[src], _randn(g, (B, T, r), factor[:, None, None] * sa)))
        layers.append((f"{n}.lora_B", _randn(g, (B, T, r)),
                       _randn(g, (B, T, o), factor[:, None, None] * sb)))
    return {"layers": layers}


def _moe_inputs(case, seed):
    """Expert rows as a top-2 router with N(0, 1) logits deals them: sorted by expert, in
    example order, with each example's row count."""
    g = _gen(seed, "moe")
    B, T, E = case["B"], case["T"], case["experts"]
    logits = torch.randn(B, T, E, generator=g, device=_device())
    expert = torch.topk(logits, 2, dim=-1).indices.reshape(B, -1)
    counts = torch.stack([(expert == e).sum(dim=1) for e in range(E)]).cpu()
    factor = _factors(g, B)
    layers = []
    for e in range(E):
        seg = counts[e].tolist()
        row_f = torch.repeat_interleave(factor, counts[e].to(_device())).unsqueeze(1)
        for n, i, o in _moe_layers(case):
            sigma = C / math.sqrt(2 * E * max(1, T * 2 // E) * i * o)
            layers.append((f"experts.{e}.{n}", _randn(g, (sum(seg), i)),
                           _randn(g, (sum(seg), o), row_f * sigma), seg))
    return {"layers": layers}


def _mlp_inputs(case, seed):
    g = _gen(seed, "mlp")
    i, h, c = case["din"], case["hidden"], case["classes"]
    f32 = torch.float32
    params = {"0.weight": _randn(g, (h, i), 1 / math.sqrt(3 * i), f32),
              "0.bias": _randn(g, (h,), 1 / math.sqrt(3 * i), f32),
              "2.weight": _randn(g, (c, h), 1 / math.sqrt(3 * h), f32),
              "2.bias": _randn(g, (c,), 1 / math.sqrt(3 * h), f32)}
    x = _randn(g, (case["B"], i), dtype=f32)
    y = torch.randint(0, c, (case["B"],), generator=g, device=_device())
    return {"params": params, "x": x, "y": y}


def _leaves_inputs(case, seed):
    g = _gen(seed, "leaves")
    B = case["B"]
    factor = _factors(g, B)
    shapes = _leaf_shapes(case)
    total = sum(math.prod(s) for s in shapes.values())
    return {"values": {n: _randn(g, (B, *s), factor.view(B, *[1] * len(s)) * (C / math.sqrt(total)),
                                 DTYPES[case["dtype"]]) for n, s in shapes.items()}}


def _noise_inputs(case, seed):
    g = _gen(seed, "noise")
    return {"tree": {n: _randn(g, s, 1e-3, DTYPES[case["dtype"]])
                     for n, s in _noise_shapes(case).items()}}


_INPUTS = {"linear": _linear_inputs, "block": _block_inputs, "lora": _lora_inputs,
           "moe": _moe_inputs, "mlp": _mlp_inputs, "leaves": _leaves_inputs,
           "noise": _noise_inputs}


def _group_map(case, names):
    """Leaf -> group and the groups' bounds (together C): a layer's leaves, dealt in order,
    or one group per expert."""
    if case["kind"] == "moe":
        groups = {n: "expert" + n.split(".")[1] for n in names}
    else:
        layers = list(dict.fromkeys(n.split(".")[0] for n in names))
        groups = {n: f"g{layers.index(n.split('.')[0]) % case['groups']}" for n in names}
    k = len(set(groups.values()))
    return groups, {v: C / math.sqrt(k) for v in sorted(set(groups.values()))}


def _mean_ce(logits, target):
    return torch.nn.functional.cross_entropy(logits, target, reduction="none")


def prepare(case, seed):
    inp = _INPUTS[case["kind"]](case, seed)
    k = case["kind"]
    state = {"case": case}
    noise_fn, noise_state = gaussian_noise(noise_multiplier=1.0, key=key(seed), stream="device")
    state["noise"] = ({"noise_fn": noise_fn, "noise_state": noise_state}
                      if k == "noise" or case["noise"] else {})
    if k in ("linear", "noise"):
        state.update(inp)
    elif k == "mlp":
        model = torch.nn.Sequential(torch.nn.Linear(case["din"], case["hidden"]), torch.nn.ReLU(),
                                    torch.nn.Linear(case["hidden"], case["classes"]))
        model.to(_device()).load_state_dict(inp["params"])
        step, clip_state = ghost_clipped_grad(model, _mean_ce, clipping_norm=C, return_aux=True)
        state.update(step=step, clip_state=clip_state, x=inp["x"], y=inp["y"])
    elif k == "leaves":
        bound = C
        if case["groups"] > 1:
            groups, bounds = _group_map(case, inp["values"])
            bound = PerGroup({(n,): v for n, v in groups.items()}, bounds)
        step, clip_state = clipped_fun(lambda grads: grads, clipping_norm=bound,
                                       return_aux=case["aux"], second_moment=case["second"])
        state.update(step=step, clip_state=clip_state, values=inp["values"])
    else:
        caps = [LinearCapture(t[0], t[1], t[2], segments=t[3] if len(t) > 3 else None)
                for t in inp["layers"]]
        if "norms" in inp:
            caps.append(DirectCapture(inp["norms"]))
        bound = C
        if k == "moe":
            groups, bounds = _group_map(case, [f"{t[0]}.weight" for t in inp["layers"]])
            bound = PerGroup({(n,): v for n, v in groups.items()}, bounds)
        state.update(captures=caps, bound=bound)
    return state


# --------------------------------------------------------------------------
# One pass
# --------------------------------------------------------------------------


def run(state):
    case, noise = state["case"], state["noise"]
    k = case["kind"]
    if k == "linear":
        out = ghost_clip_sum(state["A"], state["G"], clipping_norm=C, normalize_by=1.0,
                             bias=case["bias"], auto_s_gamma=GAMMA if case["auto"] else None,
                             dtype=torch.float32 if case["out"] == "fp32" else None,
                             return_aux=True, **noise)
        grads, aux = out[0] if noise else out
        return {**grads.pytree, "norms": aux.grad_norms, "scales": aux.clip_scales,
                "clipped": aux.num_clipped}
    if k == "mlp":
        out = state["step"](state["x"], state["y"], state=state["clip_state"], **noise)
        grads, aux = out[0]
        return {**grads.pytree, "losses": aux.loss_values, "norms": aux.grad_norms}
    if k == "noise":
        noised, _ = noise["noise_fn"](clipped(state["tree"], max_norm=C), noise["noise_state"])
        return noised.pytree
    if k == "leaves":
        out, _ = state["step"](state["values"], state=state["clip_state"])
        grads, aux = out if case["aux"] else (out, None)
        if noise:
            grads, _ = noise["noise_fn"](grads, noise["noise_state"])
        res = {}
        if case["second"]:
            res.update({f"squared.{n}": v for n, v in grads.squared_grads.pytree.items()})
            grads = grads.grads
        res.update(grads.pytree)
        if aux is not None:
            res.update(norms=aux.norms, clipped_norms=aux.clipped_norms)
        return res
    out = ghost_clip_captured(state["captures"], clipping_norm=state["bound"], return_aux=True,
                              **noise)
    grads, aux = out[0] if noise else out
    res = {**grads.pytree, "norms": aux.grad_norms, "scales": aux.clip_scales,
           "clipped": aux.num_clipped}
    if aux.group_norms is not None:
        res.update({f"norms.{n}": v for n, v in aux.group_norms.items()})
    return res


# About four times what the outputs differ by from the 64-bit result.  With 16-bit operands
# that is the clip factor's safety margin (the rounding of 16-bit gradients that it allows
# for, up to 0.5%, and a rounding bound of the norm, up to 1% at the longest sequences) where
# no noise covers it, and the outputs' own rounding; with float32 it is the order of the sums
# (and the normals' own 1e-6).
_TOLERANCE = {"linear": {"bf16": 2e-2, "fp32": 1e-5}, "block": 4e-2, "lora": 2e-2, "moe": 2e-2,
              "mlp": 1e-5, "leaves": {"bf16": 2e-2, "fp16": 4e-3, "fp32": 4e-6},
              "noise": {"bf16": 7e-3, "fp32": 4e-6}}


def tolerance(case):
    t = _TOLERANCE[case["kind"]]
    return {"rel": t if isinstance(t, float) else t[case["dtype"]]}


# --------------------------------------------------------------------------
# The same pass in 64 bits
# --------------------------------------------------------------------------


def _fold_in(seed, *data):
    for d in data:
        h = hashlib.blake2b(digest_size=8)
        for part in (seed, d):
            h.update(b"i" + part.to_bytes(16, "little", signed=True) if isinstance(part, int)
                     else b"s" + part.encode())
            h.update(b"|")
        seed = int.from_bytes(h.digest(), "little")
    return seed


def _normals(seed, leaf, rows, cols):
    """The device stream: Philox4x32-10 keyed by the step's seed, counter (block, leaf);
    Box-Muller with a 53-bit radius and a 32-bit angle; a block serves two rows."""
    block = torch.arange((rows + 1) // 2 * cols, device=_device())
    mask = 0xFFFFFFFF
    c = [block & mask, block >> 32, torch.full_like(block, leaf), torch.zeros_like(block)]
    k0, k1 = seed & mask, seed >> 32
    for _ in range(10):
        hl = []
        for m, x in ((0xD2511F53, c[0]), (0xCD9E8D57, c[2])):
            p = (m & 0xFFFF) * x  # 32 x 32 -> 64 bits in two exact pieces
            q = (m >> 16) * x + (p >> 16)
            hl.append((q >> 16, ((q & 0xFFFF) << 16) | (p & 0xFFFF)))
        (h0, l0), (h1, l1) = hl
        c = [h1 ^ c[1] ^ k0, l1, h0 ^ c[3] ^ k1, l0]
        k0, k1 = (k0 + 0x9E3779B9) & mask, (k1 + 0xBB67AE85) & mask
    u1 = ((c[0] << 21 | c[1] >> 11).double() + 0.5) * 2.0**-53
    angle = (c[2].double() + 0.5) * 2.0**-32 * (2 * math.pi)
    radius = torch.sqrt(-2 * torch.log(u1))
    z = torch.stack([radius * torch.cos(angle), radius * torch.sin(angle)])
    return z.view(2, -1, cols).transpose(0, 1).reshape(-1, cols)[:rows]


def _add_noise(tree, seed, std, *stream):
    """``tree`` plus its leaves' noise, ``std`` a number or one per leaf."""
    step = _fold_in(seed, "opake.dpsgd.gaussian", *stream, 0)
    out = {}
    for i, n in enumerate(sorted(tree)):
        x = tree[n].double()
        s = std[n] if isinstance(std, dict) else std
        z = _normals(step, i, x.shape[0], x.numel() // x.shape[0])
        out[n] = x + s * z.view(x.shape)
    return out


def _scales(case, norms, bound=C):
    if case.get("auto"):
        return bound / (norms + GAMMA)
    return torch.clamp(bound / norms, max=1.0)


def _clip_layers(layers, B, bounds, group_of):
    """Per-group norms, scales and clipped sums of ``[(name, example -> gradient)]``."""
    sq = {g: torch.zeros(B, dtype=torch.float64, device=_device()) for g in bounds}
    for n, grad in layers:
        for b in range(B):
            sq[group_of[n]][b] += grad(b).square().sum()
    norms = {g: v.sqrt() for g, v in sq.items()}
    scales = {g: torch.clamp(bounds[g] / norms[g], max=1.0) for g in bounds}
    sums = {n: sum(scales[group_of[n]][b] * grad(b) for b in range(B)) for n, grad in layers}
    return norms, scales, sums


def _dense_grad(A, G):
    return lambda b: G[b].double().t() @ A[b].double()


def _segment_grad(A, G, seg):
    starts = [0]
    for n in seg:
        starts.append(starts[-1] + n)
    return lambda b: (G[starts[b]:starts[b + 1]].double().t()
                      @ A[starts[b]:starts[b + 1]].double())


def _exact_linear(case, seed, inp):
    A, G, B = inp["A"], inp["G"], case["B"]
    grad = _dense_grad(A, G)
    cols = G.double().sum(dim=1) if case["bias"] else None
    sq = torch.stack([grad(b).square().sum() for b in range(B)])
    if case["bias"]:
        sq = sq + cols.square().sum(dim=1)
    norms = sq.sqrt()
    scales = _scales(case, norms)
    tree = {"weight": sum(scales[b] * grad(b) for b in range(B))}
    if case["bias"]:
        tree["bias"] = scales @ cols
    if case["noise"]:
        tree = _add_noise(tree, seed, C)
    return {**tree, "norms": norms, "scales": scales,
            "clipped": (norms > C).sum().reshape(1).to(torch.int32)}


def _exact_captured(case, seed, inp):
    B = case["B"]
    layers = []
    for t in inp["layers"]:
        grad = _segment_grad(*t[1:4]) if case["kind"] == "moe" else _dense_grad(t[1], t[2])
        layers.append((f"{t[0]}.weight", grad))
    for n, x in inp.get("norms", {}).items():
        layers.append((n, lambda b, x=x: x[b].double()))
    names = [n for n, _ in layers]
    per_group = case["kind"] == "moe"
    groups, bounds = (_group_map(case, names) if per_group
                      else (dict.fromkeys(names, "all"), {"all": C}))
    norms, scales, tree = _clip_layers(layers, B, bounds, groups)
    if case["noise"]:
        total = sum(bounds.values())
        tree = _add_noise(tree, seed, {n: math.sqrt(bounds[groups[n]] * total) for n in names})
    out = {n: tree[n] for n in sorted(tree)}
    out["norms"] = sum(v.square() for v in norms.values()).sqrt()
    rows = torch.stack([scales[g] for g in sorted(bounds)])
    out["scales"] = rows[:, None] if per_group else rows
    out["clipped"] = torch.stack([(norms[g] > bounds[g]).sum()
                                  for g in sorted(bounds)]).to(torch.int32)
    if per_group:
        out.update({f"norms.{g}": norms[g] for g in sorted(bounds)})
    return out


def _exact_mlp(case, seed, inp):
    p = {n: v.double() for n, v in inp["params"].items()}
    x, y = inp["x"].double(), inp["y"]
    pre = x @ p["0.weight"].t() + p["0.bias"]
    h = pre.clamp(min=0)
    logits = h @ p["2.weight"].t() + p["2.bias"]
    losses = _mean_ce(logits, y)
    g2 = torch.softmax(logits, dim=1) - torch.nn.functional.one_hot(y, case["classes"]).double()
    g1 = (g2 @ p["2.weight"]) * (pre > 0)
    sq = (x.square().sum(1) + 1) * g1.square().sum(1) + (h.square().sum(1) + 1) * g2.square().sum(1)
    norms = sq.sqrt()
    s = _scales(case, norms)[:, None]
    tree = {"0.bias": (s * g1).sum(0), "0.weight": (s * g1).t() @ x,
            "2.bias": (s * g2).sum(0), "2.weight": (s * g2).t() @ h}
    if case["noise"]:
        tree = _add_noise(tree, seed, C)
    return {**tree, "losses": losses, "norms": norms}


def _exact_leaves(case, seed, inp):
    values, B = inp["values"], case["B"]
    names = sorted(values)
    groups, bounds = (_group_map(case, values) if case["groups"] > 1
                      else (dict.fromkeys(names, "all"), {"all": C}))
    layers = [(n, lambda b, x=values[n]: x[b].double()) for n in names]
    norms, scales, tree = _clip_layers(layers, B, bounds, groups)
    squared = {}
    if case["second"]:
        for n, grad in layers:
            squared[n] = sum((scales[groups[n]][b] * grad(b)).square() for b in range(B))
    if case["noise"]:
        total = sum(bounds.values())
        std = {n: math.sqrt(bounds[groups[n]] * total) for n in names}
        if case["second"]:
            # Two streams under one budget; a squared leaf's bound is its group's squared.
            sq_bounds = {n: bounds[groups[n]] ** 2 for n in names}
            joint = total + sum(v * v for v in bounds.values())
            std = {n: math.sqrt(bounds[groups[n]] * joint) for n in names}
            squared = _add_noise(squared, seed, {n: math.sqrt(sq_bounds[n] * joint) for n in names},
                                 "opake.paired.second")
            tree = _add_noise(tree, seed, std, "opake.paired.first")
        else:
            tree = _add_noise(tree, seed, std)
    out = {f"squared.{n}": squared[n] for n in names} if case["second"] else {}
    out.update({n: tree[n] for n in names})
    if case["aux"]:
        out["norms"] = sum(v.square() for v in norms.values()).sqrt()
        out["clipped_norms"] = sum((scales[g] * norms[g]).square() for g in bounds).sqrt()
    return out


def exact(case, seed):
    inp = _INPUTS[case["kind"]](case, seed)
    k = case["kind"]
    if k == "noise":
        return _add_noise(inp["tree"], seed, C)
    if k in ("block", "lora", "moe"):
        return _exact_captured(case, seed, inp)
    return {"linear": _exact_linear, "mlp": _exact_mlp, "leaves": _exact_leaves}[k](case, seed, inp)
