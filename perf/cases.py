"""Timed cases of the pair stack: what a program that folds or trains on pair
tensors [B, N, N, C] asks of genie_tk, through the public modules and the
LayerNorm operator.

A case names an operator, a mode and its sizes:

* ``op``: ``tri_mul``, ``tri_attn``, ``transition``, ``layer`` (one
  PairTransformLayer: four triangle operators and the transition) or
  ``layernorm`` (``genie_tk._C.layernorm``);
* ``mode``: ``infer`` (no gradients) or ``train`` (forward and backward: the
  gradients of the pair tensor and of every parameter are returned);
* ``dtype``, ``B``, ``N``, ``c`` (pair channels), ``len``: the pair mask is one
  where both positions are below the sequence's length.  The first sequence of
  the batch has length ``len``, any others the full N, as in a padded batch;
* ``first``: the outgoing / starting direction, or the incoming / ending one;
* ``c_mul``, ``c_att``, ``heads``: the widths of the triangle operators.

Inputs are N(0, 1), weights N(0, 1/fan_in) and gate biases 1, as in the other
workloads of this repository; LayerNorm weights are near 1.
"""
from __future__ import annotations

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "genie-tk_amd"))

import genie_tk  # noqa: E402
from genie_tk import _ext  # noqa: E402
from genie_tk.pair_transform import PairTransition  # noqa: E402

DEVICE = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
INF = 1e9


def _case(name, op, mode, dtype, N, B=1, c=128, length=None, first=True, c_mul=128, c_att=32,
          heads=4):
    case = {"op": op, "mode": mode, "dtype": dtype, "B": B, "N": N, "c": c,
            "len": N if length is None else length, "first": first, "c_mul": c_mul,
            "c_att": c_att, "heads": heads}
    if name is not None:
        case["name"] = name
    return case


def listed():
    return [
        # one short chain in the modules' default type: three small launches and the call itself
        _case("tri_mul_fp32_n64", "tri_mul", "infer", "fp32", 64),
        # a chain of 224 residues padded to 256, the incoming direction
        _case("tri_mul_in_bf16_n256", "tri_mul", "infer", "bf16", 256, length=224, first=False),
        # the operator at the crop most folding programs use, full width
        _case("tri_mul_out_bf16_n512", "tri_mul", "infer", "bf16", 512),
        # the default attention (four heads of 8) in the modules' default type
        _case("tri_attn_fp32_n256", "tri_attn", "infer", "fp32", 256),
        # full-width attention, ending node, at the same crop as the update above
        _case("tri_attn_end_bf16_n512", "tri_attn", "infer", "bf16", 512, first=False, c_att=128),
        # one long chain of no round length
        _case("tri_attn_bf16_n1100", "tri_attn", "infer", "bf16", 1100, c_att=128),
        # the norm of a whole pair tensor: memory bandwidth
        _case("layernorm_bf16_n512", "layernorm", "infer", "bf16", 512),
        # sampling: a default layer over a padded batch of two chains
        _case("layer_bf16_b2_n384", "layer", "infer", "bf16", 384, B=2, length=300),
        # a training step of the default attention in the modules' default type
        _case("tri_attn_train_fp32_n128", "tri_attn", "train", "fp32", 128),
        # training steps of the single operators in bf16: a chain of any length,
        # the default attention, and the transition at a training crop
        _case("tri_mul_train_bf16_n301", "tri_mul", "train", "bf16", 301),
        _case("tri_attn_train_bf16_n250", "tri_attn", "train", "bf16", 250, length=230),
        _case("transition_train_bf16_n384", "transition", "train", "bf16", 384),
    ]


# The ranges of N that the listed cases stand for, by operator, mode and dtype.
_RANGES = {
    ("tri_mul", "infer", "bf16"): (48, 640),
    ("tri_mul", "infer", "fp32"): (32, 256),
    ("tri_attn", "infer", "bf16"): (48, 1100),
    ("tri_attn", "infer", "fp32"): (32, 256),
    ("layernorm", "infer", "bf16"): (64, 1024),
    ("layer", "infer", "bf16"): (48, 448),
    ("tri_mul", "train", "fp32"): (32, 192),
    ("tri_attn", "train", "fp32"): (32, 192),
    ("tri_mul", "train", "bf16"): (48, 384),
    ("tri_attn", "train", "bf16"): (48, 384),
    ("transition", "train", "bf16"): (48, 448),
}


def draw(rng):
    op, mode, dtype = rng.choice(sorted(_RANGES))
    low, high = _RANGES[op, mode, dtype]
    N = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    B = 2 if N * 3 < high * 2 and rng.random() < 0.25 else 1
    length = N if rng.random() < 0.5 else rng.randint((N + 1) // 2, N)
    c = 64 if rng.random() < 0.2 else 128
    return _case(None, op, mode, dtype, N, B=B, c=c, length=length, first=rng.random() < 0.5,
                 c_mul=c, c_att=rng.choice((32, 128)))


# ---------------------------------------------------------------------------
# What a program has in hand before the call
# ---------------------------------------------------------------------------
def _module(case):
    c = case["c"]
    if case["op"] == "tri_mul":
        cls = (genie_tk.TriangleMultiplicationOutgoing if case["first"]
               else genie_tk.TriangleMultiplicationIncoming)
        return cls(c, case["c_mul"])
    if case["op"] == "tri_attn":
        cls = (genie_tk.TriangleAttentionStartingNode if case["first"]
               else genie_tk.TriangleAttentionEndingNode)
        return cls(c, case["c_att"], case["heads"])
    if case["op"] == "transition":
        return PairTransition(c)
    # dropout off: a random mask would make every pass another one
    return genie_tk.PairTransformLayer(c, c_hidden_mul=case["c_mul"],
                                       c_hidden_tri_att=case["c_att"],
                                       n_head_tri=case["heads"], tri_dropout=0.0)


def _fill(module, gen):
    """Seeded weights in place of the constructors' (whose last layers are zero)."""
    with torch.no_grad():
        for name, p in module.named_parameters():
            x = torch.randn(p.shape, generator=gen, device=DEVICE)
            if p.dim() == 2:
                x *= 1.0 / math.sqrt(p.shape[1])
            elif "layer_norm" in name:
                x = x * 0.1 + (1.0 if name.endswith("weight") else 0.0)
            else:
                x = x * 0.1 + (1.0 if "_g." in name else 0.0)
            p.copy_(x)


def _mask(case):
    B, N = case["B"], case["N"]
    lengths = torch.full((B, 1), N, device=DEVICE)
    lengths[0] = case["len"]
    valid = (torch.arange(N, device=DEVICE)[None, :] < lengths).float()
    return valid[:, :, None] * valid[:, None, :]


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    B, N, c = case["B"], case["N"], case["c"]
    state = {"op": case["op"], "train": case["mode"] == "train",
             "z": torch.randn(B, N, N, c, generator=gen, device=DEVICE).to(dt)}
    if case["op"] == "layernorm":
        state["w"] = 1 + 0.1 * torch.randn(c, generator=gen, device=DEVICE)
        state["b"] = 0.1 * torch.randn(c, generator=gen, device=DEVICE)
        return state
    module = _module(case).to(DEVICE)
    _fill(module, gen)
    module = module.to(dt)
    state["mask"] = _mask(case)
    if state["train"]:
        state["dy"] = torch.randn(B, N, N, c, generator=gen, device=DEVICE).to(dt)
        state["z"].requires_grad_()
        state["module"] = module.train()
    else:
        state["module"] = module.eval()
    return state


def _call(module, op, z, mask):
    return module((z, mask))[0] if op == "layer" else module(z, mask)


def run(state):
    if state["op"] == "layernorm":
        return _ext.require().layernorm(state["z"], state["w"], state["b"], 1e-5)
    module, z = state["module"], state["z"]
    if not state["train"]:
        with torch.no_grad():
            return _call(module, state["op"], z, state["mask"])
    y = _call(module, state["op"], z, state["mask"])
    grads = torch.autograd.grad(y, [z, *module.parameters()], state["dy"])
    return {"y": y, "grads": list(grads)}


# ---------------------------------------------------------------------------
# What one pass cannot do without
# ---------------------------------------------------------------------------
def _flops(case, op):
    """Dense products of one forward pass."""
    B, N, c, cm, ca = case["B"], case["N"], case["c"], case["c_mul"], case["c_att"]
    pairs = B * N * N
    if op == "tri_mul":
        return 2 * pairs * c * (5 * cm + c) + 2 * pairs * N * cm
    if op == "tri_attn":
        return 2 * pairs * c * (5 * ca + case["heads"]) + 4 * pairs * N * ca
    if op == "transition":
        return 16 * pairs * c * c
    if op == "layer":
        return (2 * _flops(case, "tri_mul") + 2 * _flops(case, "tri_attn")
                + _flops(case, "transition"))
    return 0


def work(case):
    size = 2 if case["dtype"] == "bf16" else 4
    pairs = case["B"] * case["N"] ** 2
    tensor = pairs * case["c"] * size
    train = case["mode"] == "train"
    # z and y; dy and dz besides in training; the mask
    moved = tensor * (4 if train else 2)
    if case["op"] in ("tri_mul", "tri_attn", "layer"):
        moved += 4 * pairs
    return {"bytes": moved, "flops": _flops(case, case["op"]) * (3 if train else 1)}


def tolerance(case):
    """About four times what two correct implementations differ by: the kernels,
    the modules' PyTorch path and exact(), compared at the listed sizes."""
    train = case["mode"] == "train"
    if case["dtype"] == "fp32":
        # seen: 6e-7 (one forward pass), 3e-6 (forward and backward)
        return {"rel": 1e-5, "max": 1e-4} if train else {"rel": 3e-6, "max": 4e-5}
    if case["op"] == "layernorm":
        return {"rel": 7e-3, "max": 1.6e-2}  # seen: 1.7e-3; one unit in the last place is 8e-3
    if not train:
        return {"rel": 2e-2, "max": 0.2}  # seen: 5e-3 against exact(), largest 0.05
    if case["op"] == "tri_mul":
        return {"rel": 2.5e-2, "max": 0.16}  # seen: 6.3e-3, largest 0.04
    if case["op"] == "tri_attn":
        return {"rel": 3e-2, "max": 0.5}  # seen: 1.5e-2, largest 0.12
    # the transition's ReLU: a hidden value whose sign the rounding of LN(p) to
    # bf16 decides takes its whole gradient along (against exact(): 4.8e-2, largest 1;
    # implementations that round LN(p) to bf16 once flip few of the same values)
    return {"rel": 3e-2, "max": 0.9}


# ---------------------------------------------------------------------------
# The same values in 64 bits, in plain torch
# ---------------------------------------------------------------------------
def _norm(P, name, x):
    return torch.nn.functional.layer_norm(x, x.shape[-1:], P[name + ".weight"],
                                          P[name + ".bias"])


def _linear(P, name, x):
    return torch.nn.functional.linear(x, P[name + ".weight"], P.get(name + ".bias"))


def _tri_mul(P, pre, z, m, outgoing):
    zn = _norm(P, pre + "layer_norm_in", z)
    a, b = (_linear(P, pre + "linear_%s_p" % s, zn)
            * torch.sigmoid(_linear(P, pre + "linear_%s_g" % s, zn)) * m[..., None] for s in "ab")
    # [B, C, i, k] @ [B, C, k, j]
    a = a.permute(0, 3, 1, 2) if outgoing else a.permute(0, 3, 2, 1)
    b = b.permute(0, 3, 2, 1) if outgoing else b.permute(0, 3, 1, 2)
    x = torch.matmul(a.contiguous(), b.contiguous()).permute(0, 2, 3, 1)
    x = _linear(P, pre + "linear_z", _norm(P, pre + "layer_norm_out", x))
    return x * torch.sigmoid(_linear(P, pre + "linear_g", zn))


def _tri_attn(P, pre, x, m, starting, heads):
    if not starting:
        x, m = x.transpose(1, 2), m.transpose(1, 2)
    x = _norm(P, pre + "layer_norm", x)
    B, N = x.shape[:2]
    tri = _linear(P, pre + "linear", x).permute(0, 3, 1, 2)  # [B, H, Q, K]
    rows = max(1, min(N, (1 << 28) // (B * heads * N * N)))
    if torch.is_grad_enabled():
        rows = N
    out = []
    for r in range(0, N, rows):
        xr, mr = x[:, r:r + rows], m[:, r:r + rows]
        q, k, v = (_linear(P, pre + "mha.linear_" + s, xr).unflatten(-1, (heads, -1))
                   .transpose(2, 3).contiguous() for s in "qkv")  # [B, R, H, N, D]
        s = torch.matmul(q, k.transpose(-1, -2).contiguous()) / math.sqrt(q.shape[-1])
        s = s + tri[:, None]
        # where no key is valid the single-precision scores are all -INF: equal
        # weights, and the gradient of the scores passes through
        dead = (mr.sum(-1) == 0)[:, :, None, None, None]
        s = torch.where(dead, s - s.detach(), s + (INF * (mr - 1))[:, :, None, None, :])
        o = torch.matmul(torch.softmax(s, -1), v).transpose(2, 3).flatten(-2)
        out.append(_linear(P, pre + "mha.linear_o",
                           o * torch.sigmoid(_linear(P, pre + "mha.linear_g", xr))))
    y = torch.cat(out, 1)
    return y if starting else y.transpose(1, 2)


def _transition(P, pre, p):
    h = torch.relu(_linear(P, pre + "linear_1", _norm(P, pre + "layer_norm", p)))
    return _linear(P, pre + "linear_2", h)


def _forward(case, P, z, m):
    op, heads = case["op"], case["heads"]
    if op == "tri_mul":
        return _tri_mul(P, "", z, m, case["first"])
    if op == "tri_attn":
        return _tri_attn(P, "", z, m, case["first"], heads)
    if op == "transition":
        return _transition(P, "", z)
    z = z + _tri_mul(P, "tri_mul_out.", z, m, True)
    z = z + _tri_mul(P, "tri_mul_in.", z, m, False)
    z = z + _tri_attn(P, "tri_att_start.", z, m, True, heads)
    z = z + _tri_attn(P, "tri_att_end.", z, m, False, heads)
    return (z + _transition(P, "pair_transition.", z)) * m[..., None]


def exact(case, seed):
    state = prepare(case, seed)
    z = state["z"].detach().double()
    if case["op"] == "layernorm":
        return torch.nn.functional.layer_norm(z, z.shape[-1:], state["w"].double(),
                                              state["b"].double())
    P = {n: p.detach().double() for n, p in state["module"].named_parameters()}
    m = state["mask"].double()
    if not state["train"]:
        with torch.no_grad():
            return _forward(case, P, z, m)
    leaves = [z.requires_grad_(), *(p.requires_grad_() for p in P.values())]
    with torch.enable_grad():
        y = _forward(case, P, z, m)
        grads = torch.autograd.grad(y, leaves, state["dy"].double())
    return {"y": y.detach(), "grads": list(grads)}
