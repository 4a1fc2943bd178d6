"""The performance cases of this repository: the calls a user of triangle attention makes, over the sizes,
types and options that they are made with.

Two public entry points are timed.  `attention(q, k, v, bias, sm_scale[, dropout_p, seed])` is the operator
itself, for callers that bring their own projections; `TriangleAttention` is the AlphaFold2 block around it
(layer norm, projections, attention, gating, output projection).  Each is run for inference (forward under
no_grad) and for training (forward and every gradient).  Inputs are synthetic: unit-normal pair tensors and
randomly initialised weights.
"""
import math
import os
import sys

import torch

sys.path.insert(1, os.path.join(os.getcwd(), "flash-triangle-attention_amd"))

from flash_tt_attn import attention  # noqa: E402
from triangle_attention import TriangleAttention  # noqa: E402

_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


def _case(name, op, train, B, H, L, D, dtype, layout="rows", scale=0.0, bias_std=1.0, dropout=0.0, mask=False):
    """`layout` of the operator's q, k, v: "rows" contiguous (B,H,L,L,D); "proj" the permuted view of a
    (B,L,L,H*D) projection; "ending" the L1<->L2 transposed view that the ending node uses.  For the block:
    "rows" is the starting node, "ending" the ending node.  `scale` 0 stands for 1/sqrt(D).  `mask`: the last
    eighth of the keys is padding."""
    return {"name": name, "op": op, "train": train, "B": B, "H": H, "L": L, "D": D, "dtype": dtype, "layout": layout,
            "scale": scale, "bias_std": bias_std, "dropout": dropout, "mask": mask}


def listed():
    return [
        # a peptide-sized complex scored once: the smallest call, where launches and the host count
        _case("infer_peptide", "attention", False, 1, 4, 64, 32, "fp16"),
        # a training step on short chains, batched over samples and heads: the shortest row of the sequence-length sweep
        _case("train_batch_l128", "attention", True, 4, 8, 128, 32, "fp16", scale=1.3),
        # AlphaFold2's initial-training crop, bf16, read in place from the projections
        _case("train_crop256_bf16", "attention", True, 2, 4, 256, 32, "bf16", layout="proj"),
        # AlphaFold2's fine-tuning crop, fp16, read in place from the projections
        _case("train_crop384", "attention", True, 1, 4, 384, 32, "fp16", layout="proj"),
        # the operator's benchmark shape
        _case("train_b4_h8_l512", "attention", True, 4, 8, 512, 32, "fp16", scale=1.3),
        # the ending node at head dim 64, through transposed views
        _case("train_ending_d64", "attention", True, 2, 8, 512, 64, "fp16", layout="ending"),
        # a long crop with peaked softmax rows: the largest step
        _case("train_long_l1536", "attention", True, 1, 4, 1536, 32, "fp16", bias_std=3.0),
        # training with dropout on the attention weights, a length as the data gives it
        _case("train_dropout_l300", "attention", True, 1, 4, 300, 32, "bf16", layout="proj", dropout=0.25),
        # structure prediction of one protein: an arbitrary length, padded keys masked through the bias
        _case("infer_protein_l701", "attention", False, 1, 4, 701, 32, "bf16", layout="proj", mask=True),
        # the whole block in bf16 training at the fine-tuning crop
        _case("block_train_l384_bf16", "block", True, 1, 4, 384, 32, "bf16"),
        # the whole block as its docstring builds it (fp32 weights and pair tensor), one small training crop
        _case("block_train_l192_fp32", "block", True, 1, 4, 192, 32, "fp32"),
        # the whole block in inference at a protein's own length: ending node, padded keys
        _case("block_infer_l457_bf16", "block", False, 1, 4, 457, 32, "bf16", layout="ending", mask=True),
    ]


def draw(rng):
    """One case of the same ranges: lengths of 32 to 1536 spread over their logarithm, half of them odd sizes
    and half multiples of 32, with the batch cut down where the call would cost more than the largest listed one."""
    L = int(round(math.exp(rng.uniform(math.log(32), math.log(1536)))))
    if rng.random() < 0.5:
        L = max(32, (L + 16) // 32 * 32)
    elif L % 2 == 0 and rng.random() < 0.7:
        L += 1
    op = "block" if rng.random() < 0.35 else "attention"
    train = rng.random() < 0.6
    dropout = rng.choice([0.1, 0.15, 0.25]) if train and rng.random() < 0.25 else 0.0
    if op == "block":
        case = _case("", op, train, rng.choice([1, 1, 2]), 4, L, 32, rng.choice(["bf16", "bf16", "fp32"]),
                     layout=rng.choice(["rows", "ending"]), dropout=dropout, mask=rng.random() < 0.3)
    else:
        case = _case("", op, train, rng.choice([1, 1, 2, 4]), rng.choice([4, 4, 8]), L, rng.choice([32, 32, 32, 64]),
                     rng.choice(["fp16", "bf16"]), layout=rng.choice(["rows", "proj", "ending"]), dropout=dropout,
                     mask=rng.random() < 0.3)
    top = _cost(listed()[6])
    while case["B"] > 1 and _cost(case) > top:
        case["B"] //= 2
    while case["H"] > 4 and _cost(case) > top:
        case["H"] //= 2
    while _cost(case) > top:
        case["L"] = case["L"] * 7 // 8
    del case["name"]
    return case


def _cost(c):
    # (dropout and fp32 projections cost more than their operations say)
    return work(c)["flops"] * (4.0 if c["dropout"] else 1.0) * (2.0 if c["dtype"] == "fp32" else 1.0) * (1.0 if c["train"] else 1.5)


def _pair(B, H, L, D, layout, dtype, gen):
    """A (B,H,L,L,D) tensor in the memory layout that its producer leaves it in."""
    if layout == "proj":
        return torch.randn(B, L, L, H * D, device="cuda", generator=gen).to(dtype).view(B, L, L, H, D).permute(0, 3, 1, 2, 4)
    t = torch.randn(B, H, L, L, D, device="cuda", generator=gen).to(dtype)
    return t.transpose(2, 3) if layout == "ending" else t


def prepare(case, seed):
    B, H, L, D, dtype = case["B"], case["H"], case["L"], case["D"], _DTYPES[case["dtype"]]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kept = L - L // 8
    state = {"op": case["op"], "train": case["train"], "dropout": case["dropout"], "seed": seed, "mask": None}
    if case["op"] == "block":
        blk = TriangleAttention(c_z=128, c_hidden=D, n_heads=H, starting=case["layout"] != "ending", dropout_p=case["dropout"])
        blk = blk.to(device="cuda", dtype=dtype)
        with torch.no_grad():
            for p in blk.parameters():  # unit-gain weights, biases and norm parameters off their trivial values
                x = torch.randn(p.shape, device="cuda", generator=gen)
                p.copy_(x / math.sqrt(p.shape[1]) if p.dim() == 2 else 0.1 * x)
            blk.layer_norm.weight += 1.0
        state["blk"] = blk.train(case["train"]).requires_grad_(case["train"])
        state["z"] = torch.randn(B, L, L, 128, device="cuda", generator=gen).to(dtype).requires_grad_(case["train"])
        if case["mask"]:
            state["mask"] = torch.ones(B, L, device="cuda", dtype=dtype)
            state["mask"][:, kept:] = 0
        if case["train"]:
            state["dout"] = torch.randn(B, L, L, 128, device="cuda", generator=gen).to(dtype)
        return state
    q, k, v = (_pair(B, H, L, D, case["layout"], dtype, gen) for _ in range(3))
    bias = case["bias_std"] * torch.randn(B, H, L, L, device="cuda", generator=gen)
    if case["mask"]:
        bias[..., kept:] = -math.inf
    state["args"] = [q, k, v, bias.to(dtype)]
    state["scale"] = case["scale"] or 1.0 / math.sqrt(D)
    if case["train"]:
        for t in state["args"]:
            t.requires_grad_(True)
        state["dout"] = _pair(B, H, L, D, case["layout"], dtype, gen)
    return state


def run(state):
    if state["op"] == "block":
        blk, z = state["blk"], state["z"]
        if not state["train"]:
            with torch.no_grad():
                return blk(z, state["mask"])
        out = blk(z, state["mask"], state["seed"] if state["dropout"] else None)
        return out, torch.autograd.grad(out, [z, *blk.parameters()], state["dout"])
    args = state["args"]
    if not state["train"]:
        with torch.no_grad():
            return attention(*args, state["scale"])
    out = attention(*args, state["scale"], state["dropout"], state["seed"]) if state["dropout"] else attention(*args, state["scale"])
    return out, torch.autograd.grad(out, args, state["dout"])


def work(case):
    """Bytes: each input once and each output once.  Operations: the matrix products that the definition holds,
    two per score in the forward and five in the backward (scores again), and the projections of the block."""
    B, H, L, D, train = case["B"], case["H"], case["L"], case["D"], case["train"]
    size = 4 if case["dtype"] == "fp32" else 2
    pairs, scores = B * L * L, B * H * L ** 3
    flops = (14 if train else 4) * scores * D
    if case["op"] == "block":
        c, weights = 128, 128 * (5 * H * D + H) + 128 * 3 + H * D
        flops += 2 * pairs * c * (5 * H * D + H) * (3 if train else 1)
        return {"bytes": size * ((5 if train else 2) * pairs * c + (2 if train else 1) * weights), "flops": flops}
    tensor = pairs * H * D
    # forward: q, k, v, bias read, o written; backward: those and dout read, four gradients written (o made in the same pass)
    return {"bytes": size * ((8 if train else 4) * tensor + (2 if train else 1) * pairs * H), "flops": flops}


def tolerance(case):
    """The weights and score gradients pass through the 16-bit type on their way into the matrix cores: 8
    significant bits in bf16, 11 in fp16 (which also carries the attention of an fp32 block), with a softmax
    gradient that is a difference of nearly equal numbers; the bf16 block rounds at every layer besides."""
    if case["dtype"] == "bf16":
        return {"rel": 2e-2 if case["op"] == "block" else 1e-2}
    return {"rel": 5e-3}
