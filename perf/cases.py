"""What the operators of this package are timed on: chunked forward passes, training steps, decode steps and whole
mixing layers, called the way a model calls them.

``listed()`` names the cases, ``draw(rng)`` gives another one of the same ranges, ``prepare(case, seed)`` makes what a
program holds before the call, ``run(state)`` is one pass, ``work(case)`` the bytes and operations it cannot do
without and ``tolerance(case)`` how far another correct implementation of the same precision may be from it."""
import math
import os
import random
import sys

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.getcwd(), "flash-linear-attention_amd"))

from fla_amd.modules import FusedRMSNormSwishGate, ShortConvolution, l2_norm  # noqa: E402
from fla_amd.ops.gated_delta_rule import chunk_gated_delta_rule, fused_recurrent_gated_delta_rule  # noqa: E402
from fla_amd.ops.gla import chunk_gla, fused_recurrent_gla  # noqa: E402
from fla_amd.ops.simple_gla import chunk_simple_gla  # noqa: E402

CHUNK = 64        # tokens of a chunk of the chunked algorithms
CONV_WIDTH = 4    # taps of a layer's short convolutions


def _case(name, op, mode, batch, tokens, heads, dim, dtype="bf16", packed=0, l2norm=False, state=False):
    """``packed``: number of sequences in a packed batch (0: ``batch`` sequences of equal length); ``l2norm``: q and k
    arrive raw and the operator normalises them; ``state``: an initial state is given and the final one returned."""
    c = {"op": op, "mode": mode, "batch": batch, "tokens": tokens, "heads": heads, "dim": dim, "dtype": dtype,
         "packed": packed, "l2norm": l2norm, "state": state}
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # One user's next token: the smallest call, one state per head, all launch and host time.
        _case("gla_decode_one", "gla", "decode", 1, 1, 16, 128, state=True),
        # A serving batch's next token: 512 MiB of states read and written in place.
        _case("gdr_decode_batch", "gdr", "decode", 256, 1, 32, 128, state=True),
        # The forward benchmark of the package: a batch of long sequences, states carried in and out.
        _case("gla_forward", "gla", "forward", 8, 4096, 16, 128, state=True),
        # One prompt taken in before decoding: few heads, a long time axis.
        _case("gla_prompt", "gla", "forward", 1, 8192, 16, 128, state=True),
        # A pre-training step of the operator.
        _case("gla_train", "gla", "train", 4, 4096, 16, 128, state=True),
        # The smallest model's step (unit tests, fine-tuning of a toy): short sequences, 64-wide heads.
        _case("gla_train_small", "gla", "train", 2, 256, 4, 64),
        # Requests of very different lengths packed into one prefill.
        _case("gdr_packed", "gdr", "forward", 1, 32768, 16, 128, packed=12, state=True),
        # One prompt of an odd length, q and k normalised by the operator as the layer asks for.
        _case("gdr_prompt", "gdr", "forward", 1, 5003, 16, 128, l2norm=True, state=True),
        # A pre-training step of the delta rule.
        _case("gdr_train", "gdr", "train", 4, 4096, 16, 128, state=True),
        # A training step with one decay per head, many narrow heads, half precision, a ragged length.
        _case("simple_gla_train", "simple_gla", "train", 2, 2000, 32, 64, dtype="fp16"),
        # A gated-delta-net mixing layer in training: convolutions, norms, operator, gated norm, all gradients.
        _case("gdn_layer_train", "gdn_layer", "train", 2, 2048, 16, 128),
        # The same layer for the next token of a small batch: a chain of small launches.
        _case("gdn_layer_decode", "gdn_layer", "decode", 32, 1, 16, 128, state=True),
    ]


# (operator, mode) pairs with the ranges of batch and tokens they are met at
_RANGES = (
    ("gla", "decode", (1, 256), (1, 1)), ("gdr", "decode", (1, 256), (1, 1)), ("gdn_layer", "decode", (1, 256), (1, 1)),
    ("gla", "forward", (1, 16), (64, 32768)), ("gdr", "forward", (1, 16), (64, 32768)),
    ("simple_gla", "forward", (1, 16), (64, 32768)),
    ("gla", "train", (1, 8), (128, 16384)), ("gdr", "train", (1, 8), (128, 16384)),
    ("simple_gla", "train", (1, 8), (128, 16384)), ("gdn_layer", "train", (1, 8), (128, 8192)),
)


def _spread(rng, lo, hi):
    """A whole number of lo..hi, even over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        op, mode, batches, tokens = rng.choice(_RANGES)
        dim = rng.choice((64, 128, 128))
        c = _case(None, op, mode, _spread(rng, *batches), _spread(rng, *tokens), rng.choice((4, 8, 16, 32)), dim,
                  dtype=rng.choice(("bf16", "bf16", "bf16", "fp16")),
                  l2norm=op == "gdr" and mode != "train" and rng.random() < 0.5,
                  state=mode == "decode" or (op != "gdn_layer" and rng.random() < 0.5))
        if mode != "decode" and op != "gdn_layer" and c["tokens"] >= 1024 and rng.random() < 0.3:
            c.update(batch=1, packed=rng.randint(2, 16))
        if mode != "decode" and rng.random() < 0.5:
            c["tokens"] = max(64, c["tokens"] // 64 * 64)
        if _cost(c) <= most:
            return c


def _dtype(case):
    return {"bf16": torch.bfloat16, "fp16": torch.float16}[case["dtype"]]


def _offsets(case):
    """Sequence boundaries of a packed batch: lengths that differ by an order of magnitude and more."""
    n, total = case["packed"], case["tokens"]
    rng = random.Random(1000003 * n + total)
    w = [rng.uniform(256, 6000) for _ in range(n)]
    at, ends = 0.0, [0]
    for x in w:
        at += x
        ends.append(int(round(at / sum(w) * total)))
    return ends


def prepare(case, seed):
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(seed)
    dt = _dtype(case)
    op, mode, B, T, H, D = (case[k] for k in ("op", "mode", "batch", "tokens", "heads", "dim"))
    train = mode == "train"

    def normal(*shape):
        return torch.randn(*shape, device=dev, generator=gen)

    s = {"op": op, "mode": mode, "l2norm": case["l2norm"], "offsets": None, "h0": None}
    N = B
    if case["packed"]:
        ends = _offsets(case)
        s["offsets"], N = torch.tensor(ends, dtype=torch.int64, device=dev), len(ends) - 1
    if case["state"] or mode == "decode":
        s["h0"] = normal(N, H, D, D) * 0.1
    s["state"] = case["state"] or mode == "decode"
    if op == "gdn_layer":
        s["x"] = [normal(B, T, H * D).to(dt) for _ in range(3)]       # what the q, k and v projections give
        s["gate"] = normal(B, T, H * D).to(dt)
        s["g"] = F.logsigmoid(normal(B, T, H))
        s["beta"] = normal(B, T, H).sigmoid()
        s["shape"] = (B, T, H, D)
        s["convs"] = [ShortConvolution(H * D, CONV_WIDTH, activation="silu").to(dev) for _ in range(3)]
        s["norm"] = FusedRMSNormSwishGate(D).to(dev)
        with torch.no_grad():
            for c in s["convs"]:
                c.weight.copy_(torch.rand(c.weight.shape, device=dev, generator=gen) - 0.5)
            s["norm"].weight.copy_(torch.rand(D, device=dev, generator=gen) + 0.5)
        if mode == "decode":
            for c in s["convs"]:
                c.to(dt)
            s["caches"] = [normal(B, H * D, CONV_WIDTH).to(dt) for _ in range(3)]
        leaves = s["x"] + [s["gate"], s["g"], s["beta"]]
        s["leaves"] = leaves + [c.weight for c in s["convs"]] + [s["norm"].weight]
    else:
        s["q"], s["v"] = normal(B, T, H, D).to(dt), normal(B, T, H, D).to(dt)
        k = normal(B, T, H, D)
        if op == "gdr" and not case["l2norm"]:
            k = F.normalize(k, dim=-1)                                # the delta rule is defined on unit keys
        s["k"] = k.to(dt)
        s["beta"] = None
        if op == "gla":
            s["g"] = F.logsigmoid(normal(B, T, H, D)) / 16            # one decay per key channel
        else:
            s["g"] = F.logsigmoid(normal(B, T, H)) / (16 if op == "simple_gla" else 1)
        if op == "gdr":
            s["beta"] = normal(B, T, H).sigmoid()
        leaves = [s["q"], s["k"], s["v"], s["g"]]
        if op == "gdr":
            leaves.append(s["beta"])
        if s["h0"] is not None:
            leaves.append(s["h0"])
        s["leaves"] = leaves
    if train:
        for x in leaves:
            x.requires_grad_()
        s["do"] = normal(B, T, H, D).to(dt)
        s["dht"] = normal(N, H, D, D) * 0.1 if s["state"] else None
    return s


def _operator(s):
    kw = dict(initial_state=s["h0"], output_final_state=s["state"], head_first=False)
    if s["mode"] == "decode":
        if s["op"] == "gla":
            return fused_recurrent_gla(s["q"], s["k"], s["v"], s["g"], inplace_state=True, **kw)
        return fused_recurrent_gated_delta_rule(s["q"], s["k"], s["v"], s["g"], s["beta"], inplace_state=True,
                                                use_qk_l2norm_in_kernel=s["l2norm"], **kw)
    kw["cu_seqlens"] = s["offsets"]
    if s["op"] == "gla":
        return chunk_gla(s["q"], s["k"], s["v"], s["g"], **kw)
    if s["op"] == "simple_gla":
        return chunk_simple_gla(s["q"], s["k"], s["v"], s["g"], **kw)
    return chunk_gated_delta_rule(s["q"], s["k"], s["v"], s["g"], s["beta"], use_qk_l2norm_in_kernel=s["l2norm"], **kw)


def _layer(s):
    """The mixing part of a gated-delta-net layer: short convolutions of q, k and v, unit-norm q and k, the delta rule,
    the norm with the output gate."""
    decode = s["mode"] == "decode"
    q, k, v = (c(x, cache=s["caches"][i] if decode else None)[0].view(s["shape"])
               for i, (c, x) in enumerate(zip(s["convs"], s["x"])))
    gate = s["gate"].view(s["shape"])
    if decode:
        o, ht = fused_recurrent_gated_delta_rule(q, k, v, s["g"], s["beta"], initial_state=s["h0"],
                                                 output_final_state=True, head_first=False, inplace_state=True,
                                                 use_qk_l2norm_in_kernel=True)
        return s["norm"](o, gate), ht
    o, _ = chunk_gated_delta_rule(l2_norm(q), l2_norm(k), v, s["g"], s["beta"], head_first=False)
    return s["norm"](o, gate), None


def run(s):
    step = _layer if s["op"] == "gdn_layer" else _operator
    if s["mode"] != "train":
        with torch.no_grad():
            o, ht = step(s)
            if s["op"] == "gdn_layer":
                return [o, ht] + s["caches"]
            return [o] if ht is None else [o, ht]
    for x in s["leaves"]:
        x.grad = None
    o, ht = step(s)
    if ht is not None and s["dht"] is not None:
        torch.autograd.backward((o, ht), (s["do"], s["dht"]))
    else:
        o.backward(s["do"])
    return [o.detach()] + ([] if ht is None else [ht.detach()]) + [x.grad for x in s["leaves"]]


def work(case):
    op, mode, B, T, H, D = (case[k] for k in ("op", "mode", "batch", "tokens", "heads", "dim"))
    n = B * T * H
    N = case["packed"] or B
    row = 2 * D                                                      # one 16-bit row of a head
    gates = 4 * D if op == "gla" else 4 if op == "simple_gla" else 8  # fp32: per channel, per head, or g and beta
    states = N * H * D * D * 4
    if mode == "decode":
        flops = n * D * D * (4 if op == "gla" else 6)
        nbytes = n * (4 * row + gates) + 2 * states
        if op == "gdn_layer":                                        # gate, y, the convolution caches in and out
            nbytes += n * row + 3 * n * 2 * CONV_WIDTH * row
        return {"bytes": nbytes, "flops": flops}
    # state update and read-out, causal scores and their product with the values; the delta rule adds k h, the
    # key products of a chunk and its triangular inverse applied to the values
    if op in ("gla", "simple_gla"):
        flops = n * (4 * D * D + 2 * CHUNK * D)
    else:
        flops = n * (6 * D * D + 4 * CHUNK * D)
    nbytes = n * (4 * row + gates)
    if mode == "train":
        flops *= 3                                                   # two products of the backward for each of the forward
        nbytes += n * (7 * row + 2 * gates)                          # q, k, v, do and the gates in; dq, dk, dv and theirs out
        if op == "gdn_layer":                                        # forward: gate; backward: gate in, its gradient out
            nbytes += 3 * n * row
    if case["state"]:
        nbytes += states * (4 if mode == "train" else 2)
    return {"bytes": nbytes, "flops": flops}


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def tolerance(case):
    # 16-bit operands of the matrix products and 16-bit outputs, sums in fp32.  Against the same step in fp64 the largest
    # relative error of an output in bf16 is 1.7e-3 (decode), 3.3e-3 (forward), 3.7e-3 (training) and, through the three
    # further 16-bit tensors of a layer, 2.7e-3 (decode) and 5.6e-3 (training); four times that.  fp16 has three bits more.
    layer = case["op"] == "gdn_layer"
    rel = {"decode": 1.1e-2 if layer else 7e-3, "forward": 1.3e-2, "train": 2.2e-2 if layer else 1.5e-2}[case["mode"]]
    return {"rel": rel / 8 if case["dtype"] == "fp16" else rel}
