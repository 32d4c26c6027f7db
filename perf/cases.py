"""What the speed of this package is judged on: training and validation steps of the transducer losses, through the
modules and functions a training program calls.

A case is a dict of plain values:
  op        "rnnt" | "tdt" | "multiblank"            the loss modules on given logits [B, T, U, V (+ durations)]
            "wrapper"                                 RNNT through `RNNTLoss`, the wrapper a model constructs
            "logprobs"                                the compact log-prob op of the graph losses
            "joint_rnnt" | "joint_tdt" | "joint_multiblank"   joint network + loss from its inputs [B, T, H], [B, U, H]
  B, T, U, V   batch, frames, label axis (longest label sequence + 1), token outputs (blank, and big blanks, included)
  dtype     of the logits (of the joint's inputs): "float32" | "bfloat16" | "float16"
  train     forward and backward (False: forward under no_grad, a validation loss)
  ragged    lengths spread over about [T/2, T] and [U/3, U-1] as batches of speech have them (False: all full)
  std       of the logits;  fastemit, clamp, sigma: the losses' options
  steps     TDT durations, or durations of the big blanks, as text ("0 1 2 3 4"); "" where the loss has none
  H, dropout   joint cases: hidden units, dropout of the joint network
"""

import math

import torch

from speech_amd.joint import joint_multiblank_loss, joint_rnnt_loss, joint_tdt_loss
from speech_amd.k2 import rnnt_logprobs
from speech_amd.losses import RNNTLoss
from speech_amd.rnnt_loss import MultiblankRNNTLossNumba, RNNTLossNumba, TDTLossNumba

_DEFAULTS = dict(dtype="float32", train=True, ragged=True, std=1.0, fastemit=0.0, clamp=-1.0, sigma=0.0, steps="", H=0,
                 dropout=0.0)  # fmt: skip


def _case(name, op, B, T, U, V, **options):
    return {**_DEFAULTS, "name": name, "op": op, "B": B, "T": T, "U": U, "V": V, **options}


def listed():
    return [
        # the smallest batch of the benchmark configurations: a step of a few short utterances, all launches and host work
        _case("rnnt_small", "rnnt", 4, 50, 21, 129, ragged=False),
        # validation loss of one batch of short utterances: forward only
        _case("rnnt_validation", "rnnt", 8, 187, 46, 1025, train=False),
        # character vocabulary and long audio: the largest lattice, very short rows
        _case("rnnt_characters", "rnnt", 32, 1600, 451, 29),
        # 30 s of audio, 1024 subwords: the benchmark's headline step
        _case("rnnt_subwords", "rnnt", 16, 375, 121, 1025),
        # 60 s of audio under bf16 autocast, through the wrapper a model constructs: the largest tensor of 16-bit logits
        _case("rnnt_bf16_long", "wrapper", 32, 750, 201, 1025, dtype="bfloat16", std=2.0, fastemit=0.001),
        # multilingual vocabulary
        _case("rnnt_large_vocabulary", "rnnt", 8, 250, 101, 16385, fastemit=0.001, clamp=5.0),
        # token-and-duration transducer at the headline shape
        _case("tdt_subwords", "tdt", 16, 375, 121, 1025, sigma=0.05, steps="0 1 2 3 4"),
        # a small ragged batch in 16 bits with a small vocabulary
        _case("tdt_bf16_short", "tdt", 6, 157, 47, 257, dtype="bfloat16", sigma=0.05, steps="0 1 2 3 4"),
        # multi-blank transducer at the headline shape
        _case("multiblank_subwords", "multiblank", 16, 375, 121, 1028, sigma=0.05, steps="2 4 8"),
        # log-probs for a graph loss
        _case("logprobs_bf16", "logprobs", 8, 250, 83, 513, dtype="bfloat16"),
        # joint network + loss without the logits tensor, the headline lattice
        _case("joint_rnnt_subwords", "joint_rnnt", 16, 375, 121, 1025, dtype="bfloat16", H=640),
        # a sub-batch of the fused joint with dropout, as the reference's recipes train
        _case("joint_tdt_subbatch", "joint_tdt", 4, 190, 49, 1025, dtype="bfloat16", sigma=0.05, steps="0 1 2 3 4", H=640,
              dropout=0.2),
    ]  # fmt: skip


def _between(rng, lo, hi):
    """An integer of [lo, hi], uniform over its logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    """One more case of the ranges the listed ones stand for: B 1..32, T 50..1600, U 8..451, V 29..16385 for RNNT;
    T 50..750, U 8..201, V 129..4097 for the other losses and (V up to 2049, H of the kernels) the fused joint; no larger
    than the largest listed one."""
    largest = [work(c) for c in listed()]
    cells_limit = max(c["B"] * c["T"] * c["U"] for c in listed())
    while True:
        op = rng.choice(["rnnt", "rnnt", "wrapper", "tdt", "multiblank", "logprobs", "joint_rnnt", "joint_tdt",
                         "joint_multiblank"])  # fmt: skip
        joint = op.startswith("joint")
        t_max, u_max, v_min, v_max = (1600, 451, 29, 16385) if op in ("rnnt", "wrapper") else (750, 201, 129, 4097)
        case = {**_DEFAULTS, "op": op, "B": _between(rng, 1, 32), "T": _between(rng, 50, t_max),
                "U": _between(rng, 8, u_max), "V": _between(rng, v_min, 2049 if joint else v_max)}  # fmt: skip
        case["dtype"] = "bfloat16" if joint else rng.choice(["float32", "float32", "bfloat16", "float16"])
        case["ragged"] = rng.random() < 0.8
        case["train"] = joint or op == "logprobs" or rng.random() < 0.85
        case["fastemit"] = rng.choice([0.0, 0.001])
        case["clamp"] = rng.choice([-1.0, -1.0, 5.0])
        if op.endswith("tdt"):
            case["steps"] = rng.choice(["0 1 2 3 4", "0 1 2 3 4 5 6 7", "1 2 3 4", "0 1 2 4"])
            case["sigma"] = 0.05
        elif op.endswith("multiblank"):
            case["steps"] = rng.choice(["2", "2 4", "2 4 8"])
            case["sigma"] = 0.05
        if joint:
            case["H"] = rng.choice([256, 320, 384, 512, 640])
            case["dropout"] = rng.choice([0.0, 0.2])
        need = work(case)
        if (case["B"] * case["T"] * case["U"] <= cells_limit and need["bytes"] <= max(w["bytes"] for w in largest)
                and (not joint or need["flops"] <= max(w["flops"] for w in largest))):  # fmt: skip
            return case


def _steps(case):
    return [int(s) for s in case["steps"].split()]


def _row(case):
    """Outputs per cell: the tokens and, for TDT, the durations."""
    return case["V"] + (len(_steps(case)) if case["op"].endswith("tdt") else 0)


def _lengths(case):
    """(frames, labels) of each utterance; the longest of either fills the tensor.  Their pairing is fixed by the case,
    so that every seed's batch is the same amount of work; the seed decides the order in the batch."""
    B, T, U = case["B"], case["T"], case["U"]
    if not case["ragged"] or B == 1:
        return [(T, U - 1)] * B
    t_min, u_min = round(0.53 * T), round(0.33 * (U - 1))
    stride = next(s for s in range(max(1, round(0.618 * B)), B + 2) if math.gcd(s, B) == 1)
    out = []
    for i in range(B):
        j = (i * stride + B // 2) % B
        out.append((T - round((T - t_min) * i / (B - 1)), U - 1 - round((U - 1 - u_min) * j / (B - 1))))
    return out


def prepare(case, seed):
    device = torch.device("cuda")
    gen = torch.Generator(device=device).manual_seed(seed)
    host = torch.Generator().manual_seed(seed)
    B, T, U, V = case["B"], case["T"], case["U"], case["V"]
    dtype = getattr(torch, case["dtype"])
    lengths = _lengths(case)
    order = torch.randperm(B, generator=host).tolist()
    n_tokens = V - 1 - (len(_steps(case)) if case["op"].endswith("multiblank") else 0)
    state = {
        "case": case,
        "labels": torch.randint(0, n_tokens, (B, U - 1), generator=host).to(device),
        "act_lens": torch.tensor([lengths[i][0] for i in order]).to(device),
        "label_lens": torch.tensor([lengths[i][1] for i in order]).to(device),
    }
    if case["op"].startswith("joint"):
        H = case["H"]

        def normal(*shape, scale=1.0, to=torch.float32):
            x = torch.randn(*shape, generator=gen, device=device) * scale
            return x.to(to).requires_grad_(case["train"])

        state["f"] = normal(B, T, H, to=dtype)
        state["g"] = normal(B, U, H, to=dtype)
        state["weight"] = normal(_row(case), H, scale=H**-0.5)
        state["bias"] = normal(_row(case), scale=0.1)
        return state
    acts = torch.empty(B, T, U, _row(case), dtype=dtype, device=device)
    for b in range(B):
        acts[b] = torch.randn(T, U, _row(case), generator=gen, device=device) * case["std"]
    state["acts"] = acts.requires_grad_(case["train"])
    options = dict(fastemit_lambda=case["fastemit"], clamp=case["clamp"])
    if case["op"] == "rnnt":
        state["loss"] = RNNTLossNumba(blank=V - 1, reduction="none", **options)
    elif case["op"] == "wrapper":
        state["loss"] = RNNTLoss(num_classes=V - 1, loss_kwargs=options)
    elif case["op"] == "tdt":
        state["loss"] = TDTLossNumba(blank=V - 1, durations=_steps(case), reduction="none", sigma=case["sigma"], **options)
    elif case["op"] == "multiblank":
        state["loss"] = MultiblankRNNTLossNumba(blank=V - 1, big_blank_durations=_steps(case), reduction="none",
                                                sigma=case["sigma"], **options)  # fmt: skip
    else:  # logprobs: the graph loss hands back a gradient of the scores
        state["grad_scores"] = [-torch.rand(B, T, U, generator=gen, device=device) for _ in range(2)]
    return state


def run(state):
    case = state["case"]
    labels, act_lens, label_lens = state["labels"], state["act_lens"], state["label_lens"]
    blank = case["V"] - 1
    if case["op"].startswith("joint"):
        leaves = [state[k] for k in ("f", "g", "weight", "bias")]
        for x in leaves:
            x.grad = None
        args = (*leaves, labels, act_lens, label_lens, blank)
        options = dict(fastemit_lambda=case["fastemit"], clamp=max(case["clamp"], 0.0), dropout=case["dropout"], seed=7)
        if case["op"] == "joint_rnnt":
            costs = joint_rnnt_loss(*args, **options)
        elif case["op"] == "joint_tdt":
            costs = joint_tdt_loss(*args, _steps(case), sigma=case["sigma"], **options)
        else:
            costs = joint_multiblank_loss(*args, _steps(case), sigma=case["sigma"], **options)
        costs.sum().backward()
        return (costs.detach(), *(x.grad for x in leaves))
    acts = state["acts"]
    acts.grad = None
    if case["op"] == "logprobs":
        scores = rnnt_logprobs(acts, labels, blank, act_lens, label_lens)
        torch.autograd.backward(scores, state["grad_scores"])
        return scores[0].detach(), scores[1].detach(), acts.grad
    with torch.set_grad_enabled(case["train"]):
        if case["op"] == "wrapper":
            costs = state["loss"](log_probs=acts, targets=labels, input_lengths=act_lens, target_lengths=label_lens)
        else:
            costs = state["loss"](acts, labels, act_lens, label_lens)
    if not case["train"]:
        return costs
    costs.sum().backward()
    return costs.detach(), acts.grad


def work(case):
    """Valid logits read once, every gradient element (padding included) written once; the joint never needs its logits
    in memory: its inputs and their gradients, and three products over the valid cells."""
    cells = case["B"] * case["T"] * case["U"]
    valid = sum(t * (u + 1) for t, u in _lengths(case))
    row = _row(case)
    if case["op"].startswith("joint"):
        H = case["H"]
        inputs = case["B"] * (case["T"] + case["U"]) * H * 2 + row * (H + 1) * 4
        return {"bytes": 2 * inputs, "flops": 3 * 2 * valid * row * H}
    size = 4 if case["dtype"] == "float32" else 2
    nbytes = valid * row * size
    if case["train"]:
        nbytes += cells * row * size
    if case["op"] == "logprobs":
        nbytes += 2 * 4 * (cells + valid)
    # an exponential and a multiply-add per logit and direction
    return {"bytes": nbytes, "flops": valid * row * (8 if case["train"] else 4)}


def tolerance(case):
    """Four times the largest error seen against float64 (the losses at up to 1000 frames and 300 labels, the joint at
    small lattices): float32 1.5e-6 (largest single difference 4e-5), bf16 1.7e-3 (4e-3), fp16 an eighth of bf16's;
    the joint, whose gradient entries and d hidden are bf16, 2.8e-3 (2.3e-2)."""
    if case["op"].startswith("joint"):
        return {"rel": 1.1e-2, "max": 9e-2}
    if case["dtype"] == "bfloat16":
        return {"rel": 7e-3, "max": 1.6e-2}
    if case["dtype"] == "float16":
        return {"rel": 9e-4, "max": 2e-3}
    return {"rel": 6e-6, "max": 1.6e-4}
