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
        if case["steps"].startswith("1") and op.endswith("tdt") and 2 * case["U"] > case["T"]:
            continue  # no duration 0: a frame a label, and some utterances would have no alignment
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


def _inputs(case, seed):
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
    if case["op"] == "logprobs":  # the graph loss hands back a gradient of the scores
        state["grad_scores"] = [-torch.rand(B, T, U, generator=gen, device=device) for _ in range(2)]
    return state


def prepare(case, seed):
    state = _inputs(case, seed)
    V, options = case["V"], dict(fastemit_lambda=case["fastemit"], clamp=case["clamp"])
    if case["op"] == "rnnt":
        state["loss"] = RNNTLossNumba(blank=V - 1, reduction="none", **options)
    elif case["op"] == "wrapper":
        state["loss"] = RNNTLoss(num_classes=V - 1, loss_kwargs=options)
    elif case["op"] == "tdt":
        state["loss"] = TDTLossNumba(blank=V - 1, durations=_steps(case), reduction="none", sigma=case["sigma"], **options)
    elif case["op"] == "multiblank":
        state["loss"] = MultiblankRNNTLossNumba(blank=V - 1, big_blank_durations=_steps(case), reduction="none",
                                                sigma=case["sigma"], **options)  # fmt: skip
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


def _arcs(case):
    """(frames, labels, token, place of its duration or None) of every arc out of a cell; a big blank's token is its place."""
    if case["op"].endswith("tdt"):
        steps = list(enumerate(_steps(case)))
        return [(d, 0, "blank", i) for i, d in steps if d > 0] + [(d, 1, "label", i) for i, d in steps]
    arcs = [(1, 0, "blank", None), (0, 1, "label", None)]
    if case["op"].endswith("multiblank"):
        arcs += [(d, 0, i, None) for i, d in enumerate(_steps(case))]
    return arcs


def _lattice(case, lengths, tokens, durations):
    """Log-likelihood of each utterance and the posterior of every arc, from log-probs [B, T, U] in 64 bits: the forward
    and the backward recursion over anti-diagonals n = t + u, all utterances at once."""
    B, T, U, device = case["B"], case["T"], case["U"], tokens["blank"].device
    frames = torch.tensor([t for t, _ in lengths], device=device)[:, None, None]
    labels = torch.tensor([u for _, u in lengths], device=device)[:, None, None]
    t, u = torch.arange(T, device=device)[:, None], torch.arange(U, device=device)
    N = T + U - 1
    n = torch.arange(N, device=device)[:, None]
    at = (n - u).clamp(0, T - 1)  # the frame of diagonal n, column u
    on = (n >= u) & (n - u < T)

    def skew(x, fill=-math.inf):
        return x[:, at, u].masked_fill(~on, fill).transpose(0, 1).contiguous()  # [N, B, U]

    inside, ends = [], []
    for dt, du, token, place in _arcs(case):
        score = tokens[token] - case["sigma"] + (durations[..., place] if place is not None else 0.0)
        valid = (t < frames) & (u <= labels)
        inside.append(skew(score.masked_fill(~(valid & (t + dt < frames) & (u + du <= labels)), -math.inf)))
        ends.append(skew(score.masked_fill(~(valid & (t + dt == frames) & (u == labels)), -math.inf)) if du == 0 else None)
    finish = torch.logsumexp(torch.stack([e for e in ends if e is not None]), 0)
    shifts = [(dt, du) for dt, du, _, _ in _arcs(case)]
    most = max(dt + du for dt, du in shifts)
    alpha = torch.full((N + most, B, U), -math.inf, dtype=torch.float64, device=device)  # row n + most: diagonal n
    beta = torch.full((N + most, B, U + 1), -math.inf, dtype=torch.float64, device=device)
    alpha[most, :, 0] = 0.0
    for k in range(1, N):
        terms = torch.full((len(shifts), B, U), -math.inf, dtype=torch.float64, device=device)
        for i, (dt, du) in enumerate(shifts):
            if k >= dt + du:
                terms[i, :, du:] = (alpha[most + k - dt - du] + inside[i][k - dt - du])[:, : U - du]
        alpha[most + k] = torch.logsumexp(terms, 0)
    for k in reversed(range(N)):
        terms = [finish[k]] + [beta[k + dt + du][:, du : U + du] + inside[i][k] for i, (dt, du) in enumerate(shifts)]
        beta[k, :, :U] = torch.logsumexp(torch.stack(terms), 0)
    ll = beta[0, :, 0]
    posteriors = []
    for i, (dt, du) in enumerate(shifts):
        through = torch.exp(alpha[most:] + inside[i] + beta[dt + du : dt + du + N, :, du : U + du] - ll[:, None])
        if ends[i] is not None:
            through += torch.exp(alpha[most:] + ends[i] - ll[:, None])
        posteriors.append(through[t + u, :, u].permute(2, 0, 1))  # back to [B, T, U]
    return ll, posteriors


def exact(case, seed):
    """What `run` returns, in 64 bits: log-softmax, the lattice's arc posteriors and the Jacobian of the softmax, by
    definition.  None with dropout, whose mask only the joint's kernels know."""
    if case["dropout"]:
        return None
    s = _inputs(case, seed)
    B, T, U, V = case["B"], case["T"], case["U"], case["V"]
    steps = _steps(case)
    is_tdt = case["op"].endswith("tdt")
    joint = case["op"].startswith("joint")
    lengths = list(zip(s["act_lens"].tolist(), s["label_lens"].tolist()))
    ids = torch.cat([s["labels"], s["labels"].new_zeros(B, 1)], 1)

    def hidden(b):
        return torch.relu(s["f"][b].detach().double()[:, None] + s["g"][b].detach().double())

    def logits(b):
        if joint:
            return hidden(b) @ s["weight"].detach().double().T + s["bias"].detach().double()
        return s["acts"][b].detach().double()

    which = {"blank": V - 1, **{i: V - 2 - i for i in range(len(steps) if case["op"].endswith("multiblank") else 0)}}
    picked, of_durations = {k: [] for k in ("label", *which)}, []
    for b in range(B):
        x = logits(b)
        norm = torch.logsumexp(x[..., :V], -1)
        picked["label"].append(x.gather(-1, ids[b].expand(T, U)[..., None])[..., 0] - norm)
        for k, v in which.items():
            picked[k].append(x[..., v] - norm)
        of_durations.append(torch.log_softmax(x[..., V:], -1) if is_tdt else None)
    tokens = {k: torch.stack(v) for k, v in picked.items()}
    durations = torch.stack(of_durations) if is_tdt else None

    if case["op"] == "logprobs":
        t, u = torch.arange(T, device=ids.device)[:, None], torch.arange(U, device=ids.device)
        cell = (t < s["act_lens"][:, None, None]) & (u <= s["label_lens"][:, None, None])
        target = cell & (u < s["label_lens"][:, None, None])
        scores = (tokens["label"].masked_fill(~target, 0.0), tokens["blank"].masked_fill(~cell, 0.0))
        flow = {"label": -s["grad_scores"][0].double() * target, "blank": -s["grad_scores"][1].double() * cell}
        costs, of_places = None, []
    else:
        ll, posteriors = _lattice(case, lengths, tokens, durations)
        costs = -ll * (1.0 + case["fastemit"])
        flow = {k: torch.zeros(B, T, U, dtype=torch.float64, device=ids.device) for k in tokens}
        of_places = [torch.zeros_like(flow["blank"]) for _ in steps] if is_tdt else []
        for (_, _, token, place), p in zip(_arcs(case), posteriors):
            flow[token] += p * (1.0 + case["fastemit"]) if token == "label" else p
            if place is not None:
                of_places[place] += p
    scale = 1.0
    if case["op"] == "wrapper":
        costs, scale = costs.mean(), 1.0 / B
    if not case["train"]:
        return costs

    total = sum(flow.values())
    if joint:
        grads = [torch.zeros(x.shape, dtype=torch.float64, device=x.device) for x in (s["f"], s["g"], s["weight"], s["bias"])]
    else:
        grads = torch.zeros(s["acts"].shape, dtype=torch.float64, device=ids.device)
    for b in range(B):
        x = logits(b)
        x[..., :V] = torch.softmax(x[..., :V], -1) * total[b][..., None]
        x.scatter_add_(-1, ids[b].expand(T, U)[..., None], -flow["label"][b][..., None])
        for k, v in which.items():
            x[..., v] -= flow[k][b]
        if is_tdt:
            place = torch.stack([p[b] for p in of_places], -1)
            x[..., V:] = torch.exp(durations[b]) * place.sum(-1, keepdim=True) - place
        if case["clamp"] > 0.0:
            x.clamp_(-case["clamp"], case["clamp"])
        if not joint:
            grads[b] = x * scale
            continue
        h, rows = hidden(b), x.reshape(T * U, -1)
        through = (x @ s["weight"].detach().double()) * (h > 0)
        grads[0][b] = through.sum(1)
        grads[1][b] = through.sum(0)
        grads[2] += rows.T @ h.reshape(T * U, -1)
        grads[3] += rows.sum(0)
    if joint:
        return (costs, *grads)
    return (*scores, grads) if case["op"] == "logprobs" else (costs, grads)
