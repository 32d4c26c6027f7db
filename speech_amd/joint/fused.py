"""Joint network + RNNT / TDT loss without the [B,T,U,V] tensor.

The reference computes `joint_net(f.unsqueeze(2) + g.unsqueeze(1))` -- ReLU, Linear(H -> V) -- into a
[B,T,U,V] tensor (nemo/collections/asr/modules/rnnt.py:1707-1724, joint_net built at :1759-1777) and hands it
to the loss (:1573-1578); autograd then keeps that tensor and a gradient of the same size.  Here

  forward   one kernel forms the logits tile by tile on the matrix cores (bf16 operands, float32 accumulation: the
            arithmetic of bf16 autocast) and keeps only each cell's log-softmax denominator and its blank / label
            log-probs; the lattice kernel turns those into the costs.  When a backward is to follow it also keeps the
            logits as fp16 and the hidden activations as bf16, one row per lattice cell of lattices without padding
            (a bound known on the host: nothing is read back from the device);
  backward  two kernels form the gradient of the logits from the saved ones on the fly and multiply it, on the
            matrix cores, with the weights (d hidden) and with the saved activations (d weight, d bias; partial sums
            per slice of the rows, added up here); a reduction kernel sums d hidden, in one pass, over u into d f
            and over t into d g (d g as one partial sum per run of frames, added up here).  No library GEMM, no
            host wait.

`joint_rnnt_loss` is differentiable in f, g, weight and bias; `joint_rnnt_forward` is the no-grad form.
`joint_tdt_loss` / `joint_tdt_forward` are the same for the TDT loss: the Linear layer then has V + D outputs, the
token logits followed by the duration logits (rnnt_pytorch.py:563-568), the token softmax covers the first V, the
duration logits are normalised among themselves, and the lattice kernels are the TDT ones.
`joint_multiblank_loss` / `joint_multiblank_forward`: the multi-blank loss, whose big blanks are ordinary outputs of
the Linear layer just below the blank (rnnt_pytorch.py:442-510).
Dropout of the hidden activations (`jointnet.dropout`) is supported: the keep mask is a hash of (seed, cell, hidden
unit), regenerated by every kernel that needs it instead of being stored; the seed is drawn from torch's default
generator per call unless given.  Activations: ReLU (the reference's default `jointnet.activation`), tanh, sigmoid.
Limits: H in {256, 320, 384, 512, 640}.
"""

import ctypes
import random

import torch

from speech_amd import _native
from speech_amd.rnnt_loss.rnnt import _DTYPE_CODE, _durations_array, _labels_ptr, _on, _ptr, _require_gpu, _stream

__all__ = ["joint_rnnt_forward", "joint_rnnt_loss", "joint_tdt_forward", "joint_tdt_loss", "joint_multiblank_forward",
           "joint_multiblank_loss", "joint_dropout_mask", "JointRNNTLoss"]  # fmt: skip


def joint_workspace(B, T, U, H, V, device, num_durations=0, num_big_blanks=0):
    nbytes = ctypes.c_size_t()
    status = _native.lib().mi_joint_workspace_bytes(B, T, U, H, V, num_durations, num_big_blanks, ctypes.byref(nbytes))
    if status != _native.SUCCESS:
        raise RuntimeError(
            f"fused joint: unsupported shape B={B} T={T} U={U} H={H} V={V} durations={num_durations} "
            f"big blanks={num_big_blanks} (H must be one of 256, 320, 384, 512, 640; at most 8 durations / big blanks)"
        )
    return torch.empty(nbytes.value, dtype=torch.uint8, device=device)


def _check(f, g, weight, bias, labels, act_lens, label_lens):
    """Shapes, dtypes and devices (the checks certify_inputs makes for the loss modules, rnnt_pytorch.py:601-634)."""
    _require_gpu(f, "joint_rnnt_loss")
    if f.dim() != 3 or g.dim() != 3 or f.shape[0] != g.shape[0] or f.shape[2] != g.shape[2]:
        raise ValueError("f must be [B,T,H] and g [B,U,H]")
    B, U = f.shape[0], g.shape[1]
    if weight.dim() != 2 or weight.shape[1] != f.shape[2]:
        raise ValueError("weight must be [V,H]")
    if bias is not None and tuple(bias.shape) != (weight.shape[0],):
        raise ValueError("bias must be [V]")
    for name, t, shape in (("labels", labels, (B, U - 1)), ("act_lens", act_lens, (B,)), ("label_lens", label_lens, (B,))):
        if t.dtype != torch.int64:
            raise TypeError(f"{name} must be int64")
        if tuple(t.shape) != shape:
            raise ValueError(f"{name} must have shape {list(shape)}, got {list(t.shape)}")
        if not t.is_contiguous():
            raise ValueError(f"{name} must be contiguous")
    for name, t in (("g", g), ("weight", weight), ("bias", bias), ("labels", labels), ("act_lens", act_lens),
                    ("label_lens", label_lens)):  # fmt: skip
        if t is not None and t.device != f.device:
            raise ValueError(f"{name} must be on {f.device}")


_ACTIVATIONS = {"relu": 0, "tanh": 1, "sigmoid": 2}  # modules/rnnt.py:1762-1770


def _activation_code(activation):
    try:
        return _ACTIVATIONS[str(activation).lower()]
    except KeyError:
        # the reference's message (modules/rnnt.py:1763)
        raise ValueError("Unsupported activation for joint step - please pass one of [relu, sigmoid, tanh]") from None


def _sum_dtype(dtype):
    """The dtype the kernels leave a gradient in: its own, or float32 for one they do not write."""
    return dtype if dtype in _DTYPE_CODE else torch.float32


def _draw_seed(dropout, seed):
    if not 0.0 <= dropout < 1.0:
        raise ValueError(f"dropout probability has to be in [0, 1), but got {dropout}")
    if seed is not None:
        return int(seed) & 0xFFFFFFFFFFFFFFFF
    if dropout == 0.0:
        return 0
    return int(torch.randint(0, 2**62, (1,)).item())  # CPU generator: follows torch.manual_seed, no device sync


def joint_dropout_mask(B, T, U, H, dropout, seed, device):
    """The keep mask [B,T,U,H] (bool) the kernels derive from (seed, cell, hidden unit), for tests."""
    mask = torch.empty(B, T, U, H, dtype=torch.uint8, device=device)
    device = mask.device  # (whatever torch takes for a device: a name, a number)
    with _on(device):
        status = _native.lib().mi_joint_dropout_mask(_ptr(mask), float(dropout), int(seed), B, T, U, H, _stream(device))
    _native.check_status(status, "joint_dropout_mask")
    return mask.bool()


def _check_durations(durations, weight, blank):
    durations = [int(d) for d in durations]
    if not durations or len(durations) >= weight.shape[0]:
        raise ValueError("durations must be a non-empty list shorter than the joint's output size")
    if not 0 <= blank < weight.shape[0] - len(durations):
        raise ValueError("blank must index one of the token logits (the first V of the V + D outputs)")
    return durations


def _forward(f16, g16, weight, bias, labels, act_lens, label_lens, blank, fastemit_lambda, workspace, dropout=0.0,
             seed=0, durations=None, sigma=0.0, big_blanks=None, act=0, saved=None):
    """saved: (logits fp16 [rows, NP], activations bf16 [rows, H+16]) to keep for a backward call, or None."""
    B, T, H = f16.shape
    D = len(durations) if durations else 0
    U, V = g16.shape[1], weight.shape[0] - D
    device = f16.device
    wdtype = torch.float32 if weight.dtype == torch.float32 else torch.bfloat16
    weight = weight.detach().to(wdtype).contiguous()
    bias = None if bias is None else bias.detach().to(wdtype).contiguous()
    costs = torch.empty(B, dtype=torch.float32, device=device)
    tiles = torch.empty(1, dtype=torch.int32, device=device)
    wcode = _native.DTYPE_F32 if wdtype == torch.float32 else _native.DTYPE_BF16
    keep_args = (None, None, 0) if saved is None else (_ptr(saved[0]), _ptr(saved[1]), saved[0].shape[0] // 128)
    with _on(device):
        if D:
            keep, dur_ptr = _durations_array(durations)
            status = _native.lib().mi_joint_tdt_forward(
                _ptr(f16), _ptr(g16), _ptr(weight), _ptr(bias), wcode, _labels_ptr(labels), _ptr(act_lens),
                _ptr(label_lens), _ptr(costs), _ptr(tiles), float(dropout), int(seed), int(act), B, T, U, H, V, D, dur_ptr,
                int(blank), float(fastemit_lambda), float(sigma), 1, *keep_args, _ptr(workspace), workspace.numel(),
                _stream(device),
            )  # fmt: skip
            del keep
        elif big_blanks:
            keep, dur_ptr = _durations_array(big_blanks)
            status = _native.lib().mi_joint_multiblank_forward(
                _ptr(f16), _ptr(g16), _ptr(weight), _ptr(bias), wcode, _labels_ptr(labels), _ptr(act_lens),
                _ptr(label_lens), _ptr(costs), _ptr(tiles), float(dropout), int(seed), int(act), B, T, U, H, V, len(big_blanks),
                dur_ptr, int(blank), float(fastemit_lambda), float(sigma), 1, *keep_args, _ptr(workspace), workspace.numel(),
                _stream(device),
            )  # fmt: skip
            del keep
        else:
            status = _native.lib().mi_joint_rnnt_forward(
                _ptr(f16), _ptr(g16), _ptr(weight), _ptr(bias), wcode, _labels_ptr(labels), _ptr(act_lens),
                _ptr(label_lens), _ptr(costs), _ptr(tiles), float(dropout), int(seed), int(act), B, T, U, H, V, int(blank),
                float(fastemit_lambda), 1, *keep_args, _ptr(workspace), workspace.numel(), _stream(device),
            )  # fmt: skip
    _native.check_status(status, "fused joint forward")
    return costs, tiles


def joint_rnnt_forward(f, g, weight, bias, labels, act_lens, label_lens, blank, fastemit_lambda=0.0, workspace=None,
                       dropout=0.0, seed=None, activation="relu"):
    """costs [B] (float32) of the RNNT loss on logits = relu(f[:, :, None] + g[:, None]) @ weight.T + bias.

    f [B,T,H], g [B,U,H] (projected encoder / prediction outputs; rounded to bf16 if they are not), weight [V,H] and
    bias [V] of the joint's last Linear (float32 or bf16), labels [B,U-1] int64, lengths [B] int64.  Nothing is
    recorded for autograd.
    """
    _check(f, g, weight, bias, labels, act_lens, label_lens)
    f16 = f.detach().to(torch.bfloat16).contiguous()
    g16 = g.detach().to(torch.bfloat16).contiguous()
    if workspace is None:
        workspace = joint_workspace(f.shape[0], f.shape[1], g.shape[1], f.shape[2], weight.shape[0], f.device)
    seed = _draw_seed(dropout, seed)
    return _forward(f16, g16, weight, bias, labels, act_lens, label_lens, blank, fastemit_lambda, workspace, dropout,
                    seed, act=_activation_code(activation))[0]


def joint_tdt_forward(f, g, weight, bias, labels, act_lens, label_lens, blank, durations, sigma=0.0,
                      fastemit_lambda=0.0, workspace=None, dropout=0.0, seed=None, activation="relu"):
    """costs [B] (float32) of the TDT loss on the joint's V + D logits (weight [V+D,H], bias [V+D]; the last
    D = len(durations) outputs are the duration logits).  Nothing is recorded for autograd."""
    _check(f, g, weight, bias, labels, act_lens, label_lens)
    durations = _check_durations(durations, weight, blank)
    f16 = f.detach().to(torch.bfloat16).contiguous()
    g16 = g.detach().to(torch.bfloat16).contiguous()
    if workspace is None:
        workspace = joint_workspace(f.shape[0], f.shape[1], g.shape[1], f.shape[2], weight.shape[0] - len(durations),
                                    f.device, len(durations))  # fmt: skip
    seed = _draw_seed(dropout, seed)
    return _forward(f16, g16, weight, bias, labels, act_lens, label_lens, blank, fastemit_lambda, workspace, dropout,
                    seed, durations, sigma, act=_activation_code(activation))[0]


class JointRNNTLoss(torch.autograd.Function):
    """costs [B] = RNNT (durations None) or TDT loss of the ReLU joint's logits, differentiable in f, g, weight, bias."""

    @staticmethod
    def forward(ctx, f, g, weight, bias, labels, act_lens, label_lens, blank, fastemit_lambda, clamp, dropout=0.0,
                seed=None, durations=None, sigma=0.0, big_blanks=None, activation="relu"):
        _check(f, g, weight, bias, labels, act_lens, label_lens)
        if clamp < 0:
            raise ValueError("`clamp` must be 0.0 or positive float value.")
        durations = _check_durations(durations, weight, blank) if durations else None
        big_blanks = [int(d) for d in big_blanks] if big_blanks else None
        if durations and big_blanks:
            raise ValueError("durations (TDT) and big blanks (multi-blank) exclude each other")
        D = len(durations) if durations else 0
        f16 = f.detach().to(torch.bfloat16).contiguous()
        g16 = g.detach().to(torch.bfloat16).contiguous()
        B, T, H = f16.shape
        workspace = joint_workspace(B, T, g16.shape[1], H, weight.shape[0] - D, f.device, D,
                                    len(big_blanks) if big_blanks else 0)  # fmt: skip
        seed = _draw_seed(dropout, seed)
        act = _activation_code(activation)
        # What the backward works from, a row per lattice cell: the logits (fp16) and the hidden activations (bf16).
        # Sized by the number of 128-cell tiles lattices without padding would have, which is known here; the tiles
        # actually used are counted on the device and never read back.
        lib = _native.lib()
        U = g16.shape[1]
        rows = lib.mi_joint_tile_bound(B, T, U) * 128
        NP = lib.mi_joint_padded_vocabulary(weight.shape[0])
        if rows <= 0:
            raise RuntimeError(f"fused joint: unsupported shape B={B} T={T} U={U}")
        logits16 = torch.empty(rows, NP, dtype=torch.float16, device=f.device)
        acts = torch.empty(rows, H + 16, dtype=torch.bfloat16, device=f.device)
        costs, tiles = _forward(f16, g16, weight, bias, labels, act_lens, label_lens, blank, fastemit_lambda, workspace,
                                dropout, seed, durations, sigma, big_blanks, act, saved=(logits16, acts))
        ctx.tdt = (durations, float(sigma), big_blanks)
        ctx.save_for_backward(f16, g16, weight, labels, act_lens, label_lens, workspace, logits16, acts)
        ctx.has_bias = bias is not None
        ctx.bias_dtype = None if bias is None else bias.dtype
        ctx.in_dtypes = (f.dtype, g.dtype)
        ctx.args = (int(blank), float(fastemit_lambda), float(clamp), float(dropout), int(seed), act)
        return costs

    @staticmethod
    def backward(ctx, grad_costs):
        f16, g16, weight, labels, act_lens, label_lens, workspace, logits16, acts = ctx.saved_tensors
        blank, fastemit_lambda, clamp, dropout, seed, act = ctx.args
        durations, sigma, big_blanks = ctx.tdt
        D = len(durations) if durations else 0
        NB = len(big_blanks) if big_blanks else 0
        B, T, H = f16.shape
        U, V = g16.shape[1], weight.shape[0] - D
        VD = V + D  # rows of weight
        device = f16.device
        lib = _native.lib()
        rows, NP = logits16.shape
        ntiles = rows // 128
        want_bias = ctx.has_bias and ctx.needs_input_grad[3]
        want_w = ctx.needs_input_grad[2] or want_bias
        want_h = ctx.needs_input_grad[0] or ctx.needs_input_grad[1]
        # d hidden = dlogits . weight, a row per cell (for d f and d g); d weight and d bias as partial sums over
        # slices of the rows, enough slices to give every compute unit a block of 128 vocabulary rows
        d_hidden = torch.empty(rows, H, dtype=torch.bfloat16, device=device) if want_h else None
        slices = max(1, 256 // (NP // 128))
        dw_part = torch.empty(slices, NP, H, dtype=torch.float32, device=device) if want_w else None
        db_part = torch.empty(slices, NP, dtype=torch.float32, device=device) if want_w else None
        grad_costs = grad_costs.to(torch.float32)
        stride = 0 if grad_costs.numel() == 1 else (grad_costs.stride(0) if grad_costs.dim() else 0)
        d_weight = d_bias = d_f = d_g = None
        if want_w or want_h:
            outs = (_ptr(logits16), _ptr(acts), _ptr(d_hidden), _ptr(dw_part), _ptr(db_part), slices, ntiles)
            with _on(device):
                if D:
                    keep, dur_ptr = _durations_array(durations)
                    status = lib.mi_joint_tdt_backward(
                        _labels_ptr(labels), _ptr(act_lens), _ptr(label_lens), *outs, _ptr(grad_costs), int(stride), 1.0,
                        B, T, U, H, V, D, dur_ptr, blank, fastemit_lambda, clamp, sigma, _ptr(workspace),
                        workspace.numel(), _stream(device),
                    )  # fmt: skip
                    del keep
                elif NB:
                    keep, dur_ptr = _durations_array(big_blanks)
                    status = lib.mi_joint_multiblank_backward(
                        _labels_ptr(labels), _ptr(act_lens), _ptr(label_lens), *outs, _ptr(grad_costs), int(stride), 1.0,
                        B, T, U, H, V, NB, dur_ptr, blank, fastemit_lambda, clamp, sigma, _ptr(workspace),
                        workspace.numel(), _stream(device),
                    )  # fmt: skip
                    del keep
                else:
                    status = lib.mi_joint_rnnt_backward(
                        _labels_ptr(labels), _ptr(act_lens), _ptr(label_lens), *outs, _ptr(grad_costs), int(stride), 1.0,
                        B, T, U, H, V, blank, fastemit_lambda, clamp, _ptr(workspace), workspace.numel(),
                        _stream(device),
                    )  # fmt: skip
            _native.check_status(status, "fused joint backward")
        want_f, want_g = ctx.needs_input_grad[0], ctx.needs_input_grad[1]
        # Both of d f and d g wanted (the usual case): one pass over d_hidden forms d f and, per run of frames, a share of d g
        # (runs of a length that U alone decides: the sums then do not depend on how a batch is split into sub-batches).
        # A workgroup walks its run frame by frame, a barrier every four: shorter runs give more workgroups, longer ones
        # fewer partial sums to add.  Runs of 16 frames / 32, us: a step, and the reduction with the sums behind it, at
        # B=16, T=375, H=640, V=257: U=33 443 / 449, 83 / 89; U=64 703 / 710, 109 / 117; U=65 707 / 697, 124 / 115; U=121
        # 1183 / 1170, 178 / 164; U=200 1854 / 1823, 282 / 255; at B=4, T=190, U=49, V=1025 253 / 263, 31 / 41.  Few
        # utterances gain from 16 at larger U too (B=8, T=250, H=256: U=96 272 / 280, U=121 323 / 337), but their number
        # must not decide.
        run = 16 if U <= 64 else 32
        one_pass = want_f and want_g and U <= 256
        chunks = (T + run - 1) // run if one_pass else 0
        if one_pass or want_w:
            f_dtype, g_dtype = (_sum_dtype(t) for t in ctx.in_dtypes)
            if one_pass:
                d_f = torch.empty(B, T, H, dtype=f_dtype, device=device)
                d_g = torch.empty(B, U, H, dtype=g_dtype, device=device)
                dg_part = torch.empty(chunks, B, U, H, dtype=torch.float32, device=device)
            else:
                dg_part = None
            if ctx.needs_input_grad[2]:
                d_weight = torch.empty(VD, H, dtype=_sum_dtype(weight.dtype), device=device)
            if want_bias:
                d_bias = torch.empty(VD, dtype=_sum_dtype(ctx.bias_dtype), device=device)
            with _on(device):
                status = lib.mi_joint_gradient_sums(
                    _ptr(d_hidden) if one_pass else None, _ptr(f16), _ptr(g16), _ptr(act_lens), _ptr(label_lens), _ptr(d_f),
                    _DTYPE_CODE[f_dtype], _ptr(dg_part), chunks, _ptr(d_g), _DTYPE_CODE[g_dtype], _ptr(dw_part), _ptr(db_part),
                    slices, _ptr(d_weight), _DTYPE_CODE[_sum_dtype(weight.dtype)], _ptr(d_bias),
                    _DTYPE_CODE[_sum_dtype(ctx.bias_dtype)], ntiles, dropout, seed, act, B, T, U, H, V, D, NB,
                    _ptr(workspace), workspace.numel(), _stream(device),
                )  # fmt: skip
            _native.check_status(status, "fused joint backward")
            d_weight = None if d_weight is None else d_weight.to(weight.dtype)  # (nothing to do but for odd dtypes)
            d_bias = None if d_bias is None else d_bias.to(ctx.bias_dtype)
        if want_h and not one_pass:
            d_f = torch.empty(B, T, H, dtype=torch.float32, device=device) if want_f else None
            d_g = torch.empty(B, U, H, dtype=torch.float32, device=device) if want_g else None
            with _on(device):
                status = lib.mi_joint_reduce_hidden(
                    _ptr(d_hidden), _ptr(f16), _ptr(g16), _ptr(act_lens), _ptr(label_lens), _ptr(d_f), _ptr(d_g), None, 0,
                    ntiles, dropout, seed, act, B, T, U, H, V, D, NB, _ptr(workspace), workspace.numel(), _stream(device),
                )  # fmt: skip
            _native.check_status(status, "joint_rnnt_loss backward")
        d_f = None if d_f is None else d_f.to(ctx.in_dtypes[0])
        d_g = None if d_g is None else d_g.to(ctx.in_dtypes[1])
        return d_f, d_g, d_weight, d_bias, None, None, None, None, None, None, None, None, None, None, None, None


def _in_sub_batches(fused_batch_size, f, g, labels, act_lens, label_lens, seed, one):
    """The reference's fused sub-batch loop (modules/rnnt.py:1527-1587) around `one(f, g, labels, act_lens,
    label_lens, seed)`: there it bounds the joint tensor, here what the forward keeps for the backward (an fp16 row
    of the padded vocabulary and a bf16 row of activations per lattice cell).  Sub-batches are views; their padding is skipped by the kernels,
    so nothing is trimmed.  Each sub-batch gets its own dropout seed (seed + index when one is given)."""
    B = f.shape[0]
    if not fused_batch_size or fused_batch_size >= B:
        return one(f, g, labels, act_lens, label_lens, seed)
    if fused_batch_size < 1:
        raise ValueError("fused_batch_size must be positive")
    costs = []
    for i, b0 in enumerate(range(0, B, int(fused_batch_size))):
        b1 = min(B, b0 + int(fused_batch_size))
        costs.append(one(f[b0:b1], g[b0:b1], labels[b0:b1], act_lens[b0:b1], label_lens[b0:b1],
                         None if seed is None else int(seed) + i))  # fmt: skip
    return torch.cat(costs)


def joint_rnnt_loss(f, g, weight, bias, labels, act_lens, label_lens, blank, fastemit_lambda=0.0, clamp=0.0,
                    dropout=0.0, seed=None, fused_batch_size=None, activation="relu"):
    """Per-utterance RNNT costs [B] of the joint's logits, with gradients to f, g, weight and bias.

    activation: the joint network's, "relu", "tanh" or "sigmoid" (modules/rnnt.py:1762-1770).
    dropout: probability of the joint network's Dropout (pass 0.0 in eval mode); seed: the mask's 64-bit seed,
    drawn from torch's default generator when None; fused_batch_size: utterances per call of the kernels (the
    reference's `fused_batch_size`), None = the whole batch at once.
    """
    return _in_sub_batches(
        fused_batch_size, f, g, labels, act_lens, label_lens, seed,
        lambda f_, g_, lab_, al_, ll_, seed_: JointRNNTLoss.apply(
            f_, g_, weight, bias, lab_, al_, ll_, blank, fastemit_lambda, clamp, dropout, seed_, None, 0.0, None, activation
        ),
    )


def joint_tdt_loss(f, g, weight, bias, labels, act_lens, label_lens, blank, durations, sigma=0.0, fastemit_lambda=0.0,
                   clamp=0.0, omega=0.0, dropout=0.0, seed=None, fused_batch_size=None, activation="relu"):
    """Per-utterance TDT costs [B] of the joint's V + D logits, with gradients to f, g, weight and bias.

    weight [V+D,H], bias [V+D]: the joint's last Linear, whose last D = len(durations) outputs are the duration
    logits (rnnt_pytorch.py:563-568).  omega: with that probability a call uses the plain RNNT loss on the token
    logits and leaves the duration rows without gradient (gpu_rnnt.py:606-622), drawn with random.uniform as there.
    """
    durations = _check_durations(durations, weight, blank)
    if omega > 0.0 and random.uniform(0, 1) < omega:
        V = weight.shape[0] - len(durations)
        return joint_rnnt_loss(f, g, weight[:V], None if bias is None else bias[:V], labels, act_lens, label_lens,
                               blank, fastemit_lambda, clamp, dropout, seed, fused_batch_size, activation)  # fmt: skip
    return _in_sub_batches(
        fused_batch_size, f, g, labels, act_lens, label_lens, seed,
        lambda f_, g_, lab_, al_, ll_, seed_: JointRNNTLoss.apply(
            f_, g_, weight, bias, lab_, al_, ll_, blank, fastemit_lambda, clamp, dropout, seed_, durations, sigma, None,
            activation
        ),
    )


def _check_big_blanks(big_blank_durations, weight, blank):
    big_blanks = [int(d) for d in big_blank_durations]
    if not big_blanks:
        raise ValueError("big_blank_durations must not be empty (use joint_rnnt_loss without big blanks)")
    if not len(big_blanks) <= blank < weight.shape[0]:
        raise ValueError("the big blanks sit at the outputs blank-1-i: blank must leave room for them below it")
    return big_blanks


def joint_multiblank_forward(f, g, weight, bias, labels, act_lens, label_lens, blank, big_blank_durations, sigma=0.0,
                             fastemit_lambda=0.0, workspace=None, dropout=0.0, seed=None, activation="relu"):
    """costs [B] (float32) of the multi-blank loss on the joint's logits (weight [V,H], V counting the big blanks at
    outputs blank-1-i).  Nothing is recorded for autograd."""
    _check(f, g, weight, bias, labels, act_lens, label_lens)
    big_blanks = _check_big_blanks(big_blank_durations, weight, blank)
    f16 = f.detach().to(torch.bfloat16).contiguous()
    g16 = g.detach().to(torch.bfloat16).contiguous()
    if workspace is None:
        workspace = joint_workspace(f.shape[0], f.shape[1], g.shape[1], f.shape[2], weight.shape[0], f.device, 0,
                                    len(big_blanks))  # fmt: skip
    seed = _draw_seed(dropout, seed)
    return _forward(f16, g16, weight, bias, labels, act_lens, label_lens, blank, fastemit_lambda, workspace, dropout,
                    seed, None, sigma, big_blanks, act=_activation_code(activation))[0]


def joint_multiblank_loss(f, g, weight, bias, labels, act_lens, label_lens, blank, big_blank_durations, sigma=0.0,
                          fastemit_lambda=0.0, clamp=0.0, dropout=0.0, seed=None, fused_batch_size=None,
                          activation="relu"):
    """Per-utterance multi-blank costs [B] of the joint's logits (MultiblankRNNTLossNumba's arguments,
    rnnt_pytorch.py:442-510), with gradients to f, g, weight and bias."""
    big_blanks = _check_big_blanks(big_blank_durations, weight, blank)
    return _in_sub_batches(
        fused_batch_size, f, g, labels, act_lens, label_lens, seed,
        lambda f_, g_, lab_, al_, ll_, seed_: JointRNNTLoss.apply(
            f_, g_, weight, bias, lab_, al_, ll_, blank, fastemit_lambda, clamp, dropout, seed_, None, sigma, big_blanks,
            activation
        ),
    )
