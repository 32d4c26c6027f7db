"""The fused joint's forward kernel gives a wave 32 cells (few tiles) or 64 (many), and computes only the blocks of 64
vocabulary rows that are in use: both splits, for every loss and activation and with dropout, against the loss on
materialised logits, vocabularies around a block's edges."""

import pytest
import torch

from speech_amd import MultiblankRNNTLossNumba, RNNTLossNumba, TDTLossNumba
from speech_amd.joint import joint_dropout_mask, joint_multiblank_loss, joint_rnnt_loss, joint_tdt_loss

pytestmark = pytest.mark.gpu


def _inputs(B, T, U, V, H, seed):
    gen = torch.Generator().manual_seed(seed)
    f, g = (torch.randn(B, n, H, generator=gen).to(torch.bfloat16).cuda() for n in (T, U))
    weight = (torch.randn(V, H, generator=gen) / H**0.5).cuda()
    bias = torch.randn(V, generator=gen).cuda()
    labels = torch.randint(0, V - 1, (B, U - 1), generator=gen).cuda()
    act_lens = torch.randint(1, T + 1, (B,), generator=gen)
    label_lens = torch.randint(0, U, (B,), generator=gen)
    act_lens[0], label_lens[-1] = T, U - 1
    return [x.requires_grad_(True) for x in (f, g, weight, bias)], (labels, act_lens.cuda(), label_lens.cuda())


def _grads(loss, leaves):
    for x in leaves:
        x.grad = None
    costs = loss()
    costs.sum().backward()
    return costs.detach(), [x.grad.float().clone() for x in leaves]


# tiles of 128 cells without padding: 3 x 2 (one group a wave) and 9 x 58 = 522 (two; an odd number in use now and then)
@pytest.mark.parametrize("B,T,U", [(3, 21, 9), (9, 130, 57)])
@pytest.mark.parametrize("V,H", [(5, 256), (63, 320), (64, 256), (65, 384), (129, 512), (193, 640)])
def test_both_splits(B, T, U, V, H):
    leaves, rest = _inputs(B, T, U, V, H, V + B)
    f, g, weight, bias = leaves
    costs, grads = _grads(lambda: joint_rnnt_loss(f, g, weight, bias, *rest, V - 1), leaves)
    module = RNNTLossNumba(blank=V - 1, reduction="none")

    def materialised():  # the same roundings: bf16 sum and hidden vector, bf16 weights, float32 products
        hidden = torch.relu(f.unsqueeze(2) + g.unsqueeze(1)).float()
        return module(hidden @ weight.to(torch.bfloat16).float().T + bias, *rest)

    want, want_grads = _grads(materialised, leaves)
    torch.testing.assert_close(costs, want, rtol=1e-5, atol=1e-3)
    for name, got, ref in zip(("f", "g", "weight", "bias"), grads, want_grads):
        # gradient entries and d hidden are bf16 (2^-9 each, logits fp16): sums of them stay within 2^-6 of the largest
        assert (got - ref).abs().max() <= 2.0**-6 * ref.abs().max(), name


# what one group and two groups of cells compile to for the other losses, activations and dropout; duration rows (from V on)
# and big blanks (below the blank) on both sides of a block's edge
@pytest.mark.parametrize("B,T,U", [(3, 21, 9), (9, 130, 57)])
@pytest.mark.parametrize("loss,V,H", [("rnnt", 65, 640), ("tdt", 62, 640), ("tdt", 126, 512), ("tdt", 64, 320),
                                      ("multiblank", 67, 640), ("multiblank", 131, 512), ("multiblank", 66, 256)])  # fmt: skip
@pytest.mark.parametrize("activation,dropout", [("relu", 0.3), ("tanh", 0.0), ("sigmoid", 0.2)])
def test_both_splits_of_every_loss_and_activation(B, T, U, loss, V, H, activation, dropout):
    steps = {"rnnt": [], "tdt": [0, 1, 2, 3, 4], "multiblank": [2, 4, 8]}[loss]
    rows = V + len(steps) if loss == "tdt" else V
    leaves, rest = _inputs(B, T, U, rows, H, V + B + len(activation))
    f, g, weight, bias = leaves
    rest = (rest[0] % (V - 1 - len(steps)), *rest[1:])  # token ids only
    options = dict(dropout=dropout, seed=99, activation=activation)
    keep = joint_dropout_mask(B, T, U, H, dropout, 99, f.device) if dropout else None

    def fused():
        if loss == "tdt":
            return joint_tdt_loss(f, g, weight, bias, *rest, V - 1, steps, sigma=0.05, **options)
        if loss == "multiblank":
            return joint_multiblank_loss(f, g, weight, bias, *rest, V - 1, steps, sigma=0.05, **options)
        return joint_rnnt_loss(f, g, weight, bias, *rest, V - 1, **options)

    module = {
        "rnnt": lambda: RNNTLossNumba(blank=V - 1, reduction="none"),
        "tdt": lambda: TDTLossNumba(blank=V - 1, durations=steps, reduction="none", sigma=0.05),
        "multiblank": lambda: MultiblankRNNTLossNumba(blank=V - 1, big_blank_durations=steps, reduction="none", sigma=0.05),
    }[loss]()

    def rounded(x):  # to bf16 as the joint network's layers round under autocast; the gradient passes in float32
        return x + (x.detach().to(torch.bfloat16).float() - x.detach())

    def materialised():  # (a backward in bf16 would round at every layer: its error alone reaches the bound below)
        hidden = rounded(getattr(torch, activation)(rounded(f.float().unsqueeze(2) + g.float().unsqueeze(1))))
        if dropout:
            hidden = rounded(hidden * keep / (1.0 - dropout))
        return module(hidden @ rounded(weight).T + bias, *rest)

    costs, grads = _grads(fused, leaves)
    want, want_grads = _grads(materialised, leaves)
    torch.testing.assert_close(costs, want, rtol=1e-5, atol=1e-3)
    for name, got, ref in zip(("f", "g", "weight", "bias"), grads, want_grads):
        # (the bound of the test above)
        assert (got - ref).abs().max() <= 2.0**-6 * ref.abs().max(), name
    if loss == "tdt":  # the duration rows on their own: small beside the token rows
        assert (grads[2] - want_grads[2])[V:].abs().max() <= 2.0**-6 * want_grads[2][V:].abs().max()
