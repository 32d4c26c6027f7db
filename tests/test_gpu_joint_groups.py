"""The fused joint's forward kernel gives a wave 32 cells (few tiles) or 64 (many), and computes only the blocks of 64
vocabulary rows that are in use: both splits against the loss on materialised logits, vocabularies around a block's edges."""

import pytest
import torch

from speech_amd import RNNTLossNumba
from speech_amd.joint import joint_rnnt_loss

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
