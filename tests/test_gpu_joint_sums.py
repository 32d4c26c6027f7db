"""The joint backward's sums (mi_joint_gradient_sums): rounding into each gradient's dtype, vectors' remainders, few and many
partial sums, and the prefix scan that the forward's preparation launch carries, through speech_amd.joint.

The sums are formed in float32 in an order that neither the gradients' dtypes nor the other inputs decide, and rounded
once: with float32 tensors that hold the same values the same step gives the unrounded sums, so these checks are exact.
The sums themselves are held against the oracle by `check` (tolerances as in test_gpu_joint.py)."""

import pytest
import torch

from speech_amd.joint import joint_rnnt_loss, joint_tdt_loss

from gpu_utils import DEV
from test_gpu_joint import check, dev_ints, make_case

pytestmark = pytest.mark.gpu

F32, BF16, F16 = torch.float32, torch.bfloat16, torch.float16


# V = 2, 37: the fewest outputs, with the most partial sums each; V odd: a remainder of a vector in d bias
@pytest.mark.parametrize("V,durations", [(2, None), (37, None), (227, None), (300, None), (30, [0, 1, 2])])
@pytest.mark.parametrize("dtypes", [(BF16, BF16, BF16, BF16), (F16, F32, F16, F16), (F32, F16, BF16, F32)])
def test_gradients_are_the_float32_sums_rounded_once(V, durations, dtypes):
    D = len(durations) if durations else 0
    f, g, W, bias, labels, al, ll = make_case(V, 3, 37, 12, 256, V + D)
    lab, ald, lld = dev_ints(labels % max(V - 1, 1), al, ll)
    # (values that bfloat16 holds: weights of another type than float32, and the bias with them, are rounded to it)
    typed = [x.to(BF16).to(dt) for x, dt in zip((f, g, W, bias), dtypes)]

    def grads(tensors, wanted):
        t = [x.to(DEV).requires_grad_(i in wanted) for i, x in enumerate(tensors)]
        if durations:
            costs = joint_tdt_loss(*t, lab, ald, lld, V - 1, durations, sigma=0.05)
        else:
            costs = joint_rnnt_loss(*t, lab, ald, lld, V - 1)
        return torch.autograd.grad(costs.sum(), [t[i] for i in wanted])

    exact = grads([x.to(F32) for x in typed], (0, 1, 2, 3))
    for wanted in ((0, 1, 2, 3), (0, 1), (2, 3), (2,), (0, 1, 2)):
        for i, x in zip(wanted, grads(typed, wanted)):
            assert x.dtype == dtypes[i] and torch.equal(x, exact[i].to(dtypes[i])), (wanted, i)


@pytest.mark.parametrize("B", [63, 64, 65, 129])
def test_prefix_scan_over_the_utterances(B):
    check(B, B, 4, 3, 256, 7)


# label positions of a thread (2, 4 or 8: U up to 64, 128, 256) with their remainders and beyond them (two passes); frames of a
# barrier (four), of a run (16 up to U = 64, else 32), and their remainders; relu's and the other activations' slopes
@pytest.mark.parametrize("U", [1, 31, 33, 64, 65, 97, 128, 129, 256, 257])
@pytest.mark.parametrize("T,activation", [(1, "relu"), (6, "tanh"), (15, "sigmoid"), (34, "relu"), (69, "relu")])
def test_reductions_over_frames_and_label_positions(T, U, activation):
    check(1000 * T + U, 2, T, U, 256, 5, activation=activation)


@pytest.mark.parametrize("U,p", [(33, 0.2), (70, 0.5), (140, 0.2)])
def test_one_pass_over_d_hidden_is_the_two_passes(U, p):
    """With f alone (or g alone) wanted the sums are those of joint_reduce_hidden_kernel, in another order, of the same terms.
    A float32 sum of n <= 140 terms in any order is within n 2^-24 of the sum of their magnitudes; that sum is allowed to
    be 16 times the largest gradient entry, so two orders differ by no more than 2 * 140 * 16 * 2^-24 of it."""
    f, g, W, bias, labels, al, ll = make_case(U, 3, 50, U, 256, 40)
    lab, ald, lld = dev_ints(labels, al, ll)
    f, g, W, bias = (x.to(DEV, F32) for x in (f, g, W, bias))

    def grads(wanted):
        t = [f.clone().requires_grad_("f" in wanted), g.clone().requires_grad_("g" in wanted)]
        costs = joint_rnnt_loss(*t, W, bias, lab, ald, lld, 39, dropout=p, seed=7)
        return torch.autograd.grad(costs.sum(), [x for x in t if x.requires_grad])

    both = grads("fg")
    for x, one in zip(both, (grads("f")[0], grads("g")[0])):
        assert (x - one).abs().max() <= 2 * 140 * 16 * 2.0**-24 * one.abs().max()
