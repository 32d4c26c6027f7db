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
    typed = [x.to(dt) for x, dt in zip((f, g, W, bias), dtypes)]

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
