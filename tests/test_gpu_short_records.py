"""RNNT over short rows: cell records of 16 bytes, with the label id and the clamp's bound found by the gradient tile.  What it has
to find: the scale of an utterance (per utterance, broadcast, negative, none, the mean's factor), no label in the last column
or with U = 1, a label that is the blank, a tile that begins past the last label.  Tolerances as in test_gpu_tiles.py, the
absolute one times the largest scale."""

import numpy as np
import pytest
import torch

import oracle
from speech_amd import RNNTLossNumba

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("U,V", [(1, 5), (2, 29), (33, 29), (130, 9), (40, 129), (9, 257)])
@pytest.mark.parametrize("clamp", [0.0, 0.05])
@pytest.mark.parametrize("scale", ["per utterance", "broadcast", "mean"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_scales_bounds_and_labels(U, V, clamp, scale, dtype):
    rng = np.random.RandomState(10 * U + V)
    B, T = 3, 6
    x = torch.tensor(rng.randn(B, T, U, V) * 2).to(dtype)
    labels = rng.randint(0, V - 1, size=(B, U - 1))
    labels[:, ::3] = V - 1  # (the blank's own id)
    act_lens, label_lens = np.array([T, 2, 5]), np.array([U // 2 if U > 1 else 0, U - 1, 0])
    costs, grads = oracle.rnnt_loss(x.double().numpy(), labels, act_lens, label_lens, V - 1, 0.01, clamp)[:2]
    acts = x.to("cuda").requires_grad_(True)
    loss = RNNTLossNumba(blank=V - 1, reduction="mean" if scale == "mean" else "none", fastemit_lambda=0.01, clamp=clamp)
    got = loss(acts, *(torch.tensor(v, device="cuda") for v in (labels, act_lens, label_lens)))
    if scale == "per utterance":
        w = np.array([-1.5, 0.0, 2.0], dtype=np.float32)
        (got * torch.tensor(w, device="cuda")).sum().backward()
    else:
        w = np.full(B, -3.0 / (B if scale == "mean" else 1), dtype=np.float32)
        (-3.0 * got.sum()).backward()
    want = grads * w[:, None, None, None]
    assert acts.grad.dtype == dtype
    np.testing.assert_allclose(acts.grad.float().cpu().numpy(), want, rtol=0 if dtype == torch.float32 else 2.0**-8,
                               atol=3e-5)  # fmt: skip
