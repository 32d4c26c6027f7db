"""Rows of at most 64 vectors (mi_tile.inc): both passes work on tiles of 8 to 128 rows of a frame.  Every row length
class against the float64 oracle: rows shorter than a vector, tiles of every size, a last tile of one row, a label axis
just beside a tile's edge, both dtype widths, duration and big-blank entries inside a tile, gradients at another phase."""

import numpy as np
import pytest
import torch

import oracle
from speech_amd import MultiblankRNNTLossNumba, RNNTLossNumba, TDTLossNumba

pytestmark = pytest.mark.gpu

# (U, V): V + extras from below one vector to 64 whole vectors and an odd end; U around the 8 .. 128 rows of a tile
SHAPES = [(1, 2), (9, 3), (128, 5), (129, 5), (200, 11), (65, 29), (64, 33), (33, 65), (17, 127), (16, 129), (9, 255), (8, 259)]
F32, BF16 = torch.float32, torch.bfloat16


def _case(U, V, dtype, extra=0, seed=0):
    rng = np.random.RandomState(1000 * U + V + seed)
    B, T = 3, 7
    x = torch.tensor(rng.randn(B, T, U, V + extra) * 2).to(dtype)
    labels = rng.randint(0, max(V - 1 - 2 * (extra == 0 and V > 8), 1), size=(B, U - 1))
    act_lens = np.array([T, 4, 6])
    label_lens = np.array([(U - 1) // 3, U - 1, max(U - 2, 0)])
    return x, labels, act_lens, label_lens


def _run(loss, x, labels, act_lens, label_lens):
    acts = x.to("cuda").requires_grad_(True)
    costs = loss(acts, *(torch.tensor(v, device="cuda") for v in (labels, act_lens, label_lens)))
    costs.sum().backward()
    return costs.detach().float().cpu().numpy(), acts.grad.float().cpu().numpy()


def _check(got, want, dtype):
    # float32: the suite's bars; bf16 gradients (at most 2 in magnitude) to one rounding step, 2^-8 of the value
    costs, grads = got
    np.testing.assert_allclose(costs, want[0], rtol=1e-5 if dtype == F32 else 2.0**-8)
    np.testing.assert_allclose(grads, want[1], rtol=0 if dtype == F32 else 2.0**-8, atol=1e-5)


@pytest.mark.parametrize("U,V", SHAPES + [(21, 513), (8, 519)])
@pytest.mark.parametrize("dtype", [F32, BF16])
def test_rnnt(U, V, dtype):
    x, *rest = _case(U, V, dtype)
    loss = RNNTLossNumba(blank=V - 1, reduction="none", fastemit_lambda=0.01, clamp=0.4)
    want = oracle.rnnt_loss(x.double().numpy(), *rest, V - 1, 0.01, 0.4)
    _check(_run(loss, x, *rest), want, dtype)


# 16-bit rows of 57 to 64 vectors, with durations 41 to 64, give their gradient a wave each: the last rows of the tiles and
# the first of the waves, the same rows in float32
@pytest.mark.parametrize("V", [455, 456, 512])
@pytest.mark.parametrize("dtype", [BF16, torch.float16])
def test_rnnt_rows_about_the_line(V, dtype):
    x, *rest = _case(11, V, dtype)
    loss = RNNTLossNumba(blank=V - 1, reduction="none", fastemit_lambda=0.01, clamp=0.4)
    want = oracle.rnnt_loss(x.double().numpy(), *rest, V - 1, 0.01, 0.4)
    _check(_run(loss, x, *rest), want, dtype)


@pytest.mark.parametrize("V,dtype", [(327, BF16), (328, BF16), (335, torch.float16), (515, BF16), (197, F32), (255, F32)])
def test_tdt_rows_about_the_line(V, dtype):
    durations = [0, 1, 2, 3, 4]
    x, *rest = _case(11, V, dtype, extra=len(durations))
    loss = TDTLossNumba(blank=V - 1, durations=durations, reduction="none", sigma=0.05)
    want = oracle.tdt_loss(x.double().numpy(), *rest, V - 1, durations, 0.05)
    _check(_run(loss, x, *rest), (want[0], want[1]), dtype)


@pytest.mark.parametrize("U,V", [(9, 3), (65, 29), (16, 129), (8, 257)])
@pytest.mark.parametrize("dtype", [F32, BF16])
def test_tdt(U, V, dtype):
    durations = [0, 1, 2, 4]
    x, *rest = _case(U, V, dtype, extra=len(durations))
    loss = TDTLossNumba(blank=V - 1, durations=durations, reduction="none", sigma=0.05)
    want = oracle.tdt_loss(x.double().numpy(), *rest, V - 1, durations, 0.05)
    _check(_run(loss, x, *rest), want, dtype)


@pytest.mark.parametrize("U,V", [(65, 29), (16, 129), (8, 257)])
def test_multiblank(U, V):
    x, *rest = _case(U, V, F32)
    loss = MultiblankRNNTLossNumba(blank=V - 1, big_blank_durations=[2, 4], reduction="none", sigma=0.05)
    want = oracle.multiblank_loss(x.double().numpy(), *rest, V - 1, [2, 4], 0.05)
    _check(_run(loss, x, *rest), want, F32)


@pytest.mark.parametrize("U", [129, 193, 257, 500, 1000])
def test_wide_label_axis(U):
    """The RNNT recursion in workgroups of 4, 8 and 16 waves: utterances that end beside a wave's edge and fewer
    diagonals than a batch."""
    rng = np.random.RandomState(U)
    B, T, V = 4, 5, 4
    x = torch.tensor(rng.randn(B, T, U, V))
    labels = rng.randint(0, V - 1, size=(B, U - 1))
    act_lens, label_lens = np.array([T, 1, 3, 4]), np.array([U - 1, 2, 63, 128])
    loss = RNNTLossNumba(blank=V - 1, reduction="none")
    want = oracle.rnnt_loss(x.float().double().numpy(), labels, act_lens, label_lens, V - 1)
    _check(_run(loss, x.float(), labels, act_lens, label_lens), want, F32)
