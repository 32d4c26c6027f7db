"""TDT and multi-blank lattices on probabilities with shared exponents (mi_scaled.inc), against the oracle: the edges of their
groups of 64 columns, batches of diagonals and longest durations, and the inputs that send them to the same recursion on
logarithms (arcs below exp(-693), cells far below their columns, columns far apart, totals near the sentinels, values that are not numbers)."""

import numpy as np
import pytest
import torch

import oracle
from speech_amd import MultiblankRNNTLossNumba, TDTLossNumba, _native

from gpu_utils import call_loss

gpu = pytest.mark.gpu


def check(kind, acts, labels, act_lens, label_lens, steps, sigma=0.05, lam=0.01, cost_rtol=1e-6, grad_atol=1e-5):
    """grad_atol: a posterior is the exponential of a difference of sums of up to T + U float32 log-probs; each is rounded by
    2^-24 of its size, and the test's are below 64 for all but the inputs that say otherwise: 700 * 2^-24 * 4 = 1.7e-4 at
    worst, and with signs that differ the square root of that number of terms, 26 * 2^-24 * 4 = 6e-6.  Relative to the
    largest entry: where no alignment exists (no duration 0, more labels than frames) the sentinels give "posteriors" of
    thousands, rounded relative to their size."""
    acts = np.asarray(acts, dtype=np.float32)
    blank = acts.shape[-1] - 1 - (len(steps) if kind == "tdt" else 0)
    if kind == "tdt":
        fn = TDTLossNumba(blank=blank, durations=steps, reduction="none", fastemit_lambda=lam, sigma=sigma)
        ref = oracle.tdt_loss
    else:
        fn = MultiblankRNNTLossNumba(blank=blank, big_blank_durations=steps, reduction="none", fastemit_lambda=lam, sigma=sigma)
        ref = oracle.multiblank_loss
    costs, grads = call_loss(fn, acts, labels, act_lens, label_lens)
    c_ref, g_ref, _ = ref(acts, labels, act_lens, label_lens, blank, steps, sigma, lam, 0.0, num_threads=4)
    np.testing.assert_allclose(costs, c_ref, rtol=cost_rtol, atol=1e-6)
    err = np.abs(grads - g_ref).max() / max(1.0, np.abs(g_ref).max())
    assert err < grad_atol, err


def draw(seed, kind, B, T, U, steps, tokens=6):
    rng = np.random.RandomState(seed)
    acts = rng.randn(B, T, U, tokens + 1 + len(steps)) * 2
    labels = rng.randint(0, tokens, size=(B, U - 1))
    act_lens, label_lens = rng.randint(1, T + 1, size=B), rng.randint(0, U, size=B)
    act_lens[0], label_lens[0] = T, U - 1  # full, and one of each alone
    act_lens[1 % B], label_lens[-1] = T, U - 1
    return acts, labels, act_lens, label_lens


@gpu
@pytest.mark.parametrize("steps", [[0, 1, 2, 3, 4], [0, 1, 2, 4], [1, 2, 3, 4], [0, 1, 2, 3, 4, 5, 6, 7], [0, 1, 8], [1]])
@pytest.mark.parametrize("U", [1, 2, 63, 64, 65, 128, 129, 192, 193, 256])
def test_tdt_columns_and_durations(U, steps):
    check("tdt", *draw(U, "tdt", 4, 13, U, steps), steps)


@gpu
@pytest.mark.parametrize("steps", [[2], [2, 4], [2, 4, 8], [3, 5, 7], [2, 3, 4, 5, 6, 7, 8], [2, 2], [1, 3], [9]])
@pytest.mark.parametrize("U", [1, 64, 65, 129, 192, 256])
def test_multiblank_columns_and_durations(U, steps):
    check("multiblank", *draw(U, "multiblank", 4, 13, U, steps), steps)


@gpu
@pytest.mark.parametrize("T", [1, 2, 3, 4, 5, 7, 8, 9, 15, 16, 17, 33])
@pytest.mark.parametrize("kind,steps", [("tdt", [0, 1, 2, 3, 4]), ("tdt", [0, 1, 7]), ("multiblank", [2, 4, 8]), ("multiblank", [3])])
def test_frames_about_a_batch(T, kind, steps):
    check(kind, *draw(T, kind, 5, T, 9, steps), steps)


@gpu
@pytest.mark.parametrize("kind,steps", [("tdt", [0, 1, 2, 3, 4]), ("tdt", [0, 1, 2, 3, 4, 5, 6, 7]), ("multiblank", [2, 4, 8]), ("multiblank", [2])])
def test_many_diagonals(kind, steps):
    """Costs of several thousand: the exponents move over many times the range of a double."""
    acts, labels, act_lens, label_lens = draw(7, kind, 3, 600, 90, steps)
    check(kind, acts * 2, labels, act_lens, label_lens, steps, grad_atol=4e-5)


@gpu
@pytest.mark.parametrize("kind,steps,scale", [("tdt", [0, 1, 2, 3, 4], 30.0), ("tdt", [0, 1, 2, 6], 25.0),
                                              ("multiblank", [2, 4, 8], 30.0), ("multiblank", [2], 300.0)])  # fmt: skip
def test_arcs_below_the_range(kind, steps, scale):
    """Log-probs of -60 and far beyond, most of them: the recursion on logarithms decides most.  (TDT with totals above the sentinels' -10000:
    below, the oracle's own posteriors overflow.  Rounding: log-probs of 1000, 2^-24 of each.)"""
    acts, labels, act_lens, label_lens = draw(11, kind, 4, 21, 70, steps)
    check(kind, acts * scale, labels, act_lens, label_lens, steps, cost_rtol=2e-6, grad_atol=60 * 1000 * 2.0**-24)


@gpu
@pytest.mark.parametrize("value", [-70.0, -150.0, -600.0, -686.0, -700.0, -5000.0])
@pytest.mark.parametrize("kind,steps", [("tdt", [0, 1, 2, 3, 4]), ("tdt", [0, 1, 8]), ("multiblank", [2, 4, 8]), ("multiblank", [2])])
@pytest.mark.parametrize("T,U", [(40, 1), (30, 9), (21, 70), (12, 140)])
def test_few_dear_arcs_among_ordinary_ones(kind, steps, value, T, U):
    """Log-probs of `value` in one cell of a hundred, on both sides of the range's lower end.  What passes through such an arc carries
    its rounding, 2^-24 of 690 (beyond: of the gradient's share of next to nothing), and without labels a path may need three."""
    acts, labels, act_lens, label_lens = draw(13, kind, 3, T, U, steps)
    rng = np.random.RandomState(U)
    acts[rng.rand(*acts.shape) < 0.01] = value
    check(kind, acts, labels, act_lens, label_lens, steps, cost_rtol=2e-6, grad_atol=3 * 700 * 2.0**-24)


@gpu
@pytest.mark.parametrize("kind,steps", [("tdt", [0, 1, 2, 3, 4]), ("multiblank", [2, 4, 8])])
def test_columns_far_apart(kind, steps):
    """Labels cost 50 each on all but the last frames, where they are nearly free: on an anti-diagonal the mass falls by up to
    thousands of bits from column to column, further than a column's exponent is raised."""
    B, T, U, tokens = 2, 12, 80, 6
    rng = np.random.RandomState(5)
    acts = rng.randn(B, T, U, tokens + 1 + len(steps)) * 0.1
    labels = rng.randint(0, tokens, size=(B, U - 1))
    blank = acts.shape[-1] - 1 - (len(steps) if kind == "tdt" else 0)
    acts[:, : T - 2, :, :tokens] -= 50.0
    acts[:, T - 2 :, :, blank] -= 30.0
    check(kind, acts, labels, [T, T], [U - 1, 40], steps, cost_rtol=2e-6, grad_atol=1e-4)


@gpu
@pytest.mark.parametrize("value", [float("nan"), float("inf"), float("-inf"), -3.0e38])
@pytest.mark.parametrize("kind,steps", [("tdt", [0, 1, 2, 3, 4]), ("multiblank", [2, 4, 8])])
def test_values_that_are_not_ordinary_stay_with_their_utterance(value, kind, steps):
    acts, labels, act_lens, label_lens = draw(3, kind, 3, 11, 9, steps)
    blank = acts.shape[-1] - 1 - (len(steps) if kind == "tdt" else 0)
    plain = acts.copy()
    acts[0, 4, 3, blank] = value
    make = (lambda: TDTLossNumba(blank=blank, durations=steps, reduction="none", sigma=0.05)) if kind == "tdt" else (
        lambda: MultiblankRNNTLossNumba(blank=blank, big_blank_durations=steps, reduction="none", sigma=0.05))  # fmt: skip
    costs, grads = call_loss(make(), acts, labels, act_lens, label_lens)
    c_ref, g_ref = call_loss(make(), plain, labels, act_lens, label_lens)
    assert np.array_equal(costs[1:], c_ref[1:]) and np.array_equal(grads[1:], g_ref[1:])
    if value < 0:  # an arc that cannot be taken: a cost above that of the utterance with it, and still a number
        assert np.isfinite(costs[0]) and costs[0] > c_ref[0] - 1.0


def test_plan_lines():
    """Which lattice a shape gets: 256 columns, 192 with a longest duration above 4, durations up to 8."""
    for U, longest, scaled in [(121, 4, True), (256, 4, True), (257, 4, False), (192, 8, True), (193, 8, False), (64, 9, False)]:
        tdt = _native.describe_plan(0, 4, 100, U, 65, D=5, max_duration=longest)["lattice"]
        assert tdt.startswith("tdt_lattice_pair_kernel<") == scaled, (U, longest, tdt)
        mb = _native.describe_plan(0, 4, 100, U, 68, max_duration=longest, num_big_blanks=3)["lattice"]
        assert mb.startswith("multiblank_lattice_kernel<") == scaled, (U, longest, mb)


@gpu
@pytest.mark.parametrize("sigma", [0.7, 1.5, -0.8])
@pytest.mark.parametrize("value", [-1.0e10, -1.0e30, float(np.finfo(np.float32).min)])
@pytest.mark.parametrize("kind,steps,column", [
    ("tdt", [0, 1, 2, 3, 4], "blank"), ("tdt", [0, 1, 2, 3, 4], "label"), ("tdt", [0, 1, 2, 3, 4], "step"),
    ("tdt", [0, 1, 2, 6], "step"), ("multiblank", [2, 4, 8], "blank"), ("multiblank", [2, 4, 8], "label"),
    ("multiblank", [2, 4], "step")])  # fmt: skip
def test_masked_arcs_whatever_sigma(kind, steps, column, value, sigma):
    """An arc that is masked out, far below the range of a float exponent: in all cells for a duration (or big blank), in one for
    a token, of an utterance without labels, one with some and one with all of them.  Every utterance keeps a path without it."""
    acts, labels, _, _ = draw(17, kind, 3, 9, 5, steps)
    blank = acts.shape[-1] - 1 - (len(steps) if kind == "tdt" else 0)
    acts = acts.astype(np.float32)
    if column == "step":
        acts[..., acts.shape[-1] - 1 if kind == "tdt" else blank - 1] = value
    elif column == "blank":
        acts[:, 3, :, blank] = value
    else:
        for b in range(3):
            acts[b, 3, 1, labels[b, 1]] = value
    check(kind, acts, labels, [9, 9, 8], [0, 2, 4], steps, sigma=sigma)


def steep(kind, steps, level, T, U, B=2, seed=0, jitter=0.0):
    """Logits whose arcs all have log-probs of `level`, beside one likely token that is no label and, for TDT, a likely duration of
    0: long steps and runs of short ones reach the same cells with hundreds of bits between them on the way."""
    rng = np.random.RandomState(seed)
    tokens = 6
    acts = rng.randn(B, T, U, tokens + 1 + len(steps)) * jitter
    labels = rng.randint(0, tokens - 1, size=(B, U - 1))  # (token 5 is never a label)
    if kind == "tdt":
        acts[..., 5] -= level  # blank and labels at `level`
        acts[..., tokens + 1] -= level  # duration 0: of no use to a blank
    else:
        acts[..., 5] -= level
    return acts, labels


@gpu
@pytest.mark.parametrize("level", [-40.0, -50.0, -55.0, -59.0])
@pytest.mark.parametrize("kind,steps,T,U", [("tdt", [0, 1, 8], 15, 1), ("tdt", [0, 1, 8], 40, 1), ("tdt", [0, 1, 8], 31, 9), ("tdt", [0, 1, 2, 8], 30, 4), ("tdt", [0, 1, 6], 25, 7),
                                            ("tdt", [0, 1, 4], 29, 12), ("tdt", [0, 1, 8], 24, 70), ("multiblank", [8], 33, 5), ("multiblank", [2, 8], 24, 70)])  # fmt: skip
def test_long_steps_beside_runs_of_short_ones(kind, steps, T, U, level):
    """Costs of about 100 * level, each log-prob rounded by 2^-24 of its size: up to (T + U) * 60 * 2 * 2^-24 in an exponent."""
    acts, labels = steep(kind, steps, level, T, U)
    check(kind, acts, labels, [T, T - 2], [U - 1, U // 2], steps, sigma=0.05, lam=0.0, grad_atol=(T + U) * 120 * 2.0**-24)
