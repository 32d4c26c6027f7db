"""The lattice kernels on logarithms that the ones on probabilities (mi_scaled.inc) leave some shapes to: every instantiation
against the oracle, at label axes of one lane, one wave, just beyond, and the widest it takes."""

import pytest

from speech_amd import _native

from test_gpu_lattice_scaled import check, draw

pytestmark = pytest.mark.gpu


def plan(kind, U, steps):
    if kind == "tdt":
        return _native.describe_plan(0, 4, 13, U, 7, D=len(steps), max_duration=max(steps))["lattice"]
    return _native.describe_plan(0, 4, 13, U, 7 + len(steps), max_duration=max(steps), num_big_blanks=len(steps))["lattice"]


# a longest duration above 8: rings of arc scores, two threads a column, as far as LDS holds them; then one wave a lattice
@pytest.mark.parametrize("steps,widest", [([1, 9], 256), ([0, 1, 9], 256), ([0, 1, 2, 9], 128), ([1, 2, 3, 4, 9], 128), ([0, 1, 2, 3, 4, 9], 128),
                                          ([0, 1, 2, 3, 4, 5, 9], 128), ([0, 1, 2, 3, 4, 5, 6, 9], 64), ([0, 1, 12], 128)])  # fmt: skip
def test_tdt_rings(steps, widest):
    assert plan("tdt", widest, steps) == f"tdt_lattice_ring_kernel<D={len(steps)}>"
    for U in sorted({1, 2, 64, 65, widest}):
        if U <= widest:
            check("tdt", *draw(U, "tdt", 4, 13, U, steps), steps)


@pytest.mark.parametrize("steps,U", [([0, 1, 2, 3, 4, 5, 6, 9], 65), ([0, 1, 2, 3, 4, 5, 6, 7, 9], 9), ([0, 1, 2, 3, 4], 257), ([0, 1, 8], 513), ([1], 300)])
def test_tdt_one_wave_a_lattice(steps, U):
    assert plan("tdt", U, steps).startswith("tdt_lattice_kernel<K=")
    check("tdt", *draw(U, "tdt", 3, 13, U, steps), steps)


# big blanks longer than 8, or of equal durations (planes for 1, 2, 4 or 8 of them; workgroups of 256 and of 1024 threads)
@pytest.mark.parametrize("steps", [[9], [2, 9], [2, 4, 9], [9, 2, 4, 3], [2, 3, 4, 5, 9], [2, 3, 4, 5, 6, 7, 8, 9], [2, 2, 4], [1, 3, 3]])
@pytest.mark.parametrize("U", [1, 64, 65, 256])
def test_multiblank_rings(steps, U):
    planes = next(n for n in (1, 2, 4, 8) if len(steps) <= n)
    if max(steps) > 8:
        kernel = f"multiblank_lattice_ring_kernel<NBC={planes}>" if (max(steps) + 1) * (2 + planes) * max(64, U if U != 65 else 128) * 8 <= 160 * 1024 else "multiblank_lattice_pull_kernel"
        assert plan("multiblank", U, steps) == kernel
    check("multiblank", *draw(U, "multiblank", 4, 13, U, steps), steps)


@pytest.mark.parametrize("steps,U,kernel", [([2], 257, "multiblank_lattice_ring_kernel<NBC=1>"), ([2, 3], 300, "multiblank_lattice_ring_kernel<NBC=2>"), ([2, 4, 5], 400, "multiblank_lattice_ring_kernel<NBC=4>"),
                                            ([2, 3, 4, 2, 3], 257, "multiblank_lattice_pull_kernel"), ([2, 3], 600, "multiblank_lattice_ring_kernel<NBC=2>"), ([2, 2, 2, 2, 2], 300, "multiblank_lattice_ring_kernel<NBC=8>")])  # fmt: skip
def test_multiblank_wide_label_axes(steps, U, kernel):
    if kernel.endswith("pull_kernel"):
        steps = [*steps[:-1], 9]
    assert plan("multiblank", U, steps) == kernel
    check("multiblank", *draw(U, "multiblank", 3, 13, U, steps), steps)
