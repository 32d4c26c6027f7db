"""The maxima of the lengths that the first kernel of a forward call leaves in the caller's words: every kernel of pass 1, few and
many utterances (a wave takes 64 at a time), and the checks of the loss modules that read them."""

import pytest
import torch

from speech_amd import MultiblankRNNTLossNumba, RNNTLossNumba, TDTLossNumba, _native
from speech_amd.rnnt_loss import rnnt

from gpu_utils import DEV

pytestmark = pytest.mark.gpu

# V and dtype of a row: by tile, by wave, by workgroup, streamed (more than 8192 vectors of 16 bytes)
ROWS = [(29, torch.float32), (1025, torch.float32), (1025, torch.bfloat16), (2100, torch.float16), (4097, torch.float32), (16385, torch.bfloat16),
        (40000, torch.float32)]  # fmt: skip


def test_the_rows_reach_every_kernel_of_pass_1():
    code = {torch.float32: _native.DTYPE_F32, torch.bfloat16: _native.DTYPE_BF16, torch.float16: _native.DTYPE_F16}
    kernels = {_native.describe_plan(code[dtype], 3, 3, 2, V)["denominators"].split("<")[0] for V, dtype in ROWS}
    assert kernels == {"denom_tile_kernel", "denom_rows_kernel", "denom_block_kernel", "denom_gather_kernel"}


@pytest.mark.parametrize("V,dtype", ROWS)
@pytest.mark.parametrize("B,where", [(1, 0), (3, 2), (64, 63), (65, 64), (130, 70)])
def test_words_hold_the_maxima(V, dtype, B, where):
    T, U = 3, 2
    acts = torch.randn(B, T, U, V, device=DEV).to(dtype)
    act_lens = torch.ones(B, dtype=torch.int64)
    label_lens = torch.zeros(B, dtype=torch.int64)
    act_lens[where], label_lens[B - 1 - where] = T, U - 1
    act_lens, label_lens = act_lens.to(DEV), label_lens.to(DEV)
    labels = torch.zeros(B, U - 1, dtype=torch.int64, device=DEV)
    costs, unchecked = torch.empty(B, device=DEV), torch.empty(B, device=DEV)
    words = torch.full((2,), rnnt.LENGTHS_PENDING, dtype=torch.int64, pin_memory=True)
    workspace = rnnt.new_workspace(acts)
    rnnt.rnnt_forward(acts, labels, act_lens, label_lens, costs, V - 1, 0.0, True, workspace, None, words)
    rnnt.wait_lengths(words, torch.cuda.current_stream())
    assert words.tolist() == [T, U - 1]
    rnnt.rnnt_forward(acts, labels, act_lens, label_lens, unchecked, V - 1, 0.0, True, workspace)
    assert torch.equal(costs, unchecked)


@pytest.mark.parametrize("loss", ["rnnt", "tdt", "multiblank"])
@pytest.mark.parametrize("short_t,short_u", [(1, 0), (0, 1), (0, 0)])
def test_modules_refuse_and_recover(loss, short_t, short_u):
    B, T, U, V = 70, 9, 4, 40
    module = {"rnnt": lambda: RNNTLossNumba(blank=V - 1),
              "tdt": lambda: TDTLossNumba(blank=V - 4, durations=[0, 1, 2], sigma=0.05),
              "multiblank": lambda: MultiblankRNNTLossNumba(blank=V - 1, big_blank_durations=[2, 4], sigma=0.05)}[loss]()  # fmt: skip
    acts = torch.randn(B, T, U, V, device=DEV, requires_grad=True)
    labels = torch.zeros(B, U - 1, dtype=torch.int64, device=DEV)

    def call(t, u):
        return module(acts, labels, torch.full((B,), t, device=DEV), torch.full((B,), u, device=DEV))

    if short_t or short_u:
        with pytest.raises(ValueError, match="Input length mismatch" if short_t else "Output length mismatch"):
            call(T - short_t, U - 1 - short_u)
    call(T, U - 1).sum().backward()
    assert torch.isfinite(acts.grad).all()


def test_words_must_be_reachable_by_the_device():
    acts = torch.randn(1, 2, 2, 5, device=DEV)
    ones = torch.ones(1, dtype=torch.int64, device=DEV)
    for words in (torch.empty(2, dtype=torch.int64), torch.empty(3, dtype=torch.int64, device=DEV), torch.empty(2, device=DEV)):
        with pytest.raises(ValueError, match="int64"):
            rnnt.rnnt_forward(acts, ones.view(1, 1), ones + 1, ones, torch.empty(1, device=DEV), 4, 0.0, True,
                              rnnt.new_workspace(acts), None, words)  # fmt: skip
