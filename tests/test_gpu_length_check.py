"""The shape check of the loss modules reads the two maxima from two pinned words that belong to the calling thread.  Calls
on several threads and streams must each see their own maxima, a call that failed must leave nothing behind for the next
one, and a check that would have to wait inside a graph capture is refused before anything is enqueued."""

import threading

import pytest
import torch

from speech_amd import RNNTLossNumba

from gpu_utils import DEV

pytestmark = pytest.mark.gpu


def _call(loss, acts, labels, T, U, off):
    """One forward call with length tensors the module has not seen, the longest utterance `off` frames short."""
    act_lens = torch.tensor([T - off, 1], device=DEV)
    label_lens = torch.tensor([1, U - 1], device=DEV)
    return loss(acts, labels, act_lens, label_lens)


def _message(T, off):
    return f"Input length mismatch! Given T: {T}, Expected max T from input lengths: {T - off}"


def test_threads_and_streams_see_their_own_maxima():
    faults = []

    def work(index):
        try:
            T, U, V = 20 + 10 * index, 5, 31
            loss = RNNTLossNumba(blank=V - 1, reduction="none")
            with torch.cuda.stream(torch.cuda.Stream()):
                acts = torch.randn(2, T, U, V, device=DEV)
                labels = torch.ones(2, U - 1, dtype=torch.int64, device=DEV)
                want = _call(loss, acts, labels, T, U, 0)
                for i in range(25):
                    off = i % (index + 2)
                    try:
                        got = _call(loss, acts, labels, T, U, off)
                        assert off == 0 and torch.equal(got, want), (index, i)
                    except ValueError as e:
                        assert off > 0 and str(e) == _message(T, off), (index, i, str(e))
                torch.cuda.current_stream().synchronize()
        except BaseException as e:
            faults.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not faults, faults


def test_streams_of_one_thread_behind_queued_work():
    """The check of a call waits for that call's own kernel, also where its stream has work queued and another stream of the
    same thread was used just before."""
    T, U, V = 40, 6, 33
    loss = RNNTLossNumba(blank=V - 1, reduction="none")
    streams = [torch.cuda.Stream() for _ in range(2)]
    acts = torch.randn(2, T, U, V, device=DEV)
    labels = torch.ones(2, U - 1, dtype=torch.int64, device=DEV)
    busy = torch.randn(2048, 2048, device=DEV)
    torch.cuda.synchronize()
    for i in range(8):
        with torch.cuda.stream(streams[i % 2]):
            for _ in range(i):
                busy @ busy
            if i % 3:
                with pytest.raises(ValueError) as e:
                    _call(loss, acts, labels, T, U, i % 3)
                assert str(e.value) == _message(T, i % 3)
            else:
                assert torch.isfinite(_call(loss, acts, labels, T, U, 0)).all()
    torch.cuda.synchronize()


def test_new_lengths_are_refused_under_capture():
    T, U, V = 12, 4, 17
    loss = RNNTLossNumba(blank=V - 1, reduction="none")
    acts = torch.randn(2, T, U, V, device=DEV)
    labels = torch.ones(2, U - 1, dtype=torch.int64, device=DEV)
    act_lens, label_lens = torch.tensor([T, 1], device=DEV), torch.tensor([1, U - 1], device=DEV)
    graph, captured = torch.cuda.CUDAGraph(), torch.zeros(4, device=DEV)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        captured += 1
        with pytest.raises(RuntimeError, match="cannot be captured"):
            loss(acts, labels, act_lens, label_lens)
    want = loss(acts, labels, act_lens, label_lens)  # the capture went on, and so does eager work
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(captured, torch.ones(4, device=DEV)) and torch.isfinite(want).all()
