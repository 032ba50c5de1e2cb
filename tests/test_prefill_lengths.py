"""Lengths a prefill plan refuses before anything is launched (no GPU).

A negative chunk length shifts the rows of the sequences after it, so the
launch would read and write rows outside its tensors although the lengths' sum
fits; a negative prefix hides the chunk's own first keys.
"""

import pytest
import torch

from mini_vllm.attention import paged_attention_gpu as pag

CPU = torch.device("cpu")


@pytest.fixture(autouse=True)
def plan_on_the_host(monkeypatch):
    monkeypatch.setattr(pag, "_groups_per_cu", lambda *a: (2, 256))
    pag.invalidate_cached_metadata()
    yield
    pag.invalidate_cached_metadata()


def _plan(cached, qlens):
    table = torch.arange(4 * len(cached)).view(-1, 4)
    return pag._prefill_plan(table, list(range(len(cached))), cached, qlens, 16, 64, 14, 2, 64,
                             torch.bfloat16, CPU)


@pytest.mark.parametrize("cached,qlens", [
    ([0, 0], [-3, 5]), ([0, 0], [5, -3]), ([16, 0, 0], [4, -1, 4]),  # the sum fits 2, 2 and 7 rows
    ([-5], [3]), ([-20], [3]), ([16, -1], [2, 2]), ([-1, 0], [-1, 4]),
])
def test_negative_lengths_are_refused(cached, qlens):
    with pytest.raises(IndexError, match="insufficient: invalid lengths"):
        _plan(cached, qlens)


@pytest.mark.parametrize("cached", [1 << 30, 1 << 31, 1 << 40])
def test_prefixes_no_pool_holds_are_refused(cached):
    with pytest.raises(IndexError, match="insufficient to cover"):
        _plan([0, cached], [2, 2])


def test_a_sequence_without_a_chunk_needs_no_prefix(monkeypatch):
    """Accepted as before: its prefix is never read."""
    for cached in ([0, 0], [-1, 0], [-40, 0]):
        plan = _plan(cached, [0, 5])
        assert plan[1].tolist() == [[0, 0, 0, 0], [1, 0, 0, 5]]


def test_a_flagged_prefix_never_reaches_the_launch(monkeypatch):
    """Whatever the device check flags is an error, also where the look-up on
    the host finds nothing."""

    class Lib:
        def __getattr__(self, name):
            return getattr(lib, name)

        @staticmethod
        def mv_prefill_prefix_check(*a):
            return 0

    lib, stub = pag._hip.load(), Lib()
    monkeypatch.setattr(pag, "PREFILL_HOST_CHECK_SEQS", 0)
    monkeypatch.setattr(pag._hip, "load", lambda: stub)
    monkeypatch.setattr(pag, "_stream", lambda device: 0)
    real = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, **k: real(*a, **k).fill_(1))
    with pytest.raises(IndexError, match="insufficient"):
        _plan([16, 16], [2, 2])


@pytest.mark.parametrize("seqs", [1, 2])
def test_a_host_table_of_few_sequences_is_checked_on_the_host(monkeypatch, seqs):
    monkeypatch.setattr(pag, "PREFILL_HOST_CHECK_SEQS", seqs)
    assert _plan([64] * seqs, [2] * seqs)[3] > 0
    for cached in (65, 4000):  # the rows hold 4 blocks of 16
        with pytest.raises(IndexError, match="insufficient"):
            _plan([16] * (seqs - 1) + [cached], [2] * seqs)
    table = torch.tensor([[0, 1, 64, -1]] * seqs)  # 64 pool blocks
    with pytest.raises(IndexError, match="not all pool blocks"):
        pag._prefill_plan(table, list(range(seqs)), [33] * seqs, [1] * seqs, 16, 64, 14, 2, 64,
                          torch.bfloat16, CPU)
