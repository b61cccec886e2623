"""The SW queues' work items (no GPU): every candidate once, the longest
targets first, tables of a bounded size that admission counts."""
from types import SimpleNamespace

import numpy as np
import pytest

from sseqs_amd.multi import SW_QUEUE_ITEMS, MultiSearch, sw_item
from sseqs_amd.serve import query_bytes


def _plan(lens, counts, tuning=None):
    ms = MultiSearch.__new__(MultiSearch)  # no buffers
    ms.dev, ms.nq, ms.tuning = "cpu", len(lens), {}
    ms.q_len, ms.kc_q = np.array(lens, np.int64), np.array(counts, np.int64)
    ms.set_sw_tuning(tuning or {})
    return ms


@pytest.mark.parametrize("lens,counts", [
    ([50], [1]), ([60, 200, 61, 900], [16, 17, 5000, 1]), ([200] * 8, [100_000] * 8),
    ([500] * 3, [1_000_000, 7, 4_000_000]), ([33, 64, 1500], [SW_QUEUE_ITEMS * 16, 1, 999])])
def test_items_cover_every_candidate(lens, counts):
    ms = _plan(lens, counts)
    seen = [np.zeros(c, np.int8) for c in counts]
    for b in ms.buckets:
        assert b["n"] == b["item_q"].numel() == b["item_j"].numel() <= SW_QUEUE_ITEMS
        assert 1 <= b["grid"] <= b["n"]
        last = {}
        for q, j in zip(b["item_q"].tolist(), b["item_j"].tolist()):
            assert (lens[q] + 31) // 32 == b["tpt"]
            part = seen[q][j * b["item"]: (j + 1) * b["item"]]
            assert part.size and last.get(q, j + 1) == j + 1  # a query's last chunk first
            part += 1
            last[q] = j
    for q, s in enumerate(seen):
        assert (s == (1 if lens[q] <= 1024 else 0)).all()


def test_item_size_follows_the_queue():
    assert sw_item(16, [20_000]) == 16
    assert sw_item(16, [16 * SW_QUEUE_ITEMS]) == 16
    assert sw_item(16, [16 * SW_QUEUE_ITEMS + 1]) == 32
    assert sw_item(16, [4_000_000] * 2) == 256
    assert sw_item(4096, [100_000]) == 4096 and sw_item(3, [1]) == 3
    assert sw_item(1, [1] * (SW_QUEUE_ITEMS + 9)) == 1  # one candidate each: nothing to join


def test_admission_counts_the_items():
    db = SimpleNamespace(n=8_000_000, device="cpu")
    rest = lambda kc: query_bytes(db, 300, kc, 200) - 12 * kc  # noqa: E731
    for kc in (200, 20_000, 4_700_000):
        tables = sum(8 * b["n"] for b in _plan([300], [kc]).buckets)
        assert rest(kc) - (200 * (20 + 2 * 801 + 24)) >= tables
