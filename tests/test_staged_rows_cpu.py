"""Row sets of the hook and of a commit: contiguous ranges, row lists and their comparison."""

import pytest
import torch

from taomate_hd_amd import HeadMajorRingKVCache, KVContract
from taomate_hd_amd.hook import StreamingAttentionHook, _Rows


@pytest.mark.parametrize(
    "mask,condition,media",
    [
        ([], (0, 0, None), (0, 0, None)),
        ([1], (0, 0, None), (1, 5, None)),
        ([0, 0], (2, 5, None), (0, 0, None)),
        ([0, 1, 1, 1], (1, 5, None), (3, 6, None)),
        ([0, 1, 0, 1], (2, 5, [5, 7]), (2, 6, [6, 8])),
        ([1, 0, 0, 1, 0], (3, 6, [6, 7, 9]), (2, 5, [5, 8])),
    ],
)
def test_document_rows(mask, condition, media):
    hook = StreamingAttentionHook(HeadMajorRingKVCache(KVContract(layer_names=("l",))))
    full = torch.tensor([True] * 5 + [bool(m) for m in mask] + [True], dtype=torch.bool)
    got = hook._document_rows(torch, 0, 5, 5 + len(mask), full)
    for rows, (count, start, index) in zip(got, (condition, media)):
        assert (rows.count, rows.start) == (count, start)
        assert (None if rows.index is None else rows.index.tolist()) == index
        assert rows.index is None or rows.index.dtype == torch.int32


def test_staged_rows_equal():
    cache = HeadMajorRingKVCache(KVContract(layer_names=("l",)))
    rows = lambda *r: torch.tensor(r, dtype=torch.long)  # noqa: E731
    assert cache.staged_rows_host() is None and not cache.staged_rows_equal(rows(1, 2))
    cache._staged_rows_cpu = rows(4, 2, 9)  # a sink's order: video rows first
    assert cache.staged_rows_host() == (4, 2, 9)
    assert cache.staged_rows_equal(rows(2, 4, 9))
    assert not cache.staged_rows_equal(rows(2, 4)) and not cache.staged_rows_equal(rows(2, 4, 8))
    assert _Rows(torch, rows(2, 3, 4), "cpu").index is None
