"""The scoring launch's chunks per row, on the host (no GPU): the workspace holds one 8-byte slot per (row, chunk) of
the logit width with more chunks, and one 4-byte counter per row."""

import pytest

from helpers import pkg


def _chunks(rows, vocab):
    need = int(pkg("_lib").load().atlas_gather_logprobs_workspace_bytes(rows, vocab))
    assert (need - 4 * rows) % (8 * rows) == 0
    return (need - 4 * rows) // (8 * rows)


@pytest.mark.parametrize("rows,vocab,chunks", [
    (1, 128256, 32), (4, 128256, 32), (5, 128256, 16), (9, 128256, 16), (13, 128256, 11), (50, 128256, 11),
    (128, 128256, 8), (512, 128256, 2), (513, 128256, 1), (1, 32001, 8), (16, 32001, 8), (17, 32001, 4),
    (512, 32001, 2), (1, 16384, 1), (1, 16385, 5), (600, 9001, 1)])
def test_few_rows_are_cut_into_many_chunks(rows, vocab, chunks):
    """fp32 rows, which have the more chunks: single batches of 4096 logits for a handful of rows, longer chunks as the
    rows alone fill the device, one chunk when they do."""
    assert _chunks(rows, vocab) == chunks


def test_chunk_counts_stay_within_what_one_wave_combines():
    """At most 256 chunks per row at every size, never more with more rows."""
    for vocab in (1, 7, 4096, 16385, 32769, 50257, 128256, 256000, 1 << 20, 1 << 24):
        last = 256
        for rows in (1, 2, 3, 5, 9, 13, 20, 35, 64, 100, 200, 300, 512, 1000, 100000):
            c = _chunks(rows, vocab)
            assert 1 <= c <= last
            last = c
