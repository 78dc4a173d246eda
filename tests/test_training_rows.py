"""The rows of the training recurrence's states (host logic, CPU): how many columns are kept free behind a batch."""

from __future__ import annotations

import pytest


@pytest.mark.parametrize("batch,pad", [(1, 0), (2, 2), (3, 1), (4, 0), (23, 1), (24, 0), (25, 7), (32, 0), (33, 31), (36, 28),
                                       (67, 29), (256, 0)])
def test_rows_are_whole_pieces_and_from_25_positions_on_whole_lines(batch, pad):
    """A single position keeps rows of one column, which the one-column products take."""
    from chessfly.brain import _pad_columns
    assert _pad_columns(batch, 166_700) == pad


def test_rows_stay_below_2_gib_where_the_batch_alone_does():
    from chessfly.brain import _pad_columns
    rows = 2 ** 31 // (4 * 68)                   # 68 columns are the most below 2 GiB
    assert _pad_columns(66, rows) == 2           # not 96 columns
    assert _pad_columns(67, rows) == 1
    assert _pad_columns(68, rows) == 0
    assert _pad_columns(69, rows) == 0
