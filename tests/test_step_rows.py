"""BatchDecoder.step's `rows`: refused before any launch where the rows have
page lists of their own (their attention block appends and reads for all B
sequences) and outside 1..B (past the step's buffers)."""
import pytest

from g4hip.decoder import BatchDecoder


class _NoDevice:
    def __getattr__(self, name):
        raise AssertionError(f"launched {name}")


@pytest.mark.parametrize("shared,rows", [(False, 1), (False, 4), (True, 0), (True, 5), (True, -1)])
def test_rows_refused(shared, rows):
    d = BatchDecoder.__new__(BatchDecoder)
    d.ctx, d.s, d.B, d.shared_pages, d.block_attn = _NoDevice(), None, 4, shared, not shared
    with pytest.raises(ValueError, match="rows"):
        d.step(rows=rows)
