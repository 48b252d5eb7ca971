"""Tiled transposes over every walk of their tiles (plain, runs per XCD along either axis), word for
word: more and fewer tiles than the eight XCDs, counts that do not divide by eight, partly filled last tiles."""
import pytest

import test_perm_rows_gpu as rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,perm", [
    ([1301, 129], [1, 0]),       # runs, a first: 3 x 21 tiles
    ([1300, 128], [1, 0]),       # the same with aligned rows
    ([129, 2203], [1, 0]),       # runs, b first: 35 x 3 tiles
    ([2081, 2053], [1, 0]),      # runs, b first: 33 x 33 tiles
    ([70, 66], [1, 0]),          # four tiles for eight XCDs
    ([5, 3, 65, 67], [0, 1, 3, 2]),  # runs over planes
    ([1301, 95], [1, 0]),        # runs, a first, the second tile less than half full
    ([1301, 96], [1, 0]),        # half full and one short of full: plain
    ([1301, 127], [1, 0]),
    ([6, 132, 36], [0, 2, 1]),   # aligned planes: plain
    ([96, 200], [1, 0]),         # destination rows on the 128-byte grid: plain
])
@pytest.mark.parametrize("dtype,pad,offset", [("f32", 0, 0), ("u32", 3, 1), ("c64", 0, 0), ("conj", 1, 1)])
def test_tile_orders(ctx, pool, shape, perm, dtype, pad, offset):
    rows.test_rows_word_for_word(ctx, pool, shape, perm, dtype, pad, offset)
