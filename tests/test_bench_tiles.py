"""bench.py names the launches its steps ran: axes whose sweeps ran together
are not shown with tile shapes that nothing used."""
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))


class _Block:
    def __init__(self, tiles):
        self.tiles = tiles


@pytest.mark.parametrize("tiles,names,want", [
    ([0, 0, 4], ["inviscid_char_xy", "inviscid_char_z"], ["x+y march", "x+y march", "march64"]),
    ([0, 0, 0], ["inviscid_xyz", "stage_update"], ["one launch"] * 3),
    ([2, 1, 3], ["inviscid_x", "inviscid_y", "inviscid_z"], ["128x2", "16x16", "march32"]),
    ([0, 0, 0], [], ["64x4", "32x8", "32x8"]),
])
def test_tiles_desc(tiles, names, want):
    import bench
    assert bench.tiles_desc(_Block(tiles), {n: (1.0, 1) for n in names}) == want
