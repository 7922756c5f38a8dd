"""Width of the tiles of plans with line-aligned stores along the input's leading axis (no GPU)."""
import pytest


@pytest.mark.parametrize("columns,es,tiles", [
    # us with tiles 64 and 128 wide: (641,177657) 183.9 / 194.8, (650,130785) 135.4 / 143.7, (897,217633) 306.9 / 318.0,
    # (5001,26155) 214.7 / 204.9, all 4-byte elements
    (641, 4, 11), (650, 4, 11), (897, 4, 15), (999, 4, 16), (1000, 4, 8), (5001, 4, 40), (2048, 4, 32),
    # one tile up to the widest, then equal ones
    (136, 4, 1), (137, 4, 3), (68, 8, 1), (69, 8, 2), (5001, 8, 79),
])
def test_tiles_along_the_leading_axis(cutt, monkeypatch, columns, es, tiles):
    monkeypatch.setenv("CUTT_TILED_ALIGNED", "1")
    seen = 0
    with cutt.Candidates([columns, 20011], [1, 0], es) as c:
        for i in range(len(c)):
            if c.info(i).method_name == "Tiled":
                assert c.info(i).tiledAligned == 1 and c.data(i, 1)[4] == tiles
                seen += 1
    assert seen
