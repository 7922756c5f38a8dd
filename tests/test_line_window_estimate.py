"""The cost model's estimate of Tiled plans with line-aligned stores (no GPU)."""
import math

import pytest


@pytest.mark.parametrize("dim,perm,es", [
    ((1201, 60011), (1, 0), 4),        # tiles 128 wide
    ((16411, 9377), (1, 0), 4),
    ((132, 500, 2001), (2, 1, 0), 4),  # one tile along Mm
    ((75, 500, 2001), (2, 1, 0), 8),
    ((1201, 30011), (1, 0), 8),
])
def test_no_plan_has_fewer_lane_slots_than_elements(cutt, monkeypatch, dim, perm, es):
    # copy time x (1 + requested lines beyond those of the data); idle slots of a request can only add to that
    monkeypatch.setenv("CUTT_TILED_ALIGNED", "1")
    size = math.prod(dim) * es
    copy_us = 2.0 * size / (0.64 * 8.192e12) * 1e6  # the model's rate of a copy
    seen = 0
    with cutt.Candidates(list(dim), list(perm), es) as c:
        for i in range(len(c)):
            info = c.info(i)
            if info.method_name != "Tiled":
                continue
            assert info.tiledAligned == 1
            seen += 1
            read, written = info.rdLines * 128 / size, info.wrLines * 128 / size
            base, rd, wr = (1.00, 0.2, 0.1) if es == 4 else (0.95, 0.4, 0.2)
            assert info.usPredicted >= 0.999 * copy_us * (base + rd * (read - 1) + wr * (written - 1)), info.as_dict()
    assert seen
