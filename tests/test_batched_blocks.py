"""Batches of small blocks staged several at a time: every candidate's address stream against the oracle, and where such candidates exist."""
import math

import pytest

from test_planner import check_all_candidates

TENSORS = [((2, 2, 9001), (1, 0, 2)), ((5, 4, 4097), (1, 0, 2)), ((2, 3, 2, 5, 1999), (2, 0, 3, 1, 4)), ((16, 32, 77), (1, 0, 2)), ((3, 7, 2, 5, 3, 61), (2, 1, 0, 3, 4, 5)),
           ((2, 2, 2, 2, 2, 2, 2, 2, 2, 2, 2, 65), (9, 1, 6, 3, 8, 5, 2, 7, 4, 0, 10, 11))]


def stretches(cutt, dim, perm, es):
    """Candidates whose block is a stretch of the slowest rank with everything below it: both runs are the block."""
    with cutt.Candidates(dim, perm, es) as c:
        infos = [c.info(i) for i in range(len(c))]
    return [i for i in infos if i.method_name == "PackedSplit" and i.numMm == i.rank]


@pytest.mark.parametrize("es", [4, 8])
@pytest.mark.parametrize("dim,perm", TENSORS)
def test_streams(cutt, oracle_mod, dim, perm, es):
    check_all_candidates(cutt, oracle_mod, dim, perm, es)


def test_where_they_exist(cutt):
    for dim, perm in TENSORS[:4]:
        below = math.prod(dim[:-1])
        found = stretches(cutt, dim, perm, 8)
        assert found and all(i.volMmkInCont == i.volMmkOutCont >= 2 * below and i.volMbar == 1 for i in found)
    assert len(stretches(cutt, (27, 19, 997), (1, 0, 2), 8)) == 1  # (one size only)
    # a slowest rank that moves, larger blocks, too few of them
    for dim, perm in (((5, 4097, 4), (1, 0, 2)[::-1]), ((47, 49, 997), (1, 0, 2)), ((5, 4, 3), (1, 0, 2))):
        assert not stretches(cutt, dim, perm, 8)


def test_the_model_takes_them(cutt):
    for dim, perm, es in (((2, 2, 10000000), (1, 0, 2), 8), ((5, 4, 1374779), (1, 0, 2), 8), ((9, 3, 5, 222222), (2, 1, 0, 3), 4)):
        with cutt.Candidates(dim, perm, es) as c:
            best = c.info(c.best)
        assert best.numMm == best.rank and best.volMmkInCont >= 1024
