"""Which tensors the planner hands to the row-gathering kernel (leading rank stays), without a GPU: tensors timed with and
without it (us a pass with buffers in rotation) where the two differ by 15 % and more."""
import pytest

TIMED = [  # dim, perm, element bytes, row gathering, the plan without it
    ((10, 102, 6062), (0, 2, 1), 8, 33.5, 23.7),
    ((19, 4132, 100), (0, 2, 1), 4, 18.3, 13.0),
    ((9, 441, 1079), (0, 2, 1), 8, 19.4, 14.1),
    ((11, 3, 78, 5, 20, 14), (0, 5, 2, 4, 1, 3), 8, 15.7, 11.9),
    ((12, 43, 57, 134), (0, 3, 2, 1), 8, 18.2, 13.7),
    ((18, 388, 1077), (0, 2, 1), 4, 17.4, 14.0),
    ((29, 103188, 5), (0, 2, 1), 4, 21.0, 34.8),
    ((18, 1330, 629), (0, 2, 1), 4, 22.9, 35.9),
    ((24, 24, 8, 2729), (0, 2, 1, 3), 4, 17.5, 29.4),
    ((21, 2164, 263), (0, 2, 1), 4, 17.7, 29.3),
    ((16, 30, 2, 2, 21, 135), (0, 4, 3, 1, 2, 5), 8, 14.6, 21.5),
    ((1305, 599, 88), (0, 2, 1), 4, 96.4, 120.2),
]


@pytest.mark.parametrize("dim,perm,es,gather_us,other_us", TIMED)
def test_the_faster_of_the_two_is_chosen(cutt, dim, perm, es, gather_us, other_us):
    with cutt.Candidates(list(dim), list(perm), es) as c:
        assert c.info(c.best).rowGather == int(gather_us < other_us)


@pytest.mark.parametrize("dim,es,policy", [
    ((1000, 20, 30), 8, 2),       # 5 MB
    ((1000, 130, 140), 8, 2),     # 146 MB: 0.54 cache sizes
    ((1000, 155, 160), 8, 2),     # 0.74
    ((1000, 160, 160), 8, 3),     # 0.76
    ((1000, 300, 300), 8, 3),
    ((99, 500, 900), 8, 2),       # rows of 792 bytes
    ((2000, 300, 300), 4, 2),
])
def test_loads_go_past_the_caches_only_where_these_hold_little(cutt, dim, es, policy):
    with cutt.Candidates(list(dim), [0, 2, 1], es) as c:
        assert [c.info(i).cachePolicy for i in range(len(c)) if c.info(i).rowGather] == [policy]
