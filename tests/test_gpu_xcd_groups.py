"""Workgroups handed to the XCDs in groups, bit-exact against the oracle: every Tiled numbering, line-aligned stores and the packed
kernel's three item orders, group sizes from one workgroup to more than there are."""
import math

import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture
def method(monkeypatch):
    import torch  # noqa: F401  (before the library is loaded: both must share one HIP runtime)
    import cutt_amd as cutt
    yield lambda m: cutt.set_method_override(m)
    cutt.set_method_override(0)


@pytest.mark.parametrize("es", [4, 8])
@pytest.mark.parametrize("group", [1, 3, 5, 12])
def test_tiled(method, monkeypatch, es, group):
    import cutt_amd as cutt
    from gpu_util import check_case
    method(cutt.METHOD_TILED)
    monkeypatch.setenv("CUTT_XCD_GROUP", str(group))
    for order in ("0", "1", "2", "3", "5", "6", "-1"):
        for aligned in ("0", "1"):
            monkeypatch.setenv("CUTT_TILED_ALIGNED", aligned)
            monkeypatch.setenv("CUTT_TILED_ORDER", order)
            for dim, perm in [((600, 1130), (1, 0)), ((577, 130, 9), (2, 1, 0)), ((65, 4, 33, 70), (3, 2, 1, 0))]:
                info = check_case(dim, perm, es)
                assert info.method_name == "Tiled" and info.numBlocks % (8 << (group - 1)) == 0


@pytest.mark.parametrize("es", [4, 8])
@pytest.mark.parametrize("group", [1, 5, 12])
def test_packed(method, monkeypatch, es, group):
    import cutt_amd as cutt
    from gpu_util import check_case
    monkeypatch.setenv("CUTT_XCD_GROUP", str(group))
    for how in (cutt.METHOD_PACKED, cutt.METHOD_PACKEDSPLIT):
        method(how)
        for order in "012":
            monkeypatch.setenv("CUTT_ITEM_ORDER", order)
            grouped = 0
            for dim, perm in [((5, 7, 11, 13, 17, 19), (4, 2, 0, 5, 1, 3)), ((9, 1700, 5, 26), (2, 1, 0, 3)), ((3, 40, 61, 129), (1, 3, 2, 0))]:
                info = check_case(dim, perm, es)
                grouped += info.numBlocks % (8 << (group - 1)) == 0
            assert grouped >= 2


@pytest.mark.parametrize("dim,perm,es,grouped", [
    ((6000, 6080), (1, 0), 4, True),       # whole lines, past the caches
    ((8200, 5003), (1, 0), 8, True),       # line-aligned windows
    ((379, 131928), (1, 0), 4, False),     # ... of 4-byte elements in strips
    ((1201, 3001), (1, 0), 8, False),      # inside the cache: neighbours share lines
    ((3001, 2999), (1, 0), 4, False),
    # ... with an order that goes with groups: rows in few channels, few rows between the two axes, a fused axis on the line grid
    ((1024, 1056, 64), (1, 0, 2), 4, True), ((1024, 1040, 40), (1, 0, 2), 8, True), ((640, 11, 1344, 4), (2, 1, 0, 3), 8, True), ((6, 320, 8, 2400), (3, 1, 2, 0), 8, True),
    # separate matrices in strips off the line grid, by the kernel that paces its loads
    ((1822, 320, 60), (1, 0, 2), 8, False), ((2001, 448, 100), (1, 0, 2), 4, False),
])
def test_planner_takes_groups_where_lines_are_written_whole(method, monkeypatch, dim, perm, es, grouped):
    import torch
    import cutt_amd as cutt
    import sweep_runner
    st = torch.cuda.current_stream().cuda_stream
    src = sweep_runner.index_pattern(math.prod(dim), es)
    want = sweep_runner.expected_on_device(src, list(dim), list(perm))
    groups = []
    for group in (None, "0", "5"):
        if group:
            monkeypatch.setenv("CUTT_XCD_GROUP", group)
        rc, h = cutt.cuttPlan(len(dim), list(dim), list(perm), es, st)
        assert rc == cutt.CUTT_SUCCESS
        groups.append(cutt.get_plan_info(h).xcdGroup)
        dst = torch.full_like(src, -1)
        assert cutt.cuttExecute(h, src.data_ptr(), dst.data_ptr()) == cutt.CUTT_SUCCESS
        torch.cuda.synchronize()
        assert torch.equal(dst, want), (dim, es, group)
        cutt.cuttDestroy(h)
    assert groups == [5 if grouped else 0, 0, 5]
