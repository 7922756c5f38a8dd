"""The packed kernels whose arguments are decoded as a walk, one block per workgroup and several, bit-exact against the oracle: every number of elements per lane and cache policy, blocks whose
last lanes have no element of their own, slabs of two sizes on either cut rank, no Mbar rank up to the thirteenth (which the general kernel takes),
workgroups in chunks and groups."""
import pytest

pytestmark = pytest.mark.gpu

TENSORS = [((3, 5, 7), (2, 1, 0)), ((16, 4, 33), (2, 0, 1)), ((7, 67, 5, 61), (3, 0, 2, 1)), ((31, 3, 37, 5, 6), (2, 0, 4, 1, 3)),
           ((5, 2, 3, 2, 7, 2, 3, 4), (4, 2, 0, 6, 1, 7, 5, 3)), ((2, 3, 2, 3, 2, 3, 2, 3, 2, 3, 2, 3), (8, 1, 6, 3, 10, 5, 0, 7, 2, 9, 4, 11)),
           ((2, 3, 2, 2, 2, 3, 2, 2, 2, 2, 2, 2, 2, 2, 3), (14, 12, 10, 8, 6, 4, 2, 0, 13, 11, 9, 7, 5, 3, 1)), ((64, 1, 1025), (2, 1, 0)), ((6, 40009), (1, 0)), ((9, 8, 2311, 7), (1, 0, 3, 2))]


@pytest.mark.parametrize("es", [4, 8])
@pytest.mark.parametrize("method", [2, 3])
@pytest.mark.parametrize("elems", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("order", [None, 0, 1, 2])
def test_blocks_slabs_and_ranks(monkeypatch, es, method, elems, order):
    import cutt_amd as cutt
    from gpu_util import check_case
    if order is None:
        monkeypatch.setenv("CUTT_MAX_ITEMS", "1")
    else:  # (few rounds of workgroups: several blocks each)
        monkeypatch.setenv("CUTT_PACKED_ROUNDS", "1")
        monkeypatch.setenv("CUTT_ITEM_ORDER", str(order))
    monkeypatch.setenv("CUTT_ELEMS_PER_THREAD", str(elems))
    cutt.set_method_override(method)
    seen = 0
    try:
        for i, (dim, perm) in enumerate(TENSORS):
            monkeypatch.setenv("CUTT_CACHE_POLICY", str((i + elems) % 4))
            monkeypatch.setenv("CUTT_XCD_GROUP", str(3 * (i % 2)))
            rc, h = cutt.cuttPlan(len(dim), dim, perm, es, 0)
            if rc != cutt.CUTT_SUCCESS:  # (no block of this method fits)
                continue
            n = cutt.get_plan_info(h).numCandidates
            assert cutt.cuttDestroy(h) == cutt.CUTT_SUCCESS
            for c in range(0, n, max(1, n // 4)):
                info = check_case(dim, perm, es, how="candidate", candidate=c)
                assert info.method == method and (order is not None or info.itemsPerBlock == 1)
                seen += 1
    finally:
        cutt.set_method_override(0)
    assert seen >= 8
