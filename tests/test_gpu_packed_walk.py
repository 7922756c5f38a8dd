"""The packed kernels whose arguments are decoded as a walk, bit-exact against the oracle: one block per workgroup and several, every number of elements per
lane and cache policy, blocks whose last lanes have no element of their own, no Mbar rank up to the thirteenth (which the general kernel takes); loops over slabs of
two sizes, in which a workgroup's slab class changes, in every item order, in chunks and groups; stretches of a batch."""
import functools

import pytest

pytestmark = pytest.mark.gpu

TENSORS = [((3, 5, 7), (2, 1, 0)), ((16, 4, 33), (2, 0, 1)), ((7, 67, 5, 61), (3, 0, 2, 1)), ((31, 3, 37, 5, 6), (2, 0, 4, 1, 3)),
           ((5, 2, 3, 2, 7, 2, 3, 4), (4, 2, 0, 6, 1, 7, 5, 3)), ((2, 3, 2, 3, 2, 3, 2, 3, 2, 3, 2, 3), (8, 1, 6, 3, 10, 5, 0, 7, 2, 9, 4, 11)),
           ((2, 3, 2, 2, 2, 3, 2, 2, 2, 2, 2, 2, 2, 2, 3), (14, 12, 10, 8, 6, 4, 2, 0, 13, 11, 9, 7, 5, 3, 1)), ((64, 2, 1025), (2, 1, 0)), ((6, 40009), (1, 0)), ((9, 8, 2311, 7), (1, 0, 3, 2)),
           ((5, 4, 4097), (1, 0, 2)), ((2, 2, 9001), (1, 0, 2))]
METHOD_PACKED, METHOD_PACKEDSPLIT = 2, 3


@pytest.mark.parametrize("es", [4, 8])
@pytest.mark.parametrize("method", [METHOD_PACKED, METHOD_PACKEDSPLIT])
@pytest.mark.parametrize("elems", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("order", [None, 0, 1, 2])
def test_blocks_slabs_and_ranks(monkeypatch, es, method, elems, order):
    import cutt_amd as cutt
    from gpu_util import check_case
    if order is None:
        monkeypatch.setenv("CUTT_MAX_ITEMS", "1")
    else:  # (few rounds of workgroups: several blocks each, where there are that many)
        monkeypatch.setenv("CUTT_PACKED_ROUNDS", "1")
        monkeypatch.setenv("CUTT_ITEM_ORDER", str(order))
    monkeypatch.setenv("CUTT_ELEMS_PER_THREAD", str(elems))
    cutt.set_method_override(method)
    seen = refused = stretches = 0
    try:
        for i, (dim, perm) in enumerate(TENSORS):
            monkeypatch.setenv("CUTT_CACHE_POLICY", str((i + elems) % 4))
            rc, h = cutt.cuttPlan(len(dim), dim, perm, es, 0)
            if rc != cutt.CUTT_SUCCESS:
                assert rc == cutt.CUTT_INTERNAL_ERROR  # (no block of this method fits)
                refused += 1
                continue
            n = cutt.get_plan_info(h).numCandidates
            assert cutt.cuttDestroy(h) == cutt.CUTT_SUCCESS
            for c in range(0, n, 1 if perm[-1] == len(perm) - 1 else max(1, n // 4)):
                info = check_case(dim, perm, es, how="candidate", candidate=c)
                assert info.method == method and (order is not None or info.itemsPerBlock == 1)
                seen += 1
                stretches += info.numMm == info.rank
    finally:
        cutt.set_method_override(0)
    assert seen >= 8 and refused <= len(TENSORS) - 6 and (stretches >= 4 if method == METHOD_PACKEDSPLIT else not stretches)


# Tensors whose PackedSplit plans loop over slabs of two sizes: on two cut ranks, on one or two beside many Mbar positions, stretches of a batch.
# (The last has no Mbar position for a workgroup to walk, which is order 1.)
LOOPS = [(dim, perm, order) for dim, perm, orders in (((331, 7, 1999), (2, 1, 0), (0, 1, 2)), ((37, 2, 41, 3, 29, 2, 17), (4, 2, 6, 0, 1, 5, 3), (0, 1, 2)), ((5, 4, 300007), (1, 0, 2), (0, 2)))
         for order in orders]


@functools.lru_cache(maxsize=None)
def transposed(dim, perm, es):
    import gpu_util
    import numpy as np
    import oracle
    data = gpu_util.seeded(int(np.prod(dim)), es, seed=es)
    return data, oracle.transpose_mt(list(dim), list(perm), data, 8)


@pytest.mark.parametrize("dim,perm,order", LOOPS)
@pytest.mark.parametrize("es,elems", [(4, 4), (4, 8), (4, 16), (8, 4), (8, 8)])
@pytest.mark.parametrize("group", [0, 3])
def test_loops_over_slabs_of_two_sizes(monkeypatch, dim, perm, es, elems, order, group):
    import cutt_amd as cutt
    from gpu_util import check_case
    for name, value in (("PACKED_ROUNDS", 1), ("ITEM_ORDER", order), ("ELEMS_PER_THREAD", elems), ("XCD_GROUP", group), ("CACHE_POLICY", (elems + order) % 4)):
        monkeypatch.setenv("CUTT_" + name, str(value))
    data, expect = transposed(dim, perm, es)
    cutt.set_method_override(METHOD_PACKEDSPLIT)
    try:
        info = check_case(dim, perm, es, data=data, expect=expect)
    finally:
        cutt.set_method_override(0)
    assert (info.method, info.itemOrder, info.xcdGroup) == (METHOD_PACKEDSPLIT, order, group) and info.itemsPerBlock > 1 and info.elemsPerThread >= 4
    # slabs of two sizes; in orders 0 and 2 a workgroup takes several of them one after the other
    assert info.splitDim % info.numSplit or (info.numSplit2 > 1 and info.splitDim2 % info.numSplit2)
    assert (info.numMm == info.rank) == (perm[-1] == len(perm) - 1)
