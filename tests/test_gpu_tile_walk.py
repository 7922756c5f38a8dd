"""The Tiled kernel at the edges of its 64x64 tiles and strips, bit-exact against the oracle: every number of rows and columns in
the last tile that takes another piece of code, strips with a narrower last one, one to nine Mbar ranks, axes over fused ranks, and tile
orders 0 to 6 with every cache policy, through the kernel of the walk and through the general one."""
import math

import pytest

pytestmark = pytest.mark.gpu

EDGES = [2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 80, 113, 128]


@pytest.fixture
def tiled(monkeypatch):
    import torch  # noqa: F401  (before the library is loaded: both must share one HIP runtime)
    import cutt_amd as cutt
    cutt.set_method_override(cutt.METHOD_TILED)
    yield monkeypatch
    cutt.set_method_override(0)


@pytest.mark.parametrize("es", [4, 8])
def test_rows_and_columns_of_the_last_tile(tiled, es):
    from gpu_util import check_case
    for i, m in enumerate(EDGES):
        for j, k in enumerate(EDGES):
            tiled.setenv("CUTT_CACHE_POLICY", str((i + j) % 4))
            dim, perm = [((m, k), (1, 0)), ((m, 3, k), (2, 1, 0)), ((m, k, 5), (1, 0, 2))][(i + 2 * j) % 3]
            assert check_case(dim, perm, es).method_name == "Tiled"


@pytest.mark.parametrize("es", [4, 8])
@pytest.mark.parametrize("order", [0, 1, 2, 3, 5, 6])
def test_strips_and_mbar_ranks(tiled, es, order):
    from gpu_util import check_case
    tiled.setenv("CUTT_TILED_ORDER", str(order))
    for dim, perm in [((600, 530), (1, 0)), ((577, 130, 3), (1, 0, 2)), ((1100, 2, 70, 3), (2, 1, 0, 3)), ((5, 3, 30, 7, 4, 33), (3, 5, 1, 0, 4, 2)),
                      ((66, 2, 3, 2, 65, 3, 2), (4, 3, 1, 0, 6, 2, 5)), ((65, 2, 2, 3, 2, 2, 64, 2, 2, 2, 2), (6, 4, 2, 9, 0, 7, 1, 10, 3, 8, 5))]:
        for c in range(min(4, check_case(dim, perm, es).numCandidates)):
            info = check_case(dim, perm, es, how="candidate", candidate=c)
            assert info.method_name == "Tiled" and math.prod(dim) == info.volMmk * info.volMbar


@pytest.mark.parametrize("es", [4, 8])
@pytest.mark.parametrize("order", range(7))
def test_edges_in_every_order_policy_and_kernel(tiled, es, order):
    from gpu_util import check_case
    tiled.setenv("CUTT_TILED_ORDER", str(order))
    for i, m in enumerate(EDGES):
        for j, k in enumerate(EDGES):
            policy, paced = (i + 2 * j) % 4, (i // 4 + j) % 2
            tiled.setenv("CUTT_CACHE_POLICY", str(policy))
            tiled.setenv("CUTT_TILED_PACED", str(paced))
            tiled.setenv("CUTT_TILED_GROUPED", str(int(i == j)))
            dim, perm = [((m, k), (1, 0)), ((m, 3, k), (2, 1, 0)), ((m, 2, k, 3), (3, 2, 0, 1))][(i + j) % 3]
            info = check_case(dim, perm, es)
            assert info.method_name == "Tiled" and (info.tiledOrder, info.cachePolicy, info.tiledPaced) == (order, policy, paced)
