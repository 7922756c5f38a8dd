"""Tiles of 128x128 4-byte elements (CUTT_TILED_WIDE), bit-exact against the oracle: one tile and several on either axis, strips with a
narrower last one, one to eight Mbar ranks, every cache policy; axes that are no multiple of 128 and 8-byte elements keep the 64x64
tiles."""
import pytest

pytestmark = pytest.mark.gpu

CASES = [((128, 128), (1, 0)), ((128, 1408), (1, 0)), ((1408, 128), (1, 0)), ((2304, 640), (1, 0)), ((256, 3, 384), (2, 1, 0)), ((384, 256, 5), (1, 0, 2)),
         ((128, 2, 3, 2, 128, 3, 2, 2), (4, 3, 1, 0, 6, 2, 5, 7)), ((256, 2, 2, 3, 2, 2, 128, 2, 2, 2), (6, 4, 2, 9, 0, 7, 1, 3, 8, 5))]


@pytest.fixture
def tiled(monkeypatch):
    import torch  # noqa: F401  (before the library is loaded: both must share one HIP runtime)
    import cutt_amd as cutt
    cutt.set_method_override(cutt.METHOD_TILED)
    monkeypatch.setenv("CUTT_TILED_WIDE", "1")
    yield monkeypatch
    cutt.set_method_override(0)


@pytest.mark.parametrize("group", [0, 1, 5])
@pytest.mark.parametrize("order", [1, 2, 3, 5])
def test_wide_tiles(tiled, order, group):
    from gpu_util import check_case
    tiled.setenv("CUTT_TILED_ORDER", str(order))
    tiled.setenv("CUTT_XCD_GROUP", str(group))
    wide = 0
    for i, (dim, perm) in enumerate(CASES):
        tiled.setenv("CUTT_CACHE_POLICY", str((i + order) % 4))
        info = check_case(dim, perm, 4)
        assert info.method_name == "Tiled"
        wide += info.numThreads == 1024
    assert wide >= 6


@pytest.mark.parametrize("dim,perm,es", [((128, 192), (1, 0), 4), ((192, 128), (1, 0), 4), ((128, 130), (1, 0), 4), ((128, 256), (1, 0), 8), ((16, 8, 128), (2, 1, 0), 4)])
def test_other_axes_keep_the_small_tiles(tiled, dim, perm, es):
    from gpu_util import check_case
    assert check_case(dim, perm, es).numThreads == 256


def test_planner_takes_them_beyond_the_cache_only(tiled):
    import torch
    import cutt_amd as cutt
    tiled.delenv("CUTT_TILED_WIDE")
    for n, threads in [(4096, 256), (8192, 1024)]:
        src = torch.arange(n * n, device="cuda", dtype=torch.int32)
        for how in ("plan", "measure"):
            dst = torch.full_like(src, -1)
            st = torch.cuda.current_stream().cuda_stream
            if how == "plan":
                rc, h = cutt.cuttPlan(2, [n, n], [1, 0], 4, st)
                assert rc == cutt.CUTT_SUCCESS and cutt.get_plan_info(h).numThreads == threads
            else:
                rc, h = cutt.cuttPlanMeasure(2, [n, n], [1, 0], 4, st, src.data_ptr(), dst.data_ptr())
                assert rc == cutt.CUTT_SUCCESS
            dst.fill_(-1)
            assert cutt.cuttExecute(h, src.data_ptr(), dst.data_ptr()) == cutt.CUTT_SUCCESS
            torch.cuda.synchronize()
            assert torch.equal(dst, src.view(n, n).t().contiguous().view(-1))
            cutt.cuttDestroy(h)
