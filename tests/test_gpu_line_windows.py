"""Line-aligned stores of the Tiled kernel (CUTT_TILED_ALIGNED): every row of a tile stores the window of its output
run that starts on a 128-byte line.  Bit-exact against a permute on the device at the edges of the tile widths, with axes over
fused ranks, runs around one window long, buffers off the line grid, and on tensors where the planner takes it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def transpose_on_device(x, dim, perm):
    # (the oracle takes seconds for 1e8 elements; tests/test_oracle.py compares it with numpy's transpose)
    r = len(dim)
    return x.view(tuple(reversed(dim))).permute([r - 1 - perm[r - 1 - k] for k in range(r)]).contiguous().view(-1)


def run(dim, perm, es, shift_in=0, shift_out=0, candidate=None):
    import torch
    import cutt_amd as cutt
    vol = int(np.prod(dim, dtype=np.int64))
    dt = torch.int64 if es == 8 else torch.int32
    src = torch.arange(vol + shift_in, device="cuda", dtype=dt)[shift_in:]
    big = torch.full((vol + shift_out + 64,), -1, dtype=dt, device="cuda")
    dst = big[shift_out:shift_out + vol]
    st = torch.cuda.current_stream().cuda_stream
    if candidate is None:
        rc, h = cutt.cuttPlan(len(dim), list(dim), list(perm), es, st)
    else:
        rc, h = cutt.cuttPlanFromCandidate(len(dim), list(dim), list(perm), es, st, candidate)
    assert rc == cutt.CUTT_SUCCESS
    info = cutt.get_plan_info(h)
    print("%s %s es=%d %s aligned %d policy %d" % (dim, perm, es, info.method_name, info.tiledAligned, info.cachePolicy), flush=True)
    assert cutt.cuttExecute(h, src.data_ptr(), dst.data_ptr()) == cutt.CUTT_SUCCESS
    torch.cuda.synchronize()
    assert cutt.cuttDestroy(h) == cutt.CUTT_SUCCESS
    assert torch.equal(dst, transpose_on_device(src, dim, perm))
    assert bool((big[:shift_out] == -1).all()) and bool((big[shift_out + vol:] == -1).all())
    return info


WIDTHS = [1, 2, 33, 63, 64, 65, 67, 68, 69, 75, 96, 128, 132, 136, 137, 200, 639, 641, 1024, 1300]
RUNS = [1, 31, 33, 63, 64, 65, 97, 191]


@pytest.mark.parametrize("es", [4, 8])
@pytest.mark.parametrize("policy", [0, 2, 3])
def test_widths_and_run_lengths(monkeypatch, es, policy):
    import torch  # noqa: F401  (before the library is loaded: both must share one HIP runtime)
    import cutt_amd as cutt
    monkeypatch.setenv("CUTT_TILED_ALIGNED", "1")
    monkeypatch.setenv("CUTT_CACHE_POLICY", str(policy))
    cutt.set_method_override(cutt.METHOD_TILED)
    try:
        for i, m in enumerate(WIDTHS):
            for j, k in enumerate(RUNS):
                dim, perm = [((m, k), (1, 0)), ((m, 3, k), (2, 1, 0)), ((m, k, 5), (1, 0, 2))][(i + j) % 3]
                if all(d > 1 for d in dim):
                    info = run(dim, perm, es, shift_out=(5 * i + j) % 33, shift_in=(i + j) % 3)
                    assert info.method_name == "Tiled" and info.tiledAligned == 1
    finally:
        cutt.set_method_override(0)


@pytest.mark.parametrize("es", [4, 8])
def test_axes_over_fused_ranks(monkeypatch, es):
    import torch  # noqa: F401  (before the library is loaded: both must share one HIP runtime)
    import cutt_amd as cutt
    monkeypatch.setenv("CUTT_TILED_ALIGNED", "1")
    cutt.set_method_override(cutt.METHOD_TILED)
    fused = 0
    try:
        for dim, perm in [((7, 9, 5, 11, 13), (3, 4, 0, 2, 1)), ((6, 5, 3, 40, 9), (3, 2, 4, 1, 0)), ((12, 11, 67, 3), (2, 3, 1, 0)),
                          ((132, 11, 3, 47), (2, 1, 3, 0)), ((3, 50, 7, 2, 33), (4, 2, 3, 0, 1)), ((16, 8, 64, 32), (2, 3, 0, 1))]:
            for i in range(run(dim, perm, es, shift_out=3).numCandidates):
                info = run(dim, perm, es, shift_out=i % 5, candidate=i)
                assert info.tiledAligned == 1
                fused += (info.numMm > 1) + 2 * (info.numMk > 1) == 3
    finally:
        cutt.set_method_override(0)
    assert fused >= 2  # both axes fused


@pytest.mark.parametrize("dim,perm,es,aligned", [
    ((1201, 30011), (1, 0), 4, 1), ((1201, 30011), (1, 0), 8, 1), ((777, 51, 905), (2, 1, 0), 4, 1), ((8192, 5003), (1, 0), 4, 1),
    ((50, 7, 13, 6007), (3, 1, 2, 0), 8, 1), ((132, 11, 3, 47, 14, 2, 9), (2, 1, 3, 6, 5, 0, 4), 4, 1),
    ((1201, 3001), (1, 0), 8, 0),       # fits the memory-side cache
    ((96000, 407), (1, 0), 4, 0),       # runs of 1.6 KB
    ((1216, 30016), (1, 0), 4, 0),      # rows on the line grid
])
def test_planner_takes_it_for_long_rows_off_the_line_grid(dim, perm, es, aligned):
    import torch
    import cutt_amd as cutt
    info = run(dim, perm, es, shift_out=1)
    assert (info.method_name == "Tiled" and info.tiledAligned == 1) == bool(aligned)
    if aligned:
        rc, h = cutt.cuttPlan(len(dim), list(dim), list(perm), es, torch.cuda.current_stream().cuda_stream)
        assert rc == cutt.CUTT_SUCCESS
        dev, mod = cutt.count_address_stream(h, 0)
        d, m = dev.as_dict(), mod.as_dict()
        cutt.cuttDestroy(h)
        for k in ("rdInstr", "wrInstr", "rdLines", "wrLines", "rdSectors", "wrSectors", "wrPartialLines"):
            assert d[k] == m[k], (k, d[k], m[k])
