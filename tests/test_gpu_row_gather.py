"""Tensors whose leading rank stays: the kernel that writes the output front to back, block by block
from one 128-byte line to another (kernels.hip: rowGatherKernel), against the CPU oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# rows of 64 bytes (the shortest it takes), just below / at / above a block of 1024 elements, rows longer
# than several blocks; tensors smaller than a block, ending on and off a block boundary; up to six ranks
CASES = [((16, 3, 2), (0, 2, 1)), ((17, 5, 7), (0, 2, 1)), ((31, 4, 8, 3), (0, 3, 2, 1)), ((1023, 3, 5), (0, 2, 1)),
         ((1024, 4, 3), (0, 2, 1)), ((1025, 3, 4), (0, 2, 1)), ((5000, 2, 3), (0, 2, 1)), ((32, 8, 4), (0, 2, 1)),
         ((19, 3, 2, 5, 4, 7), (0, 5, 2, 4, 1, 3)), ((40, 300, 400), (0, 2, 1)), ((333, 150, 200), (0, 2, 1)),
         # enough blocks for groups per XCD
         ((333, 160, 180), (0, 2, 1)), ((18, 60, 5, 41, 43), (0, 2, 4, 1, 3))]


@pytest.mark.parametrize("es", [4, 8])
def test_row_gather_against_the_oracle(es):
    import torch
    import cutt_amd as cutt
    import gpu_util as gpu
    import oracle
    st = gpu.stream_handle()
    groups = set()
    for dim, perm in CASES:
        vol = int(np.prod(dim))
        data = gpu.seeded(vol, es, seed=vol % 997)
        want = torch.from_numpy(oracle.transpose_mt(list(dim), list(perm), data, 8).view(np.int32 if es == 4 else np.int64))
        with cutt.Candidates(list(dim), list(perm), es) as c:
            index = [i for i in range(len(c)) if c.info(i).rowGather]
        assert len(index) == 1, (dim, es)
        rc, h = cutt.cuttPlanFromCandidate(len(dim), list(dim), list(perm), es, st, index[0])
        assert rc == cutt.CUTT_SUCCESS
        info = cutt.get_plan_info(h)
        assert info.rowGather == 1, (dim, es)
        groups.add(info.numBlocks % 512 == 0)
        # the buffers' first elements at several places of a line, the elements around the output untouched
        for shift_in, shift_out in ((0, 0), (1, 0), (3, 1), (0, 128 // es - 1), (5, 128 // es // 2 + 1)):
            print("dim=%s perm=%s es=%d shifts=%d,%d" % (dim, perm, es, shift_in, shift_out), flush=True)
            a = torch.full((vol + 64,), -7, dtype=want.dtype, device="cuda")
            b = torch.full((vol + 64,), -1, dtype=want.dtype, device="cuda")
            src, dst = a[shift_in:shift_in + vol], b[shift_out:shift_out + vol]
            src.copy_(gpu.to_device(data))
            assert cutt.cuttExecute(h, src.data_ptr(), dst.data_ptr()) == cutt.CUTT_SUCCESS
            torch.cuda.synchronize()
            assert torch.equal(dst.cpu(), want), (dim, perm, es, shift_in, shift_out)
            assert bool((b[:shift_out] == -1).all()) and bool((b[shift_out + vol:] == -1).all())
        assert cutt.cuttDestroy(h) == cutt.CUTT_SUCCESS
    assert groups == {False, True}
