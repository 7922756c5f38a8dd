"""Index tables built on the device for cuttExecuteNoAlloc, against the oracle: lists of few, of up to eight and of more ranks, with
the Packed method and, on a tensor that has such a plan, with PackedSplit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SPLIT = (20000, 2, 50)


@pytest.mark.parametrize("es", [4, 8])
@pytest.mark.parametrize("dim,perm", [
    (SPLIT, (2, 1, 0)), ((5, 7, 11, 13, 3), (4, 2, 0, 3, 1)), ((3, 2, 5, 4, 3, 2, 7, 5), (7, 5, 3, 1, 6, 4, 2, 0)),
    ((2, 3, 2, 3, 2, 3, 2, 3, 2, 3), (9, 7, 5, 3, 1, 8, 6, 4, 2, 0)),
    ((2, 2, 3, 2, 2, 3, 2, 2, 2, 3, 2, 2), (11, 9, 7, 5, 3, 1, 10, 8, 6, 4, 2, 0)),
])
def test_tables_built_on_the_device(dim, perm, es):
    import torch
    import cutt_amd as cutt
    import gpu_util
    import oracle
    data = gpu_util.seeded(int(np.prod(dim)), es, seed=len(dim))
    d_in = gpu_util.to_device(data)
    expect = oracle.transpose(list(dim), list(perm), data)
    try:
        for method in (cutt.METHOD_PACKED, cutt.METHOD_PACKEDSPLIT):
            if (method == cutt.METHOD_PACKEDSPLIT) != (dim == SPLIT):
                continue
            cutt.set_method_override(method)
            d_out = torch.full_like(d_in, -1)
            rc = cutt.cuttExecuteNoAlloc(len(dim), list(dim), list(perm), es, gpu_util.stream_handle(), d_in.data_ptr(), d_out.data_ptr())
            torch.cuda.synchronize()
            assert rc == cutt.CUTT_SUCCESS and np.array_equal(gpu_util.to_host(d_out, es), expect), (dim, perm, es, method)
    finally:
        cutt.set_method_override(0)


@pytest.mark.parametrize("es,dim,perm", [
    (4, (331, 2, 270), (2, 1, 0)),                                   # two slab classes, lists of up to four ranks
    (8, (5, 4, 4097), (1, 0, 2)),                                    # two classes of a stretch of a batch
    (4, (6, 613, 252), (0, 2, 1)),                                   # four classes of different sizes
    (8, (2, 3, 2, 2, 5, 2, 7, 2, 301), (8, 6, 4, 2, 0, 1, 7, 5, 3)),   # two, up to eight ranks
    (4, (2, 2, 2, 5, 2, 2, 2, 2, 11, 2, 2, 2, 13, 2, 2), (6, 10, 2, 1, 12, 11, 3, 0, 14, 4, 7, 13, 9, 5, 8)),   # two, up to twelve
])
def test_the_tables_of_several_slab_classes(es, dim, perm):
    import torch
    import cutt_amd as cutt
    import gpu_util
    import oracle
    data = gpu_util.seeded(int(np.prod(dim)), es, seed=len(dim))
    d_in = gpu_util.to_device(data)
    expect = oracle.transpose(list(dim), list(perm), data)
    try:
        cutt.set_method_override(cutt.METHOD_PACKEDSPLIT)
        for call in range(3):  # (the tables of the call before are in the scratch memory)
            d_out = torch.full_like(d_in, -1)
            rc = cutt.cuttExecuteNoAlloc(len(dim), list(dim), list(perm), es, gpu_util.stream_handle(), d_in.data_ptr(), d_out.data_ptr())
            torch.cuda.synchronize()
            assert rc == cutt.CUTT_SUCCESS and np.array_equal(gpu_util.to_host(d_out, es), expect), (dim, perm, es, call)
    finally:
        cutt.set_method_override(0)
