"""Transposes as users of the library run them: plan once, execute many times on device buffers.

The callers are tensor-contraction codes (transpose, matrix product, transpose) and data-layout
changes: ranks 2 to 12, arbitrary extents, arbitrary permutations, 8-byte elements (double, complex
float) and 4-byte ones, from tensors of a million elements, where the call itself counts, to
tensors of 2e8 elements per buffer.  Three ways of calling it are in use: a plan from the cost model
(`plan`), a plan found by timing (`measure`) and one call that plans and executes without allocating
(`one_call`).
"""
import math

import torch

import cutt_amd as cutt

MIN_ELEMS, MAX_ELEMS = 1.0e6, 2.0e8


def listed():
    return [
        # The smallest calls: blocks of a contraction over small index ranges, launch and call overhead count.
        case("r4_small_f64", (24, 32, 36, 43), (3, 1, 2, 0), 8),
        # A small matrix off every alignment, 4-byte elements.
        case("r2_small_f32", (2011, 1163), (1, 0), 4),
        # Amplitude blocks of a contraction code: short ranks, 4e6 elements, both buffers inside the caches.
        case("r5_medium_f64", (24, 32, 16, 36, 9), (4, 1, 3, 2, 0), 8, "one_call"),
        # An ordinary layout change that keeps the leading rank, of 7e7 elements.
        case("r3_lead_f32", (1305, 599, 88), (0, 2, 1), 4),
        # An ordinary contraction tensor, 5e7 elements, leading rank moves to the end.
        case("r4_ttc_f64", (96, 75, 96, 75), (2, 1, 3, 0), 8),
        # The large square matrix, on every alignment.
        case("r2_square_f32", (8192, 8192), (1, 0), 4),
        # A large matrix with odd extents (rows start anywhere in a cache line).
        case("r2_ragged_f64", (23425, 8538), (1, 0), 8),
        # Batched transposes inside a large tensor; the largest case, and the headline benchmark.
        case("r4_batched_f64", (1024, 64, 1024, 3), (2, 1, 0, 3), 8),
        # Short odd leading ranks.
        case("r6_short_f32", (5, 7, 11, 13, 17, 1093), (4, 2, 0, 5, 1, 3), 4),
        # A very long leading rank beside a tiny one.
        case("r3_long_f64", (200000, 2, 500), (2, 1, 0), 8),
        # A large random tensor of odd extents, 4-byte elements, cost-model plan.
        case("r6_ragged_f32", (132, 11, 3, 47, 14, 2, 35), (2, 1, 3, 6, 5, 0, 4), 4),
        # A large random tensor in a program that runs one transpose many times and lets the planner time it.
        case("r5_measured_f32", (40, 14881, 4, 6, 14), (3, 2, 0, 1, 4), 4, "measure"),
    ]


def case(name, dim, perm, elem_bytes, how="plan"):
    d = {"rank": len(dim), "dim": ",".join(map(str, dim)), "perm": ",".join(map(str, perm)), "elem_bytes": elem_bytes,
         "how": how}
    return dict(d, name=name) if name else d


def draw(rng):
    """A random tensor: the volume spread over its logarithm, the extents random shares of it."""
    while True:
        target = math.exp(rng.uniform(math.log(MIN_ELEMS), math.log(MAX_ELEMS)))
        rank = rng.choice((2, 2, 3, 3, 4, 4, 5, 5, 6, 6, 7, 7, 8, 12))
        share = [rng.gammavariate(2.0, 1.0) for _ in range(rank)]
        dim = [max(2, round(math.exp(s / sum(share) * math.log(target)))) for s in share]
        big = dim.index(max(dim))
        dim[big] = max(2, round(target * dim[big] / math.prod(dim)))
        perm = list(range(rank))
        rng.shuffle(perm)
        if perm != sorted(perm) and MIN_ELEMS <= math.prod(dim) <= MAX_ELEMS:
            return case(None, dim, perm, rng.choice((4, 8)), rng.choice(("plan",) * 6 + ("measure", "one_call")))


def ints(text):
    return [int(x) for x in text.split(",")]


class Transpose:
    """What a program holds: the two buffers and, unless it makes one call of it all, the plan."""

    def __init__(self, case, seed):
        self.dim, self.perm = ints(case["dim"]), ints(case["perm"])
        self.elem_bytes = case["elem_bytes"]
        self.stream = torch.cuda.current_stream().cuda_stream
        dtype = torch.float64 if self.elem_bytes == 8 else torch.float32
        gen = torch.Generator(device="cuda").manual_seed(seed)
        self.idata = torch.randn(math.prod(self.dim), dtype=dtype, device="cuda", generator=gen)
        self.odata = torch.empty_like(self.idata)
        self.handle = None
        if case["how"] == "plan":
            rc, self.handle = cutt.cuttPlan(len(self.dim), self.dim, self.perm, self.elem_bytes, self.stream)
        elif case["how"] == "measure":
            rc, self.handle = cutt.cuttPlanMeasure(len(self.dim), self.dim, self.perm, self.elem_bytes, self.stream,
                                                   self.idata.data_ptr(), self.odata.data_ptr())
        else:
            rc = cutt.CUTT_SUCCESS
        check(rc)

    def run(self):
        if self.handle is None:
            check(cutt.cuttExecuteNoAlloc(len(self.dim), self.dim, self.perm, self.elem_bytes, self.stream,
                                          self.idata.data_ptr(), self.odata.data_ptr()))
        else:
            check(cutt.cuttExecute(self.handle, self.idata.data_ptr(), self.odata.data_ptr()))
        return self.odata

    def __del__(self):
        if getattr(self, "handle", None) is not None:
            torch.cuda.synchronize()
            cutt.cuttDestroy(self.handle)


def check(rc):
    if rc != cutt.CUTT_SUCCESS:
        raise RuntimeError("cutt returned %d" % rc)


def prepare(case, seed):
    return Transpose(case, seed)


def run(state):
    return state.run()


def work(case):
    # every element read once and written once
    return {"bytes": 2 * math.prod(ints(case["dim"])) * case["elem_bytes"], "flops": 0}


def tolerance(case):
    # elements are moved, not computed with
    return "exact"
