"""cuttPlan without a GPU: the library's planner linked against the stand-in HIP layer (fake_hip_layer.cpp), for tests that look at what a
finished plan is - the candidates of cuttCandidatesCreate stop before tile forms, cache policy and XCD groups are decided."""
import contextlib
import ctypes
import os
import subprocess

from cutt_amd import api

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "cutt_amd", "csrc")


def build(directory):
    path = os.path.join(str(directory), "libplanner.so")
    subprocess.check_call(["g++", "-O1", "-shared", "-fPIC", "-std=c++17", "-pthread", "-I" + os.path.join(os.path.dirname(HERE), "include"), "-I" + CSRC,
                           os.path.join(HERE, "fake_hip_layer.cpp")] +
                          [os.path.join(CSRC, n) for n in ("cutt_api.cpp", "plan.cpp", "model.cpp", "layer_math.cpp", "slab.cpp")] + ["-o", path])
    return Planner(path)


class Planner:
    def __init__(self, path):
        self.lib = ctypes.CDLL(path)
        self.lib.cuttPlan.argtypes = [ctypes.POINTER(ctypes.c_uint), ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p]

    def plan(self, dim, perm, elem_size, method=0, **env):
        """PlanInfo of cuttPlan with the given environment variables."""
        ints = lambda v: (ctypes.c_int * len(v))(*v)
        handle = ctypes.c_uint()
        info = api.PlanInfo()
        with environment(**env):
            self.lib.cuttSetMethodOverride(method)
            assert self.lib.cuttPlan(ctypes.byref(handle), len(dim), ints(dim), ints(perm), elem_size, None) == 0, (dim, perm, elem_size)
        assert self.lib.cuttGetPlanInfo(handle, ctypes.byref(info)) == 0
        assert self.lib.cuttDestroy(handle) == 0
        return info


@contextlib.contextmanager
def environment(**env):
    # (the C library's environment: what the planner reads)
    saved = {k: os.environ.get(k) for k in env}
    os.environ.update({k: str(v) for k, v in env.items()})
    try:
        yield
    finally:
        for k, v in saved.items():
            os.environ.pop(k) if v is None else os.environ.__setitem__(k, v)
