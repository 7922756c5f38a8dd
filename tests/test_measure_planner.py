"""What cuttPlanMeasure picks from timings that are known beforehand: on the CPU, with a simulated device clock
(measure_planner.cpp)."""
import os
import re
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(ROOT, "cutt_amd", "csrc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("measure") / "measure_planner")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-pthread", "-I" + os.path.join(ROOT, "include"), "-I" + CSRC,
                           os.path.join(HERE, "measure_planner.cpp")] +
                          [os.path.join(CSRC, n) for n in ("cutt_api.cpp", "plan.cpp", "model.cpp", "layer_math.cpp", "slab.cpp")] +
                          ["-o", exe])
    return exe


def measured(program, scenario):
    out = subprocess.check_output([program, scenario], text=True, timeout=120)
    m = re.search(r"method (\d+) measured ([\d.]+) policy (\d+) order (\d+) super (\d+)x(\d+) lines (\d+) grouped (\d+) launches (\d+)", out)
    assert m, out
    print(out)
    return dict(zip(("method", "us", "policy", "order", "superM", "superK", "lines", "grouped", "launches"),
                    (float(m.group(2)) if k == 2 else int(m.group(k)) for k in range(1, 10))))


METHOD_PACKED, METHOD_TILED = 2, 4


def test_first_launch_of_a_kernel_instance_does_not_decide(program):
    p = measured(program, "cold")
    assert p["method"] == METHOD_PACKED and p["us"] == 6.0


def test_line_aligned_plans_are_not_timed_again_with_rows_in_groups(program):
    # the switch changes nothing about them: whichever launch came later would win
    p = measured(program, "drift")
    assert p["lines"] == 1 and p["grouped"] == 0


@pytest.mark.parametrize("scenario,lines", [("plain", 0), ("lines", 1)])
def test_both_forms_of_a_tiled_plan_are_timed_as_the_planner_builds_them(program, scenario, lines):
    # ... also where a Packed plan is ahead of the form that the rules prefer
    p = measured(program, scenario)
    assert p["method"] == METHOD_TILED and p["lines"] == lines and p["us"] == 60.0


def test_row_gathering_takes_no_other_candidate_its_refinement(program):
    # the order of the Mbar ranks is refined for the three best candidates that have any
    out = subprocess.check_output([program, "predicted"], text=True, timeout=120)
    (with_us, gathered), (without_us, _) = [(float(a), int(b)) for a, b in re.findall(r"predicted ([\d.]+) gathered (\d)", out)]
    assert gathered == 0 and with_us == without_us, out


def test_rows_in_groups_go_with_loads_past_the_caches(program):
    out = subprocess.check_output([program, "accesses"], text=True, timeout=120)
    plans = [tuple(map(int, m)) for m in re.findall(r"accesses method (\d) policy (\d) grouped (\d)", out)]
    assert plans == [(METHOD_TILED, 0, 0)] * 2 + [(METHOD_TILED, 1, 1)] * 2, out


@pytest.mark.parametrize("scenario,launches", [("groups", 18), ("narrow", 6)])
def test_no_plan_is_timed_again_as_a_variant_of_itself(program, scenario, launches):
    # groups of workgroups for plans that have none: three timings of six launches, for itself and two orders of the Mbar ranks that are
    # the same here, not five; "64x64 instead of wide" for a winner that has 64x64 tiles: one timing, not two
    out = subprocess.check_output([program, scenario], text=True, timeout=120)
    assert int(re.search(r"most launches of one plan (\d+)", out).group(1)) == launches, out


@pytest.mark.parametrize("scenario,us", [("tie98", 98.0), ("tie99", 100.0)])
def test_the_heuristic_plan_wins_ties(program, scenario, us):
    # half a per cent is what two timings of one plan differ by, two per cent are not
    assert measured(program, scenario)["us"] == us


@pytest.mark.parametrize("scenario,own", [("bits", (0, 5)), ("nobits", (1, 0))])
def test_both_numberings_of_packed_work_items_are_timed(program, scenario, own):
    # by address bits in one chunk per XCD, and the default one in groups of workgroups, whichever cuttPlan takes
    p = measured(program, scenario)
    out = subprocess.check_output([program, scenario], text=True, timeout=120)
    assert tuple(map(int, re.search(r"own numbered (\d) group (\d)", out).groups())) == own
    assert p["us"] == 50.0
