"""Which places of a list the exact method computes gains at (csrc/exact_filter.h), compiled for the host."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("exact") / "check_exact_filter")
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-o", out,
                           os.path.join(HERE, "native", "check_exact_filter.cpp")])
    return out


def run(program, *args):
    return [int(x) for x in subprocess.check_output([program, *map(str, args)], timeout=100).split()]


# ordinary sums, sums of 160 magnitudes, tiny hessians, denominators about 2^63
@pytest.mark.parametrize("kind", [0, 1, 2, 3])
def test_no_place_that_counts_is_left_out(program, kind):
    nodes, wrong, places, looked, pruned = run(program, kind, 20000)
    assert nodes == 80000 and wrong == 0
    if kind == 0:
        assert looked < places / 2      # (a filter, and not all places)
    assert pruned == nodes if kind in (0, 2) else 0 < pruned < nodes


def test_the_margin_is_needed(program):
    # without it the check finds nodes whose best place is left out
    assert run(program, 0, 20000, 0.0)[1] > 0
