"""Levels of many nodes, whose slabs are added up and scanned by one kernel: every layout of the slabs (fused pass, ids of 256,
rows in place in one histogram of few bins and in groups), one, two and four bins per lane, empty nodes; with the histograms of
every level against the checker's."""
import numpy as np
import pytest

from test_gpu_parity import assert_same_training, make_data
from test_gpu_fused_sizes import _same

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def arb():
    import arboretum_amd
    return arboretum_amd


@pytest.mark.parametrize("n,F,objective,bins,depth,nan_frac", [
    (3000, 5, 1, 255, 8, 0.3), (40000, 17, 0, 64, 7, 0.0), (20000, 29, 1, 256, 8, 0.1), (500, 3, 0, 100, 9, 0.1),
    (9000, 50, 1, 255, 7, 0.0), (6000, 40, 0, 256, 8, 0.1), (30000, 130, 0, 64, 8, 0.3), (7000, 210, 0, 32, 6, 0.0),
    (12000, 36, 1, 255, 8, 0.0)])
@pytest.mark.parametrize("double_precision", [True, False])
def test_deep_trees(arb, oracle, n, F, objective, bins, depth, nan_frac, double_precision):
    X, y = make_data(n, F, objective, seed=n + F, nan_frac=nan_frac)
    cfg = {"objective": objective, "method": 1, "internals": {"hist_size": bins, "double_precision": double_precision},
           "tree": {"max_depth": depth, "eta": 0.3, "lambda": 1.0, "min_child_weight": 0.5}}
    _same(arb, oracle, X, y, cfg, 2)


@pytest.mark.parametrize("F,objective,bins,nan_frac", [(5, 1, 256, 0.2), (20, 0, 64, 0.1), (70, 0, 60, 0.1), (50, 1, 255, 0.0)])
def test_histograms_of_deep_levels(arb, oracle, F, objective, bins, nan_frac):
    X, y = make_data(3000, F, objective, seed=F, nan_frac=nan_frac)
    cfg = {"objective": objective, "method": 1, "internals": {"hist_size": bins, "double_precision": True},
           "tree": {"max_depth": 7, "eta": 0.3, "lambda": 1.0, "min_child_weight": 0.5}}
    assert_same_training(arb, oracle, X, y, cfg, 2)
