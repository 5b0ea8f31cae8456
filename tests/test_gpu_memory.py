"""Device memory that boosters hold and leave behind."""
import gc

import numpy as np
import pytest

from hipmem import free_device_bytes
from test_gpu_parity import make_data

pytestmark = pytest.mark.gpu
MB = 1 << 20


@pytest.fixture(scope="module")
def arb():
    import arboretum_amd
    if arboretum_amd.device_count() < 1:
        pytest.fail("no HIP device")
    return arboretum_amd


def _config(depth, bins=64, **tree):
    return {"objective": 1, "method": 1, "internals": {"hist_size": bins, "double_precision": True},
            "tree": dict({"max_depth": depth, "eta": 0.3, "lambda": 1.0}, **tree)}


def test_release_memory(arb):
    X, y = make_data(600000, 28, 1, seed=4)
    def use():
        data = arb.DMatrix(X, y=y)
        g = arb.train(_config(5), data, 2)
        return g.predict(data)
    first = use()                        # (code objects and the runtime's own memory)
    gc.collect()
    arb.release_memory()
    before = free_device_bytes()
    data = arb.DMatrix(X, y=y)
    g = arb.train(_config(5), data, 2)
    assert free_device_bytes() < before - 100 * MB
    arb.release_memory()                 # takes nothing that is in use
    assert np.array_equal(g.predict(data), first)
    del g, data
    gc.collect()
    assert free_device_bytes() < before - 100 * MB
    arb.release_memory()
    assert free_device_bytes() > before - 16 * MB
    assert np.array_equal(use(), first)
