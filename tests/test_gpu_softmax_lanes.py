"""Trees of a soft-max round grown side by side: the checker's trees, leaves and predictions for fewer classes
than streams, more, and more than the ring of tree records holds; with inspection switched on and off between rounds."""
import numpy as np
import pytest

from test_gpu_parity import make_data

pytestmark = pytest.mark.gpu


def _problem(n, F, K, seed):
    X, _ = make_data(n, F, 1, seed=seed)
    rng = np.random.default_rng(seed)
    labels = np.argmax(rng.gumbel(size=(n, K)) + 2 * np.nan_to_num(X[:, np.arange(K) % F]), axis=1).astype(np.uint8)
    labels[0] = K - 1
    return X, labels


@pytest.mark.parametrize("n,F,K,rounds,bins,depth", [(5000, 9, 2, 4, 64, 5), (3000, 40, 7, 3, 255, 4), (2000, 6, 70, 2, 16, 3),
                                                     (4000, 12, 3, 3, 300, 4), (1000, 5, 4, 2, 256, 1)])
def test_trees_of_a_round(oracle, n, F, K, rounds, bins, depth):
    import arboretum_amd as arb
    X, labels = _problem(n, F, K, seed=n)
    cfg = {"objective": 4, "method": 1, "internals": {"hist_size": bins, "double_precision": True},
           "tree": {"max_depth": depth, "eta": 0.3, "lambda": 1.0, "labels_count": K}}
    ob = oracle.Booster(X, labels=labels, config=cfg)
    data = arb.DMatrix(X, labels=labels)
    g = arb.Garden(cfg, data)
    g.labels_count = K
    for r in range(rounds):
        if r == 1:
            g.set_inspect(True)
        elif r == 2:
            g.set_inspect(False)
        ob.grow(1)
        g.grow_tree()
        for t in range(r * K, (r + 1) * K):
            to, tg = ob.tree(t), g.tree(t)
            for key in ("fid", "quantized", "gain", "weights"):
                assert np.array_equal(to[key], tg[key], equal_nan=True), (key, t)
        assert np.array_equal(ob.leaf(), g.leaves())
        assert np.array_equal(ob.yhat(), g.train_yhat())


def test_a_round_that_fails_leaves_the_booster_usable(oracle):
    # an error that another user of the runtime left in this thread is found by the check behind the first
    # tree's kernels, which belong to another stream's state: that tree goes, and the next round grows the
    # trees it would have grown
    import hipmem
    import arboretum_amd as arb
    X, labels = _problem(4000, 9, 3, seed=11)
    cfg = {"objective": 4, "method": 1, "internals": {"hist_size": 64, "double_precision": True},
           "tree": {"max_depth": 5, "eta": 0.3, "lambda": 1.0, "labels_count": 3}}
    ob = oracle.Booster(X, labels=labels, config=cfg)
    data = arb.DMatrix(X, labels=labels)
    g = arb.Garden(cfg, data)
    g.labels_count = 3
    g.grow_tree()
    assert hipmem.hip().hipSetDevice(99) != 0
    with pytest.raises(arb.ArboretumError):
        g.grow_tree()
    assert g.num_trees() == 3
    for _ in range(2):
        g.grow_tree()
    ob.grow(3)
    assert g.num_trees() == 9
    for t in range(9):
        to, tg = ob.tree(t), g.tree(t)
        for key in ("fid", "quantized", "gain", "weights"):
            assert np.array_equal(to[key], tg[key], equal_nan=True), (key, t)
    assert np.array_equal(ob.leaf(), g.leaves())
    assert np.array_equal(ob.yhat(), g.train_yhat())
