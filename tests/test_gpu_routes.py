"""Branches of the split search and of the predictions that ordinary tables do not reach, against
the CPU restatement and numpy."""
import numpy as np
import pytest

import catboost_rs_amd as cb
from oracle import oracle as O
from tests.trees import same_partition

pytestmark = pytest.mark.gpu


def _close(a, b, rel=1e-9):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    assert np.abs(a - b).max() <= rel * max(np.abs(b).max(), 1e-300)


@pytest.mark.parametrize("n_float,loss,score", [(3, "RMSE", "Cosine"), (62, "RMSE", "L2"), (130, "RMSE", "Cosine"),
                                                (3, "MultiClass", "Cosine"), (130, "MultiClass", "L2")])
def test_wide_one_hot_columns_match_oracle(n_float, loss, score):
    """One-hot columns of 65, 128, 129 and 200 values: their scoring windows of 64, 128 and 256 bins (by the
    table's features) start past bin 0, where a bin's own rows are the difference to the bin before
    the window, and end inside a slice.  The target makes the first and last bins of windows win."""
    g = np.random.default_rng(n_float + len(loss))
    n, cards = 6_000, [65, 128, 129, 200]
    bins = np.stack([g.integers(0, 20, n) for _ in range(n_float)] + [g.integers(0, c, n) for c in cards]).astype(np.uint8)
    one_hot = np.array([0] * n_float + [1] * 4, np.uint8)
    nb = np.array([19] * n_float + [c - 1 for c in cards], np.uint32)     # oracle convention
    c65, c128, c129, c200 = bins[n_float:]
    y = (0.05 * g.standard_normal(n) + 9.0 * (c65 == 64) + 7.0 * (c129 == 128) - 6.0 * (c200 == 64) - 5.0 * (c200 == 128) +
         4.0 * (c128 == 127) + 3.0 * (c200 == 199))
    K = 1
    if loss == "MultiClass":
        K, y = 3, np.digitize(y, [-2.0, 2.0]).astype(np.float64)
    p = dict(loss=loss, depth=4, learning_rate=0.5, l2_leaf_reg=1.0, score=score, bootstrap_type="No", approx_dim=K,
             leaf_method="Newton" if K > 1 else "Gradient")
    exp = O.train(bins, nb, y, iterations=3, one_hot=one_hot, **p)
    tr = cb.Trainer(bins, 200, y, real_folds=nb + 1, one_hot_flags=one_hot, **p)
    try:
        splits, leaves, kinds = tr.fit(3, with_one_hot=True)
    finally:
        tr.close()
    won = {tuple(s) for t in range(3) for s, k in zip(splits[t].tolist(), kinds[t]) if k}
    assert len(won & {(n_float, 64), (n_float + 1, 127), (n_float + 2, 128), (n_float + 3, 64), (n_float + 3, 128)}) >= 4, won
    for t in range(3):
        ok, flip = same_partition(bins, splits[t], kinds[t], exp["splits"][t], exp["one_hot"][t])
        assert ok, (t, splits[t].tolist(), exp["splits"][t].tolist())
        assert np.array_equal(splits[t], exp["splits"][t])
        _close(np.asarray(leaves[t]), exp["leaf_values"][t], 1e-5)


def test_best_split_of_more_features_than_the_partition_repeats():
    """Over 4096 features the best candidate is found by a launch of its own.  The second half of the
    columns repeats the first, so every level's winner is a tie that the first column must take."""
    g = np.random.default_rng(3)
    n, half = 800, 2_100
    bins = g.integers(0, 4, (half, n)).astype(np.uint8)
    bins = np.concatenate([bins, bins])
    nb = np.full(2 * half, 3, np.uint32)
    y = g.standard_normal(n)
    p = dict(loss="RMSE", depth=4, learning_rate=0.3, l2_leaf_reg=3.0, score="Cosine", bootstrap_type="No",
             leaf_method="Gradient")
    exp = O.train(bins, nb, y, iterations=2, **p)
    tr = cb.Trainer(bins, 4, y, real_folds=nb + 1, **p)
    try:
        splits, leaves = tr.fit(2)
    finally:
        tr.close()
    assert np.array_equal(splits, exp["splits"]) and np.asarray(splits)[..., 0].max() < half
    _close(leaves, exp["leaf_values"], 1e-5)


def test_best_split_of_many_features_in_several_windows():
    """Three classes, 1100 features of 255 bins, depth 7: two windows a feature at 32 parents and four at
    64, 4400 entries at the last level, so that the search over them is a launch of its own.  No row has a
    bin in 60 .. 70 or 120 .. 135, so the borders either side of a window's edge tie and the lower one
    must win.  Splits equal the oracle's."""
    g = np.random.default_rng(4)
    n, F, K = 900, 1_100, 3
    values = np.array([v for v in range(255) if not (60 <= v <= 70 or 120 <= v <= 135)])
    bins = values[g.integers(0, len(values), (F, n))].astype(np.uint8)
    nb = np.full(F, 254, np.uint32)
    # the best borders lie at the gaps; a third of the classes at random, so that no level's leaves are
    # pure (there every candidate would tie in exact arithmetic, and rounding alone decide)
    y = ((bins[1_000] > 64).astype(int) + (bins[1_001] > 127)).astype(np.float64)
    y = np.where(g.random(n) < 0.35, g.integers(0, K, n), y).astype(np.float64)
    p = dict(loss="MultiClass", depth=7, learning_rate=0.3, l2_leaf_reg=3.0, score="Cosine", bootstrap_type="No",
             leaf_method="Newton", approx_dim=K)
    exp = O.train(bins, nb, y, iterations=2, **p)
    tr = cb.Trainer(bins, 255, y, real_folds=nb + 1, **p)
    try:
        splits, leaves = tr.fit(2)
    finally:
        tr.close()
    assert np.array_equal(splits, exp["splits"])
    assert {(1_000, 59), (1_001, 119)} <= {tuple(s) for s in np.asarray(splits[0]).tolist()}
    for t in range(2):
        _close(leaves[t], exp["leaf_values"][t], 1e-5)


@pytest.mark.parametrize("stumps", [0, 1])
def test_predictions_with_leaf_values_either_side_of_the_pinned_size(stumps):
    """512 KiB of leaf values go up with the model in one pinned copy, one value more from the caller's
    memory (the value is that of a tree without splits).  Sums in tree order: equal bit by bit."""
    g = np.random.default_rng(6 + stumps)
    n, F, D, T = 1_500, 20, 14, 4
    x = g.standard_normal((F, n), dtype=np.float32)
    sf = g.integers(0, F, T * D).astype(np.uint32)
    sb = g.standard_normal(T * D).astype(np.float32).astype(np.float64)
    so = np.concatenate([np.arange(0, T * D + 1, D), [T * D] * stumps]).astype(np.uint32)
    lo = np.concatenate([np.arange(0, (T << D) + 1, 1 << D), (T << D) + 1 + np.arange(stumps)]).astype(np.uint32)
    lv = g.standard_normal(int(lo[-1]))
    assert lv.nbytes == (512 << 10) + 8 * stumps
    exp = np.zeros(n)
    for t in range(T + stumps):
        leaf = np.zeros(n, np.int64)
        for i, s in enumerate(range(so[t], so[t + 1])):
            leaf |= (x[sf[s]].astype(np.float64) > sb[s]).astype(np.int64) << i
        exp += lv[lo[t] + leaf]
    got = cb.apply_oblivious(x, sf, sb, so, lv, lo, approx_dim=1)
    assert np.array_equal(np.asarray(got).reshape(-1), exp)


def test_predictions_past_the_kept_sizes():
    """A result of 72 MB loses its device block with the call, the calls after it and beside it (three host
    threads, small and large) start from what is kept.  Equal bit by bit to the same sums on the host."""
    from concurrent.futures import ThreadPoolExecutor
    g = np.random.default_rng(9)
    sf, sb = np.zeros(2, np.uint32), np.array([-0.5, 0.75])
    so, lo, lv = np.array([0, 1, 2], np.uint32), np.array([0, 2, 4], np.uint32), np.array([0.1, 0.7, -0.3, 1.1])
    big = g.standard_normal((1, 9_000_001), dtype=np.float32)

    def one(n):
        x = big[:, :n]
        exp = np.where(x[0] > -0.5, 0.7, 0.1) + np.where(x[0] > 0.75, 1.1, -0.3)
        got = np.asarray(cb.apply_oblivious(np.ascontiguousarray(x), sf, sb, so, lv, lo, approx_dim=1)).reshape(-1)
        return np.array_equal(got, exp)

    assert one(9_000_001) and one(100)
    with ThreadPoolExecutor(3) as ex:
        assert all(ex.map(one, [9_000_001, 63, 4_000_000, 1, 8_500_000, 70_000] * 2))


@pytest.mark.parametrize("n,T", [(2_100_000, 3), (3_900_001, 3), (5_600_000, 700)])
def test_predictions_of_chunked_tables(n, T):
    """A table in two, three and four chunks of 1.57M objects, their kernels on three streams: every chunk
    sees the whole model and the results wait for every chunk, also where the kernels (700 trees) take
    longer than the uploads.  One feature, so a tree's leaf follows from the value's place between
    its borders; the sums are in tree order, equal bit by bit."""
    g = np.random.default_rng(T)
    x = g.standard_normal((1, n), dtype=np.float32)
    sb = np.sort(g.standard_normal((T, 2)).astype(np.float32).astype(np.float64), axis=1).reshape(-1)
    sf = np.zeros(2 * T, np.uint32)
    so, lo = np.arange(0, 2 * T + 1, 2, dtype=np.uint32), np.arange(0, 4 * T + 1, 4, dtype=np.uint32)
    lv = g.standard_normal(4 * T)
    rows = np.unique(np.concatenate([g.integers(0, n, 60_000), np.arange(64), n - 1 - np.arange(64)])) if T > 100 else np.arange(n)
    v = x[0, rows].astype(np.float64)
    for _ in range(2):
        got = np.asarray(cb.apply_oblivious(x, sf, sb, so, lv, lo, approx_dim=1)).reshape(-1)
        exp = np.zeros(len(rows))
        for t in range(T):
            exp += lv[4 * t + (v > sb[2 * t]).astype(np.int64) + 2 * (v > sb[2 * t + 1])]
        assert np.array_equal(got[rows], exp)


@pytest.mark.parametrize("n,F,T", [(3_900_001, 1, 3), (100_001, 100, 3), (100_001, 100, 900), (94_080, 100, 900),
                                   (40_001, 600, 900), (31_361, 250, 900)])
def test_predictions_of_chunked_tables(n, F, T):
    """Tables in pinned chunks of 6 MB: a launch a chunk at small models, one launch over several chunks at
    large ones (three of 100 features, ten of 600 whose values are read through the caches, two of 250),
    with a last group of one chunk, a last chunk of one object, or none left over, and device buffers
    that are used again.  Sums in tree order, equal bit by bit."""
    g = np.random.default_rng(n)
    x = g.standard_normal((F, n), dtype=np.float32)
    sf = g.integers(0, F, 2 * T).astype(np.uint32)
    sb = g.standard_normal(2 * T).astype(np.float32).astype(np.float64)
    so, lo = np.arange(0, 2 * T + 1, 2, dtype=np.uint32), np.arange(0, 4 * T + 1, 4, dtype=np.uint32)
    lv = g.standard_normal(4 * T)
    exp = np.zeros(n)
    for t in range(T):
        a, b = 2 * t, 2 * t + 1
        exp += lv[4 * t + (x[sf[a]] > sb[a]).astype(np.int64) + 2 * (x[sf[b]] > sb[b])]
    for _ in range(2):
        got = np.asarray(cb.apply_oblivious(x, sf, sb, so, lv, lo, approx_dim=1)).reshape(-1)
        assert np.array_equal(got, exp)
