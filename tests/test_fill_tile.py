"""Which fill a session took, as its stats and the benchmark's line tell it."""
import numpy as np
import pytest

import bench
import catboost_rs_amd as cb


def test_benchmark_names_the_fill_by_the_sessions_stats():
    """The two exact fills share fill_mode 2: the tile width tells them apart, whatever the sizes."""
    def named(mode, tile):
        return bench._fill_kernel(dict(fill_mode=mode, fill_tile=tile, fill_pack_bits=18))

    assert named(2, 8)[0] == "fill_narrow_kernel" and "exact 8-feature" in named(2, 8)[1]
    assert named(2, 32)[0] == "fill_exact_kernel" and "exact 32-feature" in named(2, 32)[1]
    assert [named(m, 32)[0] for m in (0, 3, 4)] == ["fill_kernel", "fill_pkk_kernel", "fill_pks_kernel"]
    assert [named(m, 64)[0] for m in (1, 5)] == ["fill_packed_kernel"] * 2


@pytest.mark.gpu
@pytest.mark.parametrize("n,F,B,depth,fill,mode,tile", [
    (70_000, 40, 65, 4, "", 2, 8), (70_000, 40, 65, 4, "tiled", 2, 32), (70_000, 40, 65, 4, "count", 5, 64),
    (70_000, 40, 65, 4, "packed", 1, 64), (70_000, 40, 65, 4, "generic", 0, 40),
    (70_000, 1_500, 33, 4, "", 2, 32)])   # more (row, feature) pairs than the narrow tiles' line
def test_stats_tell_the_tile(n, F, B, depth, fill, mode, tile, monkeypatch):
    monkeypatch.setenv("CBH_FILL", fill)
    g = np.random.default_rng(1)
    bins = g.integers(0, B, (F, n), dtype=np.uint8)
    tr = cb.Trainer(bins, B, g.standard_normal(n), depth=depth, bootstrap_type="No", real_folds=np.full(F, B, np.uint32))
    try:
        tr.step()
        st = tr.stats()
    finally:
        tr.close()
    assert (st["fill_mode"], st["fill_tile"]) == (mode, tile)
