"""bsscl_build_tree's row lists, checked and sorted on the device from 65,536
rows on: any order and repeated rows give the oracle's tree, rows and
gradients that are not allowed are refused on both sides of that size."""
import numpy as np
import pytest

import treecmp
from oracle import model as om

pytestmark = pytest.mark.gpu

N = {"host": 65_535, "device": 65_536, "device_odd": 70_001}


def _inputs(n, seed=3):
    rng = np.random.default_rng(seed)
    codes = rng.integers(0, 40, (n, 5)).astype(np.uint8)
    g, h = rng.standard_normal(n), rng.random(n) + 0.1
    return rng, codes, g, h


ARGS = dict(max_leaves=15, max_depth=4, min_samples_leaf=5, min_child_weight=1.0,
            bin_counts=np.full(5, 40, np.int32), max_bins=40, reg_lambda=1.0, gamma=0.0)


@pytest.mark.parametrize("size", list(N))
@pytest.mark.parametrize("kind", ["shuffled", "all_sorted", "one", "last_row", "repeated"])
def test_tree_from_row_list(engine, size, kind):
    n = N[size]
    print(f"[case] tree rows {size} {kind}", flush=True)
    rng, codes, g, h = _inputs(n)
    rows = {"shuffled": rng.permutation(n)[: n // 2], "all_sorted": np.arange(n),
            "one": np.array([n // 3]), "last_row": np.arange(n - 4097, n),
            "repeated": rng.integers(0, n, n)}[kind]
    feats = np.arange(5, dtype=np.int32)
    engine.load_codes(0, codes)
    got = engine.build_tree(g, h, rows, feats, *ARGS.values())
    want = om.build_tree(codes, g, h, np.asarray(rows, np.int64), feats, *ARGS.values())
    assert treecmp.compare(want, got) == "equal"


@pytest.mark.parametrize("size", list(N))
def test_bad_rows_and_gradients_are_refused(engine, size):
    n = N[size]
    rng, codes, g, h = _inputs(n)
    feats = np.arange(5, dtype=np.int32)
    engine.load_codes(0, codes)
    rows = np.arange(n)
    for bad in (-1, n, 2**40):
        r = rows.copy()
        r[n // 2] = bad
        with pytest.raises(ValueError, match="out of range"):
            engine.build_tree(g, h, r, feats, *ARGS.values())
    for a, v in ((0, np.nan), (1, np.inf), (0, -np.inf)):
        gh = [g.copy(), h.copy()]
        gh[a][n - 1] = v
        with pytest.raises(ValueError, match="finite"):
            engine.build_tree(*gh, rows, feats, *ARGS.values())
    got = engine.build_tree(g, h, rows, feats, *ARGS.values())
    want = om.build_tree(codes, g, h, rows, feats, *ARGS.values())
    assert treecmp.compare(want, got) == "equal"


@pytest.mark.parametrize("F", [1, 4, 5, 8, 33])
@pytest.mark.parametrize("n", [900, 5003, 140_001])
def test_scatter_shares_a_tiles_features(engine, n, F):
    """The partition's rows move with every feature of a tile, whichever
    blocks share them: batches of four, a last one of one, one block each."""
    print(f"[case] scatter {n} x {F}", flush=True)
    rng = np.random.default_rng(n + F)
    # (Few enough bins that no node has an empty one: splits on its two sides
    # part the same rows and their gains tie.)
    bins = 4 if n < 2000 else 12 if n < 50_000 else 60
    codes = rng.integers(0, bins, (n, F)).astype(np.uint8)
    g, h = rng.standard_normal(n) + 0.02 * codes.sum(1), rng.random(n) + 0.1
    args = dict(ARGS, max_leaves=31, max_depth=6, min_samples_leaf=20,
                bin_counts=np.full(F, bins, np.int32), max_bins=bins)
    feats = np.arange(F, dtype=np.int32)
    engine.load_codes(0, codes)
    got = engine.build_tree(g, h, np.arange(n), feats, *args.values())
    want = om.build_tree(codes, g, h, np.arange(n), feats, *args.values())
    assert treecmp.compare(want, got) == "equal"


@pytest.mark.parametrize("F", [64, 65, 80, 113, 128, 129])
def test_planner_takes_every_feature(engine, F):
    """The planner's waves take four or eight features each up to 128: the
    best split may lie in any of them, and of two equal columns the first
    wins."""
    print(f"[case] planner {F} features", flush=True)
    n, bins = 6007, 10
    rng = np.random.default_rng(F)
    codes = rng.integers(0, bins, (n, F)).astype(np.uint8)
    codes[:, F - 1] = codes[:, 3]
    codes[:, F - 2] = codes[:, F // 2]
    steer = codes[:, [3, F // 2, F - 3, 4, 60]].astype(np.float64)
    g = rng.standard_normal(n) + steer @ [0.2, -0.15, 0.1, 0.05, -0.05]
    h = rng.random(n) + 0.1
    args = dict(ARGS, max_leaves=31, max_depth=6, min_samples_leaf=20,
                bin_counts=np.full(F, bins, np.int32), max_bins=bins)
    feats = np.arange(F, dtype=np.int32)
    engine.load_codes(0, codes)
    got = engine.build_tree(g, h, np.arange(n), feats, *args.values())
    want = om.build_tree(codes, g, h, np.arange(n), feats, *args.values())
    assert treecmp.compare(want, got) == "equal"
