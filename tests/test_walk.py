"""The ensemble walk in LDS (csrc/walk.hip) against the oracle's traversal,
bit for bit: tile edges of every launch shape, tree sizes on both sides of a
window, column counts at the tile choices' limits, and trees that need the
general path (a child with two parents, too many nodes or columns)."""
import numpy as np
import pytest

from oracle import model as om

pytestmark = pytest.mark.gpu


def _tree(rng, n_split, F, bins, skew=False, loose=False):
    """A random tree of n_split splits as (features, thresholds, values, left,
    right); children after their parent, side by side unless `loose`."""
    n = 2 * n_split + 1
    f, t = np.full(n, -1, np.int16), np.zeros(n, np.int64)
    l, r = np.full(n, -1, np.int32), np.full(n, -1, np.int32)
    ids = iter(range(1, n))
    open_, leaves = [0], n_split
    pairs = []
    while leaves:
        at = open_.pop(-1 if skew else int(rng.integers(len(open_))))
        pairs.append(at)
        kids = [next(ids), next(ids)]
        f[at], t[at] = rng.integers(F), rng.choice([-1, 0, bins - 2, bins - 1, 255, 300]) \
            if rng.random() < 0.1 else rng.integers(bins)
        l[at], r[at] = kids
        open_ += kids
        leaves -= 1
    if loose and n > 3:  # some pairs the other way round
        for at in pairs[::2]:
            l[at], r[at] = r[at], l[at]
    return f, t, rng.standard_normal(n), l, r


def _pack(trees):
    out = {k: np.concatenate([x[i] for x in trees]) for i, k in
           enumerate(("features", "thresholds", "values", "left", "right"))}
    out["offsets"] = np.concatenate([[0], np.cumsum([len(x[0]) for x in trees])]).astype(np.int32)
    return out


# (rows, columns, trees, splits per tree, options)
CASES = {
    "one_row": (1, 5, 3, [0, 1, 2], {}),
    "leaves_only": (130, 4, 9, [0], {}),
    "short_tile": (65, 28, 11, [62], {}),
    "wide": (4097, 208, 17, [1, 30, 62], {}),
    "too_wide": (300, 230, 40, [62], {}),
    "window_63_64": (700, 20, 10, [63, 5], {}),
    "window_127_128": (700, 20, 10, [127, 128], {}),
    "window_255_256": (700, 20, 5, [255, 256], {}),
    "slot_1023": (700, 20, 3, [511], {}),
    "too_many_nodes": (700, 20, 3, [512], {}),
    "skewed": (1000, 12, 9, [62, 100], {"skew": True}),
    "right_before_left": (1000, 12, 9, [40], {"loose": True}),
    "tile256_edge": (65536 + 257, 28, 9, [62], {}),
    "shared_edge": (131072, 9, 9, [62, 5], {}),
    "not_shared": (131072 + 257, 28, 9, [62], {}),
    "rows4": (400001, 52, 9, [62, 3], {}),
    "rows4_too_wide": (400001, 53, 5, [62], {}),
    "rows4_tile_edge": (400384, 30, 3, [62], {}),
    "rows4_window": (400000, 12, 5, [127], {}),
    "rows4_large_trees": (400000, 12, 3, [128, 400], {}),
    "tiers": (3000, 30, 9, [62], {"bins": 600}),
}


@pytest.mark.parametrize("case", list(CASES))
def test_walk_equals_oracle(engine, case):
    n, F, T, splits, opt = CASES[case]
    print(f"[case] walk {case}: {n} x {F}, {T} trees", flush=True)
    rng = np.random.default_rng(len(case) + n)
    opt = dict(opt)
    bins = opt.pop("bins", 255)
    codes = rng.integers(0, bins, (n, F)).astype(np.uint8 if bins < 256 else np.uint16)
    p = _pack([_tree(rng, splits[i % len(splits)], F, bins, **opt) for i in range(T)])
    engine.load_codes(1, codes)
    want = om.predict_all_trees(codes, p, T, 0.1)
    np.testing.assert_array_equal(engine.predict(1, n, p, T, 0.1), want)
    # Probabilities from the walk's own epilogue, and a class without trees
    # beside one with them.
    proba = engine.predict_proba(1, n, p, T, 0.1, 0.25)
    np.testing.assert_allclose(proba[:, 1], om.binary_proba(want + 0.25), rtol=1e-15, atol=0)
    mc = engine.predict_proba_mc(1, n, [p, None, p], [T, 0, max(1, T - 2)], 0.1)
    F3 = np.stack([want, np.zeros(n), om.predict_all_trees(codes, p, max(1, T - 2), 0.1)], 1)
    e = np.exp(F3 - F3.max(1, keepdims=True))
    np.testing.assert_allclose(mc, e / e.sum(1, keepdims=True), rtol=1e-14, atol=0)


def test_walk_shared_child_takes_general_path(engine):
    """A child with two parents is accepted (every walk ends) and walked in
    HBM; the result is the traversal's."""
    rng = np.random.default_rng(5)
    f = np.array([0, 1, 2, 3, -1, -1], np.int16)
    t = np.array([100, 50, 150, 80, 0, 0], np.int64)
    l = np.array([1, 3, 3, 4, -1, -1], np.int32)
    r = np.array([2, 4, 5, 5, -1, -1], np.int32)
    p = _pack([(f, t, rng.standard_normal(6), l, r)])
    codes = rng.integers(0, 200, (500, 4)).astype(np.uint8)
    engine.load_codes(1, codes)
    np.testing.assert_array_equal(engine.predict(1, 500, p, 1, 0.5),
                                  om.predict_all_trees(codes, p, 1, 0.5))


def test_large_models_and_edges_pin_no_more(engine):
    """Host tables of any size leave the engine's pinned staging memory at
    its 16 MB, and give the same codes and sums."""
    from bsscl_gbm import _native
    rng = np.random.default_rng(8)
    n, F, nb, T = 500, 40, 60_000, 15_000
    eng = _native.Engine(0)
    try:
        E = np.sort(rng.standard_normal((F, nb + 1)), axis=1)  # 19 MB
        X = rng.standard_normal((n, F)).astype(np.float32)
        counts, nan_id = np.full(F, nb, np.int32), np.full(F, -1, np.int32)
        eng.bin_features(1, X, E, counts, nan_id)
        want = om.bin_features(X, E, counts, nan_id, "standard")
        np.testing.assert_array_equal(eng.get_codes(1, n, F, u16=True), want)
        codes = rng.integers(0, 200, (n, F)).astype(np.uint8)
        p = _pack([_tree(rng, 14, F, 200) for _ in range(T)])  # 435,000 nodes, 14 MB
        eng.load_codes(1, codes)
        np.testing.assert_array_equal(eng.predict(1, n, p, T, 0.1),
                                      om.predict_all_trees(codes, p, T, 0.1))
        assert eng.stats()["staging_bytes"] <= 16 << 20
    finally:
        eng.close()


@pytest.mark.parametrize("n", [300, 131_201, 400_003])
@pytest.mark.parametrize("splits", [9, 20, 21, 62, 130, 300, 511])
@pytest.mark.parametrize("stay", [0.5, 0.97])
def test_walk_of_chains(engine, n, splits, stay):
    """Trees deep on one side: walks that end early and walks that go to the
    bottom, in every launch shape, on both sides of the steps a wave takes
    before it looks for the end."""
    print(f"[case] walk of chains: {n} rows, {splits} splits, {stay}", flush=True)
    rng = np.random.default_rng(splits)
    codes = rng.integers(0, 200, (n, 9)).astype(np.uint8)
    trees = []
    for k in range(5):
        f, t, v, l, r = _tree(rng, splits if k % 2 == 0 else 5, 9, 200, skew=True)
        t[f >= 0] = int(200 * (1 - stay)) - 1  # the deeper side is the right one
        trees.append((f, t, v, l, r))
    p = _pack(trees)
    engine.load_codes(1, codes)
    np.testing.assert_array_equal(engine.predict(1, n, p, 5, 0.1),
                                  om.predict_all_trees(codes, p, 5, 0.1))


MIXED = {
    "large_then_stumps": [511] + [1] * 700,
    "one_per_group": [511, 400, 300, 511],
    "exact_groups": [255, 255, 127, 127, 127, 127, 511, 255, 62],
    "odd_tails": [255, 1, 1, 0, 200, 3, 300, 0],
    "leaves_between": [300, 0, 0, 0, 255, 0, 130, 0],
    "up_to_256_slots": [127, 1, 100, 0, 63, 64, 127, 5, 2],
}


@pytest.mark.parametrize("n", [257, 131_300, 400_011])
@pytest.mark.parametrize("case", list(MIXED))
def test_walk_of_mixed_sizes(engine, case, n):
    """Trees of more than 127 nodes lie beside small ones in slots of their
    own size: group ends, odd tails, classes of different sizes."""
    splits = MIXED[case]
    print(f"[case] walk of mixed sizes {case}: {n} rows", flush=True)
    rng = np.random.default_rng(len(splits) + n)
    codes = rng.integers(0, 250, (n, 11)).astype(np.uint8)
    p = _pack([_tree(rng, s, 11, 250) for s in splits])
    q = _pack([_tree(rng, s, 11, 250) for s in splits[::-1][:5]])
    T, U = len(splits), len(splits[::-1][:5])
    engine.load_codes(1, codes)
    want = om.predict_all_trees(codes, p, T, 0.1)
    np.testing.assert_array_equal(engine.predict(1, n, p, T, 0.1), want)
    proba = engine.predict_proba_mc(1, n, [q, None, p], [U, 0, T], 0.1)
    F = np.stack([om.predict_all_trees(codes, q, U, 0.1), np.zeros(n), want], 1)
    e = np.exp(F - F.max(1, keepdims=True))
    np.testing.assert_allclose(proba, e / e.sum(1, keepdims=True), rtol=1e-13, atol=1e-300)
