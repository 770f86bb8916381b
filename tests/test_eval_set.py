"""Validation losses of a binary fit, kept on the device with the round's
tree: equal to the reference's expressions (est:2898-2903) over the fitted
trees, on the pipelined, synchronous and host-replay paths."""
import numpy as np
import pytest

from conftest import make_data
from oracle import model as om

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_val", [1, 255, 1025, 20_011])
@pytest.mark.parametrize("path", ["pipelined", "synchronous", "host_replay", "small_table", "graphs"])
def test_val_loss_equals_reference_expression(engine, monkeypatch, n_val, path):
    from bsscl_gbm import HybridHistGBMNumbaV1_0_1
    print(f"[case] eval set {n_val} {path}", flush=True)
    X, y = make_data(9000, 9, seed=4, nan_frac=0.05, nan_cols=[1, 2])
    Xv, yv = make_data(n_val, 9, seed=5, nan_frac=0.1)
    if path == "host_replay":
        monkeypatch.setenv("BSSCL_TEST_HOST_REPLAY", "1")
    if path == "small_table":
        monkeypatch.setenv("BSSCL_TEST_NODE_CAP", "9")
    if path == "graphs":
        monkeypatch.setenv("BSSCL_GRAPHS", "1")
    m = HybridHistGBMNumbaV1_0_1(n_estimators=9, max_depth=5, n_bins=300, random_state=1,
                                 verbose=False)
    m._pipeline_rounds = path != "synchronous"
    m.fit(X, y, eval_set=[(Xv, yv)])
    ref = HybridHistGBMNumbaV1_0_1(n_estimators=9, max_depth=5, n_bins=300, random_state=1,
                                   verbose=False).fit(X, y)
    np.testing.assert_array_equal(m.train_loss_history_, ref.train_loss_history_)
    codes = om.bin_features(Xv, m.bin_edges, m.feature_bin_counts, m._nan_bin_id, "standard")
    F, want = np.full(n_val, m.base_score_), []
    for t in m.trees:
        F = F + m.learning_rate * om.predict_tree(codes, t)
        want.append(om.binary_logloss(yv, F))
    # (n_val float64 terms of one sign, added in another order.)
    np.testing.assert_allclose(m.val_loss_history_, want, rtol=1e-13, atol=0)


def test_early_stopping_drops_the_round_in_flight(engine):
    from bsscl_gbm import HybridHistGBMNumbaV1_0_1
    X, y = make_data(6000, 8, seed=8)
    rng = np.random.default_rng(0)
    yv = rng.integers(0, 2, 500)  # noise: the loss soon rises
    Xv = rng.standard_normal((500, 8)).astype(np.float32)
    kw = dict(n_estimators=60, max_depth=4, learning_rate=0.5, random_state=2, verbose=False)
    full = HybridHistGBMNumbaV1_0_1(**kw).fit(X, y, eval_set=[(Xv, yv)])
    m = HybridHistGBMNumbaV1_0_1(early_stopping_rounds=3, **kw).fit(X, y, eval_set=[(Xv, yv)])
    k = len(m.val_loss_history_)
    assert k < 60 and m.best_iteration_ == int(np.argmin(full.val_loss_history_[:k]))
    assert len(m.trees) == m.best_iteration_ + 1
    np.testing.assert_array_equal(m.val_loss_history_, full.val_loss_history_[:k])
    again = HybridHistGBMNumbaV1_0_1(**kw).fit(X, y)  # the engine is ready for another run
    np.testing.assert_array_equal(again.train_loss_history_, full.train_loss_history_)


def test_val_rows_must_match_the_run(engine):
    rng = np.random.default_rng(1)
    engine.load_codes(0, rng.integers(0, 9, (300, 4)).astype(np.uint8))
    engine.load_codes(1, rng.integers(0, 9, (50, 4)).astype(np.uint8))
    engine.boost_begin(rng.integers(0, 2, 300), 1.0, 1.0, 0.0)
    with pytest.raises(ValueError, match="length"):
        engine.boost_val_begin(np.zeros(49, np.int64), 0.0)
    with pytest.raises(ValueError, match="0 or 1"):
        engine.boost_val_begin(np.full(50, 2), 0.0)
    with pytest.raises(ValueError, match="no validation rows"):
        engine.boost_val_loss()
    engine.load_codes(1, rng.integers(0, 9, (50, 5)).astype(np.uint8))
    with pytest.raises(ValueError, match="not binned"):
        engine.boost_val_begin(np.zeros(50, np.int64), 0.0)
