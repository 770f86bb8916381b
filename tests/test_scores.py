"""Boosting scores on the device against the reference's expression
(est:2896-2903, est:3027-3029): F += lr * value, the product and the sum
rounded apart, tree by tree, bit for bit; the validation rows go through the
same update as the training rows."""
import numpy as np
import pytest

from conftest import make_data
from oracle import model as om

pytestmark = pytest.mark.gpu


def _mode(monkeypatch, path):
    if path == "host_replay":
        monkeypatch.setenv("BSSCL_TEST_HOST_REPLAY", "1")
    if path == "graphs":
        monkeypatch.setenv("BSSCL_GRAPHS", "1")


@pytest.mark.parametrize("path", ["pipelined", "synchronous", "host_replay", "graphs"])
@pytest.mark.parametrize("n,depth", [(1025, 3), (9001, 6)])
def test_binary_scores_round_twice(monkeypatch, path, n, depth):
    from bsscl_gbm import HybridHistGBMNumbaV1_0_1
    from bsscl_gbm import estimator as est_mod
    print(f"[case] scores {n} rows, depth {depth}, {path}", flush=True)
    _mode(monkeypatch, path)
    X, y = make_data(n, 9, seed=4, nan_frac=0.05, nan_cols=[1, 2])
    m = HybridHistGBMNumbaV1_0_1(n_estimators=12, max_depth=depth, random_state=1,
                                 learning_rate=0.1, verbose=False)
    m._pipeline_rounds = path != "synchronous"
    m.fit(X, y, eval_set=[(X, y)])
    codes = om.bin_features(X, m.bin_edges, m.feature_bin_counts, m._nan_bin_id, "standard")
    F = np.full(n, m.base_score_)
    for t in m.trees:
        F = F + m.learning_rate * om.predict_tree(codes, t)
    np.testing.assert_array_equal(est_mod._engine(0).boost_get_F(n), F)
    # The validation rows are the training rows: the same scores, the same
    # terms in the same blocks, the same loss to the last bit.
    np.testing.assert_array_equal(m.val_loss_history_, m.train_loss_history_)


@pytest.mark.parametrize("path", ["device", "host_replay"])
def test_multiclass_scores_round_twice(monkeypatch, path):
    from bsscl_gbm import HybridHistGBMNumbaV1_0_1
    from bsscl_gbm import estimator as est_mod
    print(f"[case] multiclass scores {path}", flush=True)
    _mode(monkeypatch, path)
    rng = np.random.default_rng(6)
    n, K = 5001, 4
    X = rng.standard_normal((n, 7)).astype(np.float32)
    y = (X @ rng.standard_normal((7, K)) + rng.gumbel(size=(n, K))).argmax(1)
    m = HybridHistGBMNumbaV1_0_1(n_estimators=8, max_depth=5, random_state=2, learning_rate=0.1,
                                 verbose=False).fit(X, y)
    codes = om.bin_features(X, m.bin_edges, m.feature_bin_counts, m._nan_bin_id, "standard")
    F = np.zeros((n, K))
    for k in range(K):
        for t in m.mc_trees[k]:
            F[:, k] = F[:, k] + m.learning_rate * om.predict_tree(codes, t)
    np.testing.assert_array_equal(est_mod._engine(0).mc_scores(), F)


@pytest.mark.parametrize("start", [np.nan, np.inf, -np.inf, 600.0])
@pytest.mark.parametrize("path", ["pipelined", "host_replay"])
def test_validation_loss_of_scores_past_the_clip(monkeypatch, path, start):
    """A NaN score gives a NaN loss, as np.clip and the mean keep it;
    infinities are clipped."""
    from bsscl_gbm import HybridHistGBMNumbaV1_0_1, _native
    print(f"[case] validation scores from {start}, {path}", flush=True)
    _mode(monkeypatch, path)
    begin = _native.Engine.boost_val_begin
    monkeypatch.setattr(_native.Engine, "boost_val_begin",
                        lambda self, y, base: begin(self, y, start))
    X, y = make_data(3000, 6, seed=9)
    m = HybridHistGBMNumbaV1_0_1(n_estimators=3, max_depth=3, random_state=1, verbose=False)
    m.fit(X, y, eval_set=[(X[:700], y[:700])])
    codes = om.bin_features(X[:700], m.bin_edges, m.feature_bin_counts, m._nan_bin_id, "standard")
    F, want = np.full(700, start), []
    for t in m.trees:
        F = F + m.learning_rate * om.predict_tree(codes, t)
        want.append(om.binary_logloss(y[:700], F))
    np.testing.assert_allclose(m.val_loss_history_, want, rtol=1e-13, atol=0)
    assert np.isfinite(m.train_loss_history_).all()


def test_one_validation_label_for_all_rows():
    """A single label stands for every validation row; other lengths that
    differ from the rows are refused."""
    from bsscl_gbm import HybridHistGBMNumbaV1_0_1
    X, y = make_data(2000, 5, seed=10)
    kw = dict(n_estimators=4, max_depth=3, random_state=1, verbose=False)
    one = HybridHistGBMNumbaV1_0_1(**kw).fit(X, y, eval_set=[(X[:50], [1])])
    full = HybridHistGBMNumbaV1_0_1(**kw).fit(X, y, eval_set=[(X[:50], np.ones(50, int))])
    assert one.val_loss_history_ == full.val_loss_history_
    with pytest.raises(ValueError):
        HybridHistGBMNumbaV1_0_1(**kw).fit(X, y, eval_set=[(X[:50], y[:49])])
